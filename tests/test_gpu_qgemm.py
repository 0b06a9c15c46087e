"""GPU parity of the quantized GEMM, get_rows and argmax against the oracle.

Bar: bit-exact.  The GEMM contract sums exact integers, so the HIP kernel must
reproduce the oracle's f32 outputs bit for bit at every shape, including the
27B-class verify shapes (K, N) in {(5120, 7168), (5120, 5120), (5120, 17408),
(17408, 5120)} with M in {1, 5, 8, 16}; up to 16 rows share one pass over
the weights (12 and 24 rows check the partial and split launches; Q4_K above
8 rows runs on the 16x16x32 MFMA kernel).  Above 16 rows (Q4_K) or 8 rows
(Q6_K, Q8_0) every type runs on its wide (prefill) kernel, held to the same
bar.
"""
import ctypes

import numpy as np
import pytest
import torch

from oracle import cpvo

pytestmark = pytest.mark.gpu

TYPES = {"q8_0": cpvo.Q8_0, "q4_k": cpvo.Q4_K, "q6_k": cpvo.Q6_K}


@pytest.fixture(scope="module")
def ctx():
    from codpiece_amd.runtime import Context
    c = Context(0)
    yield c
    c.close()


_weights = {}


def weights(t, n, k, seed=0):
    key = (t, n, k, seed)
    if key not in _weights:
        rng = np.random.default_rng(seed + 1000 * t + n + 7 * k)
        wf = rng.normal(0, 0.02, size=(n, k)).astype(np.float32)
        _weights[key] = cpvo.quantize(t, wf)
    return _weights[key]


def run_case(ctx, t, n, k, m, seed=0, xscale=1.0):
    wq = weights(t, n, k)
    rng = np.random.default_rng(seed)
    x = (rng.normal(0, 1, size=(m, k)) * xscale).astype(np.float32)
    print(f"case type={t} n={n} k={k} m={m}", flush=True)
    w = ctx.upload_weight(t, wq, n, k)
    y = ctx.qgemm(w, torch.from_numpy(x).cuda()).cpu().numpy()
    ref = cpvo.qgemm(t, wq, x)
    w.free()
    return y, ref


@pytest.mark.parametrize("tname", list(TYPES))
@pytest.mark.parametrize("n,k", [(64, 256), (48, 512), (1000, 768), (33, 1024), (160, 4096)])
@pytest.mark.parametrize("m", [1, 3, 5, 9, 12, 13, 16, 24])
def test_qgemm_bit_exact_small(ctx, tname, n, k, m):
    t = TYPES[tname]
    y, ref = run_case(ctx, t, n, k, m)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), np.abs(y - ref).max()


@pytest.mark.parametrize("tname", ["q4_k", "q8_0"])
@pytest.mark.parametrize("k,n", [(5120, 7168), (5120, 5120), (5120, 17408), (17408, 5120)])
@pytest.mark.parametrize("m", [1, 5, 8, 16])
def test_qgemm_bit_exact_verify_shapes(ctx, tname, k, n, m):
    t = TYPES[tname]
    y, ref = run_case(ctx, t, n, k, m)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), np.abs(y - ref).max()


@pytest.mark.parametrize("m", [1, 2, 3, 5, 8, 16])
def test_qgemm_lm_head_q6_k(ctx, m):
    # the output projection of the 27B-class layout: Q6_K, K = 5120, a slice of
    # the 151,936 vocabulary rows (full vocab is covered by the e2e test); 16
    # rows are a draft tree's; below 8 rows the code-sum term is summed ahead
    # of the group loop, at 8 inside it
    y, ref = run_case(ctx, cpvo.Q6_K, 4096, 5120, m)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("tname", ["q4_k", "q6_k"])
@pytest.mark.parametrize("m", [4, 9, 16])
def test_qgemm_extreme_scales_and_zero_rows(ctx, tname, m):
    # 4 rows: the 4x4x4 kernel; 9 and 16: the 16x16x32 ones
    t = TYPES[tname]
    n, k = 32, 1024
    rng = np.random.default_rng(3)
    wf = rng.normal(0, 0.02, size=(n, k)).astype(np.float32)
    wf[5] = 0.0                                   # an all-zero weight row
    wf[7] *= 1e3                                  # a row with huge scales
    wq = cpvo.quantize(t, wf)
    x = rng.normal(0, 1, size=(m, k)).astype(np.float32)
    x[1] = 0.0                                    # an all-zero activation row
    x[2] *= 1e-6
    w = ctx.upload_weight(t, wq, n, k)
    y = ctx.qgemm(w, torch.from_numpy(x).cuda()).cpu().numpy()
    ref = cpvo.qgemm(t, wq, x)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))
    assert np.all(y[1] == 0) and np.all(y[:, 5] == 0)


# ---- the wide kernels (the prompt prefill's rows; here 32 and more)

@pytest.mark.parametrize("tname", ["q4_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("n,k", [(64, 256), (1000, 768), (33, 1024), (160, 4096)])
@pytest.mark.parametrize("m", [32, 37, 64, 100, 256])
def test_qgemm_wide_bit_exact_small(ctx, tname, n, k, m):
    y, ref = run_case(ctx, TYPES[tname], n, k, m)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), np.abs(y - ref).max()


@pytest.mark.parametrize("tname", ["q4_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("m", [9, 16, 17, 33, 49, 65, 81, 97, 113, 128, 129, 145, 255])
def test_qgemm_wide_row_blocks(ctx, tname, m):
    # few tiles: 1 to 3 16-row blocks a workgroup, K in slices (11 units, which
    # no slice count divides), with one row in the last block or all; weight
    # rows past a tile
    y, ref = run_case(ctx, TYPES[tname], 131, 2816, m)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), np.abs(y - ref).max()


@pytest.mark.parametrize("m", [5, 40])
def test_qgemm_units_below_the_scale_range(ctx, m):
    # a unit whose largest value is below 127 / FLT_MAX has an infinite inverse
    # scale: its term is zero, on the skinny path and on the wide one's f16 sums
    t, n, k = cpvo.Q4_K, 70, 1024
    wq = weights(t, n, k)
    x = np.random.default_rng(9).normal(0, 1, size=(m, k)).astype(np.float32)
    x[1, 256:512] *= np.float32(1e-38)
    x[2, :256] = np.float32(-3e-39)
    w = ctx.upload_weight(t, wq, n, k)
    y = ctx.qgemm(w, torch.from_numpy(x).cuda()).cpu().numpy()
    w.free()
    z = x.copy()
    z[1, 256:512] = 0
    z[2, :256] = 0
    assert np.array_equal(y, cpvo.qgemm(t, wq, z))


def raw_blocks(t, n, k, seed=0):
    """ggml blocks of n rows [n][bytes]: random codes and sub-block scales, a
    tenth of the block scales 30 times the others."""
    rng = np.random.default_rng(seed)
    size, elems, at = {cpvo.Q8_0: (34, 32, (0,)), cpvo.Q4_K: (144, 256, (0, 2)), cpvo.Q6_K: (210, 256, (208,))}[t]
    raw = rng.integers(0, 256, size=(n * (k // elems), size), dtype=np.uint8)
    for o in at:
        d = rng.uniform(0.5, 1.5, raw.shape[0]) * np.where(rng.random(raw.shape[0]) < 0.1, 3e-2, 1e-3)
        raw[:, o:o + 2] = d.astype(np.float16).view(np.uint8).reshape(-1, 2)
    return raw.reshape(n, -1)


def wide_plan(ctx, t, n, k, m):
    """cpv_qgemm_wide_plan: 16-row blocks per workgroup, row blocks, pairs over
    all of K, K slices of the other pairs, units a slice."""
    ctx.lib.cpv_qgemm_wide_plan.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_int, ctypes.c_int * 5]
    out = (ctypes.c_int * 5)()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert ctx.lib.cpv_qgemm_wide_plan(t, n, k, m, cus, out)
    return list(out)


@pytest.mark.parametrize("tname,nmt", [(t, b) for t, lo, hi in (("q4_k", 2, 8), ("q6_k", 1, 8), ("q8_0", 1, 4))
                                       for b in range(lo, hi + 1)])
def test_qgemm_wide_whole_and_sliced(ctx, tname, nmt):
    # every number of 16-row blocks a workgroup may hold: whole rounds of
    # workgroups over all of K (9 units, in both staging buffers) and one pair
    # past them in two K slices through the accumulator, which has to be zero
    # again for the next row count; one row in the last block, then all.  Every
    # output against the skinny kernels', some tiles' against the oracle's.
    t = TYPES[tname]
    tiles = 1536 if (tname, nmt) == ("q8_0", 4) else 768 if tname == "q8_0" or nmt <= 2 else 512
    n, k = 64 * tiles + 3, 2304
    wq = raw_blocks(t, n, k)
    rows = np.r_[0:64, n // 2:n // 2 + 64, n - 130:n]
    w = ctx.upload_weight(t, wq, n, k)
    for m in (max(9, 16 * nmt - 15), 16 * nmt):
        assert wide_plan(ctx, t, n, k, m) == [nmt, 1, tiles, 2, 5]
        print(f"case type={tname} n={n} k={k} m={m}", flush=True)
        x = np.random.default_rng(m).normal(0, 1, size=(m, k)).astype(np.float32)
        x[m // 2] *= 1e-3
        xt = torch.from_numpy(x).cuda()
        y = ctx.qgemm(w, xt)
        for r in range(0, m, 8):
            ys = ctx.qgemm(w, xt[r:r + 8].contiguous())
            assert torch.equal(y[r:r + 8].view(torch.int32), ys.view(torch.int32)), r
        ref = cpvo.qgemm(t, wq[rows], x)
        assert np.array_equal(y.cpu().numpy()[:, rows].view(np.uint32), ref.view(np.uint32))
    w.free()


def test_qgemm_wide_many_weight_rows():
    # 131,100 tiles by 16 row blocks: the first, a middle and the last weight
    # rows against the same rows on their own (a context of its own: 17 GB of
    # accumulator)
    from codpiece_amd.runtime import Context
    ctx = Context(0)
    n, k, m = 64 * 131099 + 7, 32, 256
    gen = torch.Generator(device="cuda").manual_seed(3)
    raw = torch.randint(0, 256, (n, 34), dtype=torch.uint8, device="cuda", generator=gen)
    raw[:, :2] = (0.001 + 0.01 * torch.rand(n, 1, device="cuda", generator=gen)).half().view(torch.uint8)
    x = torch.randn(m, k, device="cuda", generator=gen)
    w = ctx.upload_weight(cpvo.Q8_0, raw.view(-1), n, k)
    print(f"case n={n} k={k} m={m}", flush=True)
    y = ctx.qgemm(w, x)
    w.free()
    for r0 in (0, 4_000_003, n - 1000):
        part = ctx.upload_weight(cpvo.Q8_0, raw[r0:r0 + 1000].reshape(-1).contiguous(), 1000, k)
        assert torch.equal(y[:, r0:r0 + 1000], ctx.qgemm(part, x))
        part.free()
    ctx.close()


@pytest.mark.parametrize("m", [32, 100])
def test_qgemm_wide_q8_0_partial_unit(ctx, m):
    # K = 800: 25 blocks of 32, so the last 256-element unit holds one block
    y, ref = run_case(ctx, cpvo.Q8_0, 40, 800, m)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), np.abs(y - ref).max()


@pytest.mark.parametrize("tname", ["q4_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("k,n", [(5120, 7168), (5120, 5120), (5120, 17408), (17408, 5120)])
@pytest.mark.parametrize("m", [64, 256])
def test_qgemm_wide_bit_exact_prefill_shapes(ctx, tname, k, n, m):
    y, ref = run_case(ctx, TYPES[tname], n, k, m)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), np.abs(y - ref).max()


@pytest.mark.parametrize("tname", ["q4_k", "q6_k", "q8_0"])
def test_qgemm_wide_rows_match_the_skinny_kernel(ctx, tname):
    # a row's outputs do not depend on the rows batched with it: the wide
    # launch over 96 rows against the skinny kernel on 8-row slices
    t = TYPES[tname]
    n, k = 5120, 17408
    wq = weights(t, n, k)
    x = torch.from_numpy(np.random.default_rng(11).normal(0, 1, size=(96, k)).astype(np.float32)).cuda()
    w = ctx.upload_weight(t, wq, n, k)
    yw = ctx.qgemm(w, x).cpu().numpy()
    for r in range(0, 96, 8):
        ys = ctx.qgemm(w, x[r:r + 8].contiguous()).cpu().numpy()
        assert np.array_equal(yw[r:r + 8].view(np.uint32), ys.view(np.uint32)), r
    w.free()


@pytest.mark.parametrize("tname", ["q4_k", "q6_k", "q8_0"])
def test_qgemm_wide_extreme_scales_and_zero_rows(ctx, tname):
    t = TYPES[tname]
    n, k = 96, 1280
    rng = np.random.default_rng(4)
    wf = rng.normal(0, 0.02, size=(n, k)).astype(np.float32)
    wf[5] = 0.0
    wf[70] *= 1e3
    wq = cpvo.quantize(t, wf)
    x = rng.normal(0, 1, size=(70, k)).astype(np.float32)
    x[1] = 0.0
    x[2] *= 1e-6
    x[65] *= 1e4
    w = ctx.upload_weight(t, wq, n, k)
    y = ctx.qgemm(w, torch.from_numpy(x).cuda()).cpu().numpy()
    ref = cpvo.qgemm(t, wq, x)
    w.free()
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))
    assert np.all(y[1] == 0) and np.all(y[:, 5] == 0)


def test_qgemm_rejects_bad_shapes(ctx):
    from codpiece_amd import CpvError
    w = ctx.upload_weight(cpvo.Q8_0, weights(cpvo.Q8_0, 16, 64), 16, 64)
    x = torch.zeros((257, 64), dtype=torch.float32, device="cuda")
    with pytest.raises(CpvError):
        ctx.qgemm(w, x)
    with pytest.raises(CpvError):
        ctx.upload_weight(cpvo.Q4_K, np.zeros(144, np.uint8), 1, 100)


@pytest.mark.parametrize("tname,k", [(t, k) for t in TYPES for k in (512, 5120)] + [("q8_0", 800)])
def test_get_rows_matches_ggml_dequant(ctx, tname, k):
    # four elements per thread; 800 = 25 Q8_0 blocks (a partial 256-element
    # unit); ids outside the table give zero rows
    t = TYPES[tname]
    n = 300
    wq = weights(t, n, k)
    w = ctx.upload_weight(t, wq, n, k)
    ids = [0, 7, 299, 150, 7, 64, 63]
    rows = torch.tensor(ids + [-1, n], dtype=torch.int32, device="cuda")
    got = ctx.get_rows(w, rows).cpu().numpy()
    w.free()
    ref = cpvo.dequantize(t, wq, k)[ids]
    assert np.array_equal(got[:len(ids)].view(np.uint32), ref.view(np.uint32))
    assert not got[len(ids):].any()


def test_argmax_first_maximum_and_noise(ctx):
    rng = np.random.default_rng(1)
    x = rng.normal(size=(7, 151936)).astype(np.float32)
    x[0, 100] = x[0, 90000] = 50.0               # tie: the lower index wins
    x[1, :] = -np.inf
    x[1, 12] = -1e30
    nz = rng.normal(size=x.shape).astype(np.float32)
    xt, nt = torch.from_numpy(x).cuda(), torch.from_numpy(nz).cuda()
    got = ctx.argmax_rows(xt).cpu().numpy()
    want = [cpvo.argmax(r) for r in x]
    assert got.tolist() == want and got[0] == 100 and got[1] == 12
    got2 = ctx.argmax_rows(xt, nt).cpu().numpy()
    assert got2.tolist() == [cpvo.argmax((a + b).astype(np.float32)) for a, b in zip(x, nz)]
