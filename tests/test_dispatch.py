"""What the library's dispatch picks, by its host queries (no GPU): the rules
that a retuned estimate must not move past what was measured, and the forms
that the GPU parity tests are meant to reach."""
import ctypes

import pytest

from codpiece_amd import _lib


@pytest.fixture(scope="module")
def lib():
    lib = _lib.load()
    lib.cpv_attn_takes_limbs.argtypes = [ctypes.c_int64] + [ctypes.c_int] * 4
    lib.cpv_qgemm_wide_plan.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_int, ctypes.c_int * 5]
    return lib


def wide_plan(lib, tname, n, k, m, cus=256):
    """(16-row blocks per workgroup, row blocks, pairs over all of K, K slices
    of the others, units a slice), or None where the wide GEMM refuses."""
    out = (ctypes.c_int * 5)()
    ok = lib.cpv_qgemm_wide_plan({"q4_k": _lib.Q4_K, "q6_k": _lib.Q6_K, "q8_0": _lib.Q8_0}[tname], n, k, m, cus, out)
    return tuple(out) if ok else None


@pytest.mark.parametrize("n_past,t,h,h_kv,d,limbs", [
    (3584, 512, 40, 8, 128, 1), (3584, 102, 40, 8, 128, 0), (3584, 103, 40, 8, 128, 1),
    # 48-row blocks over the f16 caches (512 (chunk, KV head) units): d = 128
    # converts from 1536 query rows per KV head, by the limbs' bytes; d = 64 from 512
    (16384, 128, 40, 8, 128, 0), (32768, 103, 40, 8, 128, 0), (16384, 86, 24, 4, 128, 0), (8192, 256, 32, 8, 128, 0),
    (8192, 307, 40, 8, 128, 0), (8192, 308, 40, 8, 128, 1), (16384, 308, 40, 8, 128, 0), (16384, 410, 40, 8, 128, 1),
    (20000, 410, 40, 8, 128, 0), (32768, 512, 40, 8, 128, 0), (24000, 256, 24, 4, 128, 1), (12288, 2048, 16, 16, 128, 0),
    (16384, 64, 32, 4, 64, 1),
    # limbs of more than 256 MB
    (42000, 1024, 16, 16, 64, 1), (43000, 1024, 16, 16, 64, 0)])
def test_prompt_chunks_over_f16_caches(lib, n_past, t, h, h_kv, d, limbs):
    assert lib.cpv_attn_takes_limbs(n_past, t, h, h_kv, d) == limbs


@pytest.mark.parametrize("tname", ["q4_k", "q6_k", "q8_0"])
def test_wide_gemm_limits(lib, tname):
    # every weight that a grid of 2^32 - 1 threads can deal: 64-row tiles by
    # blocks of at least 64 activation rows; K up to 2^31 / 64 elements
    for n, m in ((8_400_000, 256), (200_000_000, 256), (60_000_000, 1024)):
        nmt, mblocks, nfull, ksplit, upk = wide_plan(lib, tname, n, 256, m)
        pairs = (n + 63) // 64 * mblocks
        assert nmt * mblocks * 16 >= m and 0 <= nfull <= pairs and (nfull + (pairs - nfull) * ksplit) * 256 < 2**32
    assert wide_plan(lib, tname, 64, 2**31 // 64 - 256, 256) and not wide_plan(lib, tname, 64, 2**31 // 64, 256)
    assert not wide_plan(lib, tname, 2**31, 256, 256)


@pytest.mark.parametrize("tname", ["q4_k", "q6_k", "q8_0"])
def test_wide_gemm_slices_cover_k(lib, tname):
    for tiles in (1, 3, 40, 272, 513, 811, 2374):
        for U in (1, 3, 11, 20, 68):
            for m in (17, 64, 100, 201, 256, 512):
                nmt, mblocks, nfull, ksplit, upk = wide_plan(lib, tname, 64 * tiles, 256 * U, m)
                assert 1 <= nmt <= (4 if tname == "q8_0" else 8) and nmt * mblocks * 16 >= m > nmt * 16 * (mblocks - 1)
                assert (ksplit - 1) * upk < U <= ksplit * upk and (ksplit == 1 or nfull < tiles * mblocks)
                assert ksplit > 1 or nfull == tiles * mblocks
