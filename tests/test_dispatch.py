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
    return lib


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
