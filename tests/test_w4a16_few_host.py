"""CPU tier: the rules by which shapes reach the few-row W4A16 GEMM
(csrc/w4a16_few.hpp, compiled with g++) and its entry point's refusals."""
import ctypes
import os
import subprocess

import pytest

from cudaforge_amd import _lib

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "w4a16_few_host.cpp")
LIB = os.path.join(HERE, "native", "libw4a16_few_host.so")
HDR = os.path.join(os.path.dirname(HERE), "cudaforge_amd", "csrc", "w4a16_few.hpp")


@pytest.fixture(scope="module")
def few():
    if not os.path.exists(LIB) or os.path.getmtime(LIB) < max(os.path.getmtime(f) for f in (SRC, HDR)):
        subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", SRC, "-o", LIB], check=True)
    return ctypes.CDLL(LIB)


@pytest.mark.parametrize("M", [1, 16, 17, 128, 129])
def test_word_offsets_fit_32_bits(few, M):
    """Lane offsets of w4few_kernel: 4 * (row N + 4 l) bytes, row <= 15, l <=
    31, and the 16 bytes from there.  Every N that 17 rows and more are taken
    for has to keep them below 2^32; up to 16 rows no such offset is formed."""
    assert few.few_takes(M, 256, 128) == (M <= 128)
    for N in (2 ** 26, 2 ** 26 + 128, 71582720, 71582848, 2 ** 28, 2 ** 31 - 128):
        fits = 4 * (15 * N + 4 * 31) + 16 <= 2 ** 32
        assert few.few_takes(M, N, 128) <= (M <= 16 or fits)
    assert few.few_takes(M, 2 ** 26, 128) == (M <= 128)
    assert few.few_takes(M, 2 ** 31 - 128, 128) == (M <= 16)


@pytest.mark.parametrize("M", [17, 128])
def test_entry_refuses_wider_weights(M):
    lib = _lib.load()
    rc = lib.cfa_w4a16_gemm_few(16, 16, 16, 16, M, 2 ** 26 + 128, 128, 128, 0, 16, None, 0, None)
    assert rc == _lib.CFA_ERR_ARG and "2^26" in _lib.last_error()
    assert lib.cfa_w4a16_gemm_few_workspace_size(M, 2 ** 26 + 128, 128) == 0


@pytest.mark.parametrize("spg", [1, 2, 3, 4, 5, 7, 127, 4099, 65535, 65537, 65900, 131071, 2 ** 20 + 1,
                                 2 ** 25 - 1, 2 ** 25 + 1, 2 ** 26 - 1, 2 ** 26])
def test_scale_group_of_a_slice(few, spg):
    """slice / spg at every slice next to a multiple of spg, for K up to the
    entry points' bound of 2^31 (2^26 slices); one slice into another group
    would read past the scales (spg = 65900 at K = 2108800 did)."""
    few.few_group.restype = few.few_group_wrong.restype = ctypes.c_uint32
    top = 2 ** 26
    assert few.few_group_wrong(0, min(top, 1 << 18), spg) == min(top, 1 << 18)
    assert few.few_group_wrong(top - (1 << 18), top, spg) == top
    step = max(1, top // spg // 3000)
    for q in list(range(0, top // spg, step)) + [top // spg]:
        for sl in (q * spg - 1, q * spg, q * spg + spg - 1):
            if 0 <= sl < top:
                assert few.few_group(sl, spg) == sl // spg


def test_workspace_for_more_rows_serves_fewer():
    """A buffer sized for a call's largest M (up to one 256-row tile) is large
    enough for every smaller one, whichever kernel each takes."""
    lib = _lib.load()
    rows = (1, 4, 15, 16, 17, 32, 33, 63, 64, 65, 100, 127, 128, 129, 160, 200, 256)
    for N in (256, 512, 768, 1024, 1280, 2048, 3072, 4096, 6144, 12288, 14336, 28672):
        for K in (128, 256, 1024, 1152, 4096, 8192, 8320, 14336, 16384, 20480, 32768, 65536, 131072):
            size = [lib.cfa_w4a16_gemm_zp_workspace_size(M, N, K) for M in rows]
            assert size == sorted(size), (N, K, size)
            part = [lib.cfa_w4a16_gemm_zp_splits(M, N, K) * M for M in rows]
            assert part == sorted(part), (N, K, part)
            assert max(lib.cfa_w4a16_gemm_zp_splits(M, N, K) for M in rows) <= 16
            for M in rows[:13]:
                assert lib.cfa_w4a16_gemm_few_workspace_size(M, N, K) <= 16 * 4 * M * N


@pytest.mark.parametrize("M", [4, 100])
def test_small_workspace_names_the_entrys_own_size_function(M):
    lib = _lib.load()
    N, K = 384, 4096                       # not a width that cfa_w4a16_gemm_zp takes
    need = lib.cfa_w4a16_gemm_few_workspace_size(M, N, K)
    assert need > 0 and lib.cfa_w4a16_gemm_zp_workspace_size(M, N, K) == 0
    rc = lib.cfa_w4a16_gemm_few(16, 16, 16, 16, M, N, K, 128, 0, 16, 16, need - 16, None)
    assert rc == _lib.CFA_ERR_ARG and "cfa_w4a16_gemm_few_workspace_size" in _lib.last_error()
    rc = lib.cfa_w4a16_gemm_zp(16, 16, 16, 16, M, 256, K, 128, 16, 16, 16, None)
    assert rc == _lib.CFA_ERR_ARG and "cfa_w4a16_gemm_zp_workspace_size" in _lib.last_error()
