"""The choice among the prefill GEMM kernels, through the measurement library and
without a device, for a card of 256 CUs."""
import ctypes as C

import pytest

from edgerunner_amd import _ffi

TYPE = {"q4_k": 12, "q8_0": 8}
SPLIT, LOADER128, LOADER256, GROUPED = range(4)


def plan(fmt, T, N, K):
    """(kernel, tokens per tile, splits of K over workgroups)"""
    p = (C.c_uint32 * 3)()
    assert _ffi.load_probe().er_hip_probe_gemm_plan(TYPE[fmt], T, N, K, 256, p) == 0
    return tuple(p)


@pytest.mark.parametrize("fmt,T,N,K,kernel", [
    # few tiles of a long K: 16.8 us split against 18.5 K-grouped, 19.7 against 24.2, 22.1 against 24.8
    ("q4_k", 13, 6192, 4608, SPLIT), ("q4_k", 10, 6456, 6656, SPLIT), ("q8_0", 10, 6456, 6656, SPLIT),
    ("q4_k", 16, 2048, 2048, SPLIT), ("q8_0", 32, 4096, 4096, SPLIT),
    # small matrices: 4.9 us K-grouped against 7.0, 5.6 against 7.2, 6.0 against 7.1
    ("q8_0", 11, 264, 768, GROUPED), ("q8_0", 51, 264, 1024, GROUPED), ("q4_k", 51, 264, 1024, GROUPED),
    ("q8_0", 16, 1024, 1024, GROUPED), ("q8_0", 100, 4096, 4096, GROUPED), ("q4_k", 256, 3072, 1024, GROUPED),
    ("q4_k", 100, 14336, 2048, LOADER128), ("q4_k", 512, 4096, 4096, LOADER128), ("q4_k", 512, 14336, 4096, LOADER256)])
def test_kernel_of_a_shape(fmt, T, N, K, kernel):
    assert plan(fmt, T, N, K)[0] == kernel


def test_no_split_without_the_zero_fill():
    """T N not a multiple of 4: Y cannot be cleared by the fill, so K stays whole."""
    for T in (1, 3, 33, 129):
        assert plan("q8_0", T, 4097, 4096)[2] == 1
