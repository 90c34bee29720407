"""Which kernel serves a GEMV-size matrix: points on both sides of each line, by the library's own function.

0 is the v_dot2 GEMV, 1 the matrix-core GEMV with an LDS ring, 2 the one staged through registers.  The lines
are where the two were measured to cross; the points below are sizes at which one side was clearly faster, or
at which a batch of matrices that share their activations would fall apart into more launches.
"""

import ctypes

import pytest

import qmm

F16, Q4_0, Q8_0, Q4_K, Q6_K = 1, 2, 8, 12, 14
H, F = qmm.DTYPE_F16, qmm.DTYPE_F32

_kind = getattr(qmm.lib(), "_ZN3qmm14gemv_mfma_kindEiPKviiiib")
_kind.restype = ctypes.c_int
_kind.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_bool]


def kind(t, M, N, K, a=H, identity=False, W=4096):
    return _kind(t, W, M, N, K, a, identity)


@pytest.mark.parametrize("t", [Q8_0, Q4_0, Q6_K, F16])
def test_fp32_activations_stay_on_v_dot2_up_to_many_rows(t):
    K = 14080 if t == Q6_K else 14336
    for M in (3, 4, 5, 8, 16):
        for N in (64, 1024, 2048):
            assert kind(t, M, N, K, F) == 0, (M, N)
    assert kind(t, 8, 28672, 4352, F) == 2 and kind(t, 3, 28672, 4352, F) == (2 if t == F16 else 0)
    assert kind(Q8_0, 6, 14336, 8192, F) == 0 and kind(Q4_0, 6, 8192, 8192, F) == 2


@pytest.mark.parametrize("t", [Q8_0, Q4_0, Q6_K])
def test_matrices_that_share_activations_agree(t):
    """q with k and v of few rows: one kernel, so one launch, where that is the faster one for each of them."""
    for h in (2048, 4096, 8192):
        K = h + 256 if t == Q6_K else h
        for kv in (64, 128, 512, 1024):
            for M in (3, 4, 5, 6, 8, 13, 16):
                assert kind(t, M, h, K) == kind(t, M, kv, K), (h, kv, M)
        for M in (9, 12):
            assert kind(t, M, 1024, K) == kind(t, M, h, K) == 2 and kind(t, M, 512, K) == 0


def test_large_matrices_at_three_and_four_rows():
    for t in (Q8_0, Q4_0):
        assert kind(t, 3, 14336, 4096) == kind(t, 4, 28672, 8192) == kind(t, 3, 8192, 28672) == kind(t, 4, 14336, 14336) == 2
        assert kind(t, 3, 8192, 8192) == kind(t, 4, 4096, 4096) == kind(t, 3, 8192, 4096) == kind(t, 2, 28672, 8192) == 0
    assert kind(Q8_0, 3, 4096, 14336) == 2 and kind(Q4_0, 3, 4096, 14336) == 0
    assert kind(Q6_K, 4, 28672, 14080) == 0


def test_f16_rows():
    for M in (3, 5, 8, 9, 16):
        assert kind(F16, M, 4096, 4096) == kind(F16, M, 1024, 4096) == kind(F16, M, 3072, 2048) == 2
        assert kind(F16, M, 2048, 2048) == kind(F16, M, 512, 2048) == kind(F16, M, 1023, 4096) == 0
    assert kind(F16, 2, 8192, 8192) == 0


def test_other_conditions():
    assert kind(Q8_0, 8, 4096, 4096, identity=True) == kind(Q8_0, 8, 4096, 4096, W=4097) == 0
    assert kind(F16, 8, 4096, 4104) == 0 and kind(Q6_K, 8, 512, 2048) == 1 and kind(Q6_K, 8, 512, 2048, W=4098) == 2
    assert kind(Q4_K, 1, 64, 256) == 0 and kind(Q4_K, 1, 64, 256, identity=True) == kind(Q4_K, 2, 64, 256, F) == 1
    assert kind(Q8_0, 20, 512, 4096) == 0 and kind(Q8_0, 20, 1024, 4096) == 2
