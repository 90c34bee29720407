"""Matrix-core GEMV of Q4_0, Q8_0 and F16 weights, and of Q6_K rows that are not whole 16-byte pieces.

Against fp64 on the exact weights: fp16 activations and codes enter exactly, so only fp32 sums remain; fp32
activations are rounded to fp16 first (at most 2^-11 of each).
"""

import numpy as np
import pytest

import gguf_oracle as O

pytestmark = pytest.mark.gpu
F16 = 1


def _case(t, N, K, M, a_dtype, seed):
    r = np.random.default_rng(seed)
    if t == F16:
        raw = (r.standard_normal((N, K)) / 32).astype(np.float16)
    else:
        raw = O.synth_weights(t, N, K, r)
    x = r.standard_normal((M, K)).astype(a_dtype)
    return raw, x


def _want(t, raw, x, N, K):
    if t == F16:
        return x.astype(np.float64) @ raw.astype(np.float64).T
    return O.matmul_f64(t, x.astype(np.float32), raw, N, K)


def _gemm(dev, t, raw, x, N, K, off=0):
    import torch
    import qmm
    b = torch.from_numpy(np.ascontiguousarray(raw).view(np.uint8).reshape(-1))
    buf = torch.empty(b.numel() + off, dtype=torch.uint8, device=dev)
    buf[off:] = b.to(dev)
    W = buf[off:].view(torch.float16).view(N, K) if t == F16 else buf[off:]
    C = qmm.gemm(t, torch.from_numpy(x).to(dev), W, N, K, out_dtype=torch.float32)
    torch.cuda.synchronize()
    return C.cpu().numpy()


# Rows of 1024 and 1025 (a last row tile of one row), K from one block to several windows with partial
# units and windows, odd block counts (rows 2 bytes off), a matrix whose last piece is not whole.
CASES = [(O.GGML_Q8_0, 1025, 32), (O.GGML_Q8_0, 1024, 2048), (O.GGML_Q8_0, 1025, 2080), (O.GGML_Q8_0, 1031, 4544),
         (O.GGML_Q4_0, 1025, 32), (O.GGML_Q4_0, 1024, 2048), (O.GGML_Q4_0, 1057, 2336), (O.GGML_Q4_0, 1025, 5280),
         (F16, 1025, 32), (F16, 1024, 1024), (F16, 1041, 2144), (O.GGML_Q6_K, 1025, 256), (O.GGML_Q6_K, 1030, 2304),
         (O.GGML_Q6_K, 1024, 5888)]


@pytest.mark.parametrize("t,N,K", CASES)
@pytest.mark.parametrize("a_dtype", [np.float16, np.float32])
def test_staged_gemv_vs_fp64(cuda, t, N, K, a_dtype):
    for M in (5, 16):
        raw, x = _case(t, N, K, M, a_dtype, 31 * N + K + M)
        y64 = _want(t, raw, x, N, K)
        err = np.abs(_gemm(cuda, t, raw, x, N, K) - y64).max() / np.abs(y64).max()
        bound = 2.0 ** -11 if a_dtype == np.float32 else 1e-5
        assert err <= bound, (M, err)


@pytest.mark.parametrize("t,N,K", [(O.GGML_Q8_0, 1025, 2080), (O.GGML_Q4_0, 1025, 2336), (F16, 1030, 1056), (O.GGML_Q6_K, 1027, 2304)])
def test_staged_gemv_rows_and_alignment(cuda, t, N, K):
    """Each row is the same for every M that the kernel serves, and for weights 2 bytes off a 16-byte
    boundary."""
    raw, x = _case(t, N, K, 16, np.float16, N + K)
    full = _gemm(cuda, t, raw, x, N, K)
    for M in (5, 6, 9):
        assert np.array_equal(_gemm(cuda, t, raw, x[:M], N, K), full[:M]), M
    assert np.array_equal(_gemm(cuda, t, raw, x, N, K, off=2), full)


# Few rows: the activation rows run in passes of four and more beside each other, the last one shorter.
@pytest.mark.parametrize("t,N,K", [(O.GGML_Q8_0, 16, 2048), (O.GGML_Q8_0, 513, 2080), (O.GGML_Q4_0, 1, 32), (O.GGML_Q4_0, 515, 4640),
                                   (O.GGML_Q6_K, 33, 2304), (O.GGML_Q6_K, 1000, 256), (F16, 1040, 2080)])
def test_few_rows_in_several_passes(cuda, t, N, K):
    raw, x = _case(t, N, K, 16, np.float16, N + K)
    y64 = _want(t, raw, x, N, K)
    full = _gemm(cuda, t, raw, x, N, K)
    assert np.abs(full - y64).max() / np.abs(y64).max() <= 1e-5
    for M in (5, 7, 8, 13, 14):
        assert np.array_equal(_gemm(cuda, t, raw, x[:M], N, K), full[:M]), M


@pytest.mark.parametrize("M", [17, 20, 33, 40, 100])
def test_more_rows_than_one_pass(cuda, M):
    """With the GEMV / prefill threshold raised: passes without a row are not launched."""
    import qmm
    t, N, K = O.GGML_Q8_0, 1024, 544
    raw, x = _case(t, N, K, M, np.float16, M)
    y64 = _want(t, raw, x, N, K)
    qmm.set_thread_gemv_max_m(256)
    try:
        got = _gemm(cuda, t, raw, x, N, K)
    finally:
        qmm.set_thread_gemv_max_m(0)
    assert np.abs(got - y64).max() / np.abs(y64).max() <= 1e-5
    assert np.array_equal(got[:16], _gemm(cuda, t, raw, x[:16], N, K))
