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


def _sample(t, raw, N, K, r, n=40):
    """Row numbers (the first, the last and n others) and their part of the matrix."""
    rows = np.unique(np.concatenate([[0, N - 1], r.choice(N, size=n, replace=False)]))
    if t == F16:
        return rows, raw[rows]
    rb = O.weight_bytes(t, 1, K)
    return rows, np.concatenate([raw[i * rb:(i + 1) * rb] for i in rows])


# More than four row groups per workgroup: a second batch takes over the partial sums' LDS and the pending
# request, with one window of K and with several; the last workgroups have fewer groups.
@pytest.mark.parametrize("t,N,K", [(O.GGML_Q8_0, 36009, 256), (O.GGML_Q8_0, 34001, 2336), (O.GGML_Q4_0, 36009, 512), (O.GGML_Q4_0, 33001, 4640),
                                   (F16, 33003, 160), (F16, 20001, 2144), (O.GGML_Q6_K, 36009, 256), (O.GGML_Q6_K, 33001, 2304)])
@pytest.mark.parametrize("a_dtype", [np.float16, np.float32])
def test_several_batches_per_workgroup(cuda, t, N, K, a_dtype):
    raw, x = _case(t, N, K, 16, a_dtype, N + K)
    rows, sub = _sample(t, raw, N, K, np.random.default_rng(K))
    y64 = _want(t, sub, x, rows.size, K)
    full = _gemm(cuda, t, raw, x, N, K)
    bound = 2.0 ** -11 if a_dtype == np.float32 else 1e-5
    assert np.abs(full[:, rows] - y64).max() / np.abs(y64).max() <= bound
    assert np.array_equal(_gemm(cuda, t, raw, x[:5], N, K), full[:5])


# fp32 rows outside f16's range are scaled per unit of K by a power of two that is undone exactly, so each row
# keeps the error of its rounding to f16, 2^-11 of the terms' magnitude.
@pytest.mark.parametrize("t,N,K", [(O.GGML_Q8_0, 20501, 2336), (O.GGML_Q4_0, 6161, 4640), (F16, 4099, 2144), (O.GGML_Q6_K, 12301, 2304)])
def test_staged_fp32_rows_beyond_f16_range(cuda, t, N, K):
    r = np.random.default_rng(N)
    raw, x = _case(t, N, K, 7, np.float32, N)
    x[0] *= 1e6
    x[1, :100] *= 3e5        # units of one row scaled differently
    x[2] *= 1e-7
    x[3] *= 1e30
    x[4] *= 1e-30
    x[5, 700:] *= 1e-12
    rows, sub = _sample(t, raw, N, K, r)
    y64 = _want(t, sub, x, rows.size, K) if t == F16 else x.astype(np.float64) @ O.dequantize_f64(t, sub, rows.size * K).reshape(rows.size, K).T
    got = _gemm(cuda, t, raw, x, N, K)[:, rows].astype(np.float64)
    for m in range(7):
        assert np.isfinite(got[m]).all()
        assert np.abs(got[m] - y64[m]).max() <= 2.0 ** -11 * np.abs(y64[m]).max(), m


@pytest.mark.parametrize("t,K", [(O.GGML_Q8_0, 2080), (O.GGML_Q4_0, 2336), (F16, 2080), (O.GGML_Q6_K, 2304)])
@pytest.mark.parametrize("M,ns", [(5, (1025, 1031, 1040)), (8, (1027, 1039)), (16, (1024, 1500, 1033, 1025))])
def test_staged_batch_equals_single_calls(cuda, t, K, M, ns):
    """Matrices with odd row counts in one launch: row groups never cross from one to the next."""
    import torch
    import qmm
    r = np.random.default_rng(K + M)
    raws = [_case(t, n, K, 1, np.float16, n)[0] for n in ns]
    A = torch.from_numpy(r.standard_normal((M, K)).astype(np.float16)).to(cuda)
    Ws = [torch.from_numpy(np.ascontiguousarray(w).view(np.uint8).reshape(-1)).to(cuda) for w in raws]
    Cs = [torch.full((M, n), float("nan"), device=cuda) for n in ns]
    d = (qmm.GemmDesc * len(ns))()
    for x, n, W, C in zip(d, ns, Ws, Cs):
        x.ggml_type, x.A, x.a_dtype, x.W, x.C, x.c_dtype = t, A.data_ptr(), qmm.DTYPE_F16, W.data_ptr(), C.data_ptr(), qmm.DTYPE_F32
        x.M, x.N, x.K = M, n, K
    qmm.gemm_batch(d)
    for n, W, C in zip(ns, Ws, Cs):
        w = W.view(torch.float16).view(n, K) if t == F16 else W
        assert torch.equal(C, qmm.gemm(t, A, w, n, K, out_dtype=torch.float32)), n


@pytest.mark.parametrize("t,N,K", [(O.GGML_Q8_0, 10241, 3296), (O.GGML_Q4_0, 14337, 2368), (O.GGML_Q8_0, 3073, 10944), (F16, 3073, 2048)])
@pytest.mark.parametrize("M", [3, 4])
def test_large_matrices_at_three_and_four_rows(cuda, t, N, K, M):
    raw, x = _case(t, N, K, M, np.float16, N + M)
    rows, sub = _sample(t, raw, N, K, np.random.default_rng(M))
    y64 = _want(t, sub, x, rows.size, K)
    assert np.abs(_gemm(cuda, t, raw, x, N, K)[:, rows] - y64).max() / np.abs(y64).max() <= 1e-5
