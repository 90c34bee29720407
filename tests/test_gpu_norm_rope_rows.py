"""RMSNorm rows held in registers (K % 8 == 0, K <= 16384) and their neighbours, and RoPE blocks of several heads.

Bars as in test_gpu_layer.py: 2e-3 absolute of the CPU restatement, for outputs of order 1.
"""

import numpy as np
import pytest

import layer_oracle as L

pytestmark = pytest.mark.gpu


def _dev(x, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


@pytest.mark.parametrize("K", [8, 2056, 4096, 4104, 8192, 8200, 16384, 16392, 1001])
@pytest.mark.parametrize("wdt", [np.float16, np.float32])
def test_rmsnorm_row_sizes(cuda, K, wdt):
    import torch
    import qmm
    r = np.random.default_rng(K)
    x, res = (r.standard_normal((3, K)).astype(np.float16) for _ in range(2))
    w = (1 + 0.1 * r.standard_normal(K)).astype(wdt)
    X, R, W = _dev(x, cuda), _dev(res, cuda), _dev(w, cuda)
    s = torch.cuda.current_stream().cuda_stream
    dt = qmm.DTYPE_F32 if wdt == np.float32 else qmm.DTYPE_F16
    out = torch.empty_like(X)
    qmm.check(qmm.lib().qmm_rmsnorm(X.data_ptr(), W.data_ptr(), dt, out.data_ptr(), 3, K, 1e-5, s))
    torch.cuda.synchronize()
    assert np.abs(out.cpu().numpy().astype(np.float32) - L.rmsnorm(x, w, 1e-5).astype(np.float32)).max() < 4e-3
    h = torch.empty_like(X)
    qmm.check(qmm.lib().qmm_rmsnorm_residual(X.data_ptr(), R.data_ptr(), W.data_ptr(), dt, h.data_ptr(), out.data_ptr(), 3, K, 1e-5, s))
    torch.cuda.synchronize()
    wh, wn = L.rmsnorm_residual(x, res, w, 1e-5)
    assert np.array_equal(h.cpu().numpy(), wh)
    assert np.abs(out.cpu().numpy().astype(np.float32) - wn.astype(np.float32)).max() < 4e-3


@pytest.mark.parametrize("seq,heads,d,neox", [(1, 3, 2, False), (1, 40, 128, True), (300, 9, 96, False), (700, 64, 128, True), (5, 33, 256, False)])
def test_rope_head_blocks(cuda, seq, heads, d, neox):
    import torch
    import qmm
    x = np.random.default_rng(seq + d).standard_normal((seq, heads, d)).astype(np.float16)
    X = _dev(x, cuda)
    out = torch.empty_like(X)
    qmm.check(qmm.lib().qmm_rope(X.data_ptr(), out.data_ptr(), seq, heads, d, 7, 10000.0, int(neox), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert np.abs(out.cpu().numpy().astype(np.float32) - L.rope(x, 7, 10000.0, neox).astype(np.float32)).max() < 4e-3


@pytest.mark.parametrize("seq,heads,d,neox", [(1, 1, 128, False), (7, 1, 128, True), (1001, 1, 64, False), (13, 2, 2, True), (9, 5, 64, False), (3, 127, 4, True)])
def test_rope_few_heads(cuda, seq, heads, d, neox):
    """Blocks of several positions, the last one not full."""
    test_rope_head_blocks(cuda, seq, heads, d, neox)
