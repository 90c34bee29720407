"""Prefill of Q8_0 and Q4_0 rows read as runs of two blocks: K tails with one block of a run, or none.

Against the fp64 product of the kernel's own f16 operands: only fp32 sums remain (1e-5, the bar of
test_gpu_prefill.py).
"""

import numpy as np
import pytest

import gguf_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [O.GGML_Q8_0, O.GGML_Q4_0])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 160, 192, 224, 1184])
def test_block_run_tails(cuda, t, K):
    import torch
    import qmm
    N = 37
    r = np.random.default_rng(K + t)
    raw = O.synth_weights(t, N, K, r)
    W = torch.from_numpy(np.ascontiguousarray(raw)).to(cuda)
    for M in (20, 130):
        x = r.standard_normal((M, K)).astype(np.float16)
        got = qmm.gemm(t, torch.from_numpy(x).to(cuda), W, N, K, out_dtype=torch.float32).cpu().numpy()
        want = O.matmul_f16_operands(t, x.astype(np.float32), raw, N, K)
        assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max(), M
