"""Attention and prefill calls of several host threads on one stream: each call's workspace is its own.

Every result equals the single-threaded one bit for bit, with calls of different sizes (so that the scratch
grows while another thread is at work), and with the scratch released in between.
"""

import threading

import pytest

pytestmark = pytest.mark.gpu

CASES = [(40, 1500, 32, 8, 128), (17, 3000, 8, 2, 64), (3, 2000, 32, 8, 128), (64, 4000, 16, 4, 128)]


def _call(q, k, v, out, case, stream):
    import qmm
    n, pos, heads, kvh, d = case
    qmm.check(qmm.lib().qmm_gqa_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), n, pos + n, heads, kvh, d, pos,
                                          0.0, 1, stream))


@pytest.mark.parametrize("per_thread", [False, True])
def test_threads_on_one_stream_handle(cuda, per_thread):
    import torch
    import qmm
    g = torch.Generator(device=cuda)
    g.manual_seed(11)
    stream = 2 if per_thread else torch.cuda.current_stream().cuda_stream  # 2: hipStreamPerThread
    ins, want = [], []
    for n, pos, heads, kvh, d in CASES:
        ins.append([torch.randn(s, generator=g, device=cuda).half() for s in ((n, heads * d), (pos + n, kvh * d), (pos + n, kvh * d))])
    torch.cuda.synchronize()
    qmm.check(qmm.lib().qmm_release_workspace())
    for t, c in zip(ins, CASES):
        out = torch.empty_like(t[0])
        torch.cuda.synchronize()
        _call(*t, out, c, stream)
        torch.cuda.synchronize()
        want.append(out)
    qmm.check(qmm.lib().qmm_release_workspace())
    outs = [[torch.empty_like(t[0]) for _ in range(40)] for t in ins]
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            torch.cuda.set_device(cuda)
            for j, out in enumerate(outs[i]):
                _call(*ins[i], out, CASES[i], stream)
                if i == 2 and j % 13 == 12:
                    qmm.check(qmm.lib().qmm_release_workspace())
        except Exception as e:  # reported by the main thread
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(CASES))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    for i, w in enumerate(want):
        for out in outs[i]:
            assert torch.equal(out, w), CASES[i]


def test_prefill_threads_on_one_stream(cuda):
    """Prefill products whose activations are converted into, and whose K is split over, the stream's workspace."""
    import torch
    import qmm
    g = torch.Generator(device=cuda)
    g.manual_seed(12)
    stream = torch.cuda.current_stream().cuda_stream
    cases = [(20, 512, 4096), (100, 384, 8192), (40, 2048, 2080), (130, 256, 14336)]  # M, N, K
    A = [torch.randn((m, k), generator=g, device=cuda) for m, _, k in cases]
    W = [(torch.randn((n, k), generator=g, device=cuda) / k ** 0.5).half() for _, n, k in cases]

    def call(i, out):
        m, n, k = cases[i]
        qmm.check(qmm.lib().qmm_gemm(1, A[i].data_ptr(), qmm.DTYPE_F32, W[i].data_ptr(), out.data_ptr(), qmm.DTYPE_F32, m, n, k, stream))
    want = []
    for i, (m, n, _) in enumerate(cases):
        want.append(torch.empty((m, n), device=cuda))
        call(i, want[i])
    torch.cuda.synchronize()
    for i, (m, n, k) in enumerate(cases):
        y64 = A[i].double() @ W[i].double().t().contiguous()
        assert float((want[i] - y64).abs().max() / y64.abs().max()) < 1e-3
    qmm.check(qmm.lib().qmm_release_workspace())
    outs = [[torch.empty_like(want[i]) for _ in range(40)] for i in range(len(cases))]
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            torch.cuda.set_device(cuda)
            for j, out in enumerate(outs[i]):
                call(i, out)
                if i == 1 and j % 13 == 12:
                    qmm.check(qmm.lib().qmm_release_workspace())
        except Exception as e:  # reported by the main thread
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    for i in range(len(cases)):
        assert all(torch.equal(out, want[i]) for out in outs[i]), cases[i]
