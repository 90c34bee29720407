"""Attention with its keys split over workgroups, and the 16-row matrix-core kernel of short calls.

Against the CPU restatement (oracle/layer_oracle.py).  Both sides round to fp16 once (half an ulp each,
2^-11 of the largest output together twice that); the 128-row kernel also rounds each weight p to fp16,
at most 2^-11 sum(p |v|) / sum(p) <= 2^-11 max |v|.  fp32 sums of up to a few thousand terms add 1e-5 max |v|.
"""

import numpy as np
import pytest

import layer_oracle as L

pytestmark = pytest.mark.gpu


def _run(dev, Q, K, V, start, causal):
    import torch
    import qmm
    q_len, heads, d = Q.shape
    kv_len, kvh, _ = K.shape
    t = [torch.from_numpy(x).to(dev) for x in (Q, K, V)]
    out = torch.full((q_len, heads, d), 7.0, dtype=torch.float16, device=dev)
    qmm.check(qmm.lib().qmm_gqa_attention(t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), out.data_ptr(), q_len, kv_len, heads,
                                          kvh, d, start, 0.0, int(causal), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _inputs(q_len, kv_len, heads, kvh, d, seed):
    r = np.random.default_rng(seed)
    return [r.standard_normal(s).astype(np.float16) for s in ((q_len, heads, d), (kv_len, kvh, d), (kv_len, kvh, d))]


# 16-row tiles: one row to several tiles, 32-key blocks, 128-key ranges and their edges, groups that do
# not divide the tile, start positions past the keys; 128-row tiles: ranges of two 64-key tiles and more,
# rows that see no key of their tile's last range.
@pytest.mark.parametrize("q_len,kv_len,start,heads,kvh,d,causal", [
    (1, 1, 0, 4, 4, 128, True), (1, 32, 31, 8, 2, 64, True), (1, 33, 32, 8, 1, 128, True), (1, 128, 127, 32, 8, 128, True),
    (1, 129, 128, 32, 8, 128, True), (1, 4001, 4000, 32, 8, 128, True), (2, 257, 255, 8, 8, 64, True), (3, 500, 497, 21, 3, 128, True),
    (15, 15, 0, 64, 8, 128, True), (15, 1200, 1185, 8, 1, 64, True), (9, 300, 0, 8, 2, 128, False), (4, 70, 500, 8, 2, 128, True),
    (5, 40, 0, 8, 2, 128, True), (40, 600, 560, 6, 2, 128, True), (17, 4096, 4079, 20, 4, 64, True),
    (16, 129, 113, 8, 8, 128, True), (40, 3040, 3000, 32, 8, 128, True), (130, 700, 570, 4, 4, 64, True), (33, 777, 0, 8, 2, 128, False),
    (257, 257, 0, 4, 4, 128, True), (64, 2048, 100, 16, 2, 64, True),
    # ranges that a tile's first rows do not see, merged by a thread group of their own
    (700, 800, 100, 4, 4, 128, True), (700, 790, 90, 8, 2, 64, True)])
def test_split_attention(cuda, q_len, kv_len, start, heads, kvh, d, causal):
    Q, K, V = _inputs(q_len, kv_len, heads, kvh, d, 7 * q_len + kv_len + d)
    got = _run(cuda, Q, K, V, start, causal).astype(np.float32)
    want = L.gqa_attention(Q, K, V, start, 0.0, causal).astype(np.float32)
    vmax = float(np.abs(V).max())
    p16 = q_len >= 16 and 128 % (heads // kvh) == 0
    bound = 2.0 ** -10 * float(np.abs(want).max()) + (2.0 ** -11 if p16 else 0.0) * vmax + 1e-5 * vmax
    assert float(np.abs(got - want).max()) <= bound


# both sides of the line between one range and several, last ranges of one key, and ranges that only the
# last rows of their tile see
@pytest.mark.parametrize("q_len,kv_len,start,heads,kvh,d,causal", [
    (1, 640, 639, 32, 8, 128, True), (1, 641, 640, 32, 8, 128, True), (1, 769, 768, 32, 8, 128, True), (1, 1025, 1024, 24, 8, 64, True),
    (15, 1281, 1266, 64, 8, 128, True), (15, 1281, 1266, 20, 4, 64, True), (16, 257, 241, 8, 8, 128, True), (16, 577, 561, 8, 8, 128, True),
    (40, 1089, 1049, 32, 8, 64, True), (100, 833, 733, 4, 4, 64, True), (200, 1025, 825, 8, 2, 128, True), (320, 1000, 680, 4, 1, 128, True)])
def test_split_edges(cuda, q_len, kv_len, start, heads, kvh, d, causal):
    test_split_attention(cuda, q_len, kv_len, start, heads, kvh, d, causal)


@pytest.mark.parametrize("q_len", [3, 40])
def test_negative_scale(cuda, q_len):
    import torch
    import qmm
    Q, K, V = _inputs(q_len, 200, 8, 2, 128, 5)
    t = [torch.from_numpy(x).to(cuda) for x in (Q, K, V)]
    out = torch.empty_like(t[0])
    qmm.check(qmm.lib().qmm_gqa_attention(t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), out.data_ptr(), q_len, 200, 8, 2, 128,
                                          200 - q_len, -0.07, 1, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    want = L.gqa_attention(Q, K, V, 200 - q_len, -0.07, True).astype(np.float32)
    vmax = float(np.abs(V).max())
    bound = 2.0 ** -10 * float(np.abs(want).max()) + 2.0 ** -11 * vmax + 1e-5 * vmax
    assert float(np.abs(out.cpu().numpy().astype(np.float32) - want).max()) <= bound


def test_rows_ignore_values_they_do_not_see(cuda):
    """A later position's infinite or NaN value reaches only the rows that see it."""
    Q, K, V = _inputs(5, 140, 8, 2, 128, 3)
    clean = _run(cuda, Q, K, V, 135, True)
    V[138, 1, 5], V[139, 0, 9] = np.inf, np.nan
    got = _run(cuda, Q, K, V, 135, True)
    assert np.array_equal(got[:3].view(np.uint16), clean[:3].view(np.uint16))
    assert not np.isfinite(got[3:, 4:, 5]).any() and np.isfinite(got[3, :4]).all() and np.isnan(got[4, :4, 9]).all()


@pytest.mark.parametrize("q_len,kv_len", [(1, 140), (5, 140), (3, 4000)])
@pytest.mark.parametrize("d", [64, 128])
def test_infinite_values_that_a_row_sees(cuda, q_len, kv_len, d):
    """An infinite value gives an infinite output of its sign, +inf and -inf together NaN, a NaN value NaN, and
    the other outputs do not change."""
    Q, K, V = _inputs(q_len, kv_len, 8, 2, d, 5)
    clean = _run(cuda, Q, K, V, kv_len - q_len, True)
    V[10, 1, 5] = V[20, 1, 9] = V[100, 1, 50] = np.inf
    V[40, 1, 7] = V[77, 1, 9] = -np.inf
    V[33, 1, 11] = np.nan
    got = _run(cuda, Q, K, V, kv_len - q_len, True)
    assert (got[:, 4:, [5, 50]] == np.inf).all() and (got[:, 4:, 7] == -np.inf).all() and np.isnan(got[:, 4:, [9, 11]]).all()
    keep = np.ones(got.shape, bool)
    keep[:, 4:, [5, 50, 7, 9, 11]] = False
    assert np.array_equal(got[keep].view(np.uint16), clean[keep].view(np.uint16))


@pytest.mark.parametrize("q_len,kv_len", [(3, 140), (3, 4000)])
def test_nan_scores_stay_with_their_row(cuda, q_len, kv_len):
    """A NaN query makes its own row NaN; a NaN key every row that sees it."""
    Q, K, V = _inputs(q_len, kv_len, 8, 2, 128, 6)
    clean = _run(cuda, Q, K, V, kv_len - q_len, True)
    Q[1, 2, 7] = np.nan
    K[kv_len - 1, 1, 3] = np.nan  # the last position's key of the second KV head
    got = _run(cuda, Q, K, V, kv_len - q_len, True)
    want_nan = np.zeros(got.shape, bool)
    want_nan[1, 2] = want_nan[q_len - 1, 4:] = True
    assert np.array_equal(np.isnan(got), want_nan)
    assert np.array_equal(got[~want_nan].view(np.uint16), clean[~want_nan].view(np.uint16))


@pytest.mark.parametrize("off", [0, 1])
def test_cache_append_alignment(cuda, off):
    """The new rows reach the cache from 16-byte aligned and from 2-byte aligned sources alike."""
    import layer
    import torch
    import qmm
    pool = layer.DeviceKVCache(2, 64, 2, 64)  # noqa: F841  (the pool lives as long as the object)
    Q, K, V = _inputs(20, 20, 4, 2, 64, 11)
    src = [torch.zeros(K.size + 8, dtype=torch.float16, device=cuda) for _ in range(2)]
    for s, x in zip(src, (K, V)):
        s[off:off + x.size] = torch.from_numpy(x.reshape(-1)).to(cuda)
    q = torch.from_numpy(Q).to(cuda)
    out = torch.empty_like(q)
    qmm.check(qmm.lib().qmm_gqa_attention_cached(q.data_ptr(), src[0].data_ptr() + 2 * off, src[1].data_ptr() + 2 * off,
                                                 out.data_ptr(), 1, 20, 0, 4, 2, 64, 0.0, 1, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint16), _run(cuda, Q, K, V, 0, True).view(np.uint16))


def test_graphs_of_shorter_contexts_after_the_longest_call(cuda):
    """One eager call at the longest context is enough for captures at every shorter one: none of them
    allocates, and replays after further eager calls give the eager results."""
    import torch
    import qmm
    heads, kvh, d, longest = 32, 8, 128, 12000
    g = torch.Generator(device=cuda)
    g.manual_seed(3)
    q = torch.randn((1, heads * d), generator=g, device=cuda).half()
    k, v = (torch.randn((longest, kvh * d), generator=g, device=cuda).half() for _ in range(2))
    qmm.check(qmm.lib().qmm_release_workspace())
    stream = torch.cuda.Stream()

    def call(kv, out):
        qmm.check(qmm.lib().qmm_gqa_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), 1, kv, heads, kvh, d, kv - 1,
                                              0.0, 1, stream.cuda_stream))
    torch.cuda.synchronize()
    eager, replayed, graphs = {}, {}, {}
    with torch.cuda.stream(stream):
        for kv in (longest, 8192, 8193, 6000, 4097, 1000, 129):
            eager[kv] = torch.empty_like(q)
            call(kv, eager[kv])
            if kv == longest:
                stream.synchronize()
                free = torch.cuda.mem_get_info()[0]
    stream.synchronize()
    assert torch.cuda.mem_get_info()[0] == free
    for kv in (8192, 8193, 6000, 4097, 1000, 129):
        replayed[kv], graphs[kv] = torch.zeros_like(q), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graphs[kv], stream=stream):
            call(kv, replayed[kv])
    for _ in range(3):
        for kv, graph in graphs.items():
            replayed[kv].zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                graph.replay()
                call(longest, eager[longest])
            torch.cuda.synchronize()
            assert torch.equal(replayed[kv], eager[kv]), kv
