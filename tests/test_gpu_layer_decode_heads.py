"""Decode steps of whole layers with head_dim 64 and 128: the matrix-core attention that rotates the query and the
new key itself and writes the cache row.

Against the CPU restatement (oracle/layer_oracle.py), 5e-3 absolute as in test_gpu_layer.py.  One new key among
many moves the output little, so its cache row is also read back: a query of 40 times the expected key makes
the softmax choose that row, and the output is its value.  A key in the other pair layout, unrotated, or at
another position scores far below.
"""

import numpy as np
import pytest

import gguf_oracle as O
import layer_oracle as L
from test_gpu_layer import host, make_layer, maxerr, stream, t16

pytestmark = pytest.mark.gpu


# positions: the first key of all, edges of the 32-key blocks and of the 128-key ranges, one range and several;
# groups of 1, 3, 8 query heads and of 24 (two row tiles)
@pytest.mark.parametrize("heads,kvh,d,neox", [(4, 4, 128, False), (8, 1, 128, True), (6, 2, 128, True), (24, 1, 128, False), (24, 1, 128, True),
                                              (4, 4, 64, True), (8, 1, 64, False), (24, 1, 64, True)])
def test_decode_rotates_attends_and_writes_the_cache(cuda, heads, kvh, d, neox):
    import torch
    import qmm
    r = np.random.default_rng(heads + kvh + d)
    hidden, inter, cap = 256, 512, 1100
    types = {"q": O.GGML_Q4_K, "k": O.GGML_Q4_K, "v": O.GGML_Q6_K, "o": O.GGML_Q8_0, "gate": O.GGML_Q4_K, "up": O.GGML_Q4_K, "down": O.GGML_Q6_K}
    packed, deq = make_layer(r, hidden, inter, heads, kvh, d, types)
    dev_w = {n: t16(raw, cuda) for n, (t, raw) in packed.items()}
    norms = {n: t16(deq[n], cuda) for n in ("attn_norm", "ffn_norm")}
    w = qmm.LayerWeights()
    w.attn_norm, w.attn_norm_dtype = norms["attn_norm"].data_ptr(), qmm.DTYPE_F16
    w.ffn_norm, w.ffn_norm_dtype = norms["ffn_norm"].data_ptr(), qmm.DTYPE_F16
    for f, n in (("wq", "q"), ("wk", "k"), ("wv", "v"), ("wo", "o"), ("wgate", "gate"), ("wup", "up"), ("wdown", "down")):
        setattr(w, f, dev_w[n].data_ptr())
        setattr(w, f + "_type", packed[n][0])
    c = qmm.LayerConfig()
    c.hidden_size, c.intermediate_size, c.num_heads, c.num_kv_heads, c.head_dim = hidden, inter, heads, kvh, d
    c.rms_norm_eps, c.rope_freq_base, c.rope_neox, c.scale = 1e-5, 10000.0, int(neox), 0.0
    cfg = {"num_heads": heads, "num_kv_heads": kvh, "head_dim": d, "rms_norm_eps": 1e-5, "rope_freq_base": 10000.0, "rope_neox": neox}
    past = [r.standard_normal((cap, kvh, d)).astype(np.float16) for _ in range(2)]
    lib = qmm.lib()
    qmm.check(lib.qmm_kv_cache_init(2, cap + 1, kvh, d))
    try:
        P = [t16(p, cuda) for p in past]
        q0 = torch.zeros((cap, heads * d), dtype=torch.float16, device=cuda)
        o0 = torch.empty_like(q0)
        for pos in (0, 1, 31, 32, 63, 127, 128, 300, 511, 1024):
            # the cache's rows before `pos`, and old rows behind it that must not be seen
            qmm.check(lib.qmm_gqa_attention_cached(q0.data_ptr(), P[0].data_ptr(), P[1].data_ptr(), o0.data_ptr(), 1, cap, 0, heads, kvh, d,
                                                   0.0, 1, stream()))
            kc, vc = (p.copy() for p in past)
            x = (r.standard_normal((2, hidden)) * 0.5).astype(np.float16)
            X = t16(x, cuda)
            Y = torch.empty_like(X)
            for i in range(2):  # the second step reads the row that the first one wrote
                want = L.layer_forward(x[i:i + 1], deq, cfg, kc, vc, pos + i)
                qmm.check(lib.qmm_forward_layer(c, w, X[i:].data_ptr(), Y[i:].data_ptr(), 1, 1, pos + i, stream()))
                assert maxerr(host(Y)[i:i + 1], want) < 5e-3, (pos, i)
            for row in (pos, pos + 1):
                probe = np.repeat(40 * kc[row].astype(np.float32), heads // kvh, axis=0).astype(np.float16)
                out = torch.empty((1, heads * d), dtype=torch.float16, device=cuda)
                new = torch.zeros((1, kvh * d), dtype=torch.float16, device=cuda)
                Q = t16(probe.reshape(1, -1), cuda)
                qmm.check(lib.qmm_gqa_attention_cached(Q.data_ptr(), new.data_ptr(), new.data_ptr(), out.data_ptr(), 1, 1, pos + 2, heads, kvh, d,
                                                       0.0, 1, stream()))
                got = host(out).reshape(heads, d)
                assert maxerr(got, np.repeat(vc[row], heads // kvh, axis=0)) < 5e-3, (pos, row)
    finally:
        qmm.check(lib.qmm_kv_cache_free())
