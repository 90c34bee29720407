"""The scratch of a split attention call grows with the context and with the rows of the call, never the other way.

A caller that runs its largest call first (to have the buffer in place before it captures a graph) must not
meet a smaller call that needs more.  Host arithmetic only: the library's own function, by its C++ symbol.
"""

import ctypes

import pytest

import qmm

_bytes = getattr(qmm.lib(), "_ZN3qmm25attention_workspace_bytesEPKvS1_S1_iiiiiibb")
_bytes.restype = ctypes.c_size_t
_bytes.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_int] * 6 + [ctypes.c_bool] * 2


def need(q, kv, heads, kvh, d, causal=True, may_split=True):
    return _bytes(1024, 2048, 4096, q, kv, heads, kvh, d, kv - q if causal else 0, causal, may_split)


@pytest.mark.parametrize("heads,kvh,d", [(32, 8, 128), (64, 8, 128), (8, 8, 64), (24, 8, 128), (32, 1, 64), (28, 4, 128)])
@pytest.mark.parametrize("causal", [True, False])
def test_grows_with_context_and_rows(heads, kvh, d, causal):
    rows = [1, 2, 4, 5, 8, 15, 16, 17, 40, 100, 200, 513, 1023]
    before = dict.fromkeys(rows, 0)
    for kv in sorted([*range(1, 700, 31), *range(1024, 20000, 487), 8191, 8192, 8193]):
        last = 0
        for q in rows:
            if q > kv:
                continue
            n = need(q, kv, heads, kvh, d, causal)
            assert n >= before[q], (q, kv)
            assert n >= last, (q, kv)
            before[q] = last = n


def test_never_more_than_the_unbounded_partials():
    """At most one partial result per row and 64 keys, and none for a call that may not be split."""
    for q, kv in [(1, 12000), (15, 4000), (16, 129), (40, 12040), (1023, 1023), (4000, 16000)]:
        for heads, kvh, d in [(32, 8, 128), (24, 8, 128), (4, 4, 64)]:
            assert need(q, kv, heads, kvh, d) <= q * heads * -(-kv // 64) * (d + 2) * 4
            assert need(q, kv, heads, kvh, d, may_split=False) == 0
