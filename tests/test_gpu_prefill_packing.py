"""Workgroups of the streaming prefill kernel as four (row block, head) pairs: numbers of heads per KV head that are no multiple of
two or four (pairs of a workgroup in one, two or four row blocks, pairs that do not exist), and numbers of head groups around the
eight XCDs that whole rounds are dealt to (one group, a round less one, a round, a round and some).  Oracle and tolerance as in
test_gpu_prefill.py."""

import pytest
import torch

import test_gpu_prefill as P
from oracle import paged_ops as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    P.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("b,hq,hkv,d,s,window", [
    (1, 3, 1, 128, 32, 0), (1, 3, 1, 128, 160, 0), (1, 5, 1, 128, 96, 0), (3, 15, 3, 64, 224, 0), (1, 7, 1, 64, 64, 0), (2, 12, 2, 128, 288, 0),
    (1, 9, 1, 256, 96, 0), (7, 1, 1, 128, 160, 0), (9, 4, 1, 64, 96, 0), (5, 4, 2, 128, 64, 0), (11, 2, 1, 64, 352, 0),
    (2, 10, 2, 128, 224, 40), (3, 3, 1, 64, 192, 100),
])
def test_dense(b, hq, hkv, d, s, window):
    g = torch.Generator().manual_seed(b + hq + s + window + d)
    q, k, v = P._bf(g, b, hq, s, d), P._bf(g, b, hkv, s, d), P._bf(g, b, hkv, s, d)
    want = O.sdpa_windowed(q, k, v, sliding_window=window) if window else O.sdpa(q, k, v, None, True, None)
    got = torch.ops.tt.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), is_causal=True, sliding_window_size=window or None)
    P._check(f"dense b{b} h{hq}x{hkv} d{d} s{s} window{window}", got.cpu(), want)


@pytest.mark.parametrize("stream", ["1", "0"])
@pytest.mark.parametrize("users,hq,hkv,d,bs,start,lc", [
    (1, 5, 1, 128, 64, 64, 32), (3, 10, 2, 128, 32, 96, 70), (1, 3, 1, 64, 64, 1100, 96), (1, 5, 1, 128, 32, 1000, 100), (2, 6, 1, 128, 64, 700, 33),
    (9, 2, 1, 64, 32, 160, 64), (1, 4, 1, 64, 64, 2048, 40),
])
def test_paged(users, hq, hkv, d, bs, start, lc, stream, monkeypatch):
    monkeypatch.setenv("TTPA_PREFILL_STREAM", stream)  # (the plain loop has the same places and the same merge)
    g = torch.Generator().manual_seed(hq + bs + start + d)
    key, value, table = P._paged(g, users, -(-(start + lc) // bs) + 1, hkv, bs, d, False)
    q = P._bf(g, users, hq, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    want = O.chunked_sdpa(q, key, value, table, st, d**-0.5)
    got = torch.ops.tt.chunked_scaled_dot_product_attention(q.cuda(), key.cuda(), value.cuda(), table.cuda(), st.cuda(), d**-0.5)
    P._check(f"paged h{hq}x{hkv} d{d} bs{bs} start{start} len{lc}", got.cpu(), want)
