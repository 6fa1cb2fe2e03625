"""Chunks whose KV heads have three, five, six or seven query heads, with a head group's workgroups on one XCD or spread over all, and with
a workgroup per head where a chunk has one row block: around the lines of test_prefill_places.py, row blocks and parts that do not come
out even, eager and captured.  Oracle and tolerance as in test_gpu_prefill.py."""

import pytest
import torch

import test_gpu_prefill as P
from oracle import paged_ops as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    P.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("users,hq,hkv,d,bs,start,lc", [
    # spread over the XCDs, and just not (fewer workgroups, more keys)
    (1, 20, 4, 128, 64, 1216, 256), (1, 40, 8, 128, 32, 1600, 90), (2, 40, 8, 128, 64, 832, 96), (1, 12, 4, 256, 64, 1216, 250), (1, 28, 4, 128, 64, 1203, 225),
    (1, 20, 4, 128, 64, 448, 256), (1, 20, 4, 256, 64, 3500, 100),
    # one row block: a workgroup per head (per two heads), pairs
    (1, 40, 8, 128, 64, 512, 32), (2, 20, 4, 128, 32, 520, 31), (1, 10, 2, 64, 32, 600, 17), (1, 12, 4, 256, 64, 512, 32), (1, 12, 2, 128, 64, 520, 32),
    (1, 20, 4, 128, 64, 2432, 32), (3, 10, 2, 128, 32, 100, 32),
])
def test_chunks(users, hq, hkv, d, bs, start, lc):
    g = torch.Generator().manual_seed(hq + bs + start + d)
    key, value, table = P._paged(g, users, -(-(start + lc) // bs), hkv, bs, d, False)
    q = P._bf(g, users, hq, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    want = O.chunked_sdpa(q, key, value, table, st, d**-0.5)
    args = [t.cuda() for t in (q, key, value, table, st)]
    got = torch.ops.tt.chunked_scaled_dot_product_attention(*args, d**-0.5)
    P._check(f"places u{users} h{hq}x{hkv} d{d} bs{bs} start{start} len{lc}", got.cpu(), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = torch.ops.tt.chunked_scaled_dot_product_attention(*args, d**-0.5)
    for _ in range(2):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, got)
