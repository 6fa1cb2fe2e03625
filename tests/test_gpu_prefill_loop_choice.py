"""Chunks of few rows at head size 64 on either side of the line between the two prefill loops (one or two (row block, head) pairs in a
group; whether the launch is split, its keys, its groups, two workgroups to a CU).  Which loop ran is told by the bits: the plain loop's reference
moves for 64 keys at a time, the streaming one's for 32 and the 32 behind them, and every fourth block of 32 keys here has scores that
move it, so probabilities of the block in front are rounded relative to other references."""

import pytest
import torch

import test_gpu_prefill as P
from oracle import paged_ops as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    P.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("users,hq,hkv,start,lc,plain", [
    (1, 8, 8, 128, 32, False), (1, 8, 8, 384, 32, True), (1, 8, 8, 512, 64, True), (1, 8, 8, 384, 65, False),
    (6, 8, 8, 768, 64, True), (7, 8, 8, 768, 64, False), (5, 8, 8, 192, 64, False), (4, 16, 8, 512, 32, True), (1, 8, 8, 1408, 64, True), (1, 8, 8, 1536, 64, False),
    (4, 8, 8, 8192, 32, False), (5, 8, 8, 8192, 32, True), (5, 8, 8, 8192, 64, False), (1, 5, 1, 512, 32, True),
])
def test_which_loop(users, hq, hkv, start, lc, plain, monkeypatch):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are those of 256 CUs")
    d, bs = 64, 64
    g = torch.Generator().manual_seed(users + hq + start + lc)
    width = -(-(start + lc) // bs)
    key, value, table = P._paged(g, users, width, hkv, bs, d, False)
    q = P._bf(g, users, hq, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    moving = key.clone().view(-1, hkv, 2, 32, d)  # (pages hold two blocks: the odd pages' second)
    moving[table[:, 1::2].flatten().long(), :, 1] *= 4

    def run(k):
        return torch.ops.tt.chunked_scaled_dot_product_attention(q.cuda(), k.view_as(key).cuda(), value.cuda(), table.cuda(), st.cuda(), d**-0.5)

    P._check(f"u{users} h{hq}x{hkv} start{start} len{lc}", run(key).cpu(), O.chunked_sdpa(q, key, value, table, st, d**-0.5))
    got = run(moving)
    monkeypatch.setenv("TTPA_PREFILL_STREAM", "0")
    assert torch.equal(got, run(moving)) == plain
