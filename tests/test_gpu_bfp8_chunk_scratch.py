"""Block-float-8 chunks of 64 features whose caller brings scratch for the copies alone, for the copies and the parts behind them, or one
byte less: copies are read where the pass is split all the same, or where the scratch does not hold the parts of the other form either.
Oracle and tolerance as in test_gpu_prefill.py."""

import pytest
import torch

import test_gpu_prefill as P
from oracle import bfp8_codec
from oracle import paged_ops as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    P.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("users,hq,hkv,start,lc,alone", [
    (4, 8, 2, 8700, 256, False),  # the parts of the other form fit into the room of the copies
    (4, 8, 2, 700, 256, True),    # they do not
    (1, 64, 8, 40, 250, True),    # neither form is split
])
def test_scratch(users, hq, hkv, start, lc, alone, monkeypatch):
    from tt_xla_amd import _native as N

    d, bs = 64, 64
    width = -(-(start + lc) // bs)
    g = torch.Generator().manual_seed(users + start)
    key, value, table = P._paged(g, users, width, hkv, bs, d, False)
    q = P._bf(g, users, hq, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    packed = [bfp8_codec.pack_cache(t) for t in (key, value)]
    args = [t.cuda() for t in (q, packed[0], packed[1], table, st)]
    copies = int(N.lib().ttpa_sdpa_prefill_workspace_bytes(users, hkv, d, bs, width, 1))
    full = int(N.lib().ttpa_sdpa_prefill_scratch_bytes(users, hq, hkv, lc, d, bs, width, 1))
    assert full >= copies
    first = bfp8_codec.unpack_cache(packed[0], bs).to(torch.bfloat16)[int(table[0, 0])].flatten().cuda()
    want = O.chunked_sdpa(q, *[bfp8_codec.unpack_cache(t, bs).to(torch.bfloat16) for t in packed], table, st, d**-0.5)
    call = N.call
    for room, copied in ((copies, alone), (full, True), (copies - 1, False)):
        scratch = torch.zeros(full, dtype=torch.uint8, device="cuda")
        with monkeypatch.context() as m:
            m.setattr(N, "call", lambda name, *a: call(name, *(a[:-3] + (scratch.data_ptr(), room, a[-1]) if name == "ttpa_sdpa_prefill_expanded" else a)))
            got = torch.ops.tt.chunked_scaled_dot_product_attention(*args, d**-0.5)
        P._check(f"scratch {room} of {full}: u{users} h{hq}x{hkv} start{start}", got.cpu(), want)
        # (the scratch starts with K's copy of block 0 of user 0, or with float accumulators)
        assert torch.equal(scratch[: first.numel() * 2].view(torch.bfloat16), first) == copied
        assert not scratch[room:].any()
