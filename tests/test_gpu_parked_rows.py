"""Parked rows (position -1) of a decode step: their tokens go to the last row of the table's last
block, the last user winning where several share it (the null block), whatever the number of users and
cache format; nothing else in the caches changes."""

import pytest
import torch

import __graft_entry__ as entry
from oracle import bfp8_codec as C
from oracle import paged_ops as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("users,parked,hq,hkv,d,bs,bfp8", [
    (1, 1, 8, 2, 128, 64, False), (6, 3, 8, 2, 64, 32, False), (12, 7, 32, 8, 128, 64, True), (5, 2, 16, 8, 256, 32, True),
    (300, 280, 8, 1, 128, 16, False), (300, 299, 8, 1, 64, 32, True),
])
def test_parked_rows(users, parked, hq, hkv, d, bs, bfp8):
    from tt_xla_amd import custom_ops as ops

    g = torch.Generator().manual_seed(users + parked + d)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    active = users - parked
    nb, w = active + 3, 1
    table = torch.zeros(users, w, dtype=torch.int32)
    table[:active, 0] = torch.arange(active) + 1
    pos = torch.full((users,), -1, dtype=torch.int32)
    pos[:active] = torch.randint(0, bs, (active,), generator=g)
    if parked > 1:  # one parked row with a block of its own
        table[active, 0] = nb - 1
    kc, vc, q, k, v = bf(nb, hkv, bs, d), bf(nb, hkv, bs, d), bf(1, users, hq, d), bf(1, users, hkv, d), bf(1, users, hkv, d)
    pack = ops.bfp8_pack_cache if bfp8 else (lambda t: t.clone())
    kd, vd = pack(kc.cuda()), pack(vc.cuda())
    out = torch.ops.tt.paged_update_kv_decode_(q.cuda(), kd, vd, k.cuda(), v.cuda(), table.cuda(), pos.cuda(), scale=d**-0.5)
    trip = C.roundtrip if bfp8 else (lambda t: t)
    for got, cache, new in ((kd, kc, k), (vd, vc, v)):
        for u in range(users):  # one after the other: which of several writes to a slot wins
            cache = O.paged_update_cache(cache, new[:, u : u + 1], pos[u : u + 1], table[u : u + 1])
        want = trip(cache)
        got = (ops.bfp8_unpack_cache(got) if bfp8 else got).cpu()
        assert torch.equal(got, want)
    assert torch.isnan(out[0, active:].float()).all() and torch.isfinite(out[0, :active].float()).all()
