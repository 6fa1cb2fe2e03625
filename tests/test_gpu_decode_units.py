"""Decode where the leading unit per segment depends on the length of the tile list (ranges of the 16x16 matrix kernel): lists
that just fill the ranges and just do not, users without tokens, 64 and 65 users, a window; against the oracle's tolerance,
and against the same step with the unit forced on, which cuts the list elsewhere where there is none (other ranges
round to other bits) and nowhere else."""

import pytest
import torch

import test_gpu_decode as D
from oracle import paged_ops as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    D.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


# the list fills the 768 ranges of 256 CUs (3 per CU), or has a tile per segment more
@pytest.mark.parametrize("hq,hkv,d,bs,pos,window,unit", [
    (32, 8, 128, 64, [3071], 0, False), (32, 8, 128, 64, [3072], 0, True), (8, 2, 64, 32, [233, -1, 1960, 0], 0, False),
    (8, 4, 64, 64, [6143, 6143], 0, False), (8, 4, 64, 64, [6143, 6144], 0, True), (16, 8, 256, 32, [3071], 0, False),
    (16, 8, 256, 32, [3072], 0, True), (8, 2, 128, 64, [20 + 7 * i for i in range(64)], 0, True),
    (8, 2, 128, 64, [20 + 3 * i for i in range(64)], 0, False), (8, 2, 128, 64, [20 + 3 * i for i in range(65)], 0, True),
    (32, 8, 128, 64, [5119, -1, 2047, 3999], 1024, False), (32, 8, 128, 64, [5119, -1, 2047, 4000], 1024, True),
])
def test_unit_follows_the_list(hq, hkv, d, bs, pos, window, unit, monkeypatch):
    gen = torch.Generator().manual_seed(hq + d + len(pos) + max(pos))
    users, width = len(pos), max(pos) // bs + 1
    tile = {64: 64, 128: 32, 256: 32}[d]
    ranges = 3 * torch.cuda.get_device_properties(0).multi_processor_count // 4 * 4
    tiles = hkv * sum(p // tile - max(0, p + 1 - (window or p + 1)) // tile + 1 for p in pos if p >= 0)
    if ranges == 768:
        assert (tiles > ranges or users > 64) == unit
    k = torch.randn(width * 2, hkv, bs, d, generator=gen).to(torch.bfloat16)
    v = torch.randn(width * 2, hkv, bs, d, generator=gen).to(torch.bfloat16)
    table = torch.randint(0, width * 2, (users, width), generator=gen).to(torch.int32)
    q = torch.randn(1, users, hq, d, generator=gen).to(torch.bfloat16)
    cur = torch.tensor(pos, dtype=torch.int32)
    print(f"units h{hq}x{hkv} d{d} users{users} longest{max(pos)} window{window}", flush=True)
    monkeypatch.setenv("TTPA_DECODE_KERNEL", "ranges")  # (narrow tables and windows take whole segments)

    def step():
        return torch.ops.tt.paged_scaled_dot_product_attention_decode(
            q.cuda(), k.cuda(), v.cuda(), table.cuda(), is_causal=True, cur_pos_tensor=cur.cuda(), scale=d**-0.5,
            sliding_window_size=window or None).cpu()

    got = step()
    monkeypatch.setenv("TTPA_DECODE_SEG_UNITS", "1")
    forced = step()
    live = [u for u, p in enumerate(pos) if p >= 0]
    assert got[:, [u for u in range(users) if u not in live]].isnan().all()
    if ranges == 768:
        assert torch.equal(got[:, live], forced[:, live]) == unit
    want = O.paged_sdpa_decode_windowed(q[:, live], k, v, table[live], cur[live], d**-0.5, window, None)
    for t in (got, forced):
        torch.testing.assert_close(t[:, live].float(), want.reshape(t[:, live].shape).float(), atol=2e-2, rtol=2e-2)
