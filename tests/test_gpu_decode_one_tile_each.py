"""Decode at head size 256 on either side of the lists that have a range for every tile (three and four wavefronts per CU: 768 and 1024 tiles on 256
CUs), of the group widths, of the number of segments and of users from which they do.  Outputs against the fp32 oracle, tolerance as in
test_gpu_decode_units.py; which ranges the list was cut into is told by the bits: the caller's grid of three per CU gives the same ones, unless
every tile had a range of its own where that grid has two of them share a maximum."""

import pytest
import torch

import __graft_entry__ as entry
from oracle import paged_ops as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("hq,hkv,bs,pos,window,each", [
    (16, 8, 32, [1535, 1535], 0, False), (16, 8, 32, [1535, 1536], 0, True), (16, 8, 64, [2047, 2047], 0, True), (16, 8, 32, [2047, 2048], 0, False),
    (8, 8, 32, [2047, 2047], 0, False), (16, 8, 16, [2047, -1, 0, 2000], 0, True), (16, 8, 8, [1800, 1700], 0, True),
    (24, 8, 32, [1800, 1800], 0, True), (32, 8, 32, [1800, 1800], 0, True), (40, 8, 32, [1800, 1800], 0, False),
    (4, 4, 32, [2600, 2600], 0, False), (6, 3, 32, [2500] * 4, 0, True), (16, 8, 32, [5119, 40, 3999, 2047], 1024, True),
    (16, 8, 32, [300 + 2 * i for i in range(11)], 0, True), (16, 8, 32, [40] * 64, 0, True), (16, 8, 32, [40] * 60 + [3] * 5, 0, False),
])
def test_one_tile_each(hq, hkv, bs, pos, window, each, monkeypatch):
    tiles = hkv * sum(p // 32 - max(0, p + 1 - (window or p + 1)) // 32 + 1 for p in pos if p >= 0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if cus == 256:
        assert each == (768 < tiles <= 1024 and 2 <= hq // hkv <= 4 and len(pos) * hkv >= 12 and len(pos) <= 64)
    gen = torch.Generator().manual_seed(hq + bs + len(pos) + max(pos))
    users, width, d = len(pos), max(pos) // bs + 1, 256
    k = torch.randn(width * 2, hkv, bs, d, generator=gen).to(torch.bfloat16)
    v = torch.randn(width * 2, hkv, bs, d, generator=gen).to(torch.bfloat16)
    table = torch.randint(0, width * 2, (users, width), generator=gen).to(torch.int32)
    q = torch.randn(1, users, hq, d, generator=gen).to(torch.bfloat16)
    cur = torch.tensor(pos, dtype=torch.int32)
    print(f"one tile each h{hq}x{hkv} bs{bs} users{users} longest{max(pos)} window{window}", flush=True)

    def step():
        return torch.ops.tt.paged_scaled_dot_product_attention_decode(
            q.cuda(), k.cuda(), v.cuda(), table.cuda(), is_causal=True, cur_pos_tensor=cur.cuda(), scale=d**-0.5,
            sliding_window_size=window or None).cpu()

    got = step()
    monkeypatch.setenv("TTPA_DECODE_WAVES_PER_CU", "3")
    three = step()
    live = [u for u, p in enumerate(pos) if p >= 0]
    if cus == 256:
        assert torch.equal(got[:, live], three[:, live]) != each
    assert got[:, [u for u in range(users) if u not in live]].isnan().all()
    want = O.paged_sdpa_decode_windowed(q[:, live], k, v, table[live], cur[live], d**-0.5, window, None)
    for t in (got, three):
        torch.testing.assert_close(t[:, live].float(), want.reshape(t[:, live].shape).float(), atol=2e-2, rtol=2e-2)
