"""GPU tests of how the 16x16 matrix kernel cuts a block-float-8 decode (csrc/decode.hip): long tiles and one workgroup per CU for
wide groups, for the others one or two by the length of the list.  A grid is told by its bits: the same list cut into the same ranges gives the same output, and into others
another one (partials are rounded against other maxima)."""

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


def _inputs(users, hq, hkv, d, bs, pos, width):
    from tt_xla_amd import custom_ops as ops

    gen = torch.Generator().manual_seed(users + hq + d + width)
    blocks = 64 * 64 // bs
    k, v = (ops.bfp8_pack_cache(torch.randn(blocks, hkv, bs, d, generator=gen).to(torch.bfloat16).cuda()) for _ in range(2))
    table = torch.randint(0, blocks, (users, width), generator=gen, dtype=torch.int32).cuda()
    q = torch.randn(1, users, hq, d, generator=gen).to(torch.bfloat16).cuda()
    return q, k, v, table, torch.tensor(pos, dtype=torch.int32).cuda()


def _attend(q, k, v, table, cur, window=0, sink=None):
    return torch.ops.tt.paged_scaled_dot_product_attention_decode(
        q, k, v, table, is_causal=True, cur_pos_tensor=cur, scale=q.shape[-1] ** -0.5, sliding_window_size=window or None, attention_sink=sink)


@pytest.mark.parametrize("hq,hkv,bs,pos,window,with_sink", [
    (72, 8, 64, [0, 63, 64, 65, 127, 128, -1, 1000], 0, False),  # borders of 64-token tiles, one block each
    (64, 4, 32, [0, 31, 32, 95, 96, 2047], 0, True),            # sixteen heads, tiles of two blocks
    (60, 4, 16, [15, 16, 63, 64, 500], 0, False),               # fifteen heads, tiles of four blocks
    (128, 8, 128, [127, 128, 900, 1500], 200, True),            # a window: tiles cut at both ends
])
def test_long_tiles_of_wide_groups(monkeypatch, hq, hkv, bs, pos, window, with_sink):
    monkeypatch.setenv("TTPA_DECODE_KERNEL", "ranges")
    q, k, v, table, cur = _inputs(len(pos), hq, hkv, 128, bs, pos, max(pos) // bs + 1)
    sink = (torch.randn(hq, generator=torch.Generator().manual_seed(1)) * 2).to(torch.bfloat16) if with_sink else None
    print(f"long tiles h{hq}x{hkv} bs{bs} window{window}", flush=True)
    live = [u for u, p in enumerate(pos) if p >= 0]
    k_ref, v_ref = (C.unpack_cache(t.cpu(), bs).to(torch.bfloat16) for t in (k, v))
    want = O.paged_sdpa_decode_windowed(q[:, live].cpu(), k_ref, v_ref, table[live].cpu(), cur[live].cpu(), 128**-0.5, window, sink)
    for waves in (None, "0.05"):  # ... and with several segments and tiles per wavefront
        if waves:
            monkeypatch.setenv("TTPA_DECODE_WAVES_PER_CU", waves)
        got = _attend(q, k, v, table, cur, window, None if sink is None else sink.cuda()).cpu()
        assert got[:, [u for u in range(len(pos)) if u not in live]].isnan().all()
        torch.testing.assert_close(got[:, live].float(), want.reshape(got[:, live].shape).float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("users,hq,hkv", [(40, 64, 4), (10, 64, 8)])
def test_wide_groups_have_one_workgroup_per_cu(monkeypatch, users, hq, hkv):
    args = _inputs(users, hq, hkv, 128, 64, [8000 - 77 * u for u in range(users)], 128)
    got = _attend(*args)
    outs = {}
    for waves in ("4", "8"):
        monkeypatch.setenv("TTPA_DECODE_WAVES_PER_CU", waves)
        outs[waves] = _attend(*args)
    assert torch.equal(got, outs["4"]) and not torch.equal(got, outs["8"])


@pytest.mark.parametrize("users,hq,hkv,d,n_short,n_long", [
    (16, 32, 8, 128, 31, 32),  # 512 values per partial: from 4096 tiles of 32 tokens on
    (16, 40, 8, 128, 39, 40),  # 640: from 5120
    (4, 64, 8, 64, 127, 128),  # tiles of 64 tokens
    (8, 8, 8, 128, 43, 44),    # 128: from 2816
    (65, 8, 8, 128, 4, 5),     # above 64 users the list counts the leading units as well: 5 and 6 per segment, 2816 / 520 = 5.4
])
def test_short_lists_have_one_workgroup_per_cu(monkeypatch, users, hq, hkv, d, n_short, n_long):
    """Under one page table, by the tiles that there are: the border is where the grids change."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if cus != 256:
        pytest.skip("the cases are laid out for 256 CUs")
    tile, width = 4096 // d, 512
    for n, waves, other in ((n_short, "4", "8"), (n_long, "8", "4")):
        q, k, v, table, cur = _inputs(users, hq, hkv, d, 64, [n * tile - 1] * users, width)
        monkeypatch.delenv("TTPA_DECODE_WAVES_PER_CU", raising=False)
        got = _attend(q, k, v, table, cur)
        outs = {}
        for w in (waves, other):
            monkeypatch.setenv("TTPA_DECODE_WAVES_PER_CU", w)
            outs[w] = _attend(q, k, v, table, cur)
        assert torch.equal(got, outs[waves]) and not torch.equal(got, outs[other])
