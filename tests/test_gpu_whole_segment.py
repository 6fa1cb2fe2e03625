"""GPU tests of the decode step with one workgroup per (user, KV head) segment (direct_waves in csrc/decode.hip): no
ranges, no partials, no merge launch.  Caches bit for bit and outputs against the two operators in turn with the
segments cut into ranges (TTPA_DECODE_KERNEL=ranges), and against the fp32 oracle.  The two forms sum the same
products over other groups of tokens, so a weight is rounded to bfloat16 (2^-9 relative) against another maximum
and the output is rounded once (2^-9): 2^-7 of the largest value between them."""

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


CASES = [
    # Hq, Hkv, D, bs, contexts (position written = context), bfp8, window, sink, forced
    (32, 8, 128, 64, [0, 31, 32, 63, 127, 128, 400], False, 0, False, False),     # borders of 32-token tiles
    (8, 8, 64, 32, [0, 62, 63, 64, 300, 1023], False, 0, False, False),           # one head per group: weights in two parts
    (16, 16, 128, 16, [5, 15, 16, 500], False, 0, True, False),                   # tiles of two blocks
    (40, 8, 128, 32, [250, 3, 70], False, 64, True, False),                       # five heads: some threads store nothing
    (48, 3, 64, 64, [511, 100, 900], False, 300, True, False),                    # sixteen heads, three KV heads
    (4, 2, 128, 64, [255, 256, 257, 2000], False, 0, False, True),                # as many rounds of tiles as asked for
    (32, 8, 128, 64, [0, 31, 32, 700, 1022], True, 0, False, False),              # block-float-8
    (16, 2, 64, 32, [5, 64, 2000], True, 0, True, False),
    (6, 3, 128, 32, [40, 333, 1990], True, 500, False, False),
    (32, 8, 128, 64, [(37 * i) % 250 for i in range(40)], False, 0, False, False),  # more segments than CUs: four wavefronts
    (16, 16, 64, 32, [(53 * i) % 900 for i in range(20)], True, 0, True, False),
]


@pytest.mark.parametrize("hq,hkv,d,bs,ctx,bfp8,window,with_sink,forced", CASES)
def test_whole_segments_equal_ranges(monkeypatch, hq, hkv, d, bs, ctx, bfp8, window, with_sink, forced):
    from tt_xla_amd import custom_ops as ops
    from tt_xla_amd import workloads

    users = len(ctx)
    print(f"whole segments b{users} h{hq}x{hkv} d{d} bs{bs} bfp8={bfp8} window{window}", flush=True)
    nb = sum((c + bs) // bs for c in ctx) + 3
    wl = workloads.decode_ragged("whole", hq + d + bs + users, users, hq, hkv, d, bs, nb, ctx)
    if bfp8:
        workloads.add_outlier_channels(wl, 3, fraction=0.02)
    sink = (torch.randn(hq, generator=torch.Generator().manual_seed(1)) * 2).to(torch.bfloat16) if with_sink else None
    dev = wl.to("cuda")
    pack = ops.bfp8_pack_cache if bfp8 else torch.clone
    results = {}
    for kernel in ("ranges", "direct" if forced else ""):
        monkeypatch.setenv("TTPA_DECODE_KERNEL", kernel) if kernel else monkeypatch.delenv("TTPA_DECODE_KERNEL")
        k, v = pack(dev.k_cache), pack(dev.v_cache)
        kw = dict(scale=wl.scale, sliding_window_size=window or None, attention_sink=None if sink is None else sink.cuda())
        if kernel == "ranges":
            ops.paged_update_kv_cache_(k, v, dev.k_new, dev.v_new, dev.cache_position, dev.page_table)
            out = torch.ops.tt.paged_scaled_dot_product_attention_decode(
                dev.q, k, v, dev.page_table, is_causal=True, cur_pos_tensor=dev.cache_position, **kw)
        else:
            out = torch.ops.tt.paged_update_kv_decode_(dev.q, k, v, dev.k_new, dev.v_new, dev.page_table, dev.cache_position, **kw)
        torch.cuda.synchronize()
        results[kernel == "ranges"] = (out, k, v)
    (want, k0, v0), (got, k1, v1) = results[True], results[False]
    assert torch.equal(k0.view(torch.uint8), k1.view(torch.uint8)) and torch.equal(v0.view(torch.uint8), v1.view(torch.uint8))
    assert (got.float() - want.float()).abs().max() <= 2**-7 * want.float().abs().max()
    if bfp8:
        k1, v1 = (C.unpack_cache(t.cpu(), bs).to(torch.bfloat16) for t in (k1, v1))
    ref = O.paged_sdpa_decode_windowed(wl.q, k1.cpu(), v1.cpu(), wl.page_table, wl.cache_position, wl.scale, window, sink)
    torch.testing.assert_close(got.cpu().float(), ref, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("d,bfp8", [(64, False), (128, False), (128, True)])
def test_whole_segments_with_rows_of_odd_strides_and_parked_users(d, bfp8):
    """Output rows that start on 2-byte borders (stores of single elements), int64 positions, and parked users that share
    one slot of the null block: NaN rows, the last one's token stays; replayed, with eager work in between."""
    from tt_xla_amd import custom_ops as ops
    from tt_xla_amd import workloads

    users, hq, hkv, bs = 6, 8, 2, 32
    wl = workloads.decode_ragged("whole-parked", 5, users, hq, hkv, d, bs, 40, [40, 0, 100, 0, 95, 0])
    for u in (1, 3, 5):
        wl.cache_position[u] = -1
        wl.page_table[u] = 0
    dev = wl.to("cuda")
    dev.cache_position = dev.cache_position.long()
    pack = ops.bfp8_pack_cache if bfp8 else torch.clone
    k, v = pack(dev.k_cache), pack(dev.v_cache)
    wide = torch.full((users, hq, d + 5), 7.0, dtype=torch.bfloat16, device="cuda")
    from tt_xla_amd import _native as N

    def step(out, us, hs):
        ws = torch.empty(N.lib().ttpa_paged_decode_workspace_bytes(users, hq, hkv, d), dtype=torch.uint8, device="cuda")
        N.call(
            "ttpa_paged_update_decode", out.data_ptr(), us, hs, dev.q.data_ptr(), hq * d, d, k.data_ptr(), v.data_ptr(), dev.k_new.data_ptr(),
            dev.v_new.data_ptr(), dev.k_new.stride(1), dev.k_new.stride(2), dev.page_table.data_ptr(), dev.page_table.stride(0),
            dev.cache_position.data_ptr(), 1, users, hq, hkv, d, bs, dev.page_table.shape[1], k.shape[0], float(wl.scale), int(bfp8), 0,
            None, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
        return ws

    plain = torch.empty(users, hq, d, dtype=torch.bfloat16, device="cuda")
    keep = step(plain, hq * d, d)
    keep2 = step(wide, hq * (d + 5), d + 5)
    torch.cuda.synchronize()
    assert torch.isnan(plain[[1, 3, 5]]).all() and torch.isfinite(plain[[0, 2, 4]]).all()
    assert torch.equal(wide[..., :d].nan_to_num(9.0), plain.nan_to_num(9.0)) and (wide[..., d:] == 7).all()
    written = (C.unpack_cache(k.cpu(), bs) if bfp8 else k.cpu().float())[0, :, bs - 1]
    want = wl.k_new[0, 5, :hkv].float()
    if bfp8:
        want = C.unpack_cache(ops.bfp8_pack_cache(dev.k_new[0, 5, :hkv].reshape(1, hkv, 1, d).expand(1, hkv, bs, d).contiguous()).cpu(), bs)[0, :, 0]
    assert torch.equal(written.float(), want.float())
    eager, graph = plain.clone(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        keep3 = step(plain, hq * d, d)
    for _ in range(4):
        plain.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(plain.nan_to_num(9.0), eager.nan_to_num(9.0))
        (dev.q.float() @ dev.q.float().transpose(-1, -2)).sum().item()
    del keep, keep2, keep3


@pytest.mark.parametrize("hq,hkv,d,window", [(16, 8, 64, 0), (12, 4, 64, 256), (16, 8, 128, 0), (24, 8, 128, 256)])
def test_attention_alone_over_two_or_three_heads_stays_with_the_dot_product_kernel(monkeypatch, hq, hkv, d, window):
    """Whatever the page table's width or the window: its weights are rounded against the maxima of sixteen tokens, so it is
    closer to 64 bits than a whole segment (tests of closeness would need a margin; the same kernel gives the same bits)."""
    gen = torch.Generator().manual_seed(hq + d)
    users, bs = 5, 32
    width = 272 * 1024 // (4 * d * bs)
    k = torch.randn(users * width, hkv, bs, d, generator=gen).to(torch.bfloat16).cuda()
    v = torch.randn(users * width, hkv, bs, d, generator=gen).to(torch.bfloat16).cuda()
    table = torch.arange(users * width, dtype=torch.int32).reshape(users, width).cuda()
    q = torch.randn(1, users, hq, d, generator=gen).to(torch.bfloat16).cuda()
    cur = torch.tensor([0, 63, 127, 300, width * bs - 1], dtype=torch.int32).cuda()
    got = []
    for kernel in (None, "valu"):
        monkeypatch.setenv("TTPA_DECODE_KERNEL", kernel) if kernel else monkeypatch.delenv("TTPA_DECODE_KERNEL", raising=False)
        got.append(torch.ops.tt.paged_scaled_dot_product_attention_decode(
            q, k, v, table, is_causal=True, cur_pos_tensor=cur, scale=d**-0.5, sliding_window_size=window or None))
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("kernel", ["direct", "ranges"])
@pytest.mark.parametrize("hq,d", [(4, 64), (4, 128), (16, 128)])  # one head per group, where the weights have two parts; four
def test_infinite_values_stay_infinite(monkeypatch, kernel, hq, d):
    """An infinite V element makes its output infinite, of the same sign, whatever its weight is rounded to; two of
    opposite signs make NaN; one behind the context makes nothing.  (Not in a segment's last partial, which the merge of
    the ranges repeats with weight 0.)"""
    monkeypatch.setenv("TTPA_DECODE_KERNEL", kernel)
    gen = torch.Generator().manual_seed(hq + d)
    users, hkv, bs, width = 3, 4, 32, 12
    k = torch.randn(users * width, hkv, bs, d, generator=gen).to(torch.bfloat16)
    v = torch.randn(users * width, hkv, bs, d, generator=gen).to(torch.bfloat16)
    table = torch.arange(users * width, dtype=torch.int32).reshape(users, width)
    cur = torch.tensor([129, 200, width * bs - 2], dtype=torch.int32)
    inf = float("inf")
    for u in range(users):
        at = lambda t: (u * width + t // bs, slice(None), t % bs)  # noqa: E731
        for column, t in enumerate(range(0, 40, 3)):
            v[at(t)][..., column] = inf if column % 2 else -inf
        v[at(7)][..., 30], v[at(31)][..., 30] = inf, -inf
        v[at(int(cur[u]) + 1)][...] = inf
    q = torch.randn(1, users, hq, d, generator=gen).to(torch.bfloat16)
    k_new, v_new = (torch.randn(1, users, hkv, d, generator=gen).to(torch.bfloat16) for _ in range(2))
    if kernel == "direct":
        v_new[..., 40], v_new[..., 41] = inf, -inf
    dev = [t.cuda() for t in (q, k, v, k_new, v_new, table, cur)]
    got = torch.ops.tt.paged_update_kv_decode_(*dev, None, d**-0.5).cpu()
    alone = torch.ops.tt.paged_scaled_dot_product_attention_decode(
        dev[0], dev[1], dev[2], dev[5], is_causal=True, cur_pos_tensor=dev[6], scale=d**-0.5).cpu()
    want = O.textbook_decode_fp32(q, dev[1].cpu(), dev[2].cpu(), table, cur, d**-0.5)
    assert want.isinf().any() and want.isnan().any()
    for t in (got, alone):
        torch.testing.assert_close(t.float(), want.reshape(t.shape).float(), atol=2e-2, rtol=2e-2, equal_nan=True)
