"""The forms of the streaming prefill kernel (head size 128) at the sizes where they can go wrong:
one, two and four query heads of a KV head per workgroup (row blocks of one workgroup that end at
different keys, row blocks that do not exist), K / V of an odd number of 32-key blocks, sliding
windows whose lower edge falls on, before and behind a block boundary.  Oracle and tolerance as in
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


@pytest.mark.parametrize("b,hq,hkv,s,window", [
    (1, 1, 1, 32, 0), (2, 3, 3, 160, 0), (1, 5, 5, 288, 0),      # one head: 128 rows of it per workgroup
    (1, 2, 1, 32, 0), (2, 6, 3, 96, 0), (1, 4, 2, 352, 0),       # two heads: 64 rows
    (1, 4, 1, 32, 0), (2, 8, 2, 96, 0), (1, 4, 1, 416, 0),       # four heads: 32 rows, odd numbers of blocks
    (1, 2, 2, 416, 31), (1, 2, 2, 416, 32), (1, 2, 2, 416, 33), (1, 3, 3, 288, 1), (2, 2, 2, 160, 200),
    (1, 4, 2, 416, 64), (1, 6, 3, 224, 97), (1, 4, 1, 416, 65), (1, 8, 2, 288, 128),
])
def test_dense_forms(b, hq, hkv, s, window):
    g = torch.Generator().manual_seed(b + hq + s + window)
    q, k, v = P._bf(g, b, hq, s, 128), P._bf(g, b, hkv, s, 128), P._bf(g, b, hkv, s, 128)
    want = O.sdpa_windowed(q, k, v, sliding_window=window) if window else O.sdpa(q, k, v, None, True, None)
    got = torch.ops.tt.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), is_causal=True,
                                                    sliding_window_size=window or None)
    P._check(f"dense b{b} h{hq}x{hkv} s{s} window{window}", got.cpu(), want)


@pytest.mark.parametrize("hq,hkv,bs,start,lc", [
    (3, 3, 64, 64, 130), (2, 1, 64, 192, 33), (4, 2, 128, 128, 200), (1, 1, 64, 0, 32), (10, 2, 64, 37, 129),
])
def test_paged_forms(hq, hkv, bs, start, lc):
    g = torch.Generator().manual_seed(hq + bs + start)
    users, nbpu = 2, -(-(start + lc) // bs) + 1
    key, value, table = P._paged(g, users, nbpu, hkv, bs, 128, False)
    q = P._bf(g, users, hq, lc, 128)
    st = torch.tensor([start], dtype=torch.int32)
    want = O.chunked_sdpa(q, key, value, table, st, 128**-0.5)
    got = torch.ops.tt.chunked_scaled_dot_product_attention(
        q.cuda(), key.cuda(), value.cuda(), table.cuda(), st.cuda(), 128**-0.5)
    P._check(f"paged h{hq}x{hkv} bs{bs} start{start} len{lc}", got.cpu(), want)


@pytest.mark.parametrize("users,hq,hkv,bs,start,lc", [
    (2, 4, 1, 32, 0, 32), (2, 4, 1, 32, 160, 33), (1, 2, 1, 96, 96, 130), (1, 3, 3, 32, 224, 64), (2, 8, 2, 160, 320, 96),
    # split over the keys: an uneven last part, parts behind the causal limit of the first rows, one row block
    # only, a start inside a block, 64-token blocks, fewer parts than the table's width allows, several row
    # blocks per workgroup of which some do not exist
    (1, 4, 1, 32, 2048, 32), (1, 4, 1, 32, 1000, 96), (1, 8, 2, 32, 512, 300), (1, 4, 1, 64, 4096, 1), (1, 4, 1, 64, 1100, 200),
    (1, 2, 1, 32, 1536, 96), (2, 3, 3, 32, 700, 200), (1, 5, 5, 128, 1280, 129),
])
def test_blocks_of_32_and_parts(users, hq, hkv, bs, start, lc):
    g = torch.Generator().manual_seed(hq + bs + start + lc)
    for spare in (1, 40):  # columns behind the pass: the host sees the table, the device the keys
        nbpu = -(-(start + lc) // bs) + spare
        key, value, table = P._paged(g, users, nbpu, hkv, bs, 128, False)
        q = P._bf(g, users, hq, lc, 128)
        st = torch.tensor([start], dtype=torch.int32)
        want = O.chunked_sdpa(q, key, value, table, st, 128**-0.5)
        got = torch.ops.tt.chunked_scaled_dot_product_attention(
            q.cuda(), key.cuda(), value.cuda(), table.cuda(), st.cuda(), 128**-0.5)
        P._check(f"paged h{hq}x{hkv} bs{bs} start{start} len{lc} spare{spare}", got.cpu(), want)


@pytest.mark.parametrize("hq,hkv,s,window", [(16, 16, 512, 0), (16, 8, 512, 0), (16, 8, 768, 256), (16, 4, 768, 200)])
def test_as_close_to_64_bits_as_the_plain_loop(hq, hkv, s, window, monkeypatch):
    """What the probabilities are relative to decides how they round: with the maximum of 64 keys, the plain loop's
    tile, the error is the same: 0.997 - 1.001 times the plain loop's on these, where the maximum of 32 keys gave 1.007 -
    1.010.  The bound lies between the two."""
    g = torch.Generator().manual_seed(s + hkv + window)
    q, k, v = P._bf(g, 1, hq, s, 128).cuda(), P._bf(g, 1, hkv, s, 128).cuda(), P._bf(g, 1, hkv, s, 128).cuda()
    i, j = torch.arange(s, device="cuda")[:, None], torch.arange(s, device="cuda")[None]
    seen = (j <= i) & (j > i - window) if window else j <= i
    scores = q[0].double() @ k[0].double().repeat_interleave(hq // hkv, 0).transpose(1, 2) * 128**-0.5
    want = torch.softmax(scores.masked_fill(~seen, float("-inf")), -1) @ v[0].double().repeat_interleave(hq // hkv, 0)
    err = []
    for loop in ("0", "1"):
        monkeypatch.setenv("TTPA_PREFILL_STREAM", loop)
        got = torch.ops.tt.scaled_dot_product_attention(q, k, v, is_causal=True, sliding_window_size=window or None)
        err.append(((got[0].double() - want).norm() / want.norm()).item())
    print(f"h{hq}x{hkv} s{s} window{window}: plain {err[0]:.4e} stream {err[1]:.4e} ratio {err[1] / err[0]:.4f}", flush=True)
    assert err[1] < 1.002 * err[0]


@pytest.mark.parametrize("hq,hkv,bs,bfp8", [(3, 3, 32, False), (4, 2, 64, False), (8, 2, 32, False), (8, 2, 64, False), (8, 2, 64, True)])
@pytest.mark.parametrize("start,lc", [(-40, 96), (-1000, 96), (-32, 32), (-2000000000, 33), (2000000000, 33)])
@pytest.mark.parametrize("slots", [None, "1"])  # a workgroup per row block; one that walks them all, the blind ones last
def test_chunk_that_starts_outside_the_sequence(hq, hkv, bs, bfp8, start, lc, slots, monkeypatch):
    """Row i sees keys up to start + i: none is NaN (softmax over nothing), as in the plain loop.  The start is in
    device memory, so no check of the host's sees it; a block count of zero or less would never count down to zero."""
    if slots:
        monkeypatch.setenv("TTPA_PREFILL_WGS_PER_GROUP", slots)
    g = torch.Generator().manual_seed(hq + bs + lc)
    users, nbpu = 2, 20
    key, value, table = P._paged(g, users, nbpu, hkv, bs, 128, False)
    q = P._bf(g, users, hq, lc, 128)
    k, v = key.cuda(), value.cuda()
    if bfp8:
        from tt_xla_amd import custom_ops as ops
        k, v = ops.bfp8_pack_cache(k), ops.bfp8_pack_cache(v)
        key, value = ops.bfp8_unpack_cache(k).cpu(), ops.bfp8_unpack_cache(v).cpu()
    got = torch.ops.tt.chunked_scaled_dot_product_attention(
        q.cuda(), k, v, table.cuda(), torch.tensor([start], dtype=torch.int32).cuda(), 128**-0.5).cpu()
    if start > 0:  # every row sees the whole table
        want = O.chunked_sdpa(q, key, value, table, torch.tensor([nbpu * bs], dtype=torch.int32), 128**-0.5)
        P._check(f"h{hq}x{hkv} bs{bs} start{start}", got, want)
        return
    blind = min(lc, -start)
    assert got[:, :, :blind].isnan().all()
    if blind < lc:  # the other rows are a chunk that starts at 0
        want = O.chunked_sdpa(q[:, :, blind:].contiguous(), key, value, table, torch.tensor([0], dtype=torch.int32), 128**-0.5)
        P._check(f"h{hq}x{hkv} bs{bs} start{start}", got[:, :, blind:].contiguous(), want)


@pytest.mark.parametrize("users,hq,hkv,nbpu,start,lc", [(1, 32, 8, 17, 960, 128), (1, 64, 8, 17, 900, 96), (1, 16, 4, 9, 330, 200)])
@pytest.mark.parametrize("slots", ["2", "3"])
def test_several_row_blocks_per_workgroup_are_not_split(users, hq, hkv, nbpu, start, lc, slots, monkeypatch):
    """TTPA_PREFILL_WGS_PER_GROUP has a workgroup walk its row blocks over all of their keys, also where the launch would
    otherwise split the keys: every row comes out of the same operations as with a workgroup per row block and no
    scratch to split with, bit for bit.  (Parts merged in float round differently.)"""
    from tt_xla_amd import custom_ops as ops

    g = torch.Generator().manual_seed(hq + start)
    key, value, table = P._paged(g, users, nbpu, hkv, 64, 128, False)
    args = [t.cuda() for t in (P._bf(g, users, hq, lc, 128), key, value, table, torch.tensor([start], dtype=torch.int32))]
    split = torch.ops.tt.chunked_scaled_dot_product_attention(*args, 128**-0.5)
    monkeypatch.setattr(ops, "_EXPANSION_LIMIT", 0)
    whole = torch.ops.tt.chunked_scaled_dot_product_attention(*args, 128**-0.5)
    monkeypatch.undo()
    monkeypatch.setenv("TTPA_PREFILL_WGS_PER_GROUP", slots)
    walked = torch.ops.tt.chunked_scaled_dot_product_attention(*args, 128**-0.5)
    assert not torch.equal(split, whole)  # (what the next line would not tell from a split)
    assert torch.equal(walked, whole)


@pytest.mark.parametrize("bs,bfp8", [(32, False), (64, False), (32, True)])
def test_parts_on_another_stream_and_replayed(bs, bfp8):
    """A chunk that is split over the keys: its partial results are scratch of the stream's, or of the graph's own."""
    from tt_xla_amd import custom_ops as ops

    g = torch.Generator().manual_seed(bs)
    key, value, table = P._paged(g, 1, 2048 // bs, 2, bs, 128, False)
    kv = [ops.bfp8_pack_cache(t.cuda()) if bfp8 else t.cuda() for t in (key, value)]
    args = (P._bf(g, 1, 8, 96, 128).cuda(), *kv, table.cuda(), torch.tensor([1500], dtype=torch.int32, device="cuda"))
    other = (P._bf(g, 1, 8, 160, 128).cuda(),) + args[1:]
    run = lambda a=args: torch.ops.tt.chunked_scaled_dot_product_attention(*a, 128**-0.5)  # noqa: E731
    want = run()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = run()
    run(other)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for _ in range(4):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        run(other)
        torch.cuda.synchronize()


@pytest.mark.parametrize("users,hq,hkv,lc,blocks", [
    # 32-key blocks from which on the last row block is split: 16, or 7 / 16 of the workgroups of the launch, or (above half of
    # the 256 CUs) half of them
    (1, 8, 2, 32, 16), (2, 2, 2, 40, 16), (1, 4, 2, 64, 16), (4, 32, 8, 64, 28), (1, 64, 8, 256, 56), (1, 64, 8, 288, 72),
    (1, 64, 8, 512, 128),
])
@pytest.mark.parametrize("bs", [32, 64])
def test_where_the_split_begins(users, hq, hkv, lc, blocks, bs, monkeypatch):
    """Under a page table far wider than the pass, one block in front of the line every row comes out of the same
    operations as without scratch to split with, bit for bit; on the line not, but within the roundings of the parts."""
    from tt_xla_amd import custom_ops as ops

    g = torch.Generator().manual_seed(hq + lc + bs)
    width = 32 * blocks // bs + 200
    key, value, _ = P._paged(g, 1, 64, hkv, bs, 128, False)
    table = torch.randint(0, 65, (users, width), generator=g).to(torch.int32).cuda()
    q, key, value = P._bf(g, users, hq, lc, 128).cuda(), key.cuda(), value.cuda()
    for n in (blocks - 1, blocks):
        start = torch.tensor([32 * n - lc], dtype=torch.int32, device="cuda")
        args = (q, key, value, table, start, 128**-0.5)
        got = torch.ops.tt.chunked_scaled_dot_product_attention(*args)
        with monkeypatch.context() as m:
            m.setattr(ops, "_EXPANSION_LIMIT", 0)
            whole = torch.ops.tt.chunked_scaled_dot_product_attention(*args)
        assert torch.equal(got, whole) == (n < blocks)
        torch.testing.assert_close(got.float(), whole.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("hq,hkv,bs", [(2, 2, 32), (4, 1, 64)])
@pytest.mark.parametrize("users,lc,width,start", [(1, 32, 8, 90), (3, 128, 40, 1000), (1, 100, 300, 64), (2, 200, 12, 150)])
def test_block_float_8_chunks(hq, hkv, bs, users, lc, width, start):
    """Through bfloat16 copies (walked by a fixed number of workgroups, only the columns that the pass reads) or tile by
    tile, whichever the pass takes: the attention over the values that the cache holds."""
    from tt_xla_amd import custom_ops as ops

    if start + lc > width * bs:
        width = -(-(start + lc) // bs)
    g = torch.Generator().manual_seed(lc + width)
    key, value = (ops.bfp8_pack_cache(P._bf(g, 60, hkv, bs, 128).cuda()) for _ in range(2))
    table = torch.randint(-1, 61, (users, width), generator=g).to(torch.int32)  # (ids outside the cache read block 0)
    q, st = P._bf(g, users, hq, lc, 128), torch.tensor([start], dtype=torch.int32)
    want = O.chunked_sdpa(q, ops.bfp8_unpack_cache(key).cpu(), ops.bfp8_unpack_cache(value).cpu(),
                          torch.where((table < 0) | (table >= 60), 0, table), st, 128**-0.5)
    got = torch.ops.tt.chunked_scaled_dot_product_attention(q.cuda(), key, value, table.cuda(), st.cuda(), 128**-0.5)
    P._check(f"bfp8 h{hq}x{hkv} bs{bs} u{users} len{lc} width{width}", got.cpu(), want)


@pytest.mark.parametrize("native", [False, True])
def test_a_pass_without_room_for_scratch_runs(native):
    """The scratch is sized by the page table, which is as wide as the longest sequence may be; memory is what the
    caches leave.  A pass that cannot have it runs without."""
    from tt_xla_amd import TTAttentionBackendImpl, TTMetadata
    from tt_xla_amd import custom_ops as ops

    g = torch.Generator().manual_seed(3)
    users, rows, start, bs, width = 2, 64, 96, 32, 4096
    kc, vc = (ops.bfp8_pack_cache(P._bf(g, 12, 2, bs, 128).cuda()) for _ in range(2))
    table = torch.zeros(users, width, dtype=torch.int32)
    table[:, :5] = torch.arange(10).view(2, 5) + 1
    q, k, v = (P._bf(g, users * rows, n * 128).cuda() for n in (2, 2, 2))
    md = TTMetadata(page_table=table.cuda(), fill_page_table=torch.roll(table, -3, 1).cuda(), num_users=users,
                    batch_idx=torch.arange(users, dtype=torch.int32).cuda(), chunk_start_idx=torch.tensor([start], dtype=torch.int32).cuda())
    impl = TTAttentionBackendImpl(2, 128, 128**-0.5, 2, None, None, "auto")
    if not native:
        impl._native_pass = lambda *a: False
    outs = []
    for room in (True, False):
        out = torch.zeros_like(q)
        ops._WORKSPACES.clear()
        torch.cuda.empty_cache()
        if not room:  # 64 MiB where the copies of 2 x 4096 blocks would be 268
            total = torch.cuda.get_device_properties(0).total_memory
            torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
        try:
            impl.forward(None, q, k, v, [kc, vc], md, output=out)
            torch.cuda.synchronize()
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        outs.append(out)
    torch.testing.assert_close(outs[1].float(), outs[0].float(), atol=1e-2, rtol=1e-2)
