"""Chunk passes of the compiler-scheduled prefill loop split over the keys (head sizes 64 and 256, cache blocks that the
streaming loop does not take, block-float-8 tiles): sizes where a split begins and ends, parts that lie behind the causal
limit of the first rows, wavefronts without rows, row blocks without keys.  Tolerance as in test_gpu_prefill.py: a bfloat16
output and bfloat16 probabilities, split or not."""

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


def _pass(q, key, value, table, start, scale):
    return torch.ops.tt.chunked_scaled_dot_product_attention(q, key, value, table, start, scale)


@pytest.mark.parametrize("users,hq,hkv,d,bs,start,lc", [
    # head size 64: blocks of whole tiles, of whole loads, smaller ones; no split, an uneven last part, a start inside a block
    (1, 8, 8, 64, 64, 1216, 224), (1, 8, 8, 64, 32, 320, 608), (2, 4, 1, 64, 64, 0, 40), (1, 8, 2, 64, 128, 4001, 33),
    (1, 2, 1, 64, 8, 700, 100), (1, 4, 1, 64, 4, 600, 50), (3, 6, 3, 64, 64, 1500, 70),
    (1, 4, 1, 64, 64, 511, 1), (1, 4, 1, 64, 64, 479, 1), (1, 4, 1, 64, 64, 512, 200),  # 16 key blocks, 15, parts behind early rows
    # head size 128 outside the streaming loop's blocks
    (1, 4, 1, 128, 16, 2048, 32), (1, 3, 3, 128, 48, 1000, 130), (2, 8, 2, 128, 2, 650, 60),
    # head size 256: one workgroup per CU
    (1, 16, 8, 256, 32, 832, 192), (1, 4, 1, 256, 64, 3000, 65), (2, 2, 2, 256, 16, 640, 20),
])
def test_split_chunks(users, hq, hkv, d, bs, start, lc):
    g = torch.Generator().manual_seed(hq + bs + start + d)
    nbpu = -(-(start + lc) // bs) + 1
    key, value, table = P._paged(g, users, nbpu, hkv, bs, d, False)
    q = P._bf(g, users, hq, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    want = O.chunked_sdpa(q, key, value, table, st, d**-0.5)
    got = _pass(q.cuda(), key.cuda(), value.cuda(), table.cuda(), st.cuda(), d**-0.5)
    P._check(f"split u{users} h{hq}x{hkv} d{d} bs{bs} start{start} len{lc}", got.cpu(), want)


@pytest.mark.parametrize("users,hq,hkv,d,bs,start,lc", [
    (1, 8, 8, 64, 32, 1300, 96), (2, 8, 2, 64, 64, 700, 33), (1, 64, 8, 128, 64, 2368, 32), (3, 4, 4, 128, 32, 900, 40),
    (1, 4, 1, 128, 16, 1100, 100),
])
def test_split_chunks_over_block_float_8(users, hq, hkv, d, bs, start, lc, monkeypatch):
    from tt_xla_amd import _native as N

    g = torch.Generator().manual_seed(hq + bs + start + d)
    nbpu = -(-(start + lc) // bs) + 1
    key, value, table = P._paged(g, users, nbpu, hkv, bs, d, False)
    q = P._bf(g, users, hq, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    packed = [bfp8_codec.pack_cache(t) for t in (key, value)]
    want = O.chunked_sdpa(q, *[bfp8_codec.unpack_cache(t, bs).to(torch.bfloat16) for t in packed], table, st, d**-0.5)
    args = [t.cuda() for t in (q, packed[0], packed[1], table, st)]
    got = _pass(*args, d**-0.5)
    P._check(f"split bfp8 u{users} h{hq}x{hkv} d{d} bs{bs} start{start} len{lc}", got.cpu(), want)
    call = N.call
    monkeypatch.setattr(N, "call", lambda name, *a: call(name, *(a[:-3] + (0, 0, a[-1]) if name == "ttpa_sdpa_prefill_expanded" else a)))
    unsplit = _pass(*args, d**-0.5)
    P._check("the same, unsplit", unsplit.cpu(), want)
    assert not torch.equal(got, unsplit), "the pass was not split"


@pytest.mark.parametrize("d,bs", [(64, 64), (64, 32), (128, 16), (256, 32)])
def test_split_closeness_and_replay(d, bs, monkeypatch):
    """Against 64 bits a split pass is as close as an unsplit one (the same probabilities, float accumulators; a quarter
    more allows for the other references of the parts), and a captured one gives the eager bits on every replay."""
    from tt_xla_amd import _native as N

    g = torch.Generator().manual_seed(d + bs)
    hq, hkv, start, lc = 4, 2, 1600, 96
    nbpu = -(-(start + lc) // bs)
    key, value, table = P._paged(g, 1, nbpu, hkv, bs, d, False)
    q = P._bf(g, 1, hq, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    k = key[table[0].long()].permute(1, 0, 2, 3).reshape(hkv, -1, d).double().repeat_interleave(hq // hkv, 0)
    v = value[table[0].long()].permute(1, 0, 2, 3).reshape(hkv, -1, d).double().repeat_interleave(hq // hkv, 0)
    s = q[0].double() @ k.transpose(1, 2) * d**-0.5
    s = s.masked_fill(torch.arange(k.shape[1])[None] > start + torch.arange(lc)[:, None], -torch.inf)
    want = (s.softmax(-1) @ v)[None]
    args = [t.cuda() for t in (q, key, value, table, st)]
    got = _pass(*args, d**-0.5)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        replayed = _pass(*args, d**-0.5)
    for _ in range(3):
        replayed.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(replayed, got)
    assert N.lib().ttpa_sdpa_prefill_scratch_bytes(1, hq, hkv, lc, d, bs, nbpu, 0) > 0
    call = N.call

    def without_scratch(name, *a):
        return call(name, *(a[:-3] + (0, 0, a[-1]) if name == "ttpa_sdpa_prefill_expanded" else a))

    monkeypatch.setattr(N, "call", without_scratch)
    unsplit = _pass(*args, d**-0.5)
    err = [((t.cpu().double() - want).norm() / want.norm()).item() for t in (got, unsplit)]
    print(f"d{d} bs{bs}: split {err[0]:.3e}, unsplit {err[1]:.3e}")
    assert not torch.equal(got, unsplit), "the pass was not split"
    assert err[0] <= 1.25 * err[1]


@pytest.mark.parametrize("d,bs", [(64, 32), (128, 16), (256, 64)])
@pytest.mark.parametrize("start", [-40, -1000, -2000000000, 2000000000])
def test_chunks_that_start_outside_the_sequence(d, bs, start):
    """Rows without a key come out as NaN, a start behind the table lets every row see all of it; as in the streaming loop."""
    g = torch.Generator().manual_seed(d)
    lc, nbpu = 96, 1280 // bs
    key, value, table = P._paged(g, 1, nbpu, 1, bs, d, False)
    q = P._bf(g, 1, 2, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    got = _pass(q.cuda(), key.cuda(), value.cuda(), table.cuda(), st.cuda(), d**-0.5).cpu()
    blind = min(max(-start, 0), lc)
    assert got[:, :, :blind].isnan().all()
    if blind < lc:
        held = torch.tensor([min(start, 1280)], dtype=torch.int32)
        want = O.chunked_sdpa(q[:, :, blind:], key, value, table, torch.clamp(held + blind, 0), d**-0.5)
        P._check(f"start {start} d{d}", got[:, :, blind:], want)


def test_block_float_8_with_room_for_the_copies_only(monkeypatch):
    """Scratch of ttpa_sdpa_prefill_workspace_bytes holds the copies and not the parts: the pass reads copies, unsplit."""
    from tt_xla_amd import _native as N

    users, hq, hkv, d, bs, start, lc = 1, 8, 8, 128, 64, 500, 100
    g = torch.Generator().manual_seed(5)
    nbpu = -(-(start + lc) // bs)
    key, value, table = P._paged(g, users, nbpu, hkv, bs, d, False)
    q = P._bf(g, users, hq, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    packed = [bfp8_codec.pack_cache(t) for t in (key, value)]
    want = O.chunked_sdpa(q, *[bfp8_codec.unpack_cache(t, bs).to(torch.bfloat16) for t in packed], table, st, d**-0.5)
    room = int(N.lib().ttpa_sdpa_prefill_workspace_bytes(users, hkv, d, bs, nbpu, 1))
    parts = int(N.lib().ttpa_sdpa_prefill_scratch_bytes(users, hq, hkv, lc, d, bs, nbpu, 1))
    blocks = torch.zeros(room, dtype=torch.uint8, device="cuda")
    call = N.call

    def with_room(size):
        def wrapped(name, *a):
            if name == "ttpa_sdpa_prefill_expanded":
                a = a[:-3] + (blocks.data_ptr(), size, a[-1])
            return call(name, *a)
        return wrapped

    args = [t.cuda() for t in (q, packed[0], packed[1], table, st)]
    assert room < parts
    for size in (room, room - 256):  # copies; neither copies nor parts
        blocks.zero_()
        monkeypatch.setattr(N, "call", with_room(size))
        got = _pass(*args, d**-0.5)
        assert bool(blocks.any()) == (size == room)
        P._check(f"copies only, {size} of {room} bytes, parts {parts}", got.cpu(), want)


@pytest.mark.parametrize("users,hq,hkv,lc,nbpu,copies", [
    (1, 16, 16, 32, 3, True), (1, 16, 16, 128, 3, True), (8, 16, 16, 256, 12, True),  # few rows to copy; two row blocks
    (4, 40, 8, 64, 6, False), (5, 40, 8, 64, 10, True),                               # one row block, five readers of few keys, of many
    (8, 16, 8, 128, 4, False), (1, 16, 16, 128, 4, True), (5, 16, 8, 64, 4, False),   # two row blocks over few keys; few rows, many
])
def test_block_float_8_under_tables_too_narrow_to_be_split(monkeypatch, users, hq, hkv, lc, nbpu, copies):
    """Where neither loop is split, a pass reads copies if they are few or read more than once: its scratch is theirs,
    and holds them behind the pass."""
    from tt_xla_amd import _native as N

    d, bs = 128, 64
    g = torch.Generator().manual_seed(users + lc)
    key, value, table = P._paged(g, users, nbpu, hkv, bs, d, False)
    q = P._bf(g, users, hq, lc, d)
    st = torch.tensor([nbpu * bs - lc], dtype=torch.int32)
    packed = [bfp8_codec.pack_cache(t) for t in (key, value)]
    want = O.chunked_sdpa(q, *[bfp8_codec.unpack_cache(t, bs).to(torch.bfloat16) for t in packed], table, st, d**-0.5)
    room = int(N.lib().ttpa_sdpa_prefill_workspace_bytes(users, hkv, d, bs, nbpu, 1))
    assert int(N.lib().ttpa_sdpa_prefill_scratch_bytes(users, hq, hkv, lc, d, bs, nbpu, 1)) == (room if copies else 0)
    blocks = torch.zeros(room, dtype=torch.uint8, device="cuda")
    call = N.call

    def with_room(name, *a):
        return call(name, *(a[:-3] + (blocks.data_ptr(), room, a[-1]) if name == "ttpa_sdpa_prefill_expanded" else a))

    monkeypatch.setattr(N, "call", with_room)
    got = _pass(*[t.cuda() for t in (q, packed[0], packed[1], table, st)], d**-0.5)
    assert bool(blocks.any()) == copies
    P._check(f"narrow u{users} h{hq}x{hkv} len{lc} width{nbpu}", got.cpu(), want)


@pytest.mark.parametrize("d,bs,start", [(64, 64, 640), (64, 32, 1216), (128, 64, 1216), (256, 32, 832)])
def test_infinite_values_of_the_last_part_stay_infinite(d, bs, start):
    """An infinite V element seen by every row makes its output infinite, in whichever part of the keys it lies (the merge
    reads parts four at a time)."""
    from tt_xla_amd import _native as N

    g = torch.Generator().manual_seed(d + start)
    lc, inf = 32, float("inf")
    nbpu = -(-(start + lc) // bs)
    key, value, table = P._paged(g, 1, nbpu, 2, bs, d, False)
    for column, t in enumerate(range(0, start, 48)):
        value[int(table[0, t // bs]), :, t % bs, column] = inf if column % 2 else -inf
    q = P._bf(g, 1, 4, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    assert N.lib().ttpa_sdpa_prefill_scratch_bytes(1, 4, 2, lc, d, bs, nbpu, 0) > 0
    got = _pass(q.cuda(), key.cuda(), value.cuda(), table.cuda(), st.cuda(), d**-0.5).cpu().float()
    want = O.chunked_sdpa(q, key, value, table, st, d**-0.5).float()
    assert want.isinf().any() and torch.equal(got.isinf(), want.isinf()) and not got.isnan().any()
    torch.testing.assert_close(got, want.reshape(got.shape), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("hq,hkv,d,rows,start,bfp8", [
    (8, 8, 64, 32, 64, False), (64, 8, 64, 512, 512, False), (16, 8, 256, 128, 64, False), (8, 8, 64, 128, 64, True),
    (16, 16, 128, 128, 64, True),  # split in place by the table, copies by the chunk
    (32, 8, 128, 32, 96, False),   # the streaming loop
])
def test_a_pass_is_laid_out_for_the_chunk_and_not_for_the_table(hq, hkv, d, rows, start, bfp8):
    """The metadata's chunk_end, which the builder knows: a wide page table makes an eager pass no other than a table that ends with
    the chunk.  It is never what is attended: a smaller number gives the same result, and a captured pass goes by the table."""
    from tt_xla_amd import TTAttentionBackendImpl, custom_ops
    from tt_xla_amd import _native as N
    from tt_xla_amd.metadata import PagedMetadataBuilder

    bs, g = 64, torch.Generator().manual_seed(hq + d + rows)
    blocks = -(-(start + rows) // bs)
    scratch = [int(N.lib().ttpa_sdpa_prefill_bounded_scratch_bytes(1, hq, hkv, rows, d, bs, 128, int(bfp8), n)) for n in (0, start + rows)]
    assert scratch[0] == int(N.lib().ttpa_sdpa_prefill_scratch_bytes(1, hq, hkv, rows, d, bs, 128, int(bfp8))) > 0
    assert scratch[1] == (2 * 128 * hkv * bs * d * 2 + 512 if d == 128 and bfp8 else 0)
    table = torch.arange(1, blocks + 1, dtype=torch.int32).view(1, blocks).numpy()
    caches = [P._bf(g, blocks + 1, hkv, bs, d).cuda() for _ in range(2)]
    if bfp8:
        caches = [custom_ops.bfp8_pack_cache(t) for t in caches]
    q, k, v = (P._bf(g, rows, n * d).cuda() for n in (hq, hkv, hkv))
    impl = TTAttentionBackendImpl(hq, d, d**-0.5, hkv, None, None, "auto")
    outs = {}
    for name, width, end in (("narrow", blocks, None), ("told", 128, start + rows), ("told less", 128, 32), ("not told", 128, None)):
        meta = PagedMetadataBuilder(bs, width, max(32, rows), device="cuda").prepare(table, [start], [rows]).metadata
        assert meta.chunk_end == start + rows
        meta.chunk_end = end
        outs[name] = torch.zeros_like(q)
        assert impl._native_pass(q, k, v, caches, meta, outs[name])
    meta.chunk_end = start + rows
    captured, graph = torch.zeros_like(q), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        impl.forward(None, q, k, v, caches, meta, output=captured)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(outs["narrow"], outs["told"])
    for name in ("told less", "not told"):
        torch.testing.assert_close(outs[name].float(), outs["told"].float(), atol=2e-2, rtol=2e-2)
    assert torch.equal(captured, outs["not told"])
