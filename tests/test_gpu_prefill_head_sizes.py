"""The streaming prefill kernel at head sizes 64 and 256 (their own register maps and rings: five slots
of 4 KiB, four of 16 KiB) at the sizes where it can go wrong: one block, as many blocks as the rings hold
and one more, several rounds of the unrolled loop, row blocks that do not exist, window edges around a
block's, cache blocks of one and several table entries, keys split over workgroups.  Oracle and tolerance as in
test_gpu_prefill.py; the relative error against 64 bits stays at that of the compiler-scheduled loop
(measured 0.999 ... 1.001 of it over 143 passes; the bound leaves 2 %)."""

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


@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("b,hq,hkv,s,window", [
    (1, 1, 1, 32, 0), (1, 2, 1, 128, 0), (2, 4, 1, 160, 0), (1, 3, 3, 192, 0), (1, 8, 2, 352, 0), (1, 2, 2, 704, 0),
    (1, 2, 2, 416, 31), (1, 4, 2, 416, 32), (1, 4, 1, 416, 33), (1, 3, 3, 288, 1), (2, 6, 3, 224, 97),
])
def test_dense(d, b, hq, hkv, s, window):
    g = torch.Generator().manual_seed(b + hq + s + window + d)
    q, k, v = P._bf(g, b, hq, s, d), P._bf(g, b, hkv, s, d), P._bf(g, b, hkv, s, d)
    want = O.sdpa_windowed(q, k, v, sliding_window=window) if window else O.sdpa(q, k, v, None, True, None)
    got = torch.ops.tt.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), is_causal=True, sliding_window_size=window or None)
    P._check(f"dense b{b} h{hq}x{hkv} d{d} s{s} window{window}", got.cpu(), want)


@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("users,hq,hkv,bs,start,lc", [
    (2, 4, 1, 32, 0, 32), (1, 2, 1, 96, 96, 130), (1, 3, 3, 32, 224, 64), (2, 2, 1, 64, 192, 33), (4, 8, 2, 160, 320, 96),
    (1, 1, 1, 64, 0, 32), (1, 4, 2, 128, 37, 200), (1, 4, 1, 32, 1000, 96), (1, 8, 2, 64, 512, 300), (1, 2, 2, 128, 1280, 129),
])
def test_paged(d, users, hq, hkv, bs, start, lc):
    g = torch.Generator().manual_seed(hq + bs + start + d)
    key, value, table = P._paged(g, users, -(-(start + lc) // bs) + 1, hkv, bs, d, False)
    q = P._bf(g, users, hq, lc, d)
    st = torch.tensor([start], dtype=torch.int32)
    want = O.chunked_sdpa(q, key, value, table, st, d**-0.5)
    got = torch.ops.tt.chunked_scaled_dot_product_attention(q.cuda(), key.cuda(), value.cuda(), table.cuda(), st.cuda(), d**-0.5)
    P._check(f"paged h{hq}x{hkv} d{d} bs{bs} start{start} len{lc}", got.cpu(), want)


@pytest.mark.parametrize("users,hq,hkv,bs,start,lc", [
    (1, 8, 8, 32, 256, 32), (4, 8, 8, 64, 512, 64), (1, 8, 8, 32, 256, 65), (5, 8, 8, 32, 64, 32), (4, 16, 8, 32, 1024, 32), (2, 2, 1, 32, 1472, 32),
    (2, 2, 1, 32, 1504, 32), (1, 3, 1, 32, 96, 32), (32, 2, 1, 64, 100, 20),
])
def test_few_rows_of_64_features(users, hq, hkv, bs, start, lc):
    """On either side of the line between the two loops where a group has one or two (row block, head) pairs."""
    test_paged(64, users, hq, hkv, bs, start, lc)


@pytest.mark.parametrize("d", [64, 256])
def test_scores_that_force_a_rescale(d):
    """The running maximum moves by more than the lazy threshold again and again."""
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, h, 256, d, generator=g) for h in (8, 2, 2))
    k = k + q[:, ::4].mean(2, keepdim=True) * torch.linspace(0, 3, 256).view(1, 1, 256, 1)
    q, k, v = q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16)
    got = torch.ops.tt.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), None, True, None)
    P._check("rescale", got.cpu(), O.sdpa(q, k, v, None, True, None))


@pytest.mark.parametrize("hq", [2, 4, 6, 8])
@pytest.mark.parametrize("window", [31, 32, 33, 64, 100, 190])
def test_window_scores_that_force_a_rescale(hq, window):
    """The same behind a window's lower edge, with workgroups of several row blocks: rows whose first keys come blocks
    after the workgroup's first have nothing to rescale, the others have it in the same wavefront."""
    g = torch.Generator().manual_seed(window)
    q, k, v = (torch.randn(1, h, 256, 256, generator=g) for h in (hq, 2, 2))
    k = k + q[:, :: hq // 2].mean(2, keepdim=True) * torch.linspace(0, 6, 256).view(1, 1, 256, 1)
    q, k, v = q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16)
    got = torch.ops.tt.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), is_causal=True, sliding_window_size=window)
    P._check(f"rescale h{hq} window{window}", got.cpu(), O.sdpa_windowed(q, k, v, sliding_window=window))


@pytest.mark.parametrize("d,window", [(64, 0), (64, 300), (256, 0), (256, 300)])
def test_error_against_64_bits(d, window, monkeypatch):
    g = torch.Generator().manual_seed(d + window)
    q, k, v = P._bf(g, 2, 8, 704, d).cuda(), P._bf(g, 2, 2, 704, d).cuda(), P._bf(g, 2, 2, 704, d).cuda()
    kk, vv = (x.double().repeat_interleave(4, 1) for x in (k, v))
    hidden = torch.ones(704, 704, dtype=torch.bool, device="cuda").triu(1)
    if window:
        hidden |= torch.ones_like(hidden).tril(-window)
    exact = (q.double() @ kk.transpose(2, 3) * d**-0.5).masked_fill(hidden, float("-inf")).softmax(-1) @ vv
    error = {}
    for stream in ("1", "0"):
        monkeypatch.setenv("TTPA_PREFILL_STREAM", stream)
        got = torch.ops.tt.scaled_dot_product_attention(q, k, v, is_causal=True, sliding_window_size=window or None)
        error[stream] = float((got.double() - exact).norm() / exact.norm())
    assert error["1"] <= 1.02 * error["0"], error


@pytest.mark.parametrize("users,hq,hkv,bs,start,lc,copies", [
    (1, 8, 8, 64, 100, 1024, True), (1, 8, 8, 32, 100, 1000, True), (1, 8, 8, 64, 100, 896, False),   # eight workgroups per head group, seven
    (4, 8, 2, 32, 64, 256, True), (3, 8, 2, 32, 64, 256, False), (1, 64, 8, 64, 70, 250, True),        # 64 workgroups in all, 48
])
def test_block_float_8_chunks_of_64_features(monkeypatch, users, hq, hkv, bs, start, lc, copies):
    """On either side of the line from which on a pass reads bfloat16 copies of its blocks."""
    from tt_xla_amd import _native as N

    g = torch.Generator().manual_seed(users + hq + lc)
    nbpu = -(-(start + lc) // bs)
    key, value, table = P._paged(g, users, nbpu, hkv, bs, 64, False)
    q = P._bf(g, users, hq, lc, 64)
    st = torch.tensor([start], dtype=torch.int32)
    packed = [bfp8_codec.pack_cache(t) for t in (key, value)]
    want = O.chunked_sdpa(q, *[bfp8_codec.unpack_cache(t, bs).to(torch.bfloat16) for t in packed], table, st, 0.125)
    room = int(N.lib().ttpa_sdpa_prefill_workspace_bytes(users, hkv, 64, bs, nbpu, 1))
    blocks = torch.zeros(room, dtype=torch.uint8, device="cuda")
    call = N.call
    monkeypatch.setattr(N, "call", lambda name, *a: call(name, *(a[:-3] + (blocks.data_ptr(), room, a[-1]) if name == "ttpa_sdpa_prefill_expanded" else a)))
    got = torch.ops.tt.chunked_scaled_dot_product_attention(q.cuda(), packed[0].cuda(), packed[1].cuda(), table.cuda(), st.cuda(), 0.125)
    # (the scratch starts with K's copy of block 0 of user 0, of a pass that is split with float accumulators)
    k00 = bfp8_codec.unpack_cache(packed[0], bs).to(torch.bfloat16)[int(table[0, 0])]
    assert torch.equal(blocks[: k00.numel() * 2].view(torch.bfloat16).cpu(), k00.flatten()) == copies
    P._check(f"bfp8 u{users} h{hq}x{hkv} bs{bs} start{start} len{lc}", got.cpu(), want)
