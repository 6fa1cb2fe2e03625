"""The merge of few segments with many partials, whose batches are shared by slices of a workgroup: numbers of
partials around one batch (8), around one round of the slices (64) and past it, both partial formats, and
partials that an explicit mask leaves empty.

Bound: the kernels round probabilities to bfloat16 (2^-9 relative each, random signs) and the output to bfloat16
(2^-9): at most 2^-8 of the output's norm; the latent form rounds its partials as well, and a case has fewer
than 2^7 of them, whose errors add like a random walk under weights of sum 1: another 2^-9."""

import math

import pytest
import torch

import __graft_entry__ as entry

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    entry.ensure_built()
    import tt_xla_amd  # noqa: F401


def _close(got, want, bound):
    err = (got.double().cpu() - want).norm() / want.norm()
    print(f"relative error {err:.2e}", flush=True)
    assert torch.isfinite(got.float()).all() and err < bound


def _paged(g, ctx, hkv, bs, d):
    w = [-(-c // bs) for c in ctx]
    cache = [torch.randn(sum(w) + 1, hkv, bs, d, generator=g).to(torch.bfloat16) for _ in range(2)]
    ids, table, at = torch.randperm(sum(w), generator=g) + 1, torch.zeros(len(ctx), max(w), dtype=torch.int32), 0
    for u, n in enumerate(w):
        table[u, :n] = ids[at : at + n].to(torch.int32)
        at += n
    return cache, table


def _attend(q, k, v, scale, mask=None):
    """[heads, d] over [tokens, kv heads, d] in 64 bits."""
    rep = q.shape[0] // k.shape[1]
    k, v = (t.double().repeat_interleave(rep, 1) for t in (k, v))
    s = torch.einsum("hd,thd->ht", q.double(), k) * scale
    return torch.einsum("ht,thd->hd", torch.softmax(s if mask is None else s + mask.double(), 1), v)


@pytest.mark.parametrize("hq,hkv,d,ctx", [
    (4, 1, 128, [480]), (4, 1, 128, [544]), (4, 1, 64, [4096 + 64]), (8, 1, 256, [1 + 32 * 64]), (8, 2, 128, [9000, 3]),
    (3, 1, 128, [5000]), (4, 1, 128, [70, 4096, 1]),
])
@pytest.mark.parametrize("sink", [False, True])
def test_few_long_segments(hq, hkv, d, ctx, sink, monkeypatch):
    if max(ctx) <= 544:  # (short enough to be read whole, without partials)
        monkeypatch.setenv("TTPA_DECODE_KERNEL", "ranges")
    g = torch.Generator().manual_seed(sum(ctx) + d)
    bs = 32
    (k, v), table = _paged(g, ctx, hkv, bs, d)
    q = torch.randn(1, len(ctx), hq, d, generator=g).to(torch.bfloat16)
    logits = torch.randn(hq, generator=g).to(torch.bfloat16) if sink else None
    out = torch.ops.tt.paged_scaled_dot_product_attention_decode(
        q.cuda(), k.cuda(), v.cuda(), table.cuda(), is_causal=True, cur_pos_tensor=torch.tensor(ctx, dtype=torch.int32).cuda() - 1,
        scale=d**-0.5, attention_sink=logits.cuda() if sink else None)
    rows = lambda c, u: c[table[u].long()].transpose(1, 2).reshape(-1, hkv, d)[: ctx[u]]  # noqa: E731
    want = []
    for u in range(len(ctx)):
        ku, vu = rows(k, u), rows(v, u)
        ref = _attend(q[0, u], ku, vu, d**-0.5)
        if sink:
            s = torch.einsum("hd,thd->ht", q[0, u].double(), ku.double().repeat_interleave(hq // hkv, 1)) * d**-0.5
            total = torch.logsumexp(s, 1)
            ref = ref * torch.sigmoid(total - logits.double())[:, None]
        want.append(ref)
    _close(out[0], torch.stack(want), 2**-8)


@pytest.mark.parametrize("masked_from,masked_to", [(0, 3000), (1000, 4096)])
def test_partials_that_a_mask_leaves_empty(masked_from, masked_to):
    g = torch.Generator().manual_seed(masked_from)
    hq, hkv, d, bs, ctx = 4, 1, 128, 32, 4096
    (k, v), table = _paged(g, [ctx], hkv, bs, d)
    q = torch.randn(1, 1, hq, d, generator=g).to(torch.bfloat16)
    mask = torch.zeros(1, 1, 1, ctx, dtype=torch.bfloat16)
    mask[..., masked_from:masked_to] = float("-inf")
    out = torch.ops.tt.paged_scaled_dot_product_attention_decode(
        q.cuda(), k.cuda(), v.cuda(), table.cuda(), is_causal=False, attn_mask=mask.cuda(),
        cur_pos_tensor=torch.tensor([ctx - 1], dtype=torch.int32).cuda(), scale=d**-0.5)
    rows = [c[table[0].long()].transpose(1, 2).reshape(-1, hkv, d) for c in (k, v)]
    _close(out[0, 0], _attend(q[0, 0], *rows, d**-0.5, mask[0, 0]), 2**-8)


@pytest.mark.parametrize("pad", [0, 2])
@pytest.mark.parametrize("heads,ctx", [(16, [600]), (16, [5383]), (8, [2048, 17]), (128, [3000])])
def test_latent_partials(heads, ctx, pad):
    from tt_xla_amd import custom_ops as C

    g = torch.Generator().manual_seed(sum(ctx) + heads)
    bs, scale = 32, 1 / math.sqrt(192)
    (k, _), table = _paged(g, ctx, 1, bs, 576)
    q = torch.randn(len(ctx), heads, 576, generator=g).to(torch.bfloat16) * 0.5
    # (pad 2: output rows on 4-byte boundaries, one word per thread)
    out = torch.zeros(len(ctx), heads, 512 + pad, dtype=torch.bfloat16, device="cuda")[..., :512]
    C._mla_decode_launch(out, q.cuda(), k.cuda(), None, table.cuda(), torch.tensor(ctx, dtype=torch.int32).cuda() - 1, 512, scale, None)
    rows = [k[table[u].long()].reshape(-1, 1, 576)[: ctx[u]] for u in range(len(ctx))]
    want = torch.stack([_attend(q[u], rows[u], rows[u][..., :512], scale) for u in range(len(ctx))])
    _close(out, want, 2**-8 + 2**-9)
