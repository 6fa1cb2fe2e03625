"""The latent backend's passes in the forms that its own operators take or leave: outputs that are not
aligned.  Compared with the same pass in its ordinary form, bit for bit."""

import math
import types

import pytest
import torch

import __graft_entry__ as entry

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    entry.ensure_built()
    import tt_xla_amd  # noqa: F401


def _bf(gen, *shape):
    return torch.randn(*shape, generator=gen).to(torch.bfloat16)


def _impl(n, **kw):
    from tt_xla_amd import attention_mla as M

    return M.TTMLAAttentionBackendImpl(
        **{**dict(num_heads=n, head_size=576, scale=192**-0.5, num_kv_heads=1, alibi_slopes=None, sliding_window=None,
                  kv_cache_dtype="auto", logits_soft_cap=None, attn_type="decoder", kv_sharing_target_layer_name=None, kv_lora_rank=512,
                  qk_nope_head_dim=128, qk_rope_head_dim=64, qk_head_dim=192, v_head_dim=128), **kw})


def _pass(seed, n, users, s, bs=32, ctx=100):
    """Inputs of a decode step (s = 1) behind up to ctx tokens, or of a prompt pass: a dict of GPU tensors."""
    from tt_xla_amd.attention import TTMetadata

    g = torch.Generator().manual_seed(seed)
    w = -(-(max(ctx, s) + 1) // bs)
    nb = users * w + 1
    table = (torch.randperm(nb - 1, generator=g)[: users * w] + 1).view(users, w).to(torch.int32).cuda()
    pos = torch.randint(0, ctx + 1, (users,), generator=g) if s == 1 else torch.full((users,), s - 1)
    t = users * s
    return types.SimpleNamespace(
        q=(_bf(g, t, n, 128).cuda(), _bf(g, t, n, 64).cuda()), kv_c=_bf(g, t, 512).cuda(), k_pe=_bf(g, t, 1, 64).cuda(),
        cache=_bf(g, nb, 1, bs, 576).cuda(),
        layer=types.SimpleNamespace(W_UK_T=(_bf(g, n, 128, 512) / math.sqrt(128)).cuda(), W_UV=(_bf(g, n, 512, 128) / math.sqrt(512)).cuda()),
        meta=TTMetadata(cache_position=pos.to(torch.int32).cuda(), page_table=table, is_causal=True))


def _run(impl, p, out=None, layer=None, cache=None):
    cache = p.cache.clone() if cache is None else cache
    if out is None:
        out = torch.zeros(p.kv_c.shape[0], impl.num_heads * 128, dtype=torch.bfloat16, device="cuda")
    impl.forward(p.q, p.kv_c, p.k_pe, cache, p.meta, layer or p.layer, output=out)
    return out, cache


@pytest.mark.parametrize("s", [1, 32])
def test_output_that_is_not_aligned(s):
    p, impl = _pass(s, 16, 3, s), _impl(16)
    want, want_cache = _run(impl, p)
    room = torch.zeros(want.numel() + 1, dtype=torch.bfloat16, device="cuda")
    got, cache = _run(impl, p, out=room[1:].view(want.shape))
    assert torch.equal(got, want) and torch.equal(cache, want_cache) and room[0] == 0
