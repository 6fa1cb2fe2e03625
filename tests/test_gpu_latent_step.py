"""tt::latent_decode_step_ (projections, cache write and latent attention in one call) against the backend's
operators in turn on the same inputs: user counts around its tile of 32, head counts of both latent
kernels, weights that are permuted views, parked rows and positions outside the table.  The caches agree bit
for bit; the outputs within the two bfloat16 roundings (2^-8 each) of the intermediates, 2e-2 as in
test_gpu_mla.py."""

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


@pytest.mark.parametrize("users,n,bs,ctx,views", [
    (1, 16, 32, 70, False), (31, 16, 64, 40, False), (32, 8, 16, 33, True), (33, 16, 32, 300, True), (130, 16, 64, 90, False),
    (3, 1, 32, 20, False), (5, 32, 32, 64, False), (4, 128, 64, 150, True),
])
def test_step_equals_operators_in_turn(users, n, bs, ctx, views):
    from tt_xla_amd import attention_mla as M
    from tt_xla_amd.attention import TTMetadata

    g = torch.Generator().manual_seed(users + n + ctx)
    w = -(-(ctx + 1) // bs)
    nb = users * w + 1
    pos = torch.randint(0, ctx + 1, (users,), generator=g).to(torch.int32)
    if users > 3:
        pos[1], pos[2] = -1, w * bs + 5  # a parked row, a position behind the table
    table = (torch.randperm(nb - 1, generator=g)[: users * w] + 1).view(users, w).to(torch.int32)
    uk, uv = _bf(g, n, 128, 512) / math.sqrt(128), _bf(g, n, 512, 128) / math.sqrt(512)
    if views:  # the same numbers behind other strides
        uk = uk.transpose(1, 2).contiguous().cuda().transpose(1, 2)
        uv = uv.transpose(0, 1).contiguous().cuda().transpose(0, 1)
    layer = types.SimpleNamespace(W_UK_T=uk.cuda(), W_UV=uv.cuda())
    q = _bf(g, users, n, 192).cuda()
    kv_c, k_pe, cache0 = _bf(g, users, 512).cuda(), _bf(g, users, 1, 64).cuda(), _bf(g, nb, 1, bs, 576).cuda()
    got = []
    for functional in (False, True):
        impl = M.TTMLAAttentionBackendImpl(
            num_heads=n, head_size=576, scale=192**-0.5, num_kv_heads=1, alibi_slopes=None, sliding_window=None,
            kv_cache_dtype="auto", logits_soft_cap=None, attn_type="decoder", kv_sharing_target_layer_name=None, kv_lora_rank=512,
            qk_nope_head_dim=128, qk_rope_head_dim=64, qk_head_dim=192, v_head_dim=128, functional_cache_ops=functional)
        cache = cache0.clone()
        meta = TTMetadata(cache_position=pos.cuda(), page_table=table.cuda(), is_causal=True)
        out = torch.full((users, n * 128), 7.0, dtype=torch.bfloat16, device="cuda")
        impl.forward((q[..., :128], q[..., 128:]), kv_c, k_pe, cache, meta, layer, output=out)
        got.append((out.float(), cache))
    assert torch.equal(got[0][1], got[1][1])
    err = (got[0][0] - got[1][0]).nan_to_num().abs().max().item()
    print(f"latent step users{users} heads{n}: max difference {err:.3e}", flush=True)
    torch.testing.assert_close(got[0][0], got[1][0], atol=2e-2, rtol=2e-2, equal_nan=True)
