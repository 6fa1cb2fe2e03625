"""Prefill with keys of 128 + 64 features in two parts (the prompt form of the latent layers, and
tt::flash_mla_prefill with a V of its own at that size): one block to rings that wrap several times,
row blocks of a workgroup that do not exist, one / two / four heads per KV head, a rotary part that the
heads share; and the two-part cache fill.  Oracle and tolerance as in test_gpu_mla.py."""

import math

import pytest
import torch

import __graft_entry__ as entry
from oracle import paged_ops as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    entry.ensure_built()
    import tt_xla_amd  # noqa: F401


def _bf(gen, *shape):
    return torch.randn(*shape, generator=gen).to(torch.bfloat16)


@pytest.mark.parametrize("b,hq,hkv,s", [
    (1, 1, 1, 32), (1, 3, 3, 64), (2, 2, 2, 96), (1, 5, 5, 160), (1, 2, 1, 128), (2, 4, 2, 224), (1, 4, 1, 96),
    (1, 8, 2, 288), (2, 16, 16, 352), (1, 1, 1, 1184),
])
def test_explicit_value(b, hq, hkv, s):
    g = torch.Generator().manual_seed(b + hq + s)
    q, k, v = _bf(g, b, hq, s, 192), _bf(g, b, hkv, s, 192), _bf(g, b, hkv, s, 128)
    want = O.flash_mla_prefill(q, k, 128, v, None, True, None)
    got = torch.ops.tt.flash_mla_prefill(q.cuda(), k.cuda(), 128, v.cuda()).cpu()
    print(f"b{b} h{hq}x{hkv} s{s}: max-abs error {(got.float() - want.float()).abs().max().item():.3e}", flush=True)
    torch.testing.assert_close(got.float(), want.float(), atol=2e-2, rtol=2e-2)


def test_shared_rotary_part_and_strides():
    g = torch.Generator().manual_seed(3)
    b, h, s = 2, 6, 128
    q = _bf(g, b, s, h, 192)                      # token-major rows of both parts, as a projection leaves them
    k, rope, v = _bf(g, b, s, h, 128), _bf(g, b, s, 64), _bf(g, h, b, s, 128)
    out = torch.empty(b, s, h, 128, dtype=torch.bfloat16, device="cuda")
    qd = q.cuda().transpose(1, 2)
    torch.ops.tt.split_key_prefill_out(qd[..., :128], qd[..., 128:], k.cuda().transpose(1, 2), rope.cuda().unsqueeze(1),
                                       v.cuda().transpose(0, 1), out.transpose(1, 2), 192**-0.5)
    kk = torch.cat([k, rope.unsqueeze(2).expand(b, s, h, 64)], -1).transpose(1, 2)
    want = O.flash_mla_prefill(q.transpose(1, 2), kk, 128, v.transpose(0, 1), None, True, 192**-0.5)
    torch.testing.assert_close(out.cpu().transpose(1, 2).float(), want.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("users,s,bs,lat,rope,aligned", [
    (1, 1, 16, 512, 64, True), (3, 77, 32, 512, 64, True), (2, 130, 64, 64, 8, True),
    (3, 77, 32, 512, 64, False), (2, 33, 16, 60, 12, True),  # what does not come in 16-byte pieces
])
def test_two_part_fill(users, s, bs, lat, rope, aligned):
    g = torch.Generator().manual_seed(users + s)
    w = -(-s // bs) + 1
    nb = users * w + 2
    table = (torch.randperm(nb, generator=g)[: users * w]).view(users, w).to(torch.int32)
    table[0, 0] = nb + 5  # out of range: skipped
    cache, latent, rotary = _bf(g, nb, 1, bs, lat + rope), _bf(g, users, s, lat), _bf(g, users, s, rope)
    dev = cache.cuda() if aligned else torch.zeros(cache.numel() + 1, dtype=cache.dtype, device="cuda")[1:].view(cache.shape).copy_(cache)
    torch.ops.tt.paged_fill_latent_cache_(dev, latent.cuda(), rotary.cuda(), table.cuda())
    rows = torch.cat([latent, rotary], -1)
    for u in range(users):
        for t in range(s):
            if 0 <= int(table[u, t // bs]) < nb:
                cache[table[u, t // bs], 0, t % bs] = rows[u, t]
    assert torch.equal(dev.cpu(), cache)


@pytest.mark.parametrize("n,users,s", [(16, 2, 64), (4, 1, 32), (3, 3, 160)])
def test_backend_prompt_forms_agree(n, users, s):
    """The expanded and the absorbed form of a prompt pass: the same output up to the bfloat16 roundings of
    their intermediates (each within 2^-8 of a row's magnitude), the same cache bit for bit."""
    import types

    from tt_xla_amd import attention_mla as M
    from tt_xla_amd.attention import TTMetadata

    g = torch.Generator().manual_seed(n + s)
    layer = types.SimpleNamespace(W_UK_T=(_bf(g, n, 128, 512) / math.sqrt(128)).cuda(), W_UV=(_bf(g, n, 512, 128) / math.sqrt(512)).cuda())
    w = -(-s // 32)
    table = (torch.randperm(users * w, generator=g)).view(users, w).to(torch.int32).cuda()
    args = [t.cuda() for t in (_bf(g, users * s, n, 128), _bf(g, users * s, n, 64), _bf(g, users * s, 512), _bf(g, users * s, 1, 64))]
    got = []
    for functional in (False, True):
        impl = M.TTMLAAttentionBackendImpl(
            num_heads=n, head_size=576, scale=192**-0.5, num_kv_heads=1, alibi_slopes=None, sliding_window=None,
            kv_cache_dtype="auto", logits_soft_cap=None, attn_type="decoder", kv_sharing_target_layer_name=None, kv_lora_rank=512,
            qk_nope_head_dim=128, qk_rope_head_dim=64, qk_head_dim=192, v_head_dim=128, functional_cache_ops=functional)
        cache = torch.zeros(users * w, 1, 32, 576, dtype=torch.bfloat16, device="cuda")
        meta = TTMetadata(cache_position=torch.full((users,), s - 1, dtype=torch.int32).cuda(), page_table=table, is_causal=True)
        out = torch.empty(users * s, n * 128, dtype=torch.bfloat16, device="cuda")
        impl.forward((args[0], args[1]), args[2], args[3], cache, meta, layer, output=out)
        got.append((out.float(), cache))
    assert torch.equal(got[0][1], got[1][1])
    torch.testing.assert_close(got[0][0], got[1][0], atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("dh", [192, 128])  # the split-key kernel's shape, and one of the decode kernels'
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.uint8])
def test_value_of_another_type_is_refused(dh, dtype):
    """The kernels read V as bfloat16: another type's bits would be taken for numbers, a one-byte V read past its end."""
    g = torch.Generator().manual_seed(1)
    q, k = _bf(g, 1, 2, 32, dh).cuda(), _bf(g, 1, 2, 32, dh).cuda()
    with pytest.raises(ValueError, match="bfloat16"):
        torch.ops.tt.flash_mla_prefill(q, k, 128, torch.zeros(1, 2, 32, 128, dtype=dtype, device="cuda"))
