"""The latent backend's forward under a tracer and under differentiation, on fake tensors of the GPU type
(nothing is computed): decode step and prompt pass of the head shape with operators of its own, and of
another one, are one graph; where something looks at the weights' derivative or maps over them, the pass
goes through the operators in turn, whose output expansion is an ordinary product."""

import types

import pytest
import torch
from torch._subclasses import FakeTensorMode


def _forward(users, s, n=16, nope=128, rope=64, lat=512, vd=128, **kw):
    import __graft_entry__  # noqa: F401  (puts the package on sys.path)
    from tt_xla_amd import attention_mla as M
    from tt_xla_amd.attention import TTMetadata

    new = lambda *shape, dtype=torch.bfloat16: torch.empty(*shape, dtype=dtype, device="cuda")  # noqa: E731
    layer = types.SimpleNamespace(W_UK_T=new(n, nope, lat), W_UV=new(n, lat, vd))
    impl = M.TTMLAAttentionBackendImpl(
        **{**dict(num_heads=n, head_size=lat + rope, scale=(nope + rope) ** -0.5, num_kv_heads=1, alibi_slopes=None, sliding_window=None,
                  kv_cache_dtype="auto", logits_soft_cap=None, attn_type="decoder", kv_sharing_target_layer_name=None, kv_lora_rank=lat,
                  qk_nope_head_dim=nope, qk_rope_head_dim=rope, qk_head_dim=nope + rope, v_head_dim=vd), **kw})
    meta = TTMetadata(cache_position=new(users, dtype=torch.int32), page_table=new(users, 4, dtype=torch.int32), is_causal=True)
    cache, t = new(9, 1, 32, lat + rope), users * s

    def forward(q_nope, q_pe, kv_c, k_pe, out):
        impl.forward((q_nope, q_pe), kv_c, k_pe, cache, meta, layer, output=out)
        return out

    return forward, layer, (new(t, n, nope), new(t, n, rope), new(t, lat), new(t, 1, rope), new(t, n * vd))


@pytest.mark.parametrize("s,ops", [
    (1, ["tt.latent_decode_step_"]), (64, ["tt.flash_mla_prefill", "tt.paged_fill_latent_cache_"]),
    (96, ["tt.split_key_prefill_out", "tt.paged_fill_latent_cache_"])])
def test_one_graph(s, ops):
    seen = []

    def backend(gm, _):
        seen.append([str(n.target) for n in gm.graph.nodes if n.op == "call_function" and str(n.target).startswith("tt.")])
        return gm.forward

    with FakeTensorMode():
        forward, _, args = _forward(2, s)
        torch._dynamo.reset()
        torch.compile(forward, fullgraph=True, backend=backend)(*args)
    assert seen == [ops]


@pytest.mark.parametrize("s", [1, 64, 96])
def test_one_graph_of_operators(s):
    with FakeTensorMode():
        forward, _, args = _forward(2, s, nope=64)
        torch._dynamo.reset()
        torch.compile(forward, fullgraph=True, backend="eager")(*args)


@pytest.mark.parametrize("s", [1, 64, 96])
def test_output_depends_on_the_weights(s):
    with FakeTensorMode():
        forward, layer, args = _forward(2, s)
        layer.W_UV.requires_grad_()
        assert forward(*args).requires_grad
        with torch.no_grad():
            assert not forward(*args[:4], torch.empty_like(args[4])).requires_grad


@pytest.mark.parametrize("s", [1, 64, 96])
def test_forward_mode_and_vmap(s):
    fw = torch.autograd.forward_ad
    with FakeTensorMode():
        forward, layer, args = _forward(2, s)
        plain = layer.W_UV
        with fw.dual_level():
            layer.W_UV = fw.make_dual(plain, torch.empty_like(plain))
            assert fw.unpack_dual(forward(*args)).tangent is not None

        def one(w_uv, out):
            layer.W_UV = w_uv
            return forward(*args[:4], out)

        assert torch.vmap(one)(torch.stack([plain] * 3), torch.stack([args[4]] * 3)).shape == (3,) + args[4].shape


@pytest.mark.parametrize("s", [1, 64, 96])
def test_scale_of_the_operators(s):
    """Without a scale of its own the layer uses the operators' default."""
    with FakeTensorMode():
        forward, _, args = _forward(2, s, scale=None)
        forward(*args)
