"""GPU tests of the latent layer's pass in one native call (csrc/host_path.cpp: latent_pass) and of the prompt entry point behind
it: against the same pass through the operators.  Caches bit for bit.  Outputs: both sides round the same values to bfloat16
behind sums in another order, so an intermediate may fall on the other side of a rounding border (2^-8 of it); the
outputs' distance stays below one rounding (2^-8 relative, 2-norm)."""

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
    return torch.randn(*shape, generator=gen).to(torch.bfloat16).cuda()


def _impl(n):
    from tt_xla_amd import attention_mla as M

    return M.TTMLAAttentionBackendImpl(
        num_heads=n, head_size=576, scale=192**-0.5, num_kv_heads=1, alibi_slopes=None, sliding_window=None, kv_cache_dtype="auto",
        logits_soft_cap=None, attn_type="decoder", kv_sharing_target_layer_name=None, kv_lora_rank=512, qk_nope_head_dim=128,
        qk_rope_head_dim=64, qk_head_dim=192, v_head_dim=128)


def _pass(seed, n, users, s, bs=32, joint=None, slices=False):
    from tt_xla_amd.attention import TTMetadata

    g = torch.Generator().manual_seed(seed)
    w, t = -(-s // bs) + 1, users * s
    nb = users * w + 1
    table = (torch.randperm(nb - 1, generator=g)[: users * w] + 1).view(users, w).to(torch.int32).cuda()
    uk, uv = _bf(g, n, 128, 512) / 11, _bf(g, n, 512, 128) / 23
    if joint:  # views of one projection: [512, heads, 256] or [heads * 256, 512]
        both = torch.cat([uk.permute(2, 0, 1), uv.permute(1, 0, 2)], -1).contiguous()
        if joint == "heads first":
            both = both.permute(1, 2, 0).reshape(n * 256, 512).contiguous().t().view(512, n, 256)
        a, b = both.split([128, 128], -1)
        uk, uv = a.permute(1, 2, 0), b.transpose(0, 1)
    if slices:  # activations as slices of wider rows
        q, kv = _bf(g, t, n, 192), _bf(g, t, 576)
        qn, qr, lat, rope = q[..., :128], q[..., 128:], kv[:, :512], kv[:, 512:].unsqueeze(1)
    else:
        qn, qr, lat, rope = _bf(g, t, n, 128), _bf(g, t, n, 64), _bf(g, t, 512), _bf(g, t, 1, 64)
    pos = torch.randint(0, w * bs, (users,), generator=g) if s == 1 else torch.full((users,), s - 1)
    return types.SimpleNamespace(
        q=(qn, qr), lat=lat, rope=rope, cache=_bf(g, nb, 1, bs, 576), layer=types.SimpleNamespace(W_UK_T=uk, W_UV=uv),
        meta=TTMetadata(cache_position=pos.to(torch.int32).cuda(), page_table=table, fill_page_table=table, is_causal=True))


def _both(impl, p):
    results = []
    for native in (True, False):
        cache, out = p.cache.clone(), torch.zeros(p.lat.shape[0], impl.num_heads * 128, dtype=torch.bfloat16, device="cuda")
        args = (p.q, p.lat, p.rope, cache, p.meta, p.layer)
        if native:
            assert impl._forward_native(*args, out)
        else:
            impl._forward_native = lambda *a: False
            impl.forward(*args, output=out)
            del impl._forward_native
        torch.cuda.synchronize()
        results.append((out.float(), cache))
    return results


@pytest.mark.parametrize("n,users,s,bs,joint,slices", [
    (16, 1, 32, 32, None, False), (3, 5, 32, 16, "latent first", True), (16, 4, 64, 64, "heads first", False),   # absorbed
    (16, 1, 96, 32, None, False), (3, 3, 96, 64, None, True), (5, 1, 128, 32, "latent first", False),             # expanded: one tile, a
    (16, 2, 160, 16, "heads first", True), (1, 1, 4128, 64, None, False), (128, 1, 288, 32, None, False),         # remainder of one, many
    (16, 3, 1024, 64, None, False), (7, 1, 1, 32, None, True), (16, 40, 1, 64, "heads first", False),             # decode steps
])
def test_one_call_equals_the_operators(n, users, s, bs, joint, slices):
    print(f"latent pass heads{n} users{users} tokens{s} bs{bs} {joint} slices={slices}", flush=True)
    (got, cache), (want, want_cache) = _both(_impl(n), _pass(n + s, n, users, s, bs, joint, slices))
    assert torch.equal(cache, want_cache)
    assert torch.isfinite(got).all() and (got - want).norm() <= 2**-8 * want.norm()


@pytest.mark.parametrize("s", [64, 96, 1024])
def test_rows_that_are_not_written(s):
    """Blocks outside the cache and users behind the table's last row: skipped, as by the fill."""
    p = _pass(1, 16, 3, s)
    p.meta.fill_page_table = p.meta.fill_page_table[:2].clone()
    p.meta.fill_page_table[0, 1] = p.cache.shape[0]
    p.meta.fill_page_table[1, 0] = -1
    (got, cache), (want, want_cache) = _both(_impl(16), p)
    assert torch.equal(cache, want_cache) and not torch.equal(cache, p.cache)
    assert (got - want).norm() <= 2**-8 * want.norm()


@pytest.mark.parametrize("s", [64, 96, 2048])
def test_passes_repeat_themselves(s):
    """Workgroups of a launch that fills the chip several times over share nothing but the inputs."""
    p, impl = _pass(2, 16, 2, s), _impl(16)
    outs = []
    for _ in range(5):
        out = torch.zeros(2 * s, 2048, dtype=torch.bfloat16, device="cuda")
        assert impl._forward_native(p.q, p.lat, p.rope, p.cache.clone(), p.meta, p.layer, out)
        outs.append(out)
    assert all(torch.equal(o, outs[0]) for o in outs)


def test_what_is_left_to_the_operators():
    impl, p = _impl(16), _pass(3, 16, 2, 96)
    out = torch.zeros(192, 2048, dtype=torch.bfloat16, device="cuda")
    args = lambda **k: [{**dict(q=p.q, lat=p.lat, rope=p.rope, cache=p.cache, meta=p.meta, layer=p.layer, out=out), **k}[x]  # noqa: E731
                        for x in ("q", "lat", "rope", "cache", "meta", "layer", "out")]
    ns, before = types.SimpleNamespace, p.cache.clone()
    spread = torch.stack([p.layer.W_UV, p.layer.W_UV], -1)[..., 0]
    watched = p.layer.W_UV.clone().requires_grad_()
    for k in (dict(lat=p.lat.float()), dict(cache=p.cache.float()), dict(cache=torch.empty(0)), dict(cache=p.cache[:, :, :, :570]),
              dict(layer=ns(W_UK_T=p.layer.W_UK_T, W_UV=spread)), dict(layer=ns(W_UK_T=p.layer.W_UK_T, W_UV=watched)),
              dict(layer=ns(W_UK_T=p.layer.W_UK_T.cpu(), W_UV=p.layer.W_UV)), dict(out=out.t().contiguous().t()), dict(meta=None),
              dict(q=(p.q[0][:191], p.q[1][:191])), dict(rope=p.rope[:, 0])):
        assert not impl._forward_native(*args(**k))
    with torch.no_grad():
        assert impl._forward_native(*args(layer=ns(W_UK_T=p.layer.W_UK_T, W_UV=watched), cache=before.clone()))
    impl.scale = None
    assert not impl._forward_native(*args())
    assert torch.equal(p.cache, before)


def test_no_thread_takes_another_ones_scratch(monkeypatch):
    """A step's kernels hand data through scratch, and the interpreter lock is not held between their launches: what is kept
    belongs to a thread, for the operators and for the native call."""
    import threading

    from tt_xla_amd import custom_ops as ops

    kept, taken = ops._workspace, []
    monkeypatch.setattr(ops, "_workspace", lambda *a: taken.append(kept(*a)) or taken[-1])

    def step():
        for native in (True, False):
            p, impl = _pass(4, 16, 3, 1), _impl(16)
            if not native:
                impl._forward_native = lambda *a: False
            impl.forward(p.q, p.lat, p.rope, p.cache, p.meta, p.layer, output=torch.zeros(3, 2048, dtype=torch.bfloat16, device="cuda"))
        torch.cuda.synchronize()

    step()
    thread = threading.Thread(target=step)
    thread.start()
    thread.join()
    assert len(taken) == 4 and taken[0] is taken[1] and taken[2] is taken[3]
    assert taken[0].data_ptr() != taken[2].data_ptr()
