"""The backend's native host path against its operators on the same pass: every ordinary form gives the
same caches and output bit for bit; whatever is not ordinary (other dtypes or layouts, a watched gradient, a
cache of another shape) is left to the operators, untouched."""

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


HQ, HKV = 8, 2


def _pass(seed, users, s, d, bs, start, bfp8=False, window=None, sinks=False, i64=False, fused_rows=False):
    from tt_xla_amd import TTAttentionBackendImpl, TTMetadata
    from tt_xla_amd import custom_ops as ops

    g = torch.Generator().manual_seed(seed)
    w = -(-(start + s) // bs) + 1
    nb = users * w + 1
    table = (torch.randperm(nb - 1, generator=g) + 1).view(users, w).to(torch.int32).cuda()
    kc, vc = _bf(g, nb, HKV, bs, d), _bf(g, nb, HKV, bs, d)
    if bfp8:
        kc, vc = ops.bfp8_pack_cache(kc), ops.bfp8_pack_cache(vc)
    if fused_rows:  # q, k and v as slices of one projection's rows
        rows = _bf(g, users * s, (HQ + 2 * HKV) * d)
        q, k, v = rows[:, : HQ * d], rows[:, HQ * d : (HQ + HKV) * d], rows[:, (HQ + HKV) * d :]
    else:
        q, k, v = _bf(g, users * s, HQ * d), _bf(g, users * s, HKV * d), _bf(g, users * s, HKV * d)
    num = torch.int64 if i64 else torch.int32
    md = TTMetadata(
        cache_position=torch.randint(0, start + 1, (users,), generator=g).to(num).cuda() if s == 1 else None, page_table=table,
        fill_page_table=torch.roll(table, -(start // bs), 1) if s > 1 else None, batch_idx=torch.arange(users, dtype=num).cuda(),
        chunk_start_idx=torch.tensor([start], dtype=torch.int32).cuda() if s > 1 and start else None, num_users=users)
    sk = torch.randn(HQ, generator=g).cuda() if sinks else None
    impl = TTAttentionBackendImpl(HQ, d, d**-0.5, HKV, None, window, "auto", sinks=sk)
    return impl, [q, k, v, [kc, vc], md, torch.zeros(users * s, HQ * d, dtype=torch.bfloat16, device="cuda")]


def _run(impl, args, native):
    from tt_xla_amd import _native

    q, k, v, kv, md, out = args
    kv, out = [c.clone() for c in kv], out.clone()
    if native:
        assert impl._native_pass(q, k, v, kv, md, out)
    else:
        impl._native_pass = lambda *a: False
        try:
            impl.forward(None, q, k, v, kv, md, output=out)
        finally:
            del impl._native_pass
    assert _native.host() is not None
    return kv[0], kv[1], out


@pytest.mark.parametrize("case", [
    dict(users=1, s=1, d=64, bs=32, start=100), dict(users=5, s=1, d=128, bs=64, start=300, i64=True, sinks=True, window=50),
    dict(users=3, s=1, d=128, bs=32, start=90, bfp8=True, fused_rows=True), dict(users=2, s=1, d=256, bs=32, start=70),
    dict(users=1, s=32, d=128, bs=32, start=0), dict(users=3, s=96, d=64, bs=32, start=0, window=40, i64=True, fused_rows=True),
    dict(users=2, s=64, d=128, bs=32, start=128, fused_rows=True), dict(users=1, s=32, d=128, bs=64, start=2048),
    dict(users=2, s=48, d=64, bs=16, start=64, i64=True), dict(users=2, s=64, d=128, bs=32, start=96, bfp8=True),
])
def test_native_pass_equals_operators(case):
    impl, args = _pass(len(str(case)), **case)
    for a, b in zip(_run(impl, args, True), _run(impl, args, False)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_other_passes_are_left_to_the_operators():
    impl, args = _pass(1, users=2, s=1, d=128, bs=32, start=40)
    q, k, v, kv, md, out = args

    def refused(**change):
        a = dict(q=q, k=k, v=v, kv=kv, md=md, out=out)
        a.update(change)
        before = [c.clone() for c in kv]
        assert not impl._native_pass(a["q"], a["k"], a["v"], a["kv"], a["md"], a["out"])
        assert all(torch.equal(x, y) for x, y in zip(before, kv))

    refused(q=q.float())
    refused(q=q.view(2, HQ, 128))
    refused(k=k.cpu())
    refused(q=q.clone().requires_grad_())
    refused(out=torch.empty(2, HQ * 128 + 8, dtype=torch.bfloat16, device="cuda")[:, : HQ * 128])
    refused(kv=[kv[0], kv[1][1:]])
    refused(kv=[torch.tensor([]), torch.tensor([])])
    refused(kv=[kv[0].transpose(1, 2), kv[1].transpose(1, 2)])
    refused(q=torch._neg_view(q))
    with torch.autograd.forward_ad.dual_level():
        refused(q=torch.autograd.forward_ad.make_dual(q, torch.ones_like(q)))
    torch.vmap(lambda x: (refused(q=x), x)[1])(torch.stack([q, q]))
    md.num_users = None
    refused()
    md.num_users = 3
    refused()
    md.num_users, md.is_causal = 2, False
    refused()


def test_another_stream():
    impl, args = _pass(2, users=4, s=1, d=128, bs=32, start=200)
    want = _run(impl, args, False)[2]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = _run(impl, args, True)[2]
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, want)


@pytest.mark.parametrize("case,op", [
    (dict(users=2, s=1, d=128, bs=32, start=40), "paged_update_kv_decode_out_"),
    (dict(users=1, s=32, d=128, bs=32, start=0), "paged_fill_kv_prefill_out_"),
    (dict(users=1, s=32, d=128, bs=32, start=64), "chunked_scaled_dot_product_attention_out"),
])
def test_a_function_mode_sees_the_operators(case, op):
    from torch.overrides import TorchFunctionMode

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    impl, (q, k, v, kv, md, out) = _pass(3, **case)
    seen = []
    with Watch():
        impl.forward(None, q, k, v, kv, md, output=out)
    assert any(op in name for name in seen), seen


@pytest.mark.parametrize("case,names", [
    (dict(users=2, s=1, d=128, bs=32, start=40), ["tt::paged_update_kv_decode_out_"]),
    (dict(users=1, s=32, d=128, bs=32, start=0), ["tt::paged_fill_kv_prefill_out_"]),
    (dict(users=1, s=32, d=128, bs=32, start=64), ["tt::paged_fill_kv_cache_", "tt::chunked_scaled_dot_product_attention_out"]),
])
def test_a_profiler_names_the_operators(case, names):
    impl, (q, k, v, kv, md, out) = _pass(4, **case)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        assert impl._native_pass(q, k, v, kv, md, out)
    got = [e.name for e in prof.events()]
    assert [n for n in got if n.startswith("tt::")] == names


@pytest.mark.parametrize("case", [dict(users=2, s=1, d=96, bs=32, start=40), dict(users=1, s=32, d=96, bs=32, start=0),
                                  dict(users=1, s=32, d=96, bs=32, start=64)])
def test_an_error_names_the_entry_point(case):
    """A head size that is not built: refused on the host, in the words of the operators' error."""
    from tt_xla_amd import _native

    impl, args = _pass(5, **case)
    said = []
    for native in (True, False):
        with pytest.raises(_native.TtpaError) as error:
            _run(impl, args, native)
        said.append(str(error.value))
    assert said[0] == said[1]


def test_other_threads_run_while_a_launch_waits():
    """Behind a kernel that keeps the GPU busy the queue fills up and a launch waits for room: not with the
    interpreter lock held.  (The other thread's longest pause is compared with the longest wait of this one.)"""
    import threading
    import time

    impl, (q, k, v, kv, md, out) = _pass(6, users=1, s=1, d=64, bs=32, start=30)
    impl.forward(None, q, k, v, kv, md, output=out)
    torch.cuda.synchronize()
    pauses, stop = [], threading.Event()

    def tick():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(1e-3)
            now = time.perf_counter()
            pauses.append((now - last, last))
            last = now

    other = threading.Thread(target=tick)
    other.start()
    t0 = time.perf_counter()
    torch.cuda._sleep(10**6)
    torch.cuda.synchronize()
    cycles = int(10**6 * min(0.6 / max(time.perf_counter() - t0, 1e-4), 2000))  # about 0.6 s
    waits, begin = [], time.perf_counter()
    torch.cuda._sleep(cycles)
    while time.perf_counter() - begin < 2 and not any(w > 0.03 for w, _ in waits):
        t0 = time.perf_counter()
        impl.forward(None, q, k, v, kv, md, output=out)
        waits.append((time.perf_counter() - t0, t0))
    stop.set()
    other.join()
    torch.cuda.synchronize()
    wait, t0 = max(waits)
    print(f"{len(waits)} passes behind {cycles} cycles, longest {wait:.3f} s", flush=True)
    if wait < 0.03:
        pytest.skip("no launch had to wait")
    during = [p for p, at in pauses if at + p > t0 and at < t0 + wait]
    print(f"longest wait of a pass {wait:.3f} s, pauses of the other thread meanwhile up to {max(during):.3f} s", flush=True)
    assert max(during) < wait / 2


def test_a_window_that_is_no_64_bit_number_is_the_operators_to_refuse():
    impl, (q, k, v, kv, md, out) = _pass(7, users=2, s=1, d=128, bs=32, start=40, window=2**70)
    assert not impl._native_pass(q, k, v, kv, md, out)
    with pytest.raises((RuntimeError, OverflowError)):
        impl.forward(None, q, k, v, kv, md, output=out)
