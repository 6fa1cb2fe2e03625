"""A block-float-8 cache's first chunk through the native host path: the operators' results and caches, bit for bit, and
what neither serves is refused as the operators refuse it."""

import pytest
import torch

import test_gpu_host_path as H

pytestmark = pytest.mark.gpu
_pkg = H._pkg


@pytest.mark.parametrize("case", [
    dict(users=1, s=32, d=128, bs=32), dict(users=3, s=96, d=64, bs=16, window=40, i64=True, fused_rows=True),
    dict(users=2, s=160, d=256, bs=64), dict(users=1, s=352, d=128, bs=96, window=100, fused_rows=True),
])
def test_first_chunk_equals_operators(case):
    impl, args = H._pass(len(str(case)), start=0, bfp8=True, **case)
    for a, b in zip(H._run(impl, args, True), H._run(impl, args, False)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_ragged_chunk_is_left_to_the_operators():
    impl, (q, k, v, kv, md, out) = H._pass(3, users=2, s=48, d=128, bs=32, start=0, bfp8=True)
    before = [c.clone() for c in kv]
    assert not impl._native_pass(q, k, v, kv, md, out)
    assert all(torch.equal(x, y) for x, y in zip(before, kv))


@pytest.mark.parametrize("fault", ["scale", "short table"])
def test_refused_as_the_operators_refuse(fault):
    impl, (q, k, v, kv, md, out) = H._pass(4, users=2, s=64, d=128, bs=32, start=0, bfp8=True)
    if fault == "scale":  # the entry point's own error, behind the fill
        impl.scale = 0.0
    else:  # more tokens than the table has room for: not an ordinary pass
        md.fill_page_table = md.fill_page_table[:, :1].contiguous()
        assert not impl._native_pass(q, k, v, kv, md, out)
    seen = []
    for native in (True, False):
        caches = [c.clone() for c in kv]
        if not native:
            impl._native_pass = lambda *a: False
        with pytest.raises(Exception) as error:
            impl.forward(None, q, k, v, caches, md, output=out)
        seen.append((type(error.value), str(error.value), [c.cpu() for c in caches]))
    assert seen[0][:2] == seen[1][:2]
    assert all(torch.equal(x, y) for x, y in zip(seen[0][2], seen[1][2]))
