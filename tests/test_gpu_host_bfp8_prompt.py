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
