"""The cache rows that a dense prefill writes beside its attention, around the length up to which its workgroups take a quarter of their
passes (128 rows, but for head size 256) and those at which another workgroup starts (512, 256): copied bit for bit, and no others touched.  The
fill is the same on the plain loop, which takes the lengths that are no multiple of 32."""

import pytest
import torch

import test_gpu_prefill as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    P.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("keys", [1, 32, 63, 64, 65, 96, 127, 128, 129, 160, 255, 256, 257, 288, 383, 384, 385, 511, 512, 513, 640])
def test_rows(d, keys):
    users, heads, bs = 3, 2, 32
    print(f"fill rows d{d} keys{keys}", flush=True)
    g = torch.Generator().manual_seed(keys + d)
    q, k, v = P._bf(g, users, heads, 32, d), P._bf(g, users, heads, keys, d), P._bf(g, users, heads, keys, d)
    width = -(-keys // bs) + 1
    table = (torch.randperm(users * width, generator=g) + 1).view(users, width).to(torch.int32)
    caches = [torch.full((users * width + 1, heads, bs, d), x, dtype=torch.bfloat16) for x in (3.0, -3.0)]
    got = [c.cuda() for c in caches]
    out = torch.zeros(users, heads, 32, d, dtype=torch.bfloat16, device="cuda")
    torch.ops.tt.paged_fill_kv_prefill_out_(q.cuda(), k.cuda(), v.cuda(), *got, table.cuda(), torch.arange(users, dtype=torch.int32).cuda(), out, is_causal=False)
    for want, rows, have in zip(caches, (k, v), got):
        for u in range(users):
            for t in range(keys):
                want[int(table[u, t // bs]), :, t % bs] = rows[u, :, t]
        assert torch.equal(have.cpu(), want)
