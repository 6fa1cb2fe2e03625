"""The bfloat16 copies that a block-float-8 chunk pass reads, all of them, at the sizes where their launch's split can go wrong: slabs of two
pieces and of many, one and odd numbers of KV heads, fewer pieces than wavefronts and several rounds of them, table columns that the pass
does not read, entries out of range.  The decode is exact: the copies equal the codec's."""

import pytest
import torch

import __graft_entry__ as entry
from oracle import bfp8_codec as C

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("users,hq,hkv,d,bs,nbpu,start,lc", [
    (1, 4, 1, 128, 32, 2, 0, 64), (3, 24, 3, 128, 32, 9, 64, 160), (2, 40, 5, 128, 96, 7, 480, 192), (4, 32, 8, 128, 64, 40, 1216, 128),
    (2, 32, 8, 128, 64, 75, 4672, 128), (8, 64, 8, 64, 32, 12, 96, 256), (1, 24, 3, 64, 160, 8, 640, 1024 - 640), (8, 64, 8, 64, 64, 24, 1024, 256),
])
def test_copies(users, hq, hkv, d, bs, nbpu, start, lc):
    from tt_xla_amd import _native as N
    from tt_xla_amd import custom_ops as ops

    g = torch.Generator().manual_seed(users + hkv + bs + start)
    nb = users * nbpu + 1
    caches = [ops.bfp8_pack_cache(torch.randn(nb, hkv, bs, d, generator=g).to(torch.bfloat16).cuda()) for _ in range(2)]
    table = (torch.randperm(nb - 1, generator=g) + 1).view(users, nbpu).to(torch.int32)
    table[users - 1, 0], table[0, (start + lc - 1) // bs] = nb + 5, -1
    q, cs = torch.randn(users, hq, lc, d, generator=g).to(torch.bfloat16).cuda(), torch.tensor([start], dtype=torch.int32).cuda()
    need = int(N.lib().ttpa_sdpa_prefill_workspace_bytes(users, hkv, d, bs, nbpu, N.KV_BFP8))
    ws, out, tb = torch.full((need,), 0xAB, dtype=torch.uint8, device="cuda"), torch.empty_like(q), table.cuda()
    N.call("ttpa_sdpa_prefill_expanded", out.data_ptr(), out.stride(0), out.stride(1), out.stride(2),
           q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), caches[0].data_ptr(), caches[1].data_ptr(), 0, 0, 0,
           tb.data_ptr(), tb.stride(0), cs.data_ptr(), 0, 0, 0, users, hq, hkv, lc, nbpu * bs, d, bs, nbpu, nb, 1,
           d ** -0.5, 0, N.KV_BFP8, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    cols, size = -(-(start + lc) // bs), users * nbpu * hkv * bs * d * 2
    from_block = torch.where((table < 0) | (table >= nb), 0, table).long()
    for n, cache in enumerate(caches):
        copies = ws[n * size : (n + 1) * size].view(users, nbpu, -1).cpu()
        want = C.unpack_cache(cache.cpu(), bs).to(torch.bfloat16)[from_block].view(torch.uint8).view(users, nbpu, -1)
        assert torch.equal(copies[:, :cols], want[:, :cols])
        assert (copies[:, cols:] == 0xAB).all(), "columns that the pass does not read"
    identity = torch.arange(users * nbpu, dtype=torch.int32).view(users, nbpu)
    assert torch.equal(ws[2 * size : 2 * size + 4 * users * nbpu].view(torch.int32).view(users, nbpu).cpu()[:, :cols], identity[:, :cols])
