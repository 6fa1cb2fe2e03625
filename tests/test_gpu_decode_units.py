"""Decode where the leading unit per segment depends on the length of the tile list (the 16x16 matrix kernel): lists that
just fill the ranges and just do not, users without tokens, 64 and 65 users, a window; against the oracle's tolerance, and
against the same step with the unit forced on, which cuts the list elsewhere."""

import pytest
import torch

import test_gpu_decode as D
from oracle import paged_ops as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    D.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("hq,hkv,d,bs,pos", [
    (32, 8, 128, 64, [3071]), (32, 8, 128, 64, [3072]), (8, 2, 64, 32, [233, -1, 1960, 0]), (4, 4, 64, 64, [6143, 6143]),
    (4, 4, 64, 64, [6143, 6144]), (16, 8, 256, 32, [1535]), (16, 8, 256, 32, [1536]),
    (8, 2, 128, 64, [20 + 7 * i for i in range(64)]), (8, 2, 128, 64, [20 + 7 * i for i in range(65)]),
])
def test_unit_follows_the_list(hq, hkv, d, bs, pos, monkeypatch):
    gen = torch.Generator().manual_seed(hq + d + len(pos) + max(pos))
    users, width = len(pos), max(pos) // bs + 1
    k = torch.randn(width * 2, hkv, bs, d, generator=gen).to(torch.bfloat16)
    v = torch.randn(width * 2, hkv, bs, d, generator=gen).to(torch.bfloat16)
    table = torch.randint(0, width * 2, (users, width), generator=gen).to(torch.int32)
    q = torch.randn(1, users, hq, d, generator=gen).to(torch.bfloat16)
    cur = torch.tensor(pos, dtype=torch.int32)
    print(f"units h{hq}x{hkv} d{d} users{users} longest{max(pos)}", flush=True)

    def step():
        return torch.ops.tt.paged_scaled_dot_product_attention_decode(
            q.cuda(), k.cuda(), v.cuda(), table.cuda(), is_causal=True, cur_pos_tensor=cur.cuda(), scale=d**-0.5).cpu()

    got = step()
    monkeypatch.setenv("TTPA_DECODE_SEG_UNITS", "1")
    forced = step()
    live = [u for u, p in enumerate(pos) if p >= 0]
    assert got[:, [u for u in range(users) if u not in live]].isnan().all()
    want = O.paged_sdpa_decode(q[:, live], k, v, table[live], True, None, cur[live], None, d**-0.5)
    for t in (got, forced):
        torch.testing.assert_close(t[:, live].float(), want.float(), atol=2e-2, rtol=2e-2)
