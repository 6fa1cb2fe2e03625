"""Prefill through the C entry point into output rows that lie in descending order (a negative token stride), which the streaming
kernel's 32-bit row distances cannot express: the rows are those of an ascending output, and nothing else is written.  Both calls run the
plain loop, so the bits are the same."""

import pytest
import torch

import test_gpu_prefill as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    P.entry.ensure_built()
    import tt_xla_amd  # noqa: F401


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_descending_output_rows(d, paged, monkeypatch):
    from tt_xla_amd import _native as N

    b, hq, hkv, s, bs, start = 2, 4, 2, 96, 32, 64 if paged else 0
    g = torch.Generator().manual_seed(d)
    q = P._bf(g, b, hq, s, d).cuda()
    if paged:
        k, v, table = (t.cuda() for t in P._paged(g, b, (start + s) // bs, hkv, bs, d, False))
        at = torch.tensor([start], dtype=torch.int32, device="cuda")
        operands = (k.data_ptr(), v.data_ptr(), 0, 0, 0, table.data_ptr(), table.stride(0), at.data_ptr())
        sizes = (0, d, bs, table.shape[1], k.shape[0])
    else:
        k, v = P._bf(g, b, hkv, s, d).cuda(), P._bf(g, b, hkv, s, d).cuda()
        operands = (k.data_ptr(), v.data_ptr(), hkv * s * d, s * d, d, None, 0, None)
        sizes = (s, d, 0, 0, 0)
    out = torch.full((b, s + 2, hq, d), 7.0, dtype=torch.bfloat16, device="cuda")  # a row in front and one behind

    def run(first_row, token_stride):
        out.fill_(7.0)
        N.call("ttpa_sdpa_prefill", out[0, first_row].data_ptr(), (s + 2) * hq * d, d, token_stride, q.data_ptr(), hq * s * d, s * d, d,
               *operands, None, 0, 0, b, hq, hkv, s, *sizes, 1, d**-0.5, torch.cuda.current_stream().cuda_stream)
        return out.clone()

    down = run(s, -hq * d)
    monkeypatch.setenv("TTPA_PREFILL_STREAM", "0")
    up = run(1, hq * d)
    assert torch.equal(down[:, 1:-1].flip(1), up[:, 1:-1])
    assert (down[:, [0, -1]] == 7.0).all()
