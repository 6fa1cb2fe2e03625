"""The block-float-8 encoder at every shared exponent: elements of the group's own exponent and of those below it (ties,
the magnitude that rounds to 128, what is shifted out), zeros and subnormals, both sides of the line from which the encoder works
in floats, infinities and NaN.  Bytes and exponents equal the integer rule's."""

import numpy as np
import pytest
import torch

import __graft_entry__ as entry
from oracle import bfp8_codec as C

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _pkg():
    entry.ensure_built()
    import tt_xla_amd  # noqa: F401


def _groups(exponent, n):
    """[n, 16] bfloat16 bit patterns whose largest exponent field is `exponent`."""
    r = np.random.default_rng(exponent)
    ex = np.maximum(exponent - r.integers(0, 12, (n, 16)), 0)
    ex[r.random((n, 16)) < 0.05] = 0
    ex[np.arange(n), r.integers(0, 16, n)] = exponent
    frac = r.integers(0, 128, (n, 16))
    frac[r.random((n, 16)) < 0.1] = 127
    frac[r.random((n, 16)) < 0.1] = 0
    return (r.integers(0, 2, (n, 16)) << 15 | ex << 7 | frac).astype(np.uint16)


def _integers(bits):
    """The codec's rule for bit patterns of any exponent (it refuses infinities and NaN): bytes, exponents."""
    b = bits.astype(np.int64)
    ex = b >> 7 & 0xFF
    e = ex.max(-1, keepdims=True)
    sig, sh = np.where(ex == 0, 0, 128 | b & 127), np.minimum(e - ex + 1, 16)
    q, rem, half = sig >> sh, sig & (1 << sh) - 1, 1 << sh - 1
    m = np.minimum(q + ((rem > half) | (rem == half) & (q & 1 == 1)), 127)
    return np.where(b >> 15, 128 - m, 128 + m), e[:, 0]


def test_every_exponent():
    from tt_xla_amd import custom_ops as ops

    n = 128
    bits = np.concatenate([_groups(e, n) for e in range(256)])
    byte, exps = _integers(bits)
    x = torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16)
    finite = C.quantize(x[: 255 * n])
    assert np.array_equal(finite[0], byte[: 255 * n]) and np.array_equal(finite[1][:, 0], exps[: 255 * n])
    rows = x.reshape(256, 1, 16, 128)  # 128 groups: 16 rows of 8
    got = ops.bfp8_pack_cache(rows.cuda()).cpu().numpy().reshape(256, 17 * 128)
    assert np.array_equal(got[:, : 16 * 128].reshape(-1, 16), byte)
    assert np.array_equal(got[:, 16 * 128 :].reshape(-1), exps)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_cache_writes(d):
    """The same through the fill and the update, beside the packed cache's bytes."""
    from tt_xla_amd import custom_ops as ops

    bits = np.concatenate([_groups(e, 2 * d // 16) for e in range(256)])
    x = torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).view(1, 1, 512, d).cuda()
    want = ops.bfp8_pack_cache(x.view(16, 1, 32, d))
    table = torch.arange(16, dtype=torch.int32, device="cuda").view(1, 16)
    for write in (
        lambda c: torch.ops.tt.paged_fill_cache_(c, x, table, torch.zeros(1, dtype=torch.int32, device="cuda")),
        lambda c: torch.ops.tt.paged_update_cache_(
            c, x.view(1, 512, 1, d), torch.arange(512, dtype=torch.int32, device="cuda"), table.expand(512, 16).contiguous()),
    ):
        cache = torch.zeros_like(want)
        write(cache)
        assert torch.equal(cache, want)
