"""Chunks of earlier ranks that a rank step refuses: another type, device, batch or number of heads
that does not divide, last dimension not contiguous (no launch reads them)."""
import pytest
import torch

import ring_swa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("packed", [False, True], ids=["dense", "packed"])
@pytest.mark.parametrize("bad", ["fp32", "cpu", "batch", "dim", "strides"])
def test_chunks_of_another_kind_are_refused(packed, bad):
    s, hq, hk, d, b = 128, 4, 2, 64, 1 if packed else 2
    q, k, v = (torch.randn(b, s, h, d, device="cuda").bfloat16() for h in (hq, hk, hk))
    good = torch.randn(2, b, s, hk, d, device="cuda").bfloat16()
    prev = {"fp32": good.float(), "cpu": good.cpu(), "dim": good[..., :32],
            "batch": torch.cat([good, good], 1) if packed else good[:, :1],
            "strides": good.transpose(3, 4).contiguous().transpose(3, 4)}[bad]
    if packed:
        q, k, v, good = q[0], k[0], v[0], good[:, 0]
        prev = prev[:, 0] if bad != "batch" else prev  # (a dimension too many)
    with pytest.raises((AssertionError, RuntimeError, IndexError)):
        if packed:
            ring_swa.ring_rank_share_attn_varlen(q, k, v, [good, prev], s + 30, [0, 4 * s], 4, 2)
        else:
            ring_swa.ring_rank_share_attn(q, k, v, [good, prev], s + 30, 4, 2)
