"""Where kv heads times batch is no multiple of 8, the XCDs that share a head take its tiles in turn: numbers of heads
that leave groups of 2, 4 and 8, of tiles that no group divides, fewer tiles than XCDs, against the oracle."""
import pytest
import torch

from gradcheck_util import GRAD_TOL, relnorm
from oracle import attention_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["wide", "short"])
@pytest.mark.parametrize("batch,rows,hq,hk,d,window", [
    (1, 40, 1, 1, 64, 300),      # one tile for eight XCDs
    (1, 1337, 1, 1, 128, 900),   # eight XCDs, one head
    (3, 515, 6, 2, 64, 5000),    # six heads: groups of four, one and a half heads each
    (1, 1100, 8, 4, 128, 600),   # pairs
    (1, 700, 12, 12, 64, 400),   # three heads for two XCDs
    (5, 130, 3, 1, 128, 64),     # five heads for eight
])
def test_tiles_taken_in_turn_match_the_oracle(batch, rows, hq, hk, d, window, form):
    from ring_swa.ops import attn_bwd, attn_fwd

    torch.manual_seed(rows)
    q, do = (torch.randn(batch, rows, hq, d).bfloat16() for _ in range(2))
    k, v = (torch.randn(batch, rows, hk, d).bfloat16() for _ in range(2))
    ref, _, *ref_grads = O.attention_fwd_bwd(
        lambda q, k, v: O.sliding_window_attn(q, k, v, window), q, k, v, do)
    x = [t.cuda() for t in (q, k, v)]
    out, lse = attn_fwd(*x, None, (window, 0), True)
    grads = [torch.full_like(t, float("nan")) for t in x]
    attn_bwd(*x, out, lse, do.cuda(), *grads, None, (window, 0), True, dkdv_form=form)
    # (16-bit results of fp32 sums: the bounds of the other parity tests)
    assert (out.float().cpu() - ref).abs().max() <= 2e-2
    for got, want in zip(grads, ref_grads):
        assert relnorm(got, want) <= GRAD_TOL


@pytest.mark.parametrize("hq,hk", [(2, 1), (12, 12), (10, 2)])
def test_a_pack_equals_its_sequences(hq, hk):
    """... and a pack's, whose tiles the device counts, the bits of the sequences one by one."""
    from ring_swa.ops import attn_bwd, attn_fwd

    lens, window, d = [700, 1, 333, 64, 65, 900], 350, 64
    torch.manual_seed(hq)
    cu = torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
    q, do = (torch.randn(sum(lens), hq, d, device="cuda").bfloat16() for _ in range(2))
    k, v = (torch.randn(sum(lens), hk, d, device="cuda").bfloat16() for _ in range(2))

    def run(q, k, v, do, *cu):
        out, lse = attn_fwd(q, k, v, None, (window, 0), True, *cu)
        grads = [torch.full_like(x, float("nan")) for x in (q, k, v)]
        attn_bwd(q, k, v, out, lse, do, *grads, None, (window, 0), True, *cu, dkdv_form="short")
        return [out, *grads]

    packed, at = run(q, k, v, do, cu, cu), 0
    for n in lens:
        alone = run(*(t[at:at + n].unsqueeze(0) for t in (q, k, v, do)))
        for x, y in zip(packed, alone):
            assert torch.equal(x[at:at + n], y[0])
        at += n
