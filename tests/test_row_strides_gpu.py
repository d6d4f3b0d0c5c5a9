"""Rows closer together than their own bytes: the gradient of a sum over the rows (an expand, row stride 0), rows
that overlap.  The same bits as from contiguous copies, in both forms of the dK/dV kernel and both ways of addressing."""
import pytest
import torch

from gradcheck_util import GRAD_TOL, relnorm
from oracle import attention_oracle as O

pytestmark = pytest.mark.gpu


def _rows(shape, stride, seed):
    """N(0, 1) rows [.., rows, heads, dim] that start `stride` elements after each other (0: all the same)."""
    *lead, rows, heads, dim = shape
    g = torch.Generator(device="cuda").manual_seed(seed)
    head = (rows - 1) * stride + dim
    x = torch.randn(*lead, heads, head + -head % 8, device="cuda", generator=g).bfloat16()
    st = x.stride()
    return x.as_strided(shape, (*st[:-2], stride, st[-2], 1))


@pytest.mark.parametrize("addressing", ["auto", "far"])
@pytest.mark.parametrize("form", ["wide", "short"])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("rows,hq,hk,d,q_stride,do_stride", [
    (200, 4, 1, 128, None, 0),   # one head a wave, several tiles
    (200, 4, 1, 64, None, 0),
    (333, 2, 2, 128, None, 64),  # query tiles dealt to the waves; less than 1024 bytes per load
    (97, 2, 2, 64, 8, 0),        # q's rows overlap, too
    (97, 6, 3, 128, 120, 8),
    (1, 4, 4, 128, 0, 0),        # a stride that no row uses
])
@pytest.mark.parametrize("route", [{}, {"num_sink": 3}, {"handoff": True}], ids=["plain", "sinks", "handoff"])
def test_short_row_strides_equal_contiguous_rows(rows, hq, hk, d, q_stride, do_stride, route, packed, form, addressing,
                                                   monkeypatch):
    from ring_swa.ops import attn_bwd, attn_fwd

    if addressing == "far":
        monkeypatch.setenv("RSWA_ADDRESSING", "far")
    lead = () if packed else (2,)
    g = torch.Generator(device="cuda").manual_seed(rows)
    k, v = (torch.randn(*lead, rows, hk, d, device="cuda", generator=g).bfloat16() for _ in range(2))
    shape = (*lead, rows, hq, d)
    q = torch.randn(shape, device="cuda", generator=g).bfloat16() if q_stride is None else _rows(shape, q_stride, 1)
    do = _rows(shape, do_stride, 2)
    cu = [torch.tensor(sorted({0, rows // 3, rows}), device="cuda", dtype=torch.int32)] * 2 if packed else []

    def run(q, do):
        out, lse = attn_fwd(q, k, v, None, (50, 0), True, *cu, num_sink=route.get("num_sink", 0))
        grads = [torch.full_like(t, float("nan"), memory_format=torch.contiguous_format) for t in (q, k, v)]
        attn_bwd(q, k, v, out, lse, do, *grads, None, (50, 0), True, *cu, dkdv_form=form, **route)
        return [out, *grads]

    for got, want in zip(run(q, do), run(q.contiguous(), do.contiguous())):
        assert torch.equal(got, want) and not torch.isnan(got).any()


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("d", [64, 128])
def test_gradient_of_a_sum_over_the_rows(d, packed):
    """... through the entry points and autograd, against the oracle."""
    import ring_swa

    rows, hq, hk, w = 333, 4, 2, 100
    torch.manual_seed(d)
    q, k, v = (torch.randn(1, rows, h, d).bfloat16() for h in (hq, hk, hk))
    weight = torch.randn(1, 1, hq, d).bfloat16()
    ref, _, *ref_grads = O.attention_fwd_bwd(lambda q, k, v: O.sliding_window_attn(q, k, v, w), q, k, v,
                                             weight.expand(1, rows, hq, d))
    x = [(t[0] if packed else t).cuda().requires_grad_() for t in (q, k, v)]
    if packed:
        cu = torch.tensor([0, rows], device="cuda", dtype=torch.int32)
        out = ring_swa.ring_sliding_window_attn_varlen(*x, w, cu)
        total = out.sum(0, keepdim=True)
    else:
        out = ring_swa.ring_sliding_window_attn(*x, w)
        total = out.sum(1, keepdim=True)
    grads = torch.autograd.grad(total, x, (weight[0] if packed else weight).cuda())
    for got, want in zip(grads, ref_grads):
        assert relnorm(got, want[0] if packed else want) <= GRAD_TOL
