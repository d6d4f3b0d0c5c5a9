"""A block's walk over its key tiles starts at a tile that its neighbours start at, too, and wraps around:
walks of few tiles and many, of numbers that are no power of two, with sink tiles ahead of them, in 64- and
128-row blocks, with and without skipped tiles, against the oracle."""
import pytest
import torch

from gradcheck_util import GRAD_TOL, relnorm
from oracle import attention_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,window,hq,hk,d,sinks", [
    (321, 1, 1, 1, 128, 0),      # walks of 2 and 3 tiles
    (700, 64, 2, 2, 64, 0),      # of 3 and 4
    (900, 190, 4, 2, 128, 4),    # pairs of heads, sink tiles ahead
    (1300, 447, 3, 3, 64, 70),   # sinks beyond one tile
    (2100, 1000, 3, 1, 128, 0),  # 18 and 19 tiles
    (2200, 1055, 2, 1, 128, 1),  # 17 and 18 tiles
])
def test_wrapped_walks_match_the_oracle(rows, window, hq, hk, d, sinks):
    import ring_swa

    torch.manual_seed(rows)
    q, do = (torch.randn(1, rows, hq, d).bfloat16() for _ in range(2))
    k, v = (torch.randn(1, rows, hk, d).bfloat16() for _ in range(2))
    if sinks:
        ref_fn = lambda q, k, v: O.streaming_llm_attn(q, k, v, window, n_sink=sinks)
        fn = lambda q, k, v: ring_swa.ring_streaming_llm_attn(q, k, v, window, num_sink_tokens=sinks)
    else:
        ref_fn = lambda q, k, v: O.sliding_window_attn(q, k, v, window)
        fn = lambda q, k, v: ring_swa.ring_sliding_window_attn(q, k, v, window)
    ref, _, *ref_grads = O.attention_fwd_bwd(ref_fn, q, k, v, do)
    x = [t.cuda().requires_grad_() for t in (q, k, v)]
    out = fn(*x)
    grads = torch.autograd.grad(out, x, do.cuda())
    # (16-bit results of fp32 sums: the bounds of the other parity tests)
    assert (out.float().cpu() - ref).abs().max() <= 2e-2
    for got, want in zip(grads, ref_grads):
        assert relnorm(got, want) <= GRAD_TOL


def _run(q, k, v, do, window, *cu):
    from ring_swa.ops import attn_bwd, attn_fwd

    out, lse = attn_fwd(q, k, v, None, (window, 0), True, *cu)
    grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    attn_bwd(q, k, v, out, lse, do, *grads, None, (window, 0), True, *cu)
    return out, lse, grads[0]


def _inputs(rows, hq, hk, d):
    g = torch.Generator(device="cuda").manual_seed(rows)
    return [torch.randn(1, rows, h, d, device="cuda", generator=g).bfloat16() for h in (hq, hk, hk, hq)]


@pytest.mark.parametrize("window,d", [(350, 128), (447, 64), (1000, 128), (1950, 128), (1950, 64)])
def test_rows_have_the_same_bits_in_blocks_of_64_and_of_128(window, d):
    """Pairs of q heads come in blocks of 64 rows (forward; dQ), single ones in blocks of 128."""
    q, k, v, do = _inputs(4100, 2, 1, d)
    out, lse, dq = _run(q, k, v, do, window)
    for h in range(2):
        x, y, z = _run(q[:, :, h:h + 1], k, v, do[:, :, h:h + 1], window)
        assert torch.equal(x, out[:, :, h:h + 1]) and torch.equal(y, lse[:, h:h + 1])
        assert torch.equal(z, dq[:, :, h:h + 1])


@pytest.mark.parametrize("hq", [1, 2])
def test_rows_of_short_calls_and_of_long_ones_have_the_same_bits(hq):
    """Above 3200 keys a row on average dQ takes blocks of twice as many rows: a call's first rows alone, and in a pack."""
    window = 4000
    q, k, v, do = _inputs(14000, hq, 1, 128)
    whole = _run(q, k, v, do, window)
    first = _run(*(t[:, :8000] for t in (q, k, v, do)), window)
    cu = torch.tensor([0, 8000, 11000, 14000], device="cuda", dtype=torch.int32)
    pack = _run(*(t[0] for t in (q, k, v, do)), window, cu, cu)
    for a, b, c, dim in zip(whole, first, pack, (1, 2, 1)):
        assert torch.equal(a.narrow(dim, 0, 8000), b)
        assert torch.equal(c.narrow(dim - 1, 0, 8000), b[0])
