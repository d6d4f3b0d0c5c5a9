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
