"""Gradients of sink keys, whose rows a kernel of its own computes in tiles of 16 rows: sequences of a
tile, one row more and less, one chunk and several, one sink per wave and two, more sinks than a pass."""
import pytest
import torch

from oracle import attention_oracle as O
from tests.gradcheck_util import GRAD_TOL, relnorm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("lens,hq,hk,window,sinks", [
    ([1, 15, 16, 17, 0, 33], 3, 1, 4, 1), ([1, 2, 3, 40], 4, 4, 0, 2), ([130, 64, 5], 8, 2, 10, 3),
    ([700], 4, 1, 50, 4), ([515, 520], 2, 2, 30, 5), ([900, 20], 6, 2, 100, 9), ([2100], 4, 2, 64, 1),
])
def test_sink_rows(lens, hq, hk, window, sinks, d, dtype):
    from ring_swa.ops import attn_bwd, attn_fwd
    from ring_swa.ops.band_attn import bwd_workspace_bytes

    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    torch.manual_seed(sum(lens))
    q, do = (torch.randn(cu[-1], hq, d, device="cuda", dtype=dtype) for _ in range(2))
    k, v = (torch.randn(cu[-1], hk, d, device="cuda", dtype=dtype) for _ in range(2))
    cud = torch.tensor(cu, dtype=torch.int32, device="cuda")
    out, lse = attn_fwd(q, k, v, None, (window, 0), True, cud, cud, num_sink=sinks)
    ws = torch.full((bwd_workspace_bytes(q, k, cud, cud, window_size=(window, 0), causal=True, num_sink=sinks),), 255,
                    dtype=torch.uint8, device="cuda")
    got = []
    for _ in range(2):  # (twice on one workspace: the arrival counters are left at zero)
        g = [torch.full_like(x, float("nan")) for x in (q, k, v)]
        attn_bwd(q, k, v, out, lse, do, *g, None, (window, 0), True, cud, cud, num_sink=sinks, workspace=ws)
        got.append(g)
    _, _, rq, rk, rv = O.attention_fwd_bwd(
        lambda q, k, v: O.streaming_llm_attn_varlen(q, k, v, window, cu, n_sink=sinks), q, k, v, do)
    for x, again, r in zip(*got, (rq, rk, rv)):
        assert torch.equal(x, again)
        assert relnorm(x, r) <= GRAD_TOL
    at = torch.tensor([c + j for c, n in zip(cu, lens) for j in range(min(sinks, n))])
    for x, r in ((got[0][1], rk), (got[0][2], rv)):  # (and by themselves, so that no other row hides one)
        assert relnorm(x[at.cuda()], r[at]) <= GRAD_TOL


@pytest.mark.parametrize("n", [15, 16, 17, 47])
@pytest.mark.parametrize("sinks", [1, 3])
def test_an_infinity_in_the_last_row_stays_one(n, sinks):
    """dV of a key is sum P dO: an infinite dO of the last row makes it infinite in that column and leaves the
    others.  (The lanes of a tile that stand for rows past the end have P = 0, which must not meet it.)"""
    from ring_swa.ops import attn_bwd, attn_fwd

    torch.manual_seed(n)
    q, do = (torch.randn(1, n, 4, 64, device="cuda").bfloat16() for _ in range(2))
    k, v = (torch.randn(1, n, 2, 64, device="cuda").bfloat16() for _ in range(2))
    out, lse = attn_fwd(q, k, v, None, (4, 0), True, num_sink=sinks)

    def dv_of(do):
        g = [torch.empty_like(x) for x in (q, k, v)]
        attn_bwd(q, k, v, out, lse, do, *g, None, (4, 0), True, num_sink=sinks)
        return g[2]

    want = dv_of(do)
    do[0, -1, 0, 3] = float("inf")
    got = dv_of(do)
    assert (got[0, :sinks, 0, 3] == float("inf")).all()
    want[0, :, 0, 3] = got[0, :, 0, 3] = 0
    assert torch.equal(got[0, :sinks], want[0, :sinks])


@pytest.mark.parametrize("d", [64, 128])
def test_sink_rows_with_less_workspace(d):
    """Without room for a pack's key tile table the sums are chunked as with it: the same bits (fp16 and many
    sinks, so that sums in another order show: in 95 values with head_dim 128).  With the least workspace
    they are not: held to the oracle."""
    from ring_swa import _lib
    from ring_swa.ops import attn_bwd, attn_fwd
    from ring_swa.ops.band_attn import _params, bwd_workspace_bytes

    cu, hq, hk, window, sinks = [0, 300, 300, 301, 901, 1500], 4, 2, 100, 64
    torch.manual_seed(4)
    q, do = (torch.randn(cu[-1], hq, d, device="cuda", dtype=torch.float16) for _ in range(2))
    k, v = (torch.randn(cu[-1], hk, d, device="cuda", dtype=torch.float16) for _ in range(2))
    cud = torch.tensor(cu, dtype=torch.int32, device="cuda")
    out, lse = attn_fwd(q, k, v, None, (window, 0), True, cud, cud, num_sink=sinks)
    need = bwd_workspace_bytes(q, k, cud, cud, window_size=(window, 0), causal=True, num_sink=sinks)
    table = (len(cu) + 1) * 4  # the last thing in it
    p = _params(q, k, v, 1., (window, 0), True, cud, cud, sinks)
    least = _lib.lib().rswa_attn_bwd_workspace_min_bytes(p)
    assert least < need - table
    got = []
    for room in (need, need - table, need - table - 256, least):
        ws = torch.full((room,), 255, dtype=torch.uint8, device="cuda")
        g = [torch.full_like(x, float("nan")) for x in (q, k, v)]
        attn_bwd(q, k, v, out, lse, do, *g, None, (window, 0), True, cud, cud, num_sink=sinks, workspace=ws)
        got.append(g)
    for x, same in zip(*got[:2]):
        assert torch.equal(x, same)
    _, _, *ref = O.attention_fwd_bwd(
        lambda q, k, v: O.streaming_llm_attn_varlen(q, k, v, window, cu, n_sink=sinks), q, k, v, do)
    for g in got:
        for x, r in zip(g, ref):
            assert relnorm(x, r) <= GRAD_TOL
