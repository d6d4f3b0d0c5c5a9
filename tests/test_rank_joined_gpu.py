"""A rank step whose window reaches over several earlier chunks, or over one whose size the two-range
pass does not take, runs as one band over the joined keys; large steps of two blocks run block by block,
ring_dtypes in the ring's accumulators: those routes run here, too.  All ranks' shares against the oracle on
the whole sequence (out <= 2e-2 max-abs, gradients <= 1e-2 relative norm), odd chunk sizes, windows at
and around multiples of a chunk, batch 2, a pack whose sequences start anywhere, and held chunks
beyond the window's reach, whose gradient is zero."""
import pytest
import torch

from oracle import attention_oracle as O

pytestmark = pytest.mark.gpu
CP = 4


def _rel(x, ref):
    return ((x - ref).norm() / ref.norm().clamp_min(1e-30)).item()


@pytest.mark.parametrize("s,w", [(100, 30), (100, 100), (100, 101), (193, 400), (64, 1000), (256, 511)])
@pytest.mark.parametrize("packed", [False, True], ids=["dense", "packed"])
@pytest.mark.parametrize("route", ["joined", "blocks", "ring_dtypes"])
def test_shares_on_joined_keys_match_the_oracle(monkeypatch, s, w, packed, route):
    import ring_swa
    from ring_swa import rank_share

    joined, real = [], rank_share._join_keys
    monkeypatch.setattr(rank_share, "_join_keys", lambda *a: joined.append(1) or real(*a))
    if route == "blocks":
        monkeypatch.setattr(rank_share, "_joinable", lambda *a: False)
    hq, hk, d, total = 4, 2, 64, s * CP
    b = 1 if packed else 2
    cu = [0, s // 2, s // 2 + 1, 2 * s + 7, total]
    g = torch.Generator().manual_seed(31)
    q, do = (torch.randn(b, total, hq, d, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(b, total, hk, d, generator=g).bfloat16() for _ in range(2))
    if packed:
        ro, _, rq, rk, rv = O.attention_fwd_bwd(
            lambda q, k, v: O.window_attention_varlen(q, k, v, cu, cu, None, (w, 0), True),
            q[0], k[0], v[0], do[0])
        ro, rq, rk, rv = (t[None] for t in (ro, rq, rk, rv))
    else:
        ro, _, rq, rk, rv = O.attention_fwd_bwd(lambda q, k, v: O.sliding_window_attn(q, k, v, w), q, k, v, do)
    outs, dqs = [], []
    dk, dv = torch.zeros(b, total, hk, d), torch.zeros(b, total, hk, d)
    for r in range(CP):
        sl = slice(r * s, (r + 1) * s)
        own = [t[:, sl].cuda() for t in (q, k, v)]
        prev = [torch.stack([t[:, (r - i) * s:(r - i + 1) * s] for t in (k, v)]).cuda() for i in range(1, r + 1)]
        if packed:
            own, prev = [t[0] for t in own], [t[:, 0] for t in prev]
        own, prev = [t.requires_grad_() for t in own], [t.requires_grad_() for t in prev]
        kw = dict(ring_dtypes=route == "ring_dtypes")
        if packed:
            out = ring_swa.ring_rank_share_attn_varlen(*own, prev, w, cu, CP, r, **kw)
        else:
            out = ring_swa.ring_rank_share_attn(*own, prev, w, CP, r, **kw)
        with torch.no_grad():  # (joins two blocks more seldom)
            if packed:
                alone = ring_swa.ring_rank_share_attn_varlen(*own, prev, w, cu, CP, r, **kw)
            else:
                alone = ring_swa.ring_rank_share_attn(*own, prev, w, CP, r, **kw)
        want = ro[:, sl] if not packed else ro[0, sl]
        assert (alone.float().cpu() - want).abs().max().item() <= 2e-2
        grads = torch.autograd.grad(out, own + prev, do[:, sl].cuda() if not packed else do[0, sl].cuda())
        cpu = [x.float().cpu() for x in (out.detach(), *grads)]
        if packed:
            cpu = [x[None] for x in cpu[:4]] + [x[:, None] for x in cpu[4:]]
        outs.append(cpu[0])
        dqs.append(cpu[1])
        dk[:, sl] += cpu[2]
        dv[:, sl] += cpu[3]
        for i, p in enumerate(cpu[4:], 1):
            ps = slice((r - i) * s, (r - i + 1) * s)
            dk[:, ps] += p[0]
            dv[:, ps] += p[1]
            if (i - 1) * s >= w:
                assert not p.any()
    assert (torch.cat(outs, 1) - ro).abs().max().item() <= 2e-2
    assert bool(joined) == (route == "joined")
    errs = [_rel(torch.cat(dqs, 1), rq), _rel(dk, rk), _rel(dv, rv)]
    assert max(errs) <= 1e-2, f"dq / dk / dv relative norm {errs}"


@pytest.mark.parametrize("packed", [False, True], ids=["dense", "packed"])
def test_gradients_are_contiguous_tensors_of_their_inputs_type(packed):
    """Also the chunks': each a tensor of its own (a ring sends it on its way back), a chunk beyond the
    reach whatever its type."""
    import ring_swa

    s, w, hq, hk, d, b = 100, 130, 4, 2, 64, 1 if packed else 2
    g = torch.Generator().manual_seed(1)
    q, k, v, do = (torch.randn(b, s, h, d, generator=g).bfloat16().cuda() for h in (hq, hk, hk, hq))
    prev = [torch.randn(2, b, s, hk, d, generator=g).to(t).cuda() for t in (torch.bfloat16, torch.bfloat16, torch.float32)]
    if packed:
        q, k, v, do, prev = q[0], k[0], v[0], do[0], [p[:, 0] for p in prev]
    leaves = [t.contiguous().requires_grad_() for t in (q, k, v, *prev)]
    if packed:
        out = ring_swa.ring_rank_share_attn_varlen(*leaves[:3], leaves[3:], w, [0, 4 * s], 4, 3)
    else:
        out = ring_swa.ring_rank_share_attn(*leaves[:3], leaves[3:], w, 4, 3)
    grads = torch.autograd.grad(out, leaves, do)
    for t, x in zip(leaves, grads):
        assert x.is_contiguous() and x.dtype == t.dtype and x.shape == t.shape
    chunks = [x.untyped_storage().data_ptr() for x in grads[3:]]
    assert len(set(chunks)) == 3 and not set(chunks) & {x.untyped_storage().data_ptr() for x in grads[:3]}
