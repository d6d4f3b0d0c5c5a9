"""Blocks of the dK/dV kernel whose four waves share out the walk over the query tiles (64 keys per
block, partial sums added in LDS): launches small enough to take that form, at the edges of its
tiles and of the way the walk is dealt -- key counts around 64 and 256, fewer query tiles than waves,
a wave without any step, group sizes 1, 2, 3, 4, 6 and 8 -- against the fp32 oracle to the relative norm
that the 16-bit P and dS allow (their rounding alone gives 2.5e-3)."""
import pytest
import torch

from oracle import attention_oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # (B, Sq, Sk, Hq, Hkv, D, window, causal)
    (1, 33, 33, 1, 1, 128, (40, 0), True),        # two query tiles for four waves
    (1, 64, 64, 2, 1, 64, (-1, -1), False),       # exactly one block
    (2, 65, 65, 4, 1, 128, (64, 0), True),        # one key in the second block
    (1, 255, 257, 3, 1, 128, (100, 0), True),     # odd group, ragged both ways
    (1, 7, 300, 6, 1, 64, (-1, 0), True),         # one query tile: waves 2 and 3 of a pair idle
    (1, 500, 63, 8, 2, 128, (-1, -1), False),     # fewer keys than a block
    (1, 130, 400, 6, 3, 128, (31, 0), True),      # leading keys that nobody sees
    (1, 1100, 1100, 28, 4, 128, (256, 0), True),  # group of 7
    (1, 1000, 1000, 4, 4, 64, (1, 0), True),
]


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 1e-2), (torch.float16, 1.3e-3)], ids=["bf16", "fp16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(x) for x in c))
def test_blocks_whose_waves_share_the_walk(case, dtype, tol):
    from ring_swa.ops import attn_bwd, attn_fwd

    b, sq, sk, hq, hk, d, window, causal = case
    g = torch.Generator().manual_seed(7)
    q, do = (torch.randn(b, sq, hq, d, generator=g).to(dtype) for _ in range(2))
    k, v = (torch.randn(b, sk, hk, d, generator=g).to(dtype) for _ in range(2))
    _, _, rq, rk, rv = O.attention_fwd_bwd(
        lambda q, k, v: O.window_attention(q, k, v, None, window, causal, 0), q, k, v, do)
    q, k, v, do = (t.cuda() for t in (q, k, v, do))
    out, lse = attn_fwd(q, k, v, None, window, causal)
    dq, dk, dv = (torch.full_like(t, float("nan")) for t in (q, k, v))
    attn_bwd(q, k, v, out, lse, do, dq, dk, dv, None, window, causal)
    for name, x, ref in (("dq", dq, rq), ("dk", dk, rk), ("dv", dv, rv)):
        err = ((x.float().cpu() - ref).norm() / ref.norm().clamp_min(1e-30)).item()
        assert err <= tol, f"{name}: relative norm {err}"


PACKS = [
    # (lengths, Hq, Hkv, D, window): the key tile table the statistics kernel writes and its search
    ([256] * 9, 8, 8, 128, 100),                      # whole tiles, all alike (blocks in snake order)
    ([512] * 6 + [77], 4, 4, 64, 300),                # alike but for the last
    ([0, 64, 0, 1, 700, 0, 129, 0], 4, 1, 128, 50),   # empty sequences everywhere
    ([1 + i % 3 for i in range(300)], 2, 1, 64, 8),   # more than 256 sequences: two passes of the scan
    ([40] * 64 + [41], 2, 2, 128, 64),                # 65 sequences: two levels of the search
    ([1024, 1000, 970, 300], 4, 4, 64, 2000),         # most tiles in fours: wide blocks in snake order
    ([1024, 300, 700], 4, 2, 128, 150),               # fewer: plain order
]


@pytest.mark.parametrize("case", PACKS, ids=lambda c: f"{len(c[0])}seq-{c[1]}x{c[2]}x{c[3]}-w{c[4]}")
def test_packs_by_their_key_tile_table(case):
    from ring_swa.ops import attn_bwd, attn_fwd

    lens, hq, hk, d, w = case
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    t = cu[-1]
    g = torch.Generator().manual_seed(8)
    q, do = (torch.randn(t, hq, d, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(t, hk, d, generator=g).bfloat16() for _ in range(2))
    _, _, rq, rk, rv = O.attention_fwd_bwd(
        lambda q, k, v: O.window_attention_varlen(q, k, v, cu, cu, None, (w, 0), True), q, k, v, do)
    q, k, v, do = (x.cuda() for x in (q, k, v, do))
    cu = torch.tensor(cu, dtype=torch.int32, device="cuda")
    out, lse = attn_fwd(q, k, v, None, (w, 0), True, cu, cu)
    dq, dk, dv = (torch.full_like(x, float("nan")) for x in (q, k, v))
    attn_bwd(q, k, v, out, lse, do, dq, dk, dv, None, (w, 0), True, cu, cu)
    for name, x, ref in (("dq", dq, rq), ("dk", dk, rk), ("dv", dv, rv)):
        err = ((x.float().cpu() - ref).norm() / ref.norm().clamp_min(1e-30)).item()
        assert err <= 1e-2, f"{name}: relative norm {err}"
