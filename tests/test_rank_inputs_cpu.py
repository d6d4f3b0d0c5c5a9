"""What a rank step accepts: the joined-keys route copies keys and values, which would convert types
and broadcast shapes on the way, so only tensors that need neither take it.  Everything else goes to
the block route, whose checks refuse it (or which takes it as it is)."""
import pytest
import torch

import ring_swa
from ring_swa import rank_share as RS

S, HQ, HK, D = 64, 4, 2, 64


def _inputs(b=2):
    q = torch.randn(b, S, HQ, D).bfloat16()
    k, v = (torch.randn(b, S, HK, D).bfloat16() for _ in range(2))
    return q, k, v, [torch.randn(2, b, S, HK, D).bfloat16() for _ in range(2)]


def _joinable(q, k, v, prev, window=S + 30, rank=2, training=True, packed=False):
    s = q.shape[1]
    plan = RS.plan_nonvarlen(s, window, 4, rank)
    return RS._joinable(q, k, v, prev, plan, window, RS._reach(plan, s, window), training, packed)


def test_tensors_alike_are_joined():
    q, k, v, prev = _inputs()
    assert _joinable(q, k, v, prev)
    fused = torch.randn(2, S, HQ + 2 * HK, D).bfloat16()
    assert _joinable(fused[:, :, :HQ], fused[:, :, HQ:HQ + HK], fused[:, :, HQ + HK:], prev)
    # a chunk beyond the window's reach is not looked at
    assert not _joinable(q, k, v, prev[:1]) and _joinable(q, k, v, [prev[0], prev[1], prev[1].float()])


def test_what_the_copies_would_change_is_not_joined():
    q, k, v, prev = _inputs()
    shifted = torch.empty(prev[0].numel() + 4).bfloat16()[4:].view_as(prev[0])  # rows not 16-byte aligned
    for bad in (prev[1].float(), prev[1].half(), prev[1].to("meta"), prev[1][:, :1], prev[1][:, :, :, :1],
                prev[1][:, :, :S // 2], prev[1][..., :1], prev[1].transpose(3, 4).contiguous().transpose(3, 4),
                shifted):
        assert not _joinable(q, k, v, [prev[0], bad])
    for bad in (v.float(), v[:, :, :1], v[:1], v.transpose(2, 3).contiguous().transpose(2, 3)):
        assert not _joinable(q, k, bad, prev) and not _joinable(q, bad, bad if bad.shape != v.shape else v, prev)


@pytest.mark.parametrize("packed", [False, True], ids=["dense", "packed"])
def test_the_entry_points_refuse_values_of_another_kind(packed):
    """(The first block's checks come before the one for a GPU, so this runs without.)"""
    q, k, v, prev = _inputs(1)
    if packed:
        q, k, v, prev = q[0], k[0], v[0], [p[:, 0] for p in prev]
    for bad in (v.float(), v[..., :1, :]):
        with pytest.raises(AssertionError):
            if packed:
                ring_swa.ring_rank_share_attn_varlen(q, k, bad, prev, S + 30, [0, 4 * S], 4, 2)
            else:
                ring_swa.ring_rank_share_attn(q, k, bad, prev, S + 30, 4, 2)


@pytest.mark.parametrize("s,hq,hk,d,window,rank,joined", [
    (1000, 16, 4, 128, 1500, 1, True),      # two blocks, the host's launches are most of it
    (2048, 32, 8, 128, 1536, 1, True),
    (1000, 32, 32, 64, 250, 1, True),
    (8192, 8, 2, 128, 12288, 1, False),     # two launches fill the chip better than one
    (7379, 4, 4, 128, 10877, 1, False),
    (8000, 32, 8, 128, 7999, 1, True),      # even blocks, grouped heads
    (8000, 32, 32, 128, 7999, 1, False),
    (4096, 32, 8, 128, 10000, 3, True),     # four blocks, whatever the work
    (6000, 32, 32, 128, 15600, 3, True),
])
def test_two_blocks_are_joined_only_where_launches_are_the_time(s, hq, hk, d, window, rank, joined):
    q, k = torch.empty(1, s, hq, d, device="meta", dtype=torch.bfloat16), torch.empty(1, s, hk, d, device="meta", dtype=torch.bfloat16)
    prev = [torch.empty(2, 1, s, hk, d, device="meta", dtype=torch.bfloat16) for _ in range(rank)]
    assert _joinable(q, k, k, prev, window, rank) == joined


@pytest.mark.parametrize("s,hq,hk,window,dense,packed", [
    (2048, 28, 4, 1536, True, True), (2048, 32, 32, 2048, False, False), (1000, 8, 2, 250, False, True),
])
def test_a_forward_alone_joins_two_blocks_only_with_small_copies(s, hq, hk, window, dense, packed):
    q, k = (torch.empty(1, s, h, 128, device="meta", dtype=torch.bfloat16) for h in (hq, hk))
    prev = [torch.empty(2, 1, s, hk, 128, device="meta", dtype=torch.bfloat16)]
    assert _joinable(q, k, k, prev, window, 1, training=False) == dense
    assert _joinable(q, k, k, prev, window, 1, training=False, packed=True) == packed


@pytest.mark.parametrize("s,window,hops", [(64, 40, 1), (64, 128, 2), (1500, 2000, 2), (1500, 4500, 3)])
def test_joined_rows_are_the_reached_rows_in_order(s, window, hops):
    """Both ways of copying (one call per tensor for few elements, one per chunk for many)."""
    b, hk, d = 2, 4, 64
    rows = torch.randn(2, b, (hops + 1) * s, hk, d).bfloat16()
    prev = [rows[:, :, (hops - i) * s:(hops - i + 1) * s] for i in range(1, hops + 1)]
    k, v = rows[:, :, hops * s:]
    plan = RS.plan_nonvarlen(s, window, hops + 2, hops)
    reach = RS._reach(plan, s, window)
    kk, vv = RS._join_keys(k, v, prev, plan, reach)
    assert kk.shape[1] == reach + s == min(window, hops * s) + s
    assert torch.equal(kk, rows[0, :, -kk.shape[1]:]) and torch.equal(vv, rows[1, :, -kk.shape[1]:])
