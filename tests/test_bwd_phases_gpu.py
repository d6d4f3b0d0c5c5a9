"""Phases of a pack's backward spread over calls with different masks: the dK/dV launch takes the row
statistics from the earlier call and nothing else.  Its table of key tiles in particular is of its own
call's tile size and place -- the earlier call may have had another (other blocks, sink keys ahead of
it in the workspace, or what was there overwritten since)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["wide", "short"])
@pytest.mark.parametrize("prep", ["other form", "sinks", "overwritten"])
def test_dkdv_launch_makes_its_own_key_tile_table(monkeypatch, form, prep):
    from ring_swa.ops.band_attn import attn_bwd, attn_fwd, bwd_workspace_bytes

    cu = [0, 700, 700, 1300, 1301, 1900]
    hq, hk, d, w = 4, 2, 64, 200
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, do = (torch.randn(cu[-1], hq, d, device="cuda", dtype=torch.bfloat16, generator=gen) for _ in range(2))
    k, v = (torch.randn(cu[-1], hk, d, device="cuda", dtype=torch.bfloat16, generator=gen) for _ in range(2))
    cu_t = torch.tensor(cu, dtype=torch.int32, device="cuda")
    out, lse = attn_fwd(q, k, v, None, (w, 0), True, cu_t, cu_t)
    sinks = 3 if prep == "sinks" else 0
    need = max(bwd_workspace_bytes(q, k, cu_t, cu_t, window_size=(w, 0), causal=True, num_sink=n) for n in (0, sinks))
    results = []
    for split in (False, True):
        ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
        grads = [torch.zeros_like(t) for t in (q, k, v)]

        def run(phases, n_sink=0):
            attn_bwd(q, k, v, out, lse, do, *grads, None, (w, 0), True, cu_t, cu_t, num_sink=n_sink,
                     workspace=ws, phases=phases, handoff=False)

        if split:
            other = {"wide": "short", "short": "wide"}[form]
            monkeypatch.setenv("RSWA_DKDV_FORM", other if prep == "other form" else form)
            run(1, sinks)
            if prep == "overwritten":  # all behind the statistics (two arrays, each to a multiple of 256 bytes)
                ws[2 * (-(-cu[-1] * hq * 4 // 256) * 256):] = 0x11
        monkeypatch.setenv("RSWA_DKDV_FORM", form)
        run(2 if split else 7)
        results.append(grads[1:])
    for one, two in zip(*results):
        assert torch.equal(one, two)


@pytest.mark.parametrize("form", ["wide", "short"])
@pytest.mark.parametrize("sinks", [0, 2])
def test_pack_without_room_for_the_table_gets_the_same_bits(monkeypatch, form, sinks):
    from ring_swa.ops.band_attn import attn_bwd, attn_fwd, bwd_workspace_bytes

    cu = [0, 300, 300, 301, 901, 1500]
    hq, hk, d, w = 4, 2, 128, 100
    gen = torch.Generator(device="cuda").manual_seed(4)
    q, do = (torch.randn(cu[-1], hq, d, device="cuda", dtype=torch.bfloat16, generator=gen) for _ in range(2))
    k, v = (torch.randn(cu[-1], hk, d, device="cuda", dtype=torch.bfloat16, generator=gen) for _ in range(2))
    cu_t = torch.tensor(cu, dtype=torch.int32, device="cuda")
    out, lse = attn_fwd(q, k, v, None, (w, 0), True, cu_t, cu_t, num_sink=sinks)
    monkeypatch.setenv("RSWA_DKDV_FORM", form)
    need = bwd_workspace_bytes(q, k, cu_t, cu_t, window_size=(w, 0), causal=True, num_sink=sinks)
    table = (len(cu) + 1) * 4  # the last thing in it
    results = []
    for room in (need, need - table):
        ws = torch.full((room,), 0xff, dtype=torch.uint8, device="cuda")
        grads = [torch.zeros_like(t) for t in (q, k, v)]
        attn_bwd(q, k, v, out, lse, do, *grads, None, (w, 0), True, cu_t, cu_t, num_sink=sinks, workspace=ws)
        results.append(grads)
    for one, two in zip(*results):
        assert torch.equal(one, two)


@pytest.mark.parametrize("over", ["q", "out", "dout"])
@pytest.mark.parametrize("hq,hk,d,cu", [(4, 4, 64, None), (6, 2, 128, None), (4, 2, 128, [0, 130, 200, 700])])
def test_dq_over_an_input_gets_the_same_bits(over, hq, hk, d, cu):
    """The dQ kernel, which otherwise goes first, then runs behind the dK/dV kernel."""
    from ring_swa.ops.band_attn import attn_bwd, attn_fwd

    s, w = 700, 150
    lead = (s,) if cu else (2, s)
    gen = torch.Generator(device="cuda").manual_seed(6)
    q, do = (torch.randn(*lead, hq, d, device="cuda", dtype=torch.bfloat16, generator=gen) for _ in range(2))
    k, v = (torch.randn(*lead, hk, d, device="cuda", dtype=torch.bfloat16, generator=gen) for _ in range(2))
    cu_t = torch.tensor(cu, dtype=torch.int32, device="cuda") if cu else None
    out, lse = attn_fwd(q, k, v, None, (w, 0), True, cu_t, cu_t)
    apart = [torch.empty_like(t) for t in (q, k, v)]
    attn_bwd(q, k, v, out, lse, do, *apart, None, (w, 0), True, cu_t, cu_t)
    dq = {"q": q, "out": out, "dout": do}[over]
    dk, dv = torch.empty_like(k), torch.empty_like(v)
    attn_bwd(q, k, v, out, lse, do, dq, dk, dv, None, (w, 0), True, cu_t, cu_t)
    for one, two in zip(apart, (dq, dk, dv)):
        assert torch.equal(one, two)
