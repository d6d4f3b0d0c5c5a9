"""The native node of the plain attention call against the Python one: same bits, same refusals, and
everything that has to see the call (hooks, transforms, tangents, tracing, modes) still does."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(packed, hq=4, hk=2, d=64, n=200, dtype=torch.bfloat16, grad=True):
    torch.manual_seed(0)
    lead = (n,) if packed else (2, n)
    q, k, v = (torch.randn(*lead, h, d, device="cuda", dtype=dtype) for h in (hq, hk, hk))
    return [x.requires_grad_() if grad else x for x in (q, k, v)]


def _count(monkeypatch):
    """Counts the calls that take the Python node."""
    from ring_swa import sliding_window as S

    seen = []
    apply = S.BandAttnFunc.apply
    monkeypatch.setattr(S.BandAttnFunc, "apply", lambda *a: (seen.append(1), apply(*a))[1])
    return seen


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("sink", [0, 2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_same_bits_as_the_python_node(packed, sink, dtype, monkeypatch):
    from ring_swa import sliding_window as S

    cu = torch.tensor([0, 70, 70, 200], dtype=torch.int32, device="cuda") if packed else None
    for scale in (None, 0.3):
        q, k, v = _inputs(packed, dtype=dtype)
        do = torch.randn_like(q).transpose(-1, -2).contiguous().transpose(-1, -2)  # (rows not contiguous)
        ref = S.BandAttnFunc.apply(q, k, v, 31, scale, cu, sink)
        gref = torch.autograd.grad(ref, (q, k, v), do)
        seen = _count(monkeypatch)
        out = S.band_attn(q, k, v, 31, scale, cu, sink)
        got = torch.autograd.grad(out, (q, k, v), do)
        with torch.no_grad():
            alone = S.band_attn(q, k, v, 31, scale, cu, sink)
        assert not seen and not alone.requires_grad
        assert torch.equal(out, ref) and torch.equal(alone, ref)
        for x, r in zip(got, gref):
            assert torch.equal(x, r) and x.stride() == r.stride()
        monkeypatch.undo()


def test_slices_of_a_fused_projection_and_partial_grads():
    import ring_swa

    x = torch.randn(1, 150, 8, 128, device="cuda").bfloat16().requires_grad_()
    q, k, v = x[:, :, :4], x[:, :, 4:6], x[:, :, 6:]
    out = ring_swa.ring_sliding_window_attn(q, k, v, 40)
    (g,) = torch.autograd.grad(out.float().sum(), (x,))
    qc, kc, vc = (t.detach().clone().requires_grad_() for t in (q, k, v))
    ref = torch.autograd.grad(ring_swa.ring_sliding_window_attn(qc, kc, vc, 40).float().sum(), (qc, kc, vc))
    assert torch.equal(g, torch.cat(ref, 2))
    out = ring_swa.ring_sliding_window_attn(qc.detach(), kc, vc.detach(), 40)
    assert torch.equal(torch.autograd.grad(out.float().sum(), (kc,))[0], ref[1])


def test_hooks_transforms_tangents_and_modes(monkeypatch):
    from torch.utils._python_dispatch import TorchDispatchMode

    import ring_swa

    q, k, v = _inputs(False)
    seen = _count(monkeypatch)
    packs = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packs.append(1), t.clone())[1], lambda t: t):
        out = ring_swa.ring_sliding_window_attn(q, k, v, 9)
    assert len(packs) == 5 and not seen
    out.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        out.sum().backward()
    out = ring_swa.ring_sliding_window_attn(q, k, v, 9)
    with torch.no_grad():
        k.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()

    def attn(x):
        return ring_swa.ring_sliding_window_attn(x, k, v, 9)

    with pytest.raises(RuntimeError):
        torch.func.vmap(attn)(q[None])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: attn(x).sum())(q.detach())
    with pytest.raises((RuntimeError, NotImplementedError)), torch.autograd.forward_ad.dual_level():
        attn(torch.autograd.forward_ad.make_dual(q.detach(), q.detach()))

    class Mode(TorchDispatchMode):
        ops = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Mode.ops += 1
            return func(*args, **(kwargs or {}))

    with Mode(), torch.no_grad():
        attn(q)
    assert Mode.ops >= 2  # (the two outputs' allocations)


def test_what_was_refused_stays_refused():
    import ring_swa

    q, k, v = _inputs(False, grad=False)
    with pytest.raises(AssertionError):
        ring_swa.ring_sliding_window_attn(q, k[:, :-1], v[:, :-1], 9)
    with pytest.raises(AssertionError):
        ring_swa.ring_sliding_window_attn(q, k.half(), v.half(), 9)
    with pytest.raises(NotImplementedError):
        ring_swa.ring_sliding_window_attn(q.float(), k.float(), v.float(), 9)
    with pytest.raises(NotImplementedError):
        ring_swa.ring_sliding_window_attn(q[..., :32], k[..., :32], v[..., :32], 9)
    with pytest.raises(ValueError):
        ring_swa.ring_sliding_window_attn(q, k, v, 9, softmax_scale=-1.0)
    assert ring_swa.ring_sliding_window_attn(q[:, :0], k[:, :0], v[:, :0], 9).shape == (2, 0, 4, 64)
    # a gradient whose rows do not start on 16 bytes is refused in the backward, by the library
    x = [t.clone().requires_grad_() for t in (q, k, v)]
    out = ring_swa.ring_sliding_window_attn(*x, 9)
    odd = torch.randn(q.numel() + 1, device="cuda").bfloat16()[1:].view(q.shape)
    with pytest.raises(NotImplementedError, match="16-byte aligned"):
        torch.autograd.grad(out, x, odd)


def test_the_environments_switches_reach_the_backward(monkeypatch):
    import ring_swa

    q, k, v = _inputs(False, n=600)
    want = torch.autograd.grad(ring_swa.ring_sliding_window_attn(q, k, v, 300).float().sum(), (q, k, v))
    out = ring_swa.ring_sliding_window_attn(q, k, v, 300)
    monkeypatch.setenv("RSWA_DKDV_FORM", "no such form")
    with pytest.raises(KeyError):
        torch.autograd.grad(out.float().sum(), (q, k, v))
    monkeypatch.setenv("RSWA_DKDV_FORM", "wide")
    out = ring_swa.ring_sliding_window_attn(q, k, v, 300)
    for x, r in zip(torch.autograd.grad(out.float().sum(), (q, k, v)), want):
        assert (x - r).float().norm() <= 4e-3 * r.float().norm()  # (16-bit rounding of sums in another order)


def test_streams_and_threads():
    """Calls of several threads on streams of their own, forward and backward, give the bits of one call."""
    import threading

    import ring_swa

    q, k, v = _inputs(False, n=500)
    want = torch.autograd.grad(ring_swa.ring_sliding_window_attn(q, k, v, 100).float().sum(), (q, k, v))
    torch.cuda.synchronize()
    bad = []

    def work():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(10):
                got = torch.autograd.grad(ring_swa.ring_sliding_window_attn(q, k, v, 100).float().sum(), (q, k, v))
            s.synchronize()
            if not all(torch.equal(a, b) for a, b in zip(got, want)):
                bad.append(1)

    ts = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("which,change,error", [
    (0, lambda t: t.cpu(), RuntimeError), (4, lambda t: t.cpu(), RuntimeError), (3, lambda t: t.cpu(), RuntimeError),
    (4, lambda t: t.to(torch.bfloat16), AssertionError), (4, lambda t: t[..., :-8], AssertionError),
    (1, lambda t: t.float(), AssertionError), (1, lambda t: t[..., :-1, :], AssertionError),
    (2, lambda t: t.transpose(-1, -2).contiguous().transpose(-1, -2), AssertionError),
    (3, lambda t: t[..., :32], AssertionError), (0, lambda t: t.flatten(-2), AssertionError),
])
def test_saved_tensors_that_hooks_gave_back_changed_are_refused(packed, which, change, error):
    """What is unpacked need not be what was packed: another type, shape, device or layout is refused ahead of
    any launch (saved are q, k, v, out and lse, in this order); the same values in another layout that the
    kernels take are used."""
    import ring_swa

    q, k, v = _inputs(packed)
    args = (31, torch.tensor([0, 70, 200], dtype=torch.int32, device="cuda")) if packed else (31,)
    attn = ring_swa.ring_sliding_window_attn_varlen if packed else ring_swa.ring_sliding_window_attn
    want = torch.autograd.grad(attn(q, k, v, *args).float().sum(), (q, k, v))

    def grads(pack):
        n = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (n.append(1), pack(len(n) - 1, t))[1], lambda t: t):
            out = attn(q, k, v, *args)
        return torch.autograd.grad(out.float().sum(), (q, k, v))

    with pytest.raises(error):
        grads(lambda i, t: change(t.detach()) if i == which else t)
    for x, r in zip(grads(lambda i, t: torch.stack([t.detach()] * 2, -2)[..., 0, :] if i < 4 else t), want):
        assert torch.equal(x, r)


def test_backward_beside_a_thread_that_changes_the_environment():
    """The backward looks at the environment from the autograd thread, where another thread may be adding
    variables (which moves the array that getenv walks): it does so under the interpreter's lock, and says so
    itself where it does not."""
    import os
    import threading

    import ring_swa

    q, k, v = _inputs(False)
    want = torch.autograd.grad(ring_swa.ring_sliding_window_attn(q, k, v, 31).float().sum(), (q, k, v))
    stop, names = threading.Event(), [f"RSWA_TEST_{i}" for i in range(200)]

    def change():
        while not stop.is_set():
            for n in names:
                os.environ[n] = "x" * 50
            for n in names:
                del os.environ[n]

    t = threading.Thread(target=change)
    t.start()
    try:
        for _ in range(20):
            got = torch.autograd.grad(ring_swa.ring_sliding_window_attn(q, k, v, 31).float().sum(), (q, k, v))
            assert all(torch.equal(x, r) for x, r in zip(got, want))
    finally:
        stop.set()
        t.join()
