"""The backward whose dQ kernel makes the row statistics against the one whose statistics have a
kernel of their own (phases in separate calls): the same sums in the same order, so the same bits.
Sizes at the edges of the dQ blocks (32-row waves, 64 / 128 / 256-row blocks), both block sizes, packs
with empty sequences and with rows behind the last one, sink keys; workspaces that held NaN."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# batch, rows, q heads, kv heads, dim, window, sinks, cu_seqlens
CASES = [
    (1, 1, 2, 2, 64, 16, 0, None),
    (2, 33, 4, 2, 128, 8, 0, None),
    (2, 255, 3, 1, 128, 1000, 0, None),
    (1, 257, 6, 2, 64, 64, 4, None),
    (1, 3500, 2, 1, 128, -1, 0, None),      # blocks of 4 waves, unbounded window
    (1, 7000, 2, 1, 128, -1, 0, None),      # blocks of 8 waves
    (1, 200, 4, 2, 128, 50, 0, [0, 64, 64, 65, 161]),   # 39 rows of nobody
    (1, 131, 3, 1, 64, 30, 2, [0, 1, 33, 130]),         # one row of nobody, sink keys
    (1, 600, 2, 2, 128, 100, 0, [0] + list(range(1, 600, 2)) + [600]),  # more sequences than threads
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(x) for x in c[:7]) + ("pack" if c[7] else ""))
def test_statistics_in_the_dq_kernel_have_the_same_bits(case, dtype):
    from ring_swa.ops.band_attn import attn_bwd, attn_fwd, bwd_workspace_bytes

    b, s, hq, hk, d, w, sinks, cu = case
    gen = torch.Generator(device="cuda").manual_seed(5)
    lead = (s,) if cu else (b, s)

    def rand(h):
        return torch.randn(*lead, h, d, device="cuda", dtype=dtype, generator=gen)

    q, k, v, do = rand(hq), rand(hk), rand(hk), rand(hq)
    cu_t = torch.tensor(cu, dtype=torch.int32, device="cuda") if cu else None
    out, lse = attn_fwd(q, k, v, None, (w, 0), True, cu_t, cu_t, num_sink=sinks)
    if cu and cu[-1] < s:  # rows of nobody may hold anything
        out[cu[-1]:], do[cu[-1]:], lse[:, cu[-1]:] = float("nan"), float("nan"), float("nan")
    need = bwd_workspace_bytes(q, k, cu_t, cu_t, window_size=(w, 0), causal=True, num_sink=sinks)
    results = []
    for split in ((7,), (1, 2, 4)):
        ws = torch.full(((need + 3) // 4,), float("nan"), device="cuda").view(torch.uint8)
        grads = [torch.zeros_like(t) for t in (q, k, v)]
        for phases in split:
            attn_bwd(q, k, v, out, lse, do, *grads, None, (w, 0), True, cu_t, cu_t, num_sink=sinks,
                     workspace=ws, phases=phases, handoff=False)
        results.append(grads)
    owned = cu[-1] if cu else s
    for one, other in zip(*results):
        one, other = (t[:owned] if cu else t for t in (one, other))
        assert torch.isfinite(one).all() and torch.equal(one, other)
