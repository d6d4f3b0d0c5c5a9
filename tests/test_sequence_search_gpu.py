"""Every block of a pack finds its sequence among up to 64 at a time: packs of as many sequences as
one, two and three such rounds take and one more, empty ones among them, against the same rows as a
dense batch -- the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq,length", [(1, 130), (64, 70), (65, 70), (129, 33), (4096, 5), (4097, 5)])
def test_pack_with_empty_sequences_equals_its_dense_rows(n_seq, length):
    from ring_swa.ops import attn_bwd, attn_fwd

    lens = [0 if n_seq > 1 and i % 5 in (0, 3) else length for i in range(n_seq)]
    cu = torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
    full, hq, hk, d, window = sum(n > 0 for n in lens), 6, 3, 64, 20
    torch.manual_seed(n_seq)
    q, do = (torch.randn(full * length, hq, d, device="cuda").bfloat16() for _ in range(2))
    k, v = (torch.randn(full * length, hk, d, device="cuda").bfloat16() for _ in range(2))

    def run(q, k, v, do, *cu):
        out, lse = attn_fwd(q, k, v, None, (window, 0), True, *cu)
        grads = [torch.empty_like(x) for x in (q, k, v)]
        attn_bwd(q, k, v, out, lse, do, *grads, None, (window, 0), True, *cu, dkdv_form="short")
        return out, lse, grads

    out, lse, grads = run(q, k, v, do, cu, cu)
    dense = [x.view(full, length, -1, d) for x in (q, k, v, do)]
    out_d, lse_d, grads_d = run(*dense)
    assert torch.equal(out, out_d.view_as(out))
    assert torch.equal(lse, lse_d.transpose(0, 1).reshape(hq, -1))
    for x, r in zip(grads, grads_d):
        assert torch.equal(x, r.view_as(x))
