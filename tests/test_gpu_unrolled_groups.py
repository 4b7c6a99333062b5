"""Batches of the unrolled model that run in groups of different sizes: a
sample's result does not depend on its group, gradients add up over groups."""

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 6, 7])             # 4, 5, 6 dual updates
@pytest.mark.parametrize("B,H,W,T", [(1, 40, 66, 3), (5, 40, 66, 3), (8, 40, 66, 3), (9, 40, 66, 3),
                                     (6, 256, 256, 4), (7, 130, 250, 8)])
def test_groups_match_single_samples(gpu, B, H, W, T, n):
    import torch
    from pnp_sci.synthetic import unrolled_batch
    from pnp_sci.unrolled import unrolled_gap_tv
    truth, mask = (torch.as_tensor(v, dtype=torch.float32, device="cuda")
                   for v in unrolled_batch(B, H, W, T, seed=B + n, mask="logits"))
    lam0, w0 = torch.tensor([1.0, 0.9, 1.1]), torch.tensor([0.1, 0.05, 0.2])

    def run(videos):
        z, lam, w = (v.clone().requires_grad_() for v in (mask, lam0, w0))
        x = unrolled_gap_tv(z, videos, lam, w, tv_iter_max=n)
        ((x - videos) ** 2).sum().backward()
        return x.detach(), (z.grad.double(), lam.grad.double(), w.grad.double())

    x, grads = run(truth)
    singles = [run(truth[b:b + 1]) for b in range(B)]
    assert torch.equal(x, torch.cat([s[0] for s in singles]))
    for i, g in enumerate(grads):
        want = sum(s[1][i] for s in singles)
        # fp32 sums over at most 9 samples in another order, and fp64 sums of fp32
        # sums of a workgroup: 1e-5 of the largest entry
        assert float((g - want).abs().max()) <= 1e-5 * float(want.abs().max())
