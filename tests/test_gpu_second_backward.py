"""A second backward pass through a retained graph uses the area densities of the
forward pass, as the first one does: the pose gradient, summed in FP64, is the same
to an ulp (the order of its sums may differ)."""
import numpy as np
import pytest
import torch

from deepdrr_amd import phantoms
from deepdrr_amd.autograd import DifferentiableProjector
from deepdrr_amd.spectral_data import synthetic_120kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("density_grad", [False, True])
def test_second_backward(gpu, density_grad):
    n = 96  # rays of some 1000 samples: the marches' sums differ
    rng = np.random.default_rng(5)
    dens = rng.uniform(0.5, 1.5, (n, n, n)).astype(np.float32)
    labels = np.repeat(np.repeat(np.repeat(rng.integers(0, 2, (n // 8,) * 3), 8, 0), 8, 1), 8, 2).astype(np.uint8)
    W = np.eye(4)
    W[:3, 3] = -(n - 1) / 2
    projs = [phantoms.pose_projection(24, 20, 6.0, p, d, f) for p, d, f in phantoms.batch_poses(2, seed=1, radius=3.0)]
    dp = DifferentiableProjector(labels, ["soft tissue", "bone"], W, step=0.1, spectrum=synthetic_120kv())
    try:
        d = torch.tensor(dens, device=gpu, requires_grad=density_grad)
        th = torch.zeros(6, device=gpu, requires_grad=True)
        gI = torch.tensor(rng.standard_normal((2, 20, 24)).astype(np.float32), device=gpu)
        loss = (dp(d, th, projs) * gI).sum()
        grads = [torch.autograd.grad(loss, [th], retain_graph=True)[0].cpu().numpy() for _ in range(3)]
        print(grads)
        for g in grads[1:]:
            np.testing.assert_allclose(g, grads[0], rtol=1.2e-7, atol=0)
    finally:
        dp.close()
