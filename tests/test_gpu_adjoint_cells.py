"""The adjoint's closed sums over a cell's samples where every cell has several
labels: from many samples a cell to one in every other cell, on volumes thinner
than a slab, as long as one and just longer.  Density and pose gradients against
the dense FP64 model, to the bars of the other adjoint tests (1e-4 relative L2)."""
import numpy as np
import pytest
import torch

from deepdrr_amd.autograd import DifferentiableProjector
from deepdrr_amd.spectral_data import synthetic_120kv
from tests.test_gpu_adjoint import MATS, _dense, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, det, step", [
    (9, 9, 0.05),    # 20 samples a cell; thinner than one slab
    (11, 16, 0.25),  # cells -1 .. 10: one slab and one cell
    (12, 17, 0.9),   # mostly one sample a cell
    (23, 8, 2.2),    # cells passed over
])
def test_mixed_cells(gpu, n, det, step):
    dens, _, W, projs, _ = _scene(n=n, det=det, seed=n)
    rng = np.random.default_rng(n)
    labels = rng.integers(0, len(MATS), dens.shape).astype(np.uint8)
    dp = DifferentiableProjector(labels, MATS, W, step=step, spectrum=synthetic_120kv())
    try:
        gI = rng.standard_normal((len(projs), det, det))
        d_t = torch.tensor(dens, device=gpu, requires_grad=True)
        th_t = torch.zeros(6, device=gpu, requires_grad=True)
        (dp(d_t, th_t, projs) * torch.tensor(gI.astype(np.float32), device=gpu)).sum().backward()
        ref = _dense(dp, projs)
        d64 = torch.tensor(dens.astype(np.float64), requires_grad=True)
        t64 = torch.zeros(6, dtype=torch.float64, requires_grad=True)
        onehot = torch.tensor(np.stack([(labels == m).astype(np.float64) for m in range(len(MATS))]))
        (ref.render(d64, onehot, t64) * torch.tensor(gI.astype(np.float32).astype(np.float64))).sum().backward()
        for name, g, w in (("density", d_t.grad, d64.grad), ("pose", th_t.grad, t64.grad)):
            g, w = g.detach().cpu().numpy().astype(np.float64), w.numpy()
            err = np.linalg.norm(g - w) / np.linalg.norm(w)
            print(f"n {n}, step {step}: {name} relative L2 {err:.2e}")
            assert err < 1e-4, name
    finally:
        dp.close()
