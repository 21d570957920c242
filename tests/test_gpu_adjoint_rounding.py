"""The adjoint's own rounding errors where every cell has several labels: against a
dense FP64 model of the very samples that the kernel takes (its FP32 source,
directions and steps), in scenes without a sample so near a face that its FP32
position may lie on the other side (the gradient jumps there).  Bars, as geometric
means over scenes: a corner's sum is a product of three factors, some four
roundings of 2^-24, 2.4e-7; the pose takes differences of such sums, 5e-7, where the
grid is the world's (elsewhere the ray in the world and in voxels, each rounded,
differ by more)."""
import numpy as np
import pytest
import torch

from deepdrr_amd import phantoms
from deepdrr_amd.autograd import DifferentiableProjector
from deepdrr_amd.spectral_data import synthetic_120kv
from tests.dense_ref import DenseDRR, _lattice
from tests.test_gpu_adjoint import MATS, _scene

pytestmark = pytest.mark.gpu

FACE = 1e-5  # voxels; FP32 positions up to 32 are good to 2e-6


def _models(dp, projs):
    """One dense model per view, of the view's FP32 numbers: samples at source +
    alpha direction with the direction in voxels as the kernel rounds it."""
    out = []
    for view, src in dp.views(projs, np.zeros(6)):
        A32 = np.array(view.vol[0].ijk_from_world[:], np.float32).reshape(3, 4)[:, :3]
        A, s = A32.astype(np.float64), np.array(view.vol[0].source_ijk[:], np.float64)
        ijk_from_world = np.eye(4)
        ijk_from_world[:3, :3] = A
        ijk_from_world[:3, 3] = s - A @ src.astype(np.float64)
        center = np.asarray(dp.center, np.float32).astype(np.float64)
        m = DenseDRR([(view, src)], np.linalg.inv(ijk_from_world), center, dp.step, dp.E, dp.pdf, dp.mu, dp.shape)
        r, rays, alphas, _ = _lattice(view, dp.step)
        r = r.astype(np.float32)
        ri = np.stack([(A32[k, 0] * r[:, 0] + A32[k, 1] * r[:, 1]) + A32[k, 2] * r[:, 2] for k in range(3)], 1)
        p = s + alphas[:, None] * ri.astype(np.float64)[rays]
        m.views[0]["x"] = torch.tensor(np.linalg.solve(A, (p - ijk_from_world[:3, 3]).T).T)
        out.append(m)
    return out


def _clear_of_faces(models):
    for m in models:
        inv = torch.linalg.inv(m.W_from_ijk)
        p = (m.views[0]["x"] @ inv[:3, :3].T + inv[:3, 3]) - 1.0
        assert len(p) > 400, "the rays miss the volume"
        if float((p - p.round()).abs().min()) < FACE:
            return False
    return True


def _errors(seed, device):
    """(density, pose) errors, or None for a scene with samples near faces."""
    rng = np.random.default_rng(seed)
    n = int(rng.integers(8, 14))
    dens, _, W, _, _ = _scene(n=n, seed=seed)
    projs = [phantoms.pose_projection(4, 4, 0.3 * n, p, d, f)
             for p, d, f in phantoms.batch_poses(2, seed=seed, radius=0.5, cone_deg=40)]
    if seed % 2:  # an oblique, anisotropic grid
        q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        W = np.eye(4)
        W[:3, :3] = q * rng.uniform(0.7, 1.4, 3)
        W[:3, 3] = -(W[:3, :3] @ np.full(3, (n - 1) / 2))
    labels = rng.integers(0, len(MATS), dens.shape).astype(np.uint8)
    dp = DifferentiableProjector(labels, MATS, W, step=0.1, spectrum=synthetic_120kv())
    try:
        models = _models(dp, projs)
        if not _clear_of_faces(models):
            return None
        gI = rng.standard_normal((len(projs), 4, 4)).astype(np.float32)
        d_t = torch.tensor(dens, device=device, requires_grad=True)
        th_t = torch.zeros(6, device=device, requires_grad=True)
        (dp(d_t, th_t, projs) * torch.tensor(gI, device=device)).sum().backward()
        d64 = torch.tensor(dens.astype(np.float64), requires_grad=True)
        t64 = torch.zeros(6, dtype=torch.float64, requires_grad=True)
        onehot = torch.tensor(np.stack([(labels == m).astype(np.float64) for m in range(len(MATS))]))
        I64 = torch.cat([m.render(d64, onehot, t64) for m in models])
        (I64 * torch.tensor(gI.astype(np.float64))).sum().backward()
    finally:
        dp.close()
    pairs = ((d_t.grad, d64.grad), (th_t.grad, t64.grad))
    return [float((g.cpu().double() - w).norm() / w.norm()) for g, w in pairs]


def test_random_labels(gpu):
    errs = {seed: _errors(seed, gpu) for seed in range(40)}
    errs = {seed: e for seed, e in errs.items() if e is not None}
    density = np.array([e[0] for e in errs.values()])
    pose = np.array([e[1] for seed, e in errs.items() if seed % 2 == 0])
    assert len(pose) >= 10 and len(density) >= 20
    mean = [float(np.exp(np.log(e).mean())) for e in (density, pose)]
    print(f"{len(density)} scenes, geometric mean: density {mean[0]:.2e}, pose {mean[1]:.2e}; "
          f"largest {density.max():.2e}, {pose.max():.2e}")
    assert mean[0] <= 2.4e-7 and mean[1] <= 5e-7
