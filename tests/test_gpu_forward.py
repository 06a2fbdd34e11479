"""Forward model on the device against the FP64 oracle, at the sizes where the
matrix-core interpolation has edges: grids smaller than a region's reach (11 x
12 cells, several wraps), regions cut by the grid's end, fewer samples than a
batch and batches that do not fill, coil counts around the groups of 8, real
and complex bases, masked samples, and the shapes that keep one wavefront per
sample (few coils, sparse samples, U = I).  Tolerance 1e-5 relative L2 (W = 8
spreading in ComplexF32), as the other NUFFT tests."""
import numpy as np
import pytest

from conftest import load_package, rel_err
from oracle import toeplitz

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


@pytest.fixture(scope="module")
def msr():
    return load_package()


@pytest.mark.parametrize("N,K,C,nt,ns,real,masked", [
    ((3, 2), 2, 8, 4, 40, False, False),    # 6 x 4 cells: every support wraps
    ((5, 4), 1, 4, 3, 33, True, True),
    ((16, 16), 3, 9, 7, 100, False, False),
    ((27, 20), 2, 16, 5, 64, False, True),  # 54 x 40: both region sizes cut
    ((20, 27), 4, 7, 6, 64, True, False),
    ((64, 48), 2, 5, 1, 3, False, False),   # three samples: one wavefront each
    ((32, 32), 2, 2, 8, 64, False, False),  # few coils: one wavefront each
    ((32, 24), 6, 20, 6, 200, False, False),
])
def test_forward_matches_oracle(torch, msr, N, K, C, nt, ns, real, masked):
    rng = np.random.default_rng(11)
    trj = rng.uniform(-0.5, 0.5, size=(nt, ns, 2)).astype(np.float32)
    trj[0, :2] = [[-0.5, 0.5], [0.0, 0.0]]
    if ns > 40:
        trj[:, 20:40] = trj[:, 20:21] + rng.uniform(0, 1e-3, size=(nt, 20, 2)).astype(np.float32)
        trj = np.clip(trj, -0.5, 0.5)
    U = rng.normal(size=(K, nt)) + (0 if real else 1j * rng.normal(size=(K, nt)))
    U = U.astype(np.float32 if real else np.complex64)
    cm = (rng.normal(size=(C,) + N[::-1]) + 1j * rng.normal(size=(C,) + N[::-1])).astype(np.complex64)
    x = (rng.normal(size=(K,) + N[::-1]) + 1j * rng.normal(size=(K,) + N[::-1])).astype(np.complex64)
    mask = rng.uniform(size=(nt, ns)) < 0.7 if masked else None
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    traj = msr.plan_trajectory(dev(trj), None if mask is None else dev(mask))
    ref = toeplitz.forward(x, trj, U, cm, sample_mask=mask)
    first = msr.forward(dev(x), traj, cmaps=[dev(c) for c in cm], U=dev(U))
    e = rel_err(first.cpu().numpy(), ref)
    print(f"forward {N} K={K} C={C}: {e:.2e}", flush=True)
    assert e < 1e-5
    # another call on the handle: fewer coils, then the first again, bit for bit
    msr.forward(dev(x), traj, cmaps=[dev(cm[0])], U=dev(U))
    again = msr.forward(dev(x), traj, cmaps=[dev(c) for c in cm], U=dev(U))
    assert torch.equal(first, again)
