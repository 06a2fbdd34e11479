"""Forward model on the device against the FP64 oracle, at the sizes where the
matrix-core interpolation has edges: grids smaller than a region's reach (11 x
12 cells, several wraps), regions cut by the grid's end, fewer samples than a
batch and batches that do not fill, coil counts around the groups of 8, real
and complex bases, masked samples, and the shapes that keep one wavefront per
sample (few coils, sparse samples, U = I).  Tolerance 1e-5 relative L2 (W = 8
spreading in ComplexF32), as the other NUFFT tests."""
import gc
import threading

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


@pytest.mark.parametrize("N,K,C", [((64, 64), 1, 8), ((256, 256), 5, 8), ((32, 32), 8, 16), ((96, 80), 3, 12)])
def test_error_is_that_of_single_coils(torch, msr, N, K, C):
    """The matrix cores' sums against 64 bits are no further off than those of the
    same coils one by one, which run one wavefront per sample: 1 % allows for the
    spread between inputs (measured 0.3 % over three seeds each)."""
    rng = np.random.default_rng(2)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    nt, ns = 20, 1000
    trj = rng.uniform(-0.5, 0.5, size=(nt, ns, 2)).astype(np.float32)
    trj[:, ns // 2:] *= np.float32(0.1)
    U = (rng.normal(size=(K, nt)) + 1j * rng.normal(size=(K, nt))).astype(np.complex64)
    cm = msr.synth.gaussian_coil_maps(N, C)
    x = msr.synth.ellipse_phantom(N, K).astype(np.complex64)
    traj = msr.plan_trajectory(dev(trj))
    ref = toeplitz.forward(x, trj, U, cm)
    together = msr.forward(dev(x), traj, cmaps=[dev(c) for c in cm], U=dev(U)).cpu().numpy()
    single = np.stack([msr.forward(dev(x), traj, cmaps=[dev(c)], U=dev(U)).cpu().numpy()[0] for c in cm])
    e, e1 = rel_err(together, ref), rel_err(single, ref)
    print(f"forward {N} K={K} C={C}: {e:.3e}, coil by coil {e1:.3e}, {e / e1:.3f}", flush=True)
    assert e <= 1.01 * e1


def problem(torch, N, K, C, nt, ns, seed=5):
    """x, trajectory, maps and U on the device."""
    rng = np.random.default_rng(seed)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    c = lambda *sh: (rng.normal(size=sh) + 1j * rng.normal(size=sh)).astype(np.complex64)
    trj = rng.uniform(-0.5, 0.5, size=(nt, ns, len(N))).astype(np.float32)
    return dev(c(K, *N[::-1])), dev(trj), [dev(m) for m in c(C, *N[::-1])], dev(c(K, nt))


@pytest.mark.parametrize("N,K,C", [((256, 256), 4, 16), ((64, 64, 64), 2, 8)])
def test_workspace_goes_back(torch, msr, N, K, C):
    """2D (matrix cores) and 3D: after a call, nothing of its workspace (at least
    the grids' 134 and 268 MB) stays with the trajectory."""
    x, trj, cm, U = problem(torch, N, K, C, 8, 3000)
    traj = msr.plan_trajectory(trj)
    msr.forward(x, traj, cmaps=cm[:4], U=U)   # tables and the plan
    torch.cuda.synchronize()

    def available():
        gc.collect()
        torch.cuda.empty_cache()
        msr.trim()
        return torch.cuda.mem_get_info()[0]

    before = available()
    msr.forward(x, traj, cmaps=cm, U=U)
    left = before - available()
    print(f"{left >> 20} MiB stay", flush=True)
    assert left < 32 << 20


def test_coils_in_chunks(torch, msr):
    """128 x 128 x 128, K = 4: the grids of nine coils exceed the workspace's bound,
    so the coils go four at a time; the bits of three calls with those coils."""
    x, trj, cm, U = problem(torch, (128, 128, 128), 4, 9, 4, 500)
    traj = msr.plan_trajectory(trj)
    y = msr.forward(x, traj, cmaps=cm, U=U)
    for c in range(0, 9, 4):
        assert torch.equal(y[c:c + 4], msr.forward(x, traj, cmaps=cm[c:c + 4], U=U))


def test_few_coils_make_no_plan(torch, msr):
    """Three coils never take the matrix cores: 4 million samples are not sorted for
    them, and no sorted list (16 MB, and the batches) stays with the trajectory."""
    x, trj, cm, U = problem(torch, (32, 32), 1, 3, 4, 1000000)
    traj = msr.plan_trajectory(trj)
    msr.forward(x, msr.plan_trajectory(trj[:, :10].contiguous()), cmaps=cm, U=U)   # tables

    def available():
        gc.collect()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        msr.trim()
        return torch.cuda.mem_get_info()[0]

    before = available()
    msr.forward(x, traj, cmaps=cm, U=U)
    assert before - available() < 8 << 20


def test_calls_on_one_trajectory_side_by_side(torch, msr):
    """Threads with streams of their own, 2D and 3D handles shared: the bits of
    the calls one after another."""
    jobs = []
    for N, K, C in [((48, 40), 3, 9), ((24, 20, 16), 2, 5)]:
        x, trj, cm, U = problem(torch, N, K, C, 6, 500)
        traj = msr.plan_trajectory(trj)
        jobs += [(x, traj, cm[:c], U) for c in (C, 4)]
    want = [msr.forward(x, t, cmaps=cm, U=U) for x, t, cm, U in jobs]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        st = torch.cuda.Stream()
        x, t, cm, U = jobs[i]
        with torch.cuda.stream(st):
            for _ in range(10):
                y = msr.forward(x, t, cmaps=cm, U=U)
                st.synchronize()
                if not torch.equal(y, want[i]):
                    wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
