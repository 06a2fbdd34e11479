"""Fused line passes of the normal operator (every shape outside the fused
Toeplitz passes, and the Cartesian operator) against the FP64 oracle, at the
sizes where their tiling has edges: lengths of one FFT stage (2-8 points),
odd and prime-power lengths, one row or column, ragged row and column tiles,
the largest workgroup (8 lines of 1024 values), and coil groups that do not
divide.  Tolerances (relative L2): ComplexF32 apply 2e-6, ComplexF64 apply
1e-12, as for the other passes."""
import numpy as np
import pytest

from conftest import load_package, rel_err
from oracle import cartesian as ocart
from oracle import toeplitz
from test_gpu_apply import make_case

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


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def check(torch, A, x, ref):
    xd = dev(torch, x).reshape(-1)
    e32 = rel_err((A @ xd).cpu().numpy().reshape(x.shape), ref)
    y = torch.empty(x.size, dtype=torch.complex128, device="cuda")
    A.A.mul_f64_(y, xd.to(torch.complex128))
    e64 = rel_err(y.cpu().numpy().reshape(x.shape), ref)
    print(f"f32 {e32:.2e} f64 {e64:.2e}", flush=True)
    assert e32 < 2e-6 and e64 < 1e-12


@pytest.mark.parametrize("N,K,C,real,identity", [
    ((4, 2), 1, 1, False, True),         # 2N = 8 x 4: one stage each
    ((1, 3), 2, 2, True, False),         # 2 x 6
    ((16, 4), 8, 3, False, False),
    ((45, 27), 3, 5, False, False),      # 90 x 54
    ((64, 48), 5, 4, True, False),       # a shape the fused passes take too
    ((75, 81), 2, 3, False, False),      # 150 x 162
    ((24, 512), 8, 1, False, False),     # 8 lines of 1024 values
    ((512, 6), 2, 2, False, False),      # rows of 1024
    ((4, 3, 2), 2, 2, False, False),     # 8 x 6 x 4
    ((20, 18, 15), 4, 2, True, False),
    ((5, 6, 100), 8, 1, False, False),  # 2Nz = 200, K = 8: fewer columns per tile
])
def test_toeplitz_matches_oracle(torch, msr, monkeypatch, N, K, C, real, identity):
    lam, km, cm, x = make_case(np.random.default_rng(3), N, K, C, real=real, identity=identity)
    monkeypatch.setenv("MSR_APPLY_PLANES", "1")
    A = msr.NFFTNormalOp(N, dev(torch, lam), dev(torch, km + 1),
                         cmaps=None if cm is None else [dev(torch, c) for c in cm])
    l64 = lam.astype(np.float64 if real else np.complex128)
    ref = toeplitz.apply_normal(N, l64, km, None if cm is None else cm.astype(np.complex128),
                                x.astype(np.complex128))
    check(torch, A, x, ref)
    y = torch.empty(x.size, dtype=torch.complex64, device="cuda")
    A.A.mul_(y, dev(torch, x).reshape(-1), percoil=True)
    assert rel_err(y.cpu().numpy().reshape(x.shape), ref) < 2e-6


@pytest.mark.parametrize("path", ["MSR_APPLY_PLANES", "MSR_APPLY_LINES"])
@pytest.mark.parametrize("N,K,C,chunk,identity", [
    ((64, 48), 5, 7, 3, False),          # chunks of 3, 3 and 1 coils, summed in 3 groups
    ((45, 27), 2, 5, 4, False),
    ((20, 18, 15), 3, 5, 2, False),
    ((12, 10, 9), 2, 4, 1, False),       # one coil at a time
    ((24, 20), 3, 1, 1, True),
])
def test_coils_in_chunks(torch, msr, monkeypatch, path, N, K, C, chunk, identity):
    """The coils of an operator too large for one pass, taken a chunk at a time."""
    lam, km, cm, x = make_case(np.random.default_rng(6), N, K, C, identity=identity)
    monkeypatch.setenv(path, "1")
    monkeypatch.setenv("MSR_COIL_CHUNK", str(chunk))
    A = msr.NFFTNormalOp(N, dev(torch, lam), dev(torch, km + 1),
                         cmaps=None if cm is None else [dev(torch, c) for c in cm])
    ref = toeplitz.apply_normal(N, lam.astype(np.complex128), km, None if cm is None else cm.astype(np.complex128),
                                x.astype(np.complex128))
    check(torch, A, x, ref)
    y = torch.empty(x.size, dtype=torch.complex64, device="cuda")
    A.A.mul_(y, dev(torch, x).reshape(-1), percoil=True)
    assert rel_err(y.cpu().numpy().reshape(x.shape), ref) < 2e-6


@pytest.mark.parametrize("N,K,C,real", [
    ((5, 4), 2, 3, False),               # one stage each
    ((3, 25), 1, 1, True),
    ((81, 30), 5, 7, False),
    ((96, 125), 8, 2, True),
    ((250, 9), 3, 4, False),
    ((9, 8, 5), 3, 2, False),
    ((16, 10, 81), 8, 2, True),
])
def test_cartesian_dense_kernel_matches_oracle(torch, msr, N, K, C, real):
    """Full kernels that are not Hermitian, with cells off the mask."""
    rng = np.random.default_rng(4)
    V = int(np.prod(N))
    L = rng.normal(size=(V, K, K)).astype(np.float32)
    if not real:
        L = (L + 1j * rng.normal(size=L.shape)).astype(np.complex64)
    L[rng.uniform(size=V) < 0.3] = 0
    cm = (rng.normal(size=(C,) + N[::-1]) + 1j * rng.normal(size=(C,) + N[::-1])).astype(np.complex64)
    x = (rng.normal(size=(K,) + N[::-1]) + 1j * rng.normal(size=(K,) + N[::-1])).astype(np.complex64)
    dense = np.transpose(L, (0, 2, 1)).reshape(N[::-1] + (K, K))   # [q, k, j] = Julia Λ[j, k, q]
    A = msr.FFTNormalOp(dev(torch, dense), cmaps=[dev(torch, c) for c in cm])
    km = A.A.kmask_indcs.cpu().numpy() - 1
    assert np.array_equal(km, ocart.kmask_of(L))
    assert np.array_equal(A.A.Λ.cpu().numpy(), np.transpose(L[km], (0, 2, 1)))
    check(torch, A, x, ocart.apply_normal(N, L.astype(np.complex128), cm.astype(np.complex128), x))
