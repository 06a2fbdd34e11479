"""Fused 2D passes at the lengths whose lines the whole workgroup transforms
(2N = 24, 40, 48, 80, 96, 160, 192, 320, 384: few threads per line in the
wavefront plans), along x, along y and both, with ragged row tiles, against the
FP64 oracle; and an operator alone against the same operator in a batch, bit
for bit.  Tolerances (relative L2) as for the other lengths: ComplexF32 apply
2e-6, ComplexF64 1e-12, compact intermediates 2e-8."""
import numpy as np
import pytest

from conftest import load_package, rel_err
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


@pytest.mark.parametrize("N,K,C,real", [
    ((12, 20), 1, 3, False), ((20, 12), 8, 2, True), ((24, 40), 5, 9, False), ((40, 24), 3, 2, True),
    ((48, 16), 8, 3, False), ((16, 48), 2, 5, False), ((80, 96), 4, 2, False), ((96, 80), 1, 1, True),
    ((160, 8), 3, 4, False), ((8, 160), 8, 2, False), ((192, 12), 2, 3, True), ((12, 192), 6, 2, False),
    ((64, 192), 5, 2, False),
])
def test_apply_matches_oracle(torch, msr, N, K, C, real):
    lam, km, cm, x = make_case(np.random.default_rng(7), N, K, C, real=real)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    A = msr.NFFTNormalOp(N, dev(lam), dev(km + 1), cmaps=[dev(c) for c in cm])
    ref = toeplitz.apply_normal(N, lam.astype(np.float64 if real else np.complex128), km,
                                cm.astype(np.complex128), x.astype(np.complex128)).reshape(-1)
    xd = dev(x).reshape(-1)
    y32 = A @ xd
    x64 = xd.to(torch.complex128)
    y64, y64c = torch.empty_like(x64), torch.empty_like(x64)
    A.A.mul_f64_(y64, x64)
    A.A.mul_f64_(y64c, x64, compact=True)
    e = [rel_err(y.cpu().numpy(), ref) for y in (y32, y64, y64c)]
    print(f"{N} K={K}: f32 {e[0]:.1e} f64 {e[1]:.1e} f64c {e[2]:.1e}", flush=True)
    assert e[0] < 2e-6 and e[1] < 1e-12 and e[2] < 2e-8
    # a second operator of another shape in the batch
    lam2, km2, cm2, x2 = make_case(np.random.default_rng(8), (N[0], 24), K, 2, real=real)
    B = msr.NFFTNormalOp((N[0], 24), dev(lam2), dev(km2 + 1), cmaps=[dev(c) for c in cm2])
    x2d = dev(x2).reshape(-1)
    ys = [torch.empty_like(xd), torch.empty_like(x2d)]
    msr.NFFTNormalOpBatch([A, B]).mul_(ys, [xd, x2d])
    assert torch.equal(ys[0], y32) and torch.equal(ys[1], B @ x2d)
