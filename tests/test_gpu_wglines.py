"""Line passes whose lines the whole workgroup transforms (lengths with few
threads per line in the wavefront plans), against the FP64 oracle: ComplexF32
rows and columns of the backprojection, ComplexF64 ones of the kernel
construction and the 3D apply, ragged line groups, lengths on both sides of the
rule.  Tolerances (relative L2) as for the other lengths: backprojection 1e-5
(width-8 ES kernel in FP32), kernel 3e-7 (FP64 build, rounded to ComplexF32),
ComplexF32 apply 2e-6, ComplexF64 1e-12, compact intermediates 2e-8."""
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


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# 2N (backprojection) and 4N (construction): 24, 40, 48, 72, 80, 96, 120, 144, 160, 192, 240, 288,
# 320, 384, 480, 576, 600, 640, 768, 960, 1024, 1280
@pytest.mark.parametrize("N", [(12, 20), (20, 12), (24, 36), (40, 18), (48, 60), (60, 72), (80, 9), (9, 96),
                               (150, 12), (12, 150), (6, 144), (160, 6), (5, 192), (192, 5), (240, 5),
                               (6, 256), (320, 6), (10, 320), (512, 4), (4, 480), (12, 20, 9), (20, 6, 24)])
def test_backprojection_and_kernel_match_oracle(torch, msr, N):
    rng = np.random.default_rng(3)
    trj = rng.uniform(-0.5, 0.5, size=(3, 70, len(N))).astype(np.float32)
    cplx = lambda *s: (rng.normal(size=s) + 1j * rng.normal(size=s)).astype(np.complex64)
    U, cm, data = cplx(2, 3), cplx(3, *N), cplx(3, 3, 70)
    b = msr.calculate_backprojection(dev(torch, data), dev(torch, trj), [dev(torch, c) for c in cm],
                                     U=dev(torch, U)).cpu().numpy()
    e = rel_err(b, toeplitz.backprojection(data, trj, cm, U=U))
    A = msr.NFFTNormalOp(N, dev(torch, trj), dev(torch, U))
    ref, km = toeplitz.toeplitz_kernel(N, trj, U)
    assert np.array_equal(A.prod.A.kmask_indcs.cpu().numpy() - 1, km)
    k = rel_err(A.prod.A.Λ.cpu().numpy(), ref)
    print(f"{N}: backprojection {e:.1e} kernel {k:.1e}", flush=True)
    assert e < 1e-5 and k < 3e-7


@pytest.mark.parametrize("N,K,C", [((5, 12, 4), 2, 3), ((3, 20, 8), 1, 2), ((6, 48, 4), 3, 2),
                                   ((9, 96, 3), 2, 1), ((4, 160, 5), 2, 2)])
def test_apply3d_columns_match_oracle(torch, msr, N, K, C):
    lam, km, cm, x = make_case(np.random.default_rng(5), N, K, C)
    A = msr.NFFTNormalOp(N, dev(torch, lam), dev(torch, km + 1), cmaps=[dev(torch, c) for c in cm])
    ref = toeplitz.apply_normal(N, lam.astype(np.complex128), km, cm.astype(np.complex128),
                                x.astype(np.complex128)).reshape(-1)
    xd = dev(torch, x).reshape(-1)
    x64 = xd.to(torch.complex128)
    y64, y64c = torch.empty_like(x64), torch.empty_like(x64)
    A.A.mul_f64_(y64, x64)
    A.A.mul_f64_(y64c, x64, compact=True)
    e = [rel_err(y.cpu().numpy(), ref) for y in (A @ xd, y64, y64c)]
    print(f"{N} K={K}: f32 {e[0]:.1e} f64 {e[1]:.1e} f64c {e[2]:.1e}", flush=True)
    assert e[0] < 2e-6 and e[1] < 1e-12 and e[2] < 2e-8
