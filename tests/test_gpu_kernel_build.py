"""Kernel construction against the FP64 oracle at the edges of its spreading
(output tiles of 4 cells per dimension, runs of bins that wrap, 1 to 10 row
tiles of pair products) and of its mask: grids of one, two and three bins,
ragged sizes, one sample, samples on the grid's edge, real and complex bases.
The mask is bit-exact, the kernel within 3e-7 (W = 8 spreading, rounded to
ComplexF32), and a construction repeats bit for bit, alone or beside others on
threads and streams of their own (whose temporaries share recycled memory)."""
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


def protocol(N, K, nt, ns, real, seed=0):
    rng = np.random.default_rng(seed)
    trj = rng.uniform(-0.5, 0.5, size=(nt, ns, len(N))).astype(np.float32)
    trj[0, 0] = -0.5
    if ns > 2:
        trj[0, 1] = 0.5
        trj[:, 2:ns // 2] *= np.float32(0.02)  # a dense centre: many samples per tile
    U = rng.normal(size=(K, nt)) + (0 if real else 1j * rng.normal(size=(K, nt)))
    return trj, U.astype(np.float32 if real else np.complex64)


CASES = [
    ((1, 2), 2, 3, 40, False),       # 4N = 4 x 8: below three bins
    ((3, 3), 1, 2, 1, False),        # 12 x 12: three bins, two samples
    ((3, 5), 3, 5, 300, True),
    ((4, 9), 4, 6, 200, False),      # P = 10: two row tiles
    ((16, 15), 12, 4, 100, False),   # P = 78: three groups of four tiles
    ((15, 16), 9, 4, 100, True),     # P = 45 real: three tiles in a group of four
    ((64, 48), 5, 20, 400, False),
    ((3, 4, 5), 3, 4, 300, False),
    ((5, 3, 3), 4, 3, 100, True),
    ((12, 10, 9), 2, 6, 500, False),
]


@pytest.mark.parametrize("N,K,nt,ns,real", CASES)
def test_kernel_matches_oracle(torch, msr, N, K, nt, ns, real):
    trj, U = protocol(N, K, nt, ns, real)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    A = msr.NFFTNormalOp(N, dev(trj), dev(U))
    ref, km = toeplitz.toeplitz_kernel(N, trj, U)
    assert np.array_equal(A.prod.A.kmask_indcs.cpu().numpy() - 1, km)
    lam = A.prod.A.Λ
    e = rel_err(lam.cpu().numpy(), ref)
    print(f"kernel {N} K={K} real={real}: {e:.2e}", flush=True)
    assert e < 3e-7
    again = msr.NFFTNormalOp(N, dev(trj), dev(U)).prod.A.Λ
    assert torch.equal(lam, again)


def test_constructions_on_threads_and_streams(torch, msr):
    jobs = [((24, 20), 3), ((12, 10, 9), 2), ((32, 27), 4), ((16, 16), 5)]
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    inputs = [[dev(a) for a in protocol(N, K, 8, 200, False, seed=i)] for i, (N, K) in enumerate(jobs)]
    want = [msr.NFFTNormalOp(N, *inp).prod.A.Λ for (N, K), inp in zip(jobs, inputs)]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for _ in range(5):
                got = msr.NFFTNormalOp(jobs[i][0], *inputs[i]).prod.A.Λ
                st.synchronize()
                if not torch.equal(got, want[i]):
                    wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_pairs_in_several_chunks(torch, msr):
    """64 x 64 x 64, K = 6: the FP64 grids of 21 pairs exceed the construction's
    budget, so the pairs go in chunks of whole row tiles; every pair has the
    bits of a construction that takes it in one chunk."""
    N = (64, 64, 64)
    trj, U = protocol(N, 6, 3, 400, False)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    build = lambda u: msr.NFFTNormalOp(N, dev(trj), dev(u)).prod.A.Λ
    lam = build(U)
    pairs = [d for d in range(lam.ndim) if lam.shape[d] == 21][0]
    assert torch.equal(lam.narrow(pairs, 0, 15), build(U[:5]))
    assert torch.equal(lam.narrow(pairs, 20, 1).flatten(), build(U[5:]).flatten())


def test_grid_of_more_blocks_than_one_dimension_takes(torch, msr, monkeypatch):
    """256 x 256 x 256: the 1024-point spreading grid has 2^24 output tiles of 256
    threads, one more than a launch takes in one dimension.  Against the tile
    spreading of the same samples (both FP64, rounded to Float32: 1e-7)."""
    N = (256, 256, 256)
    trj, U = protocol(N, 1, 2, 1000, True)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    A = msr.NFFTNormalOp(N, dev(trj), dev(U))
    lam, km = A.prod.A.Λ, A.prod.A.kmask_indcs
    del A
    monkeypatch.setenv("MSR_KERNEL_TILES", "1")
    monkeypatch.setenv("MSR_SPREAD3D_SLAB_BUDGET", "1")
    B = msr.NFFTNormalOp(N, dev(trj), dev(U))
    assert torch.equal(km, B.prod.A.kmask_indcs)
    ref = B.prod.A.Λ.double()
    e = float((lam.double() - ref).norm() / ref.norm())
    print(f"kernel {N}: gather against tiles {e:.2e}", flush=True)
    assert e < 1e-7


def test_less_memory_than_the_larger_budget(torch, msr, monkeypatch):
    """64 x 64 x 64, K = 6 with requests above 3 GiB failing: the 4 GiB grids of 16
    pairs cannot be had, so the pairs go in chunks of 8, with the same bits; the
    failed allocation does not show up in a later call either.  With nothing
    large enough the construction fails as out of memory, and the next works."""
    N = (64, 64, 64)
    trj, U = protocol(N, 6, 3, 400, False)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    build = lambda: msr.NFFTNormalOp(N, dev(trj), dev(U)).prod.A.Λ
    lam = build()
    monkeypatch.setenv("MSR_DEVICE_ALLOC_LIMIT", str(3 << 30))
    assert torch.equal(lam, build())
    monkeypatch.setenv("MSR_DEVICE_ALLOC_LIMIT", str(64 << 20))
    with pytest.raises(Exception, match="out of memory"):
        build()
    monkeypatch.delenv("MSR_DEVICE_ALLOC_LIMIT")
    assert torch.equal(lam, build())


def test_less_memory_than_the_samples_tables(torch, msr, monkeypatch):
    """200 000 samples on a 16 x 15 image with requests above 8 MB failing: the
    gather's 25.6 MB of weights cannot be had, the tile spreading takes the
    construction (both FP64, rounded to ComplexF32: 1e-7)."""
    N = (16, 15)
    trj, U = protocol(N, 3, 4, 50000, False)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    trj, U = dev(trj), dev(U)
    build = lambda: msr.NFFTNormalOp(N, trj, U).prod.A
    A = build()
    monkeypatch.setenv("MSR_KERNEL_TILES", "1")
    T = build()
    monkeypatch.delenv("MSR_KERNEL_TILES")
    monkeypatch.setenv("MSR_DEVICE_ALLOC_LIMIT", str(8 << 20))
    B = build()
    assert torch.equal(A.kmask_indcs, B.kmask_indcs)
    assert torch.equal(B.Λ, T.Λ)
    assert rel_err(A.Λ.cpu().numpy(), B.Λ.cpu().numpy()) < 1e-7
