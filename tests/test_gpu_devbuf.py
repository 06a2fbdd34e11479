"""Device memory kept for the library's next buffers: bounded, given back on
request, and nothing large kept while the device is nearly full."""
import gc
import threading

import numpy as np
import pytest

from conftest import load_package

pytestmark = pytest.mark.gpu

N, K = (64, 64, 64), 3          # a construction's FP64 grids: 1.6 and 0.8 GB
GRIDS = 6 * 256 ** 3 * 16 * 3 // 2


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


@pytest.fixture(scope="module")
def msr():
    return load_package()


def kernel(torch, msr):
    rng = np.random.default_rng(0)
    trj = torch.from_numpy(rng.uniform(-0.5, 0.5, size=(4, 200, 3)).astype(np.float32)).cuda()
    U = torch.from_numpy(rng.normal(size=(K, 4)).astype(np.float32)).cuda()
    lam = msr.NFFTNormalOp(N, trj, U).prod.A.Λ
    gc.collect()
    torch.cuda.synchronize()
    return lam


def available(torch):
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


def test_trim_gives_idle_memory_back(torch, msr):
    first = kernel(torch, msr)       # tables and contexts that stay
    msr.trim()
    before = available(torch)
    again = kernel(torch, msr)
    assert torch.equal(first, again)
    del again
    kept = before - available(torch)
    freed = msr.trim()
    after = available(torch)
    print(f"kept {kept >> 20} MiB, freed {freed >> 20} MiB, {before - after >> 20} MiB remain", flush=True)
    assert freed >= GRIDS and kept >= GRIDS
    assert before - after < 32 << 20
    assert msr.trim() == 0
    assert torch.equal(first, kernel(torch, msr))


def test_nothing_large_stays_while_the_device_is_nearly_full(torch, msr):
    first = kernel(torch, msr)
    msr.trim()
    free, total = torch.cuda.mem_get_info()
    rest = total // 16
    if free < rest:
        pytest.skip("device in use")
    try:
        hold = torch.empty(free - rest, dtype=torch.uint8, device="cuda")
    except torch.cuda.OutOfMemoryError:
        pytest.skip("device in use")
    try:
        assert torch.equal(first, kernel(torch, msr))
        freed = msr.trim()
    finally:
        del hold
        torch.cuda.empty_cache()
    print(f"freed {freed >> 20} MiB", flush=True)
    assert freed < GRIDS // 4


def test_an_operator_takes_what_its_footprint_says(torch, msr):
    """The construction leaves idle blocks a fifth larger than the operator's
    intermediates (120 MiB, 100 MiB needed): its buffers take blocks of their own
    size, at most 1/64 and 64 KiB more than its footprint counts."""
    n, k = (256, 256), 5
    trj = torch.from_numpy(msr.synth.traj_2d_radial_goldenratio(512, 8, 40)).cuda()
    U = torch.from_numpy(msr.synth.t2_basis(40, k)).cuda()
    maps = [torch.randn(n[::-1], dtype=torch.complex64, device="cuda") for _ in range(20)]
    msr.trim()
    A = msr.NFFTNormalOp(n, trj, U, cmaps=maps)
    gc.collect()
    own, kernel_bytes = msr.footprint(A, "f32")
    msr.trim()
    with_op = available(torch)
    del A
    gc.collect()
    msr.trim()
    used = available(torch) - with_op
    print(f"used {used / 2**20:.1f} MiB, footprint {(own + kernel_bytes) / 2**20:.1f} MiB", flush=True)
    assert used <= (own + kernel_bytes) * 65 / 64 + (1 << 20)


def test_allocations_beside_a_capture(torch, msr):
    """One thread captures CG graphs of new operators while another constructs and
    destroys operators: neither fails, and the solves keep their bits."""
    rng = np.random.default_rng(3)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()

    def protocol(n, k, nt, ns):
        return n, dev(rng.uniform(-0.5, 0.5, size=(nt, ns, len(n))).astype(np.float32)), \
            dev(rng.normal(size=(k, nt)).astype(np.float32))

    solve, build = protocol((32, 24), 2, 8, 200), protocol((16, 16, 12), 2, 8, 300)
    b = torch.randn(2 * 32 * 24, dtype=torch.complex64, device="cuda")

    def solved():
        return msr.cg(msr.NFFTNormalOp(*solve), b, maxiter=20, reltol=0.0, mode="graph")

    want = solved()
    msr.NFFTNormalOp(*build)      # tables
    torch.cuda.synchronize()
    failures, stop = [], threading.Event()

    def guarded(body):
        st = torch.cuda.Stream()
        try:
            with torch.cuda.stream(st):
                body(st)
        except Exception as e:
            failures.append(repr(e))

    def solver(st):
        try:
            for _ in range(150):
                x = solved()
                st.synchronize()
                if not torch.equal(x, want):
                    failures.append("bits")
        finally:
            stop.set()

    def builder(st):
        while not stop.is_set():
            msr.NFFTNormalOp(*build)

    threads = [threading.Thread(target=guarded, args=(f,)) for f in (solver, builder)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures[:3]


def test_destroying_a_handle_waits_for_the_device(torch, msr):
    """Its buffers go to the next caller, so work queued on any stream (here 100
    matrix products, about 100 ms) has ended when a handle is gone."""
    trj = torch.zeros((2, 50, 2), dtype=torch.float32, device="cuda")
    a = torch.randn(4096, 4096, device="cuda")
    a @ a
    traj = msr.plan_trajectory(trj)
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    done = torch.cuda.Event()
    with torch.cuda.stream(st):
        for _ in range(100):
            b = a @ a
        done.record(st)
    running = not done.query()
    del traj
    gc.collect()
    assert running and done.query()
    del b
