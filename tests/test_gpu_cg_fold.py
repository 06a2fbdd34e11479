"""The scalar finish of a CG iteration is folded into the next one's search
direction within a sequence of launches: however the iterations are cut into
sequences (one graph, one device loop, a batch, batch steps of 1 or 3), the
iterates, the iteration count, the residual and the stop are the same bit for
bit, with stops by tolerance inside a sequence, at its end, at the start and
by the iteration limit."""
import numpy as np
import pytest

from conftest import load_package
from test_gpu_apply import make_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


@pytest.mark.parametrize("precision", ["f32", "mixed", "f64", "f64c"])
@pytest.mark.parametrize("maxiter,reltol", [(0, 0.0), (1, 0.0), (2, 0.0), (7, 0.0), (12, 0.3), (12, 0.05), (5, 2.0)])
def test_sequences_agree(torch, precision, maxiter, reltol):
    msr = load_package()
    lam, km, cm, x = make_case(np.random.default_rng(5), (24, 20), 3, 4)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    A = msr.NFFTNormalOp((24, 20), dev(lam), dev(km + 1), cmaps=[dev(c) for c in cm])
    b = A @ dev(x).reshape(-1)
    kw = dict(maxiter=maxiter, reltol=reltol, precision=precision)
    want, info = msr.cg_(torch.empty_like(b), A, b, initially_zero=True, mode="device", log=True, **kw)
    got, g = msr.cg_(torch.empty_like(b), A, b, initially_zero=True, mode="graph", log=True, **kw)
    assert torch.equal(got, want) and g == info
    assert info["iters"] <= maxiter
    B = msr.NFFTNormalOpBatch([A])
    for mode in ("device", "graph"):
        xs, g = B.cg_([torch.empty_like(b)], [b], initially_zero=True, mode=mode, log=True, **kw)
        assert torch.equal(xs[0], want) and g["iters"] == [info["iters"]] and g["residual"] == [info["residual"]]
    for step in (1, 3):
        xs = [torch.empty_like(b)]
        B.cg_start(xs, [b], maxiter, reltol=reltol, precision=precision)
        for _ in range(0, maxiter + 3, step):
            B.cg_iterate(step)
        its, res, done = B.cg_status()
        B.cg_finish()
        torch.cuda.synchronize()
        assert torch.equal(xs[0], want) and its == [info["iters"]] and res == [info["residual"]] and done == [True]
