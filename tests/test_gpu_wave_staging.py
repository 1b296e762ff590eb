"""Kernels whose waves hand sources or sums from lane to lane through LDS
(k_p2p, k_near_grad, k_m2l_list_packed): leaves and lists that refill a wave's
part of LDS many times, whose last fill is whole or partial.  Every pass gives
the bits of the first, beside other work in flight on another stream."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _same(run, cuda):
    import torch
    first = [t.clone() for t in run()]
    other = torch.cuda.Stream()
    a = torch.rand(1024, 1024, device=cuda)
    torch.cuda.synchronize()
    for _ in range(10):
        with torch.cuda.stream(other):
            for _ in range(4):
                a = a @ a
                a = a / a.max()
        assert all(torch.equal(x, y) for x, y in zip(first, run()))
    torch.cuda.synchronize()
    assert all(bool(torch.isfinite(t).all()) for t in first)


@pytest.mark.parametrize("prec", ["s", "d"])
@pytest.mark.parametrize("N,nrhs", [(8191, 1), (8192, 4), (30_001, 2), (20_011, 7), (3001, 1)])
def test_near_field(prec, N, nrhs, cuda):
    import torch
    import bbfmmongpu_amd as B
    dt = B.dtype(prec)
    rng = np.random.default_rng(N)
    lmod = -6 if N == 8192 else 0  # leaves of 128
    plan = B.Plan(rng.random((N, 3)) - 0.5, 4, np.zeros(64 * 32, dt), np.zeros(316 * 1024, dt), nrhs=nrhs, lmod=lmod,
                  prec=prec).set(scheme=B.SCHEME_IJ)
    q = torch.from_numpy(rng.uniform(-1, 1, (nrhs, N)).astype(dt)).to(cuda)
    _same(lambda: [plan.solve(q)], cuda)
    plan.close()


@pytest.mark.parametrize("prec,m", [("s", 1), ("s", 3), ("s", 8), ("s", 16), ("d", 2), ("d", 8)])
def test_gradient(prec, m, cuda):
    import torch
    import bbfmmongpu_amd as B
    dt = B.dtype(prec)
    rng = np.random.default_rng(m)
    N = 20_011
    plan = B.Plan(rng.random((N, 3)) - 0.5, 4, np.zeros(64 * 32, dt), np.zeros(316 * 1024, dt), nrhs=2 * m,
                  prec=prec).set(scheme=B.SCHEME_IJ)
    q, g = (torch.from_numpy(rng.uniform(-1, 1, (m, N)).astype(dt)).to(cuda) for _ in range(2))
    _same(lambda: plan.gradient(q, g), cuda)
    plan.close()


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("nrhs", [1, 5])
def test_list_m2l(nrhs, form, ops4, cuda):
    import torch
    import bbfmmongpu_amd as B
    from bbfmmongpu_amd import workloads as W
    U, K, _ = ops4
    rng = np.random.default_rng(nrhs)
    plan = B.Plan.batch([W.plummer(9001, rng), W.sphere_surface(12_000, rng)], 4, U, K, nrhs=nrhs,
                        depths=[5, 5]).set(scheme=B.SCHEME_IJ, form=form)
    q = torch.from_numpy(rng.uniform(-1, 1, (nrhs, 21_001)).astype(np.float32)).to(cuda)
    _same(lambda: [plan.solve(q)], cuda)
    plan.close()
