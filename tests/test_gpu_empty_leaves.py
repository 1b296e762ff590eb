"""Trees with more empty leaves than full ones: the full-precision dense-grid
M2L leaves out the offsets that see no particles.  Clusters, a sphere, one
occupied leaf; vector counts whose tiles end inside a row of cells; against the
same plan's basic scheme in fp64 (relative L2 1e-5 fp32, 1e-12 fp64)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
TOL = {"s": 1e-5, "d": 1e-12}


def _points(kind, N, rng):
    from bbfmmongpu_amd import workloads as W
    if kind == "sphere":
        return W.sphere_surface(N, rng)
    if kind == "leaf":
        return rng.random((N, 3)) * 0.01 + 0.2
    c = rng.random((7, 3)) * 0.9 - 0.45
    return np.clip(c[rng.integers(7, size=N)] + rng.normal(size=(N, 3)) * 0.01, -0.5, 0.4999)


@pytest.mark.parametrize("kind,n,depth,nrhs,prec,form", [
    ("sphere", 4, 5, 4, "s", 0), ("sphere", 4, 4, 1, "d", 0), ("sphere", 5, 4, 3, "s", 0), ("sphere", 4, 4, 16, "s", 2),
    ("clusters", 4, 5, 1, "s", 0), ("clusters", 4, 4, 7, "d", 0), ("clusters", 6, 3, 2, "s", 0),
    ("leaf", 4, 4, 1, "s", 0), ("leaf", 4, 2, 5, "s", 2)])
def test_empty_leaves(kind, n, depth, nrhs, prec, form, cuda):
    import torch
    import bbfmmongpu_amd as B
    dt = B.dtype(prec)
    N = 4001
    rng = np.random.default_rng(n + depth)
    pos = _points(kind, N, rng).astype(np.float32)
    q = (rng.random((nrhs, N)) - 0.5).astype(np.float32)
    U, K, _ = O.operators(n)
    lmod = next(m for m in range(-8, 9) if B.maxlev(N, m) == depth)
    U, K = U.astype(np.float32), K.astype(np.float32)

    def solve(prec, **opts):
        t = B.dtype(prec)
        plan = B.Plan(pos.astype(t), n, U.astype(t), K.astype(t), nrhs=nrhs, lmod=lmod, prec=prec).set(**opts)
        assert plan.maxlev == depth
        phi = plan.solve(torch.from_numpy(q.astype(t)).to(cuda)).cpu().numpy().reshape(nrhs, N)
        plan.close()
        return phi.astype(np.float64)

    ref = solve("d", scheme=B.SCHEME_BA)
    got = solve(prec, scheme=B.SCHEME_IJ, form=form)
    err = max(O.rel_l2(ref[j], got[j]) for j in range(nrhs))
    print(f"{kind} n={n} depth={depth} nrhs={nrhs} {prec}: {err:.2e}", flush=True)
    assert err < TOL[prec]
