"""Solves of fewer than 16 vectors: P2M gathers the charges, P2P scatters the
potentials, and the M2M and L2L of levels 2 and 3 run in one launch each
(n = 3, 4).  Depths with none, one and two levels above those, sparse leaves,
potentials over the charges; against the oracle with the usual bounds
(relative L2 1e-5 fp32, 1e-12 fp64)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
TOL = {"s": 1e-5, "d": 1e-12}


@pytest.mark.parametrize("prec", ["s", "d"])
@pytest.mark.parametrize("n,depth,nrhs", [(4, 2, 2), (4, 3, 1), (4, 4, 5), (4, 5, 1), (3, 4, 3), (3, 5, 1), (5, 4, 1)])
def test_direct_solve(n, depth, nrhs, prec, cuda):
    import torch
    import bbfmmongpu_amd as B
    dt = B.dtype(prec)
    N = 3001
    rng = np.random.default_rng(depth)
    # fp32 positions in both precisions: no leaf changes with the type
    pos = (rng.random((N, 3)) - 0.5).astype(np.float32).astype(np.float64)
    q = (rng.random((nrhs, N)) - 0.5).astype(dt)
    U, K, _ = O.operators(n)
    lmod = next(m for m in range(-8, 9) if B.maxlev(N, m) == depth)
    plan = B.Plan(pos.astype(dt), n, U.astype(dt), K.astype(dt), nrhs=nrhs, lmod=lmod, prec=prec)
    assert plan.maxlev == depth
    phi = torch.from_numpy(q).to(cuda)
    plan.solve(phi, phi)
    phi = phi.cpu().numpy().reshape(nrhs, N)
    plan.close()
    tree = O.Tree(pos, 0, "d", maxlev=depth)
    Ud, Kd = U.astype(dt).astype(np.float64), K.astype(dt).astype(np.float64)
    for j in range(nrhs):
        ref = O.fmm(tree, q[j].astype(np.float64), n, Ud, Kd, scheme="basic", l2p_exact=True)
        err = O.rel_l2(ref["phi"], phi[j])
        print(f"{prec} n={n} depth={depth} rhs={j}: {err:.2e}", flush=True)
        assert err < TOL[prec]
