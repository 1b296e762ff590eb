"""The near field and the gradient in root cells of any side: particles on an
integer lattice in [-2e6, 2e6]^3, one of them at (1e6, 1e6, 1e6), the corner of
eight leaves, and the same lattice scaled to a side of 4e-6.  Sources that only
fill up a kernel's chunks must add nothing wherever the targets are.  Zero
operators leave the near field alone: against numpy sums in fp64 (relative L2
1e-5 fp32, 1e-12 fp64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = {"s": 1e-5, "d": 1e-12}
SPECIAL = 137  # the particle at (1e6, 1e6, 1e6)


def _lattice(scale, dt):
    """401 distinct lattice points, a leaf of depth 2 holding about six; their leaves."""
    rng = np.random.default_rng(8)
    flat = rng.choice(400 ** 3, size=401, replace=False)
    p = np.stack([flat // 160_000, flat // 400 % 400, flat % 400], axis=1) * 10_000.0 - 2e6 + 5_000.0
    p[SPECIAL] = 1e6
    cell = np.minimum((p / 1e6 + 2).astype(int), 3)
    return (p * scale).astype(dt), cell


def _near(pos, cell, q, g=None):
    """Potentials of q; with g, dq and dx of the gradient."""
    d = pos[None, :, :] - pos[:, None, :]
    r = np.linalg.norm(d, axis=2)
    w = np.where((r > 0) & (np.abs(cell[None] - cell[:, None]) <= 1).all(axis=2), 1 / np.where(r > 0, r, 1), 0)
    if g is None:
        return q @ w
    c = g.T @ q + q.T @ g
    return g @ w, np.einsum("ij,ijk->ik", c * w ** 3, d)


def _plan(prec, pos, L, nrhs, **opts):
    import bbfmmongpu_amd as B
    dt = B.dtype(prec)
    plan = B.Plan(pos, 4, np.zeros(64 * 32, dt), np.zeros(316 * 1024, dt), nrhs=nrhs, L=L, prec=prec)
    assert plan.maxlev == 2
    return plan.set(scheme=B.SCHEME_IJ, **opts)


def _compare(out, ref, tol):
    assert np.isfinite(out).all()
    assert np.linalg.norm(out - ref) / np.linalg.norm(ref) < tol
    k = np.abs(ref[..., SPECIAL])
    assert (np.abs(out[..., SPECIAL] - ref[..., SPECIAL]) <= 100 * tol * np.maximum(k, np.abs(ref).max())).all()


@pytest.mark.parametrize("scale", [1.0, 1e-12])
@pytest.mark.parametrize("prec,nrhs,opts", [
    ("s", 1, {}), ("s", 4, {}), ("s", 7, {}), ("s", 16, {}), ("d", 1, {}), ("d", 4, {}), ("d", 16, {}),
    ("s", 12, dict(form=1)), ("s", 16, dict(form=1)), ("s", 16, dict(form=1, flat_loads=True)),
    ("s", 16, dict(form=1, p2p_form=1)),
])
def test_solve(prec, nrhs, opts, scale, cuda):
    import torch
    import bbfmmongpu_amd as B
    pos, cell = _lattice(scale, B.dtype(prec))
    rng = np.random.default_rng(nrhs)
    q = rng.uniform(-1, 1, (nrhs, pos.shape[0])).astype(pos.dtype)
    plan = _plan(prec, pos, 4e6 * scale, nrhs, output="potential", **opts)
    ref = _near(pos.astype(np.float64), cell, q.astype(np.float64))
    tol = 3e-5 if opts.get("p2p_form") else TOL[prec]  # split-BF16 sum: its own bound
    qd = torch.from_numpy(q).to(cuda)
    _compare(plan.solve(qd).cpu().numpy().astype(np.float64), ref, tol)
    # the copy that the 16-vector kernels read is filled up again when the particles move
    rows = np.arange(pos.shape[0]) != SPECIAL
    moved = pos.copy()
    moved[rows] += pos.dtype.type(1000 * scale)
    plan.update_positions(moved)
    ref = _near(moved.astype(np.float64), cell, q.astype(np.float64))
    _compare(plan.solve(qd).cpu().numpy().astype(np.float64), ref, tol)
    plan.close()


@pytest.mark.parametrize("scale", [1.0, 1e-12])
@pytest.mark.parametrize("prec,m", [("s", 1), ("s", 3), ("s", 8), ("s", 16), ("d", 1), ("d", 8)])
def test_gradient(prec, m, scale, cuda):
    import torch
    import bbfmmongpu_amd as B
    pos, cell = _lattice(scale, B.dtype(prec))
    rng = np.random.default_rng(m)
    q, g = (rng.uniform(-1, 1, (m, pos.shape[0])).astype(pos.dtype) for _ in range(2))
    plan = _plan(prec, pos, 4e6 * scale, 2 * m)
    dq, dx = plan.gradient(torch.from_numpy(q).to(cuda), torch.from_numpy(g).to(cuda))
    plan.close()
    rq, rx = _near(pos.astype(np.float64), cell, q.astype(np.float64), g.astype(np.float64))
    _compare(dq.cpu().numpy().astype(np.float64), rq, TOL[prec])
    _compare(dx.cpu().numpy().astype(np.float64).T, rx.T, TOL[prec])
