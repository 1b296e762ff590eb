"""The near field of the gradient (k_near_grad): position gradient and
returned potentials of 1 to 17 vectors on uneven leaves (counts around the
ends of tiles and chunks, empty leaves, coincident particles) and at the sizes
where its wave split changes.  Zero operators leave the near field alone:
against numpy sums in fp64 (relative L2 1e-5 fp32, 1e-12 fp64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = {"s": 1e-5, "d": 1e-12}


def _near(pos, q, g, depth, targets):
    side = 2 ** depth
    cell = np.minimum(((pos + 0.5) * side).astype(int), side - 1)
    dq, dx = np.empty((q.shape[0], targets.size)), np.empty((targets.size, 3))
    for k, i in enumerate(targets):
        near = np.flatnonzero((np.abs(cell - cell[i]) <= 1).all(axis=1))
        d = pos[near] - pos[i]
        r = np.linalg.norm(d, axis=1)
        w = np.zeros_like(r)
        w[r > 0] = 1 / r[r > 0]
        dq[:, k] = g[:, near] @ w
        c = g[:, i] @ q[:, near] + q[:, i] @ g[:, near]
        dx[k] = (c * w ** 3) @ d
    return dq, dx


def _check(prec, pos, depth, m, cuda, ntargets):
    import torch
    import bbfmmongpu_amd as B
    dt = B.dtype(prec)
    pos = pos.astype(dt)
    N = pos.shape[0]
    rng = np.random.default_rng(m)
    q, g = ((rng.random((m, N)) - 0.5).astype(dt) for _ in range(2))
    lmod = next(k for k in range(-6, 8) if B.maxlev(N, k) == depth)
    plan = B.Plan(pos, 4, np.zeros(64 * 32, dt), np.zeros(316 * 1024, dt), nrhs=2 * m, lmod=lmod, prec=prec)
    plan.set(scheme=B.SCHEME_IJ, form=B.FORM_BF16X2 if prec == "s" and m >= 8 else B.FORM_PLAIN)
    dq, dx = plan.gradient(torch.from_numpy(q).to(cuda), torch.from_numpy(g).to(cuda))
    dq, dx = dq.cpu().numpy().reshape(m, N), dx.cpu().numpy()
    plan.close()
    t = rng.choice(N, size=min(ntargets, N), replace=False)
    rq, rx = _near(pos.astype(np.float64), q.astype(np.float64), g.astype(np.float64), depth, t)
    eq = np.linalg.norm(dq[:, t] - rq) / np.linalg.norm(rq)
    ex = np.linalg.norm(dx[t] - rx) / np.linalg.norm(rx)
    print(f"{prec} N={N} depth={depth} m={m}: dq {eq:.2e} dx {ex:.2e}", flush=True)
    assert eq < TOL[prec] and ex < TOL[prec]


@pytest.mark.parametrize("prec", ["s", "d"])
@pytest.mark.parametrize("m", [1, 2, 3, 5, 8, 9, 16, 17])
def test_uneven_leaves(prec, m, cuda):
    rng = np.random.default_rng(m)
    counts = {0: 1, 1: 15, 2: 16, 3: 17, 5: 31, 6: 33, 8: 63, 9: 64, 10: 65, 13: 130, 20: 260, 42: 49, 63: 7}
    pos = []
    for leaf, c in counts.items():
        corner = np.array([leaf // 16, leaf // 4 % 4, leaf % 4]) / 4 - 0.5
        pos.append(corner + rng.random((c, 3)) / 4)
    pos = np.concatenate(pos)
    pos[20] = pos[19]  # coincident particles do not act on each other
    _check(prec, pos, 2, m, cuda, 200)


@pytest.mark.parametrize("prec,N,depth,m", [
    ("s", 20_000, 3, 8), ("s", 30_000, 4, 16), ("s", 30_000, 4, 2), ("s", 50_000, 5, 1), ("s", 50_000, 5, 8),
    ("s", 50_000, 5, 12), ("d", 30_000, 4, 8), ("d", 50_000, 5, 3),
])
def test_size_rules(prec, N, depth, m, cuda):
    _check(prec, np.random.default_rng(N).random((N, 3)) - 0.5, depth, m, cuda, 100)
