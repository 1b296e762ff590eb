"""The near field of 1 to 8 vectors (k_p2p) and of 16 (k_p2p_seg16) at the sizes where its tiles,
staging and splits change: leaves of 0, 1, 15 .. 17, 63 .. 65 and hundreds of
particles, coincident particles, every tile and wave count that the size rule
picks, vector counts that leave part of a group.  Zero operators leave the
near field alone: against numpy sums over the neighbour leaves in fp64
(relative L2 1e-5 fp32, 1e-12 fp64, as the parity tests)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = {"s": 1e-5, "d": 1e-12}


def _near(pos, q, depth, targets):
    """Potentials of the targets from the particles of their 27 neighbour leaves."""
    g = 2 ** depth
    cell = np.minimum(((pos + 0.5) * g).astype(int), g - 1)
    out = np.empty((q.shape[0], targets.size))
    for k, i in enumerate(targets):
        near = np.flatnonzero((np.abs(cell - cell[i]) <= 1).all(axis=1))
        d = np.linalg.norm(pos[near] - pos[i], axis=1)
        w = np.zeros_like(d)
        w[d > 0] = 1 / d[d > 0]
        out[:, k] = q[:, near] @ w
    return out


def _check(prec, pos, depth, nrhs, cuda, ntargets, output="potential", **opts):
    import torch
    import bbfmmongpu_amd as B
    dt = B.dtype(prec)
    N = pos.shape[0]
    pos = pos.astype(dt)
    rng = np.random.default_rng(3)
    q = (rng.random((nrhs, N)) - 0.5).astype(dt)
    lmod = depth - (B.maxlev(N) if B.maxlev(N) > 2 else 0)
    while B.maxlev(N, lmod) > depth:
        lmod -= 1
    while B.maxlev(N, lmod) < depth:
        lmod += 1
    plan = B.Plan(pos, 4, np.zeros(64 * 32, dt), np.zeros(316 * 1024, dt), nrhs=nrhs, lmod=lmod, prec=prec)
    assert plan.maxlev == depth
    plan.set(scheme=B.SCHEME_IJ, output=output, **opts)
    phi = plan.solve(torch.from_numpy(q).to(cuda)).cpu().numpy().reshape(nrhs, N)
    plan.close()
    t = rng.choice(N, size=min(ntargets, N), replace=False)
    ref = _near(pos.astype(np.float64), q.astype(np.float64), depth, t)
    if output == "q_phi":
        ref = ref * q[:, t]
    num = np.linalg.norm(phi[:, t] - ref, axis=1) / np.linalg.norm(ref, axis=1)
    print(f"{prec} N={N} depth={depth} nrhs={nrhs}: {num.max():.2e}", flush=True)
    assert num.max() < TOL[prec]


def _uneven(seed):
    """Depth 2: leaves of the counts where tiles and staged pieces end, the others empty."""
    rng = np.random.default_rng(seed)
    counts = {0: 1, 1: 15, 2: 16, 3: 17, 5: 31, 6: 33, 8: 63, 9: 64, 10: 65, 13: 130, 20: 260, 42: 49, 63: 7}
    pos = []
    for leaf, c in counts.items():
        corner = np.array([leaf // 16, leaf // 4 % 4, leaf % 4]) / 4 - 0.5
        pos.append(corner + rng.random((c, 3)) / 4)
    pos = np.concatenate(pos)
    pos[20] = pos[19]  # coincident particles do not act on each other
    return pos


@pytest.mark.parametrize("prec", ["s", "d"])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 4, 5, 8, 9])
def test_uneven_leaves(prec, nrhs, cuda):
    _check(prec, _uneven(nrhs), 2, nrhs, cuda, 200, output="q_phi" if nrhs == 2 else "potential")


@pytest.mark.parametrize("prec,N,depth,nrhs", [
    ("s", 20_000, 3, 1), ("s", 20_000, 3, 4), ("s", 20_000, 3, 7),  # 512 leaves: 2 tiles, 8 or 4 waves
    ("s", 30_001, 4, 1), ("s", 30_001, 4, 2), ("s", 110_001, 4, 1), ("s", 110_001, 4, 6),  # 4096: 2 and 4 tiles
    ("s", 60_000, 5, 1), ("s", 60_000, 5, 4), ("s", 790_000, 5, 1), ("s", 790_000, 5, 3),  # 32768: one wave
    ("d", 20_000, 3, 1), ("d", 20_000, 3, 7), ("d", 30_001, 4, 1), ("d", 30_001, 4, 4), ("d", 60_000, 5, 2),
])
def test_size_rules(prec, N, depth, nrhs, cuda):
    pos = np.random.default_rng(N).random((N, 3)) - 0.5
    _check(prec, pos, depth, nrhs, cuda, 100)


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("N,depth,nrhs", [
    (0, 2, 16), (0, 2, 12), (20_000, 3, 16), (30_001, 4, 16),  # 64 leaves: 8 waves; 512, 4096: 4 waves
    (60_000, 5, 16), (300_000, 5, 13), (20_000, 3, 33),  # 32768: 4 waves below 8 a leaf, else 1; two blocks of 16 and 1
])
def test_sixteen(N, depth, nrhs, flat, cuda):
    import bbfmmongpu_amd as B
    pos = np.random.default_rng(N).random((N, 3)) - 0.5 if N else _uneven(nrhs)
    _check("s", pos, depth, nrhs, cuda, 100, form=B.FORM_BF16X2, flat_loads=flat)
