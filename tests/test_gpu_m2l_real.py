"""The full-precision dense-grid M2L (k_m2l_real) at the edges of its tiles
and of its block shapes: ranks around multiples of 16, vector counts that
leave partial column tiles, every block shape the size rules pick, the
pointer form, and M and L at any alignment.  Against the list kernel of the
basic scheme in fp64 on the same values; tolerances as the parity tests'
(relative L2 1e-5 fp32, 1e-12 fp64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = {"s": 1e-5, "d": 1e-12}
ORDER = {1: 3, 15: 3, 16: 3, 17: 3, 31: 4, 32: 4, 33: 4, 48: 4, 62: 4, 108: 5, 171: 6, 256: 7, 510: 8}

# (prec, rank, depth, vectors): the comment names tile rows x columns of the block
CASES = [
    ("s", 1, 2, 1), ("s", 15, 3, 3), ("s", 16, 4, 17),  # 1x1, 1x1, 1x2 (one rank tile)
    ("s", 17, 2, 1), ("s", 32, 2, 16), ("s", 32, 4, 1),  # 1x1, 1x1, 1x2
    ("s", 31, 3, 5), ("s", 32, 4, 3), ("s", 32, 4, 16), ("s", 32, 4, 130),  # 1x1, 2x2, 2x2, 2x4
    ("s", 33, 3, 1), ("s", 48, 4, 1), ("s", 62, 4, 1), ("s", 62, 4, 3),  # 1x1, 1x2, 1x2, 1x4
    ("s", 108, 3, 1), ("s", 108, 4, 1), ("s", 108, 3, 16), ("s", 171, 4, 3),  # 1x1, 1x4, 1x4, 2x4
    ("s", 256, 3, 1), ("s", 256, 3, 10), ("s", 256, 3, 58), ("s", 510, 2, 2),  # 1x2, 2x4, 4x4, 1x1
    ("d", 15, 3, 1), ("d", 32, 2, 1), ("d", 32, 4, 1), ("d", 31, 4, 5),  # 1x1, 1x1, 1x2, 2x1
    ("d", 33, 4, 1), ("d", 108, 4, 1), ("d", 171, 3, 16), ("d", 256, 2, 1),  # 1x2, 1x4, 4x2, 1x1
]


def _m2l(B, prec, n, r, depth, nrhs, K, M, cuda, off, **opts):
    import torch
    dt = B.dtype(prec)
    # a point per leaf corner is enough: the M2L only needs the tree's depth
    pos = np.random.default_rng(0).random((64, 3)) - 0.5
    plan = B.Plan(pos, n, np.zeros(n ** 3 * r, dt), K.astype(dt), nrhs=nrhs, lmod=depth, prec=prec).set(**opts)
    assert plan.maxlev == depth and plan.r == r
    Md = torch.zeros(M.size + off, dtype=torch.float32 if prec == "s" else torch.float64, device=cuda)[off:]
    Md.copy_(torch.from_numpy(M.astype(dt).ravel()))
    Ld = torch.zeros(M.size + off, dtype=Md.dtype, device=cuda)[off:]
    plan.m2l(Md, Ld)
    out = Ld.cpu().numpy().reshape(M.shape)
    plan.close()
    return out


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("prec,r,depth,nrhs", CASES)
def test_against_list_kernel(prec, r, depth, nrhs, flat, cuda):
    import bbfmmongpu_amd as B
    n = ORDER[r]
    ncell = (8 ** (depth + 1) - 1) // 7
    rng = np.random.default_rng(r * 100 + nrhs)
    K = rng.standard_normal(316 * r * r, dtype=np.float32)
    M = rng.standard_normal((nrhs, ncell, r), dtype=np.float32)
    ref = _m2l(B, "d", n, r, depth, nrhs, K, M, cuda, 0, scheme=B.SCHEME_BA)
    got = _m2l(B, prec, n, r, depth, nrhs, K, M, cuda, 1, scheme=B.SCHEME_IJ, form=B.FORM_PLAIN, flat_loads=flat)
    first = 9  # cells of levels 0 and 1 are not written
    assert not got[:, :first].any()
    num = np.linalg.norm((got - ref)[:, first:], axis=(1, 2))
    err = (num / np.linalg.norm(ref[:, first:], axis=(1, 2))).max()
    print(f"{prec} r={r} depth={depth} nrhs={nrhs} flat={flat}: {err:.2e}", flush=True)
    assert err < TOL[prec]


@pytest.mark.parametrize("prec,r,depth,nrhs,opts", [c + (dict(form=0),) for c in CASES] + [
    ("s", 32, 2, 1, dict(form=2, variant=2)), ("s", 32, 3, 16, dict(form=2)), ("s", 32, 3, 16, dict(form=2, variant=2)),
    ("s", 32, 3, 5, dict(form=2, variant=3)), ("s", 32, 4, 16, dict(form=2, variant=3)), ("s", 256, 3, 16, dict(form=2)),
])
def test_pointer_form_same_bits(prec, r, depth, nrhs, opts, cuda):
    """Only the addressing differs: the same column tiles, offset slices and order of the sums."""
    import bbfmmongpu_amd as B
    ncell = (8 ** (depth + 1) - 1) // 7
    rng = np.random.default_rng(r + nrhs)
    K = rng.standard_normal(316 * r * r, dtype=np.float32)
    M = rng.standard_normal((nrhs, ncell, r), dtype=np.float32)
    out = [_m2l(B, prec, ORDER[r], r, depth, nrhs, K, M, cuda, 0, scheme=B.SCHEME_IJ, flat_loads=flat, **opts)
           for flat in (False, True)]
    assert np.abs(out[0]).max() > 0
    assert np.array_equal(out[0], out[1])


def test_pointer_form_same_bits_many_empty_leaves(ops4, cuda):
    """The same where offsets without particles are left out."""
    import torch
    import bbfmmongpu_amd as B
    from bbfmmongpu_amd import workloads as W
    U, K, _ = ops4
    rng = np.random.default_rng(2)
    pos = W.sphere_surface(20_001, rng)
    for nrhs in (1, 4):
        q = torch.from_numpy(rng.uniform(-1, 1, (nrhs, 20_001)).astype(np.float32)).to(cuda)
        out = []
        for flat in (False, True):
            plan = B.Plan(pos, 4, U, K, nrhs=nrhs, lmod=1).set(scheme=B.SCHEME_IJ, flat_loads=flat)
            out.append(plan.solve(q).cpu().numpy())
            plan.close()
        assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("variant,nrhs", [(0, 16), (2, 16), (3, 16), (2, 3), (3, 5)])
def test_fp32_form_variants(variant, nrhs, cuda):
    import bbfmmongpu_amd as B
    r, depth = 32, 3
    ncell = (8 ** (depth + 1) - 1) // 7
    rng = np.random.default_rng(variant)
    K = rng.standard_normal(316 * r * r, dtype=np.float32)
    M = rng.standard_normal((nrhs, ncell, r), dtype=np.float32)
    ref = _m2l(B, "d", 4, r, depth, nrhs, K, M, cuda, 0, scheme=B.SCHEME_BA)
    got = _m2l(B, "s", 4, r, depth, nrhs, K, M, cuda, 0, scheme=B.SCHEME_IJ, form=B.FORM_FP32MFMA, variant=variant)
    err = np.linalg.norm((got - ref)[:, 9:]) / np.linalg.norm(ref[:, 9:])
    assert err < TOL["s"], err


def test_values_stay_in_their_columns(cuda):
    """Infinities and NaN of one vector's multipoles reach that vector's L only."""
    import bbfmmongpu_amd as B
    r, depth, nrhs = 32, 3, 3
    ncell = (8 ** (depth + 1) - 1) // 7
    rng = np.random.default_rng(5)
    K = rng.standard_normal(316 * r * r, dtype=np.float32)
    M = rng.standard_normal((nrhs, ncell, r), dtype=np.float32)
    clean = _m2l(B, "s", 4, r, depth, nrhs, K, M, cuda, 0, scheme=B.SCHEME_IJ)
    M[1, 100, 3], M[1, 300, 0] = np.inf, np.nan
    got = _m2l(B, "s", 4, r, depth, nrhs, K, M, cuda, 0, scheme=B.SCHEME_IJ)
    ref = _m2l(B, "s", 4, r, depth, nrhs, K, M, cuda, 0, scheme=B.SCHEME_BA)
    assert np.array_equal(got[[0, 2]], clean[[0, 2]])
    assert np.array_equal(np.isfinite(got[1]), np.isfinite(ref[1]))


@pytest.mark.parametrize("depth,nrhs", [(2, 1), (2, 16), (2, 130), (3, 1), (3, 3), (3, 16), (4, 1), (4, 5), (4, 15)])
def test_split_bf16_few_columns(depth, nrhs, cuda):
    """The split-BF16 kernel of few columns (k_m2l_bf16_few): one and two
    column tiles a block, partial tiles, M and L at any alignment.  The bound
    is that of the form, as everywhere (3e-5)."""
    import bbfmmongpu_amd as B
    r = 32
    ncell = (8 ** (depth + 1) - 1) // 7
    rng = np.random.default_rng(nrhs)
    K = rng.standard_normal(316 * r * r, dtype=np.float32)
    M = rng.standard_normal((nrhs, ncell, r), dtype=np.float32)
    ref = _m2l(B, "d", 4, r, depth, nrhs, K, M, cuda, 0, scheme=B.SCHEME_BA)
    got = _m2l(B, "s", 4, r, depth, nrhs, K, M, cuda, 1, scheme=B.SCHEME_IJ, form=B.FORM_BF16X2)
    assert not got[:, :9].any()
    err = (np.linalg.norm((got - ref)[:, 9:], axis=(1, 2)) / np.linalg.norm(ref[:, 9:], axis=(1, 2))).max()
    print(f"depth={depth} nrhs={nrhs}: {err:.2e}", flush=True)
    assert err < 3e-5
