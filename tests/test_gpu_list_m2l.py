"""The list M2L of sparse forests (k_m2l_list_packed): vectors that do and do
not divide its units, more than 16 of them, blocks with few cells, units of 64
and 32 columns, both addressings; against the same forest in double precision."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,tol", [(1, 3e-5), (2, 1e-5)])
@pytest.mark.parametrize("nrhs", [1, 2, 5, 11, 16, 17, 33])
def test_list_m2l_vectors(nrhs, form, tol, ops4, cuda):
    """The bounds are those of the forms on forests (split BF16 3e-5, FP32 1e-5)."""
    import bbfmmongpu_amd as B
    from bbfmmongpu_amd import workloads as W
    U, K, _ = ops4
    rng = np.random.default_rng(nrhs)
    inst = [(W.uniform(40, rng), 2), (W.uniform(3000, rng), 3), (W.plummer(5000, rng), 5),
            (W.sphere_surface(6001, rng), 4)]
    pos_list = [p.astype(np.float32) for p, _ in inst]
    depths = [d for _, d in inst]
    n = sum(p.shape[0] for p in pos_list)
    Q = rng.uniform(-1.0, 1.0, size=(nrhs, n)).astype(np.float32)
    Ud, Kd = U.astype(np.float32).astype(np.float64), K.astype(np.float32).astype(np.float64)
    plan = B.Plan.batch([p.astype(np.float64) for p in pos_list], 4, Ud, Kd, nrhs=nrhs, depths=depths, prec="d")
    ref = plan.solve_host(Q.astype(np.float64)).reshape(nrhs, n)
    plan.close()
    out = []
    for flat in (False, True):
        plan = B.Plan.batch(pos_list, 4, U, K, nrhs=nrhs, depths=depths, prec="s").set(
            form=form, scheme=B.SCHEME_IJ, flat_loads=flat)
        out.append(plan.solve_host(Q).reshape(nrhs, n))
        plan.close()
    if nrhs < 16:  # the near field of 16 vectors rounds differently in its two addressings
        assert np.array_equal(out[0], out[1])
    err = max(O.rel_l2(ref[j], o[j]) for o in out for j in range(nrhs))
    print(f"nrhs={nrhs} form={form}: {err:.2e}", flush=True)
    assert err < tol
