"""Performance cases of the framework: what a program that uses it calls.

Each case is one pass through a public entry point: Plan.solve,
Plan.solve + Plan.gradient, a Plan.batch solve replayed as one graph, or the
drop-in anotherFMMCompute on host arrays.  listed() gives the fixed cases,
draw(rng) one more of the same ranges, prepare(case, seed) the plan and the
inputs, run(state) one pass with its whole outputs, work(case) the bytes and
operations that the pass cannot do without, and exact(case, seed) the outputs
by direct summation in 64 bits.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

import bbfmmongpu_amd as B
from bbfmmongpu_amd import workloads

PLAIN, BF16X2, FP32MFMA, FP16X3 = "plain", "bf16x2", "fp32mfma", "fp16x3"
FORMS = {PLAIN: B.FORM_PLAIN, BF16X2: B.FORM_BF16X2, FP32MFMA: B.FORM_FP32MFMA, FP16X3: B.FORM_FP16X3}
# the most source-target pairs that exact() sums (a few seconds)
EXACT_PAIRS = 2.5e11


def listed():
    return [
        # a small system, one vector, as an iterative solver of a few thousand
        # unknowns calls it: latency and launches
        dict(name="one_vector_4k", kind="solve", prec="s", n=4, N=4096, nrhs=1, form=PLAIN, points="uniform", lmod=0),
        # the ordinary call: one vector of 64K particles, depth 4, fp32
        dict(name="one_vector_64k", kind="solve", prec="s", n=4, N=65536, nrhs=1, form=PLAIN, points="uniform",
             lmod=0),
        # the same form at the largest uniform size, depth 5
        dict(name="one_vector_1m", kind="solve", prec="s", n=4, N=1 << 20, nrhs=1, form=PLAIN, points="uniform",
             lmod=0),
        # the double-precision build on an odd size
        dict(name="double_100k", kind="solve", prec="d", n=4, N=100_003, nrhs=1, form=PLAIN, points="uniform",
             lmod=0),
        # a few right-hand sides on a closed surface (boundary elements), one
        # level deeper than the rule, so that most leaves are empty
        dict(name="four_vectors_surface_150k", kind="solve", prec="s", n=4, N=150_001, nrhs=4, form=PLAIN,
             points="sphere", lmod=1),
        # the throughput form: 16 vectors of 1M particles, split-BF16 M2L
        dict(name="sixteen_vectors_1m", kind="solve", prec="s", n=4, N=1 << 20, nrhs=16, form=BF16X2,
             points="uniform", lmod=0),
        # a ragged block of 12 vectors at a middle size
        dict(name="twelve_vectors_50k", kind="solve", prec="s", n=4, N=50_021, nrhs=12, form=BF16X2,
             points="uniform", lmod=0),
        # training-like use: forward and adjoint (gradients of charges and
        # positions) of 8 vectors
        dict(name="adjoint_262k", kind="adjoint", prec="s", n=4, N=262_144, nrhs=8, form=BF16X2, points="uniform",
             lmod=0),
        # 64 uneven clustered and surface instances in one plan and one graph
        dict(name="batch_64_uneven", kind="batch", prec="s", n=4, count=64, nmin=4096, nmax=131_072, nrhs=1,
             form=BF16X2),
        # a middle order (six digits): rank 108
        dict(name="order6_80k", kind="solve", prec="s", n=6, N=80_000, nrhs=1, form=PLAIN, points="uniform", lmod=0),
        # the high order, rank 256, with 16 vectors on the fp32 matrix unit
        dict(name="order8_sixteen_vectors_131k", kind="solve", prec="s", n=8, N=131_072, nrhs=16, form=FP32MFMA,
             points="uniform", lmod=0),
        # the drop-in entry point on host arrays (tree given, everything else
        # inside the call)
        dict(name="drop_in_64k", kind="dropin", prec="s", n=4, N=65536, nrhs=1, form=PLAIN, points="uniform", lmod=0),
    ]


def _log_int(rng, lo, hi):
    """An integer between lo and hi, uniform in its logarithm, odd half of the time."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        v |= 1
    return min(max(v, lo), hi)


def draw(rng):
    kind = rng.choice(["solve"] * 7 + ["adjoint", "batch", "dropin"])
    if kind == "adjoint":
        m = rng.randint(1, 12)
        return dict(kind=kind, prec="s", n=4, N=_log_int(rng, 8192, 262_144), nrhs=m,
                    form=BF16X2 if m >= 8 else PLAIN, points="uniform", lmod=0)
    if kind == "batch":
        return dict(kind=kind, prec="s", n=4, count=rng.randint(8, 48), nmin=4096,
                    nmax=_log_int(rng, 16_384, 131_072), nrhs=rng.choice([1, 1, 2]), form=BF16X2)
    if kind == "dropin":
        return dict(kind=kind, prec=rng.choice(["s", "d"]), n=4, N=_log_int(rng, 4096, 131_072), nrhs=1, form=PLAIN,
                    points="uniform", lmod=0)
    # plain solves of 1 to 7 vectors, blocks of 8 to 16 in the matrix forms,
    # double precision, other orders
    sub = rng.choice(["few", "few", "block", "block", "double", "order", "order"])
    if sub == "block":
        return dict(kind=kind, prec="s", n=4, N=_log_int(rng, 8192, 1 << 20), nrhs=rng.randint(8, 16),
                    form=rng.choice([BF16X2, BF16X2, FP32MFMA, FP16X3]), points="uniform", lmod=0)
    if sub == "double":
        return dict(kind=kind, prec="d", n=4, N=_log_int(rng, 4096, 1 << 19), nrhs=rng.randint(1, 4), form=PLAIN,
                    points="uniform", lmod=0)
    if sub == "order":
        n = rng.choice([3, 5, 6, 8])
        return dict(kind=kind, prec=rng.choice(["s", "s", "d"]) if n < 8 else "s", n=n,
                    N=_log_int(rng, 4096, 131_072), nrhs=rng.randint(1, 4), form=PLAIN, points="uniform", lmod=0)
    surface = rng.random() < 0.3
    return dict(kind=kind, prec="s", n=4, N=_log_int(rng, 4096, 262_144 if surface else 1 << 20),
                nrhs=rng.randint(1, 7), form=PLAIN, points="sphere" if surface else "uniform", lmod=1 if surface else 0)


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=4)
def _operators(n, prec):
    """Operators of order n, which a program computes once or reads from its files."""
    U, K, _ = B.operators(n, prec=prec, device=n >= 6)
    return U, K


def _points(case, rng):
    p = workloads.sphere_surface(case["N"], rng) if case["points"] == "sphere" else workloads.uniform(case["N"], rng)
    return p.astype(B.dtype(case["prec"]))


def _charges(rng, m, N, prec):
    """One vector: positive charges (masses, charges of one sign); more: both signs."""
    q = rng.random((m, N))
    return (q if m == 1 else 2 * q - 1).astype(B.dtype(prec))


def _batch_sizes(case):
    """Sizes of a batch's instances: spread over nmin..nmax in the logarithm, in no order."""
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    return [int(math.exp(lo + (hi - lo) * ((0.5 + 0.6180339887 * i) % 1.0))) for i in range(case["count"])]


def _inputs(case, seed):
    """Host inputs of a case: positions (a list of them for a batch), charges, and the adjoint's target potentials."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "batch":
        # half Plummer spheres, half closed surfaces
        sizes = _batch_sizes(case)
        pos = [(workloads.plummer if i < len(sizes) // 2 else workloads.sphere_surface)(k, rng).astype(np.float32)
               for i, k in enumerate(sizes)]
        return pos, _charges(rng, case["nrhs"], sum(sizes), "s"), None
    pos = _points(case, rng)
    q = _charges(rng, case["nrhs"], case["N"], case["prec"])
    target = None
    if case["kind"] == "adjoint":
        # the data to fit: potentials of another set of charges, about as large
        target = (rng.standard_normal(q.shape) * math.sqrt(case["N"])).astype(q.dtype)
    return pos, q, target


class _DropIn:
    """A reference program's own state: the tree, operators and weights on the host."""

    def __init__(self, case, pos, q):
        self.lib = B.load(case["prec"])
        self.n, self.pos, self.q = case["n"], np.ascontiguousarray(pos), np.ascontiguousarray(q.reshape(-1))
        self.U, self.K = _operators(case["n"], case["prec"])
        self.r = self.U.size // case["n"] ** 3
        self.Tkz, self.Kt, self.Kw, self.Cw = B.weights(case["n"], case["prec"])
        self.tree = C.c_void_p()
        self.lib.anotherBuildFMMHierachy(1.0, self.n, 1, B.maxlev(case["N"], case["lmod"]), self.r,
                                         C.byref(self.tree), case["N"], case["N"], self._p(self.pos),
                                         self._p(self.pos))

    @staticmethod
    def _p(a):
        return a.ctypes.data_as(C.c_void_p)

    def solve(self):
        p = self._p
        phi = np.empty_like(self.q)
        self.lib.anotherFMMCompute(C.byref(self.tree), p(self.pos), p(self.pos), p(self.q), p(self.K), p(self.U),
                                   p(self.Tkz), p(self.Kt), p(self.Kw), p(self.Cw), 1.0, self.r, self.n, 1, p(phi))
        if self.lib.bbfmm_amd_last_error():
            raise RuntimeError(self.lib.bbfmm_amd_last_error_string().decode())
        return phi

    def __del__(self):
        if self.tree:
            self.lib.anotherFMMCleanup(C.byref(self.tree))


def prepare(case, seed):
    pos, q, target = _inputs(case, seed)
    kind = case["kind"]
    if kind == "dropin":
        return dict(kind=kind, dropin=_DropIn(case, pos, q))
    U, K = _operators(case["n"], case["prec"])
    form = FORMS[case["form"]]
    dev = torch.device("cuda:0")
    st = dict(kind=kind, q=torch.from_numpy(np.ascontiguousarray(q)).to(dev))
    if kind == "batch":
        st["plan"] = B.Plan.batch(pos, case["n"], U, K, nrhs=case["nrhs"]).set(scheme=B.SCHEME_IJ, form=form,
                                                                               graph=True)
        st["phi"] = torch.empty_like(st["q"])
        return st
    st["plan"] = B.Plan(pos, case["n"], U, K, nrhs=case["nrhs"], lmod=case["lmod"], prec=case["prec"]).set(
        scheme=B.SCHEME_IJ, form=form, output="potential" if kind == "adjoint" else "q_phi")
    if kind == "adjoint":
        st["adjoint"] = B.Plan(pos, case["n"], U, K, nrhs=2 * case["nrhs"], lmod=case["lmod"],
                               prec=case["prec"]).set(scheme=B.SCHEME_IJ, form=form)
        st["target"] = torch.from_numpy(target).to(dev)
    return st


def run(state):
    kind = state["kind"]
    if kind == "dropin":
        return state["dropin"].solve()
    if kind == "batch":
        return state["plan"].solve(state["q"], state["phi"])
    phi = state["plan"].solve(state["q"])
    if kind == "solve":
        return phi
    # loss 1/2 |phi - target|^2: its gradients with respect to charges and positions
    dq, dx = state["adjoint"].gradient(state["q"], phi - state["target"])
    return {"phi": phi, "dq": dq, "dx": dx}


# ------------------------------------------------------------------ work
def _interactions(maxlev):
    """M2L interactions of a complete tree, levels 2..maxlev."""
    return sum((4 * (3 * 2 ** (lv - 1) - 2)) ** 3 - (3 * 2 ** lv - 2) ** 3 for lv in range(2, maxlev + 1))


def work(case):
    s = 4 if case["prec"] == "s" else 8
    n = case["n"]
    n3, r, m = n ** 3, n ** 3 // 2, case["nrhs"]
    if case["kind"] == "batch":
        # about 0.9 cells a point, 67 interactions a cell and 60 near pairs a
        # point on these forests
        N = sum(_batch_sizes(case))
        cells = 0.9 * N
        inter, pairs = 67 * cells, 60.0 * N
    else:
        N = case["N"]
        lv = B.maxlev(N, case["lmod"])
        G = 2 ** lv
        if case["points"] == "sphere":
            # cells that the surface of radius 0.4 meets, and their lists
            cells = sum(min(8 ** k, 1.5 * 4 * math.pi * 0.16 * 4 ** k) for k in range(lv + 1))
            inter = 60 * cells
            pairs = N * max(1.0, N / (4 * math.pi * 0.16)) * 9.0 / G ** 2
        else:
            cells = (8 ** (lv + 1) - 1) // 7
            inter = _interactions(lv)
            pairs = (3 * G - 2) ** 3 * (N / G ** 3) ** 2
    # forward: the M2L product, 1/r once a pair and one addition a vector,
    # P2M and L2P (n^3 terms a particle), the two transforms of every cell
    def solve(v):
        return v * 2 * r * r * inter + pairs * (8 + 2 * v) + v * 4 * n3 * N + v * 4 * n3 * r * cells

    flops = solve(m)
    nbytes = s * (N * (3 + 2 * m) + 316 * r * r + n3 * r)
    if case["kind"] == "adjoint":
        flops += solve(2 * m) + pairs * (6 + 4 * m) + m * 8 * n3 * N
        nbytes += s * N * (2 * m + 3)
    return {"bytes": float(nbytes), "flops": float(flops)}


# ------------------------------------------------------------------ direct sums in 64 bits
def _direct(pos, Q, G=None):
    """Potentials (m x N) of the charges Q (m x N) at the points themselves,
    without self terms; with G also sum_v G_v grad Phi_Qv + Q_v grad Phi_Gv (N x 3)."""
    N = pos.shape[0]
    x = pos.t().contiguous()
    phi = torch.empty_like(Q)
    dx = torch.empty_like(pos) if G is not None else None
    step = max(1, int(1.5e8) // N)
    QT, GT = Q.t().contiguous(), None if G is None else G.t().contiguous()
    for b in range(0, N, step):
        e = min(N, b + step)
        d = [x[c][None, :] - x[c][b:e, None] for c in range(3)]
        w = d[0] * d[0]
        w.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
        w = torch.where(w > 0, w.rsqrt_(), 0.0)
        if G is None:
            phi[:, b:e] = (w @ QT).t()
            continue
        # sum over v of g_vi q_vj + q_vi g_vj, then the gradient of 1/r
        w3 = w * w * w
        w3 *= GT[b:e] @ Q + QT[b:e] @ G
        for c in range(3):
            dx[b:e, c] = (w3 * d[c]).sum(1)
    return phi if G is None else dx


def exact(case, seed):
    pos, q, target = _inputs(case, seed)
    dev = torch.device("cuda:0")

    def up(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dev).double()

    sizes = _batch_sizes(case) if case["kind"] == "batch" else [case["N"]]
    if sum(float(k) ** 2 for k in sizes) > EXACT_PAIRS:
        return None
    Q = up(q)
    if case["kind"] == "batch":
        out, b = torch.empty_like(Q), 0
        for p in pos:
            e = b + p.shape[0]
            out[:, b:e] = Q[:, b:e] * _direct(up(p), Q[:, b:e].contiguous())
            b = e
        return out
    X = up(pos)
    phi = _direct(X, Q)
    if case["kind"] == "adjoint":
        g = phi - up(target)
        return {"phi": phi, "dq": _direct(X, g), "dx": _direct(X, Q, g)}
    phi *= Q
    return phi.reshape(-1).cpu().numpy() if case["kind"] == "dropin" else phi
