"""Workloads that the speed of the evaluation pass is judged by.

A case is one evaluation as a program that uses the package makes it: a plan
made once for its points (IBFMM_Mat.prcmpt), then A q for the charges at hand,
with device arrays (apply_batch_device), host arrays (gemv), several plans in
one graph (Batch), or the sampled direct sum that checks a result (direct).
Points and charges are those of the benchmark configurations
(defmm_amd/workloads.py): sphere, edge-refined cube, clustered 4:1:1 ellipsoid
surfaces and Gaussian clusters in a volume; charges re, im ~ U(-1, 1).

A program in double precision holds complex128 arrays.  One that uses the
mixed-precision path holds complex64 charges and potentials; the entry points
take complex128, so it converts on both sides of the call.
"""
import math

import numpy as np
import torch

import defmm_amd as dm
from defmm_amd import workloads as wl

_FOUR_PI = 4.0 * math.pi


def listed():
    return [
        # a small scatterer, one solver iteration: launches and latency count
        _plan("cube4k_6l_o4_fp64", "cube_edges", 4000, 6, 4, 33, "fp64", 1),
        # 20,000 points of the edge-refined cube, 32 wavelengths across:
        # engineering accuracy (order 4) ...
        _plan("cube20k_32l_o4_fp64", "cube_edges", 20000, 32, 4, 65, "fp64", 1),
        # ... and relative error <= 1e-6 (order 8), the drop-in path,
        _plan("cube20k_32l_o8_fp64", "cube_edges", 20000, 32, 8, 65, "fp64", 1),
        # the same in mixed precision,
        _plan("cube20k_32l_o8_mixed", "cube_edges", 20000, 32, 8, 65, "mixed", 1),
        # and with 16 right-hand sides (a block solver, many incident waves)
        # and the M2L storage the autotuner keeps there: the headline workload
        _plan("cube20k_32l_o8_mixed_rhs16", "cube_edges", 20000, 32, 8, 65, "mixed", 16,
              m2l="batched"),
        # the reference's own call: gemv with host arrays, its refined cube's
        # point count and points per wavelength, order 6, 31 points a leaf
        _plan("gemv41k_10l_o6_fp64", "cube_edges", 41334, 10.2, 6, 32, "fp64", 1, call="host"),
        # many wavelengths: every level high-frequency, millions of directions
        _plan("sphere200k_64l_o5_fp64", "sphere", 200000, 64, 5, 65, "fp64", 1),
        # a million points at moderate frequency, order 7
        _plan("sphere1m_16l_o7_mixed", "sphere", 1000000, 16, 7, 65, "mixed", 1),
        # clustered points and large leaves, 16 right-hand sides
        _plan("ellipsoid100k_64l_o6_mixed_rhs16", "ellipsoid", 100000, 64, 6, 97, "mixed", 16),
        # Laplace (kappa = 0, all levels low-frequency): clusters of sources in
        # a volume, the field at other points
        _plan("laplace150k_o5_fp64", "clusters", 150000, 0, 5, 65, "fp64", 1, n_trg=90001),
        # independent uneven problems evaluated by one graph
        {"name": "batch16_mixed", "kind": "batch", "instances": 16, "n_min": 2000,
         "n_max": 20000, "draw": 4242},
        # the check of a result: FP64 direct sum at sampled targets
        {"name": "direct300k_2000", "kind": "direct", "geometry": "sphere", "n": 300000,
         "n_trg": 2000, "wavelengths": 32},
    ]


def _plan(name, geometry, n, wavelengths, order, ncrit, precision, nrhs, call="device",
          m2l="auto", n_trg=0):
    """n_trg = 0: the targets are the sources."""
    case = {"kind": "plan", "geometry": geometry, "n": n, "n_trg": n_trg,
            "wavelengths": wavelengths, "order": order, "ncrit": ncrit, "precision": precision,
            "nrhs": nrhs, "call": call, "m2l": m2l}
    if name:
        case = {"name": name, **case}
    return case


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def draw(rng):
    kind = rng.choices(["plan", "batch", "direct"], [12, 1, 1])[0]
    if kind == "batch":
        return {"kind": "batch", "instances": rng.randint(4, 20), "n_min": rng.randint(2000, 4000),
                "n_max": rng.randint(8000, 20000), "draw": rng.randint(1, 10 ** 6)}
    if kind == "direct":
        return {"kind": "direct", "geometry": rng.choice(sorted(wl.GEOMETRIES)),
                "n": int(_log(rng, 3000, 300000)), "n_trg": int(_log(rng, 50, 2500)),
                "wavelengths": round(_log(rng, 2, 64), 2)}
    while True:
        geometry = rng.choice(sorted(wl.GEOMETRIES))
        n = int(_log(rng, 4000, 200000))
        n_trg = 0 if rng.random() < 0.7 else int(_log(rng, 3000, n))
        ncrit = rng.choice([32, 33, 48, 65, 65, 97])
        # leaves of a fraction of a wavelength to about one (beyond that the
        # tree has no level whose interactions can be interpolated)
        most = min(64.0, math.sqrt((n_trg or n) / ncrit) * (0.95 if geometry == "sphere" else 1.7))
        nl = 0 if rng.random() < 0.12 else round(_log(rng, 4, max(5.0, most)), 2)
        order = rng.choice([3, 4, 4, 5, 5, 5, 6, 6, 6, 7, 7, 8, 8, 8, 9, 10])
        precision = rng.choice(["fp64", "mixed", "mixed"])
        nrhs = rng.choice([1, 1, 1, 2, 3, 4, 5, 8] + ([16, 16, 17] if precision == "mixed" else []))
        # no more than the listed cases cost: stored Fourier rows and their products
        rows = n * max(nl, 4) * (2 * order - 1) ** 3 * nrhs * (2 if precision == "fp64" else 1)
        if rows <= 0.3 * 200000 * 64 * 729 * 2:
            return _plan(None, geometry, n, nl, order, ncrit, precision, nrhs,
                         call="host" if rng.random() < 0.15 else "device",
                         m2l=rng.choice(["auto", "auto", "auto", "batched"]), n_trg=n_trg)


# ---- inputs ----------------------------------------------------------------

def _clouds(case, seed):
    """Source points, target points, wavenumber."""
    make = wl.GEOMETRIES[case["geometry"]]
    src = make(case["n"], seed=seed % 1000003 + 1)
    trg = src
    if case["n_trg"]:
        if case["kind"] == "direct":  # sampled among the points
            trg = np.ascontiguousarray(src[np.linspace(0, case["n"] - 1, case["n_trg"]).astype(np.int64)])
        else:
            trg = make(case["n_trg"], seed=seed % 1000003 + 500)
    kappa = wl.kappa_for(case["wavelengths"], src, trg) if case["wavelengths"] else 0.0
    return src, trg, kappa


def _charges(n, nrhs, seed, precision):
    q = np.stack([wl.charges(n, seed=seed % 1000003 + 7 + 100 * r) for r in range(nrhs)])
    return q.astype(np.complex64) if precision == "mixed" else q


def _instances(case, seed):
    """Parameters of a batch's instances (from the case alone), their points
    and charges (from the seed)."""
    u = wl.uniform(case["draw"], 8 * case["instances"])
    out = []
    for i in range(case["instances"]):
        lo, hi = math.log(case["n_min"]), math.log(case["n_max"])
        n = int(math.exp(lo + (hi - lo) * u[8 * i]))
        geometry = sorted(wl.GEOMETRIES)[min(3, int(u[8 * i + 1] * 4))]
        nl = min(2 ** (2 + 2 * u[8 * i + 2]), 0.9 * math.sqrt(n / 33))
        order, nrhs = 4 + min(2, int(u[8 * i + 3] * 3)), 1 + min(3, int(u[8 * i + 4] * 4))
        pts = wl.GEOMETRIES[geometry](n, seed=seed % 1000003 + 31 * i + 1)
        q = _charges(n, nrhs, seed + 17 * i, "mixed")
        out.append((pts, wl.kappa_for(nl, pts), order, nrhs, q))
    return out


def _plan_of(src, trg, order, ncrit, kappa, precision, nrhs):
    A = dm.IBFMM_Mat(precision=dm.MIXED if precision == "mixed" else dm.FP64)
    A.setSourceParticles(src)
    A.setTargetParticles(trg)
    A.prcmpt(order, ncrit, kappa)
    if nrhs > 1:
        A.set_rhs(nrhs)
    return A


class _State:
    def __init__(self, case):
        self.case = case
        self.batch = None
        self.plans = []

    def __del__(self):
        # a batch goes before its plans
        if self.batch is not None:
            self.batch.destroy()
        for A in self.plans:
            A.destroy()


def prepare(case, seed):
    s = _State(case)
    dev = torch.device("cuda:0")
    if case["kind"] == "direct":
        s.src, s.trg, s.kappa = _clouds(case, seed)
        s.q = _charges(case["n"], 1, seed, "fp64")[0]
    elif case["kind"] == "batch":
        s.q64, s.q, s.p = [], [], []
        inst = _instances(case, seed)
        for pts, kappa, order, nrhs, q in inst:
            s.plans.append(_plan_of(pts, pts, order, 33, kappa, "mixed", nrhs))
            s.q64.append(torch.from_numpy(q).to(dev))
            s.q.append(torch.zeros(q.shape, dtype=torch.complex128, device=dev))
            s.p.append(torch.zeros(q.shape, dtype=torch.complex128, device=dev))
        # the arrays' addresses are bound into the graph
        s.batch = dm.Batch(s.plans, [t.data_ptr() for t in s.q], [t.data_ptr() for t in s.p],
                           [i[3] for i in inst])
    else:
        src, trg, kappa = _clouds(case, seed)
        A = _plan_of(src, trg, case["order"], case["ncrit"], kappa, case["precision"], case["nrhs"])
        s.plans.append(A)
        if case["m2l"] == "batched":
            A.set_m2l(dm.M2L_BATCHED)
        q = _charges(case["n"], case["nrhs"], seed, case["precision"])
        if case["call"] == "host":
            s.q = q
        else:
            s.q = torch.from_numpy(q).to(dev)
            s.p = torch.zeros((case["nrhs"], A.n_trg), dtype=torch.complex128, device=dev)
    return s


# ---- one pass --------------------------------------------------------------

def run(s):
    case = s.case
    if case["kind"] == "direct":
        return dm.direct(s.src, s.q, s.trg, s.kappa)
    if case["kind"] == "batch":
        for a, b in zip(s.q, s.q64):
            a.copy_(b)
        s.batch.execute(torch.cuda.current_stream().cuda_stream)
        return [p.to(torch.complex64) for p in s.p]
    A, mixed = s.plans[0], case["precision"] == "mixed"
    if case["call"] == "host":
        p = A.apply_batch(s.q) if case["nrhs"] > 1 else dm.gemv(A, s.q[0])[None]
        return p.astype(np.complex64) if mixed else p
    q = s.q.to(torch.complex128) if mixed else s.q
    A.apply_batch_device(q.data_ptr(), s.p.data_ptr(), case["nrhs"],
                         torch.cuda.current_stream().cuda_stream)
    return s.p.to(torch.complex64) if mixed else s.p


# ---- what a pass cannot do without -----------------------------------------

def _plan_work(src, trg, order, ncrit, kappa, nrhs, scalar):
    """From the lists of the method (near-field pairs, M2L pairs, slots)."""
    st = dm.build_plan_stats(src, trg, order, ncrit, kappa)
    pp, ll = (2 * order - 1) ** 3, order ** 3
    slots = st["src_slots"] + st["trg_slots"]
    rows = st["m2f_slots"] + st["m2l_targets"]
    flops = st["p2p_pairs"] * (25 + 8 * nrhs)
    flops += nrhs * (8 * pp * st["m2l_entries"] + 5 * pp * math.log2(pp) * rows)
    flops += nrhs * (12 * order * ll * slots + 4 * ll * (len(src) + len(trg)))
    tables = (st["hf_tables"] + st["lf_tables"]) * pp * 2 * scalar
    return (24 * (len(src) + len(trg)) + 2 * scalar * nrhs * (len(src) + len(trg)) + tables, flops)


def work(case):
    if case["kind"] == "direct":
        n, m = case["n"], case["n_trg"]
        return {"bytes": 40 * n + 40 * m, "flops": 33 * n * m}
    if case["kind"] == "batch":
        w = [_plan_work(pts, pts, order, 33, kappa, nrhs, 4)
             for pts, kappa, order, nrhs, _ in _instances(case, 1)]
    else:
        src, trg, kappa = _clouds(case, 1)
        w = [_plan_work(src, trg, case["order"], case["ncrit"], kappa, case["nrhs"],
                        4 if case["precision"] == "mixed" else 8)]
    return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}


# ---- the sums themselves, in 64 bits ---------------------------------------

def _direct_sum(src, trg, q, kappa):
    """sum_j exp(i kappa r) / (4 pi r) q_j, terms with r^2 < 1e-16 left out."""
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    x, y = (torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in (trg, src))
    q = torch.from_numpy(np.ascontiguousarray(q.astype(np.complex128))).to(dev)
    qr, qi = q.real.t().contiguous(), q.imag.t().contiguous()
    step = max(1, 40_000_000 // len(src))
    out = torch.empty((q.shape[0], len(trg)), dtype=torch.complex128, device=dev)
    for i in range(0, len(trg), step):
        t = x[i:i + step]
        r2 = (t[:, None, 0] - y[None, :, 0]).square()
        r2 += (t[:, None, 1] - y[None, :, 1]).square()
        r2 += (t[:, None, 2] - y[None, :, 2]).square()
        k = torch.where(r2 < 1e-16, torch.zeros_like(r2), r2.rsqrt() / _FOUR_PI)
        r = r2.sqrt_().mul_(kappa)
        c, s = r.cos().mul_(k), r.sin().mul_(k)
        out[:, i:i + step] = torch.complex(c @ qr - s @ qi, c @ qi + s @ qr).t()
    return out.cpu().numpy()


def exact(case, seed):
    if case["kind"] == "direct":
        src, trg, kappa = _clouds(case, seed)
        return _direct_sum(src, trg, _charges(case["n"], 1, seed, "fp64"), kappa)[0]
    if case["kind"] == "batch":
        return [_direct_sum(pts, pts, q, kappa) for pts, kappa, _, _, q in _instances(case, seed)]
    if case["n"] * (case["n_trg"] or case["n"]) > 5e10:
        return None
    src, trg, kappa = _clouds(case, seed)
    return _direct_sum(src, trg, _charges(case["n"], case["nrhs"], seed, case["precision"]), kappa)
