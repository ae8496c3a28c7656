"""The solver's work as a user's program calls it, as cases that can be prepared, run and checked.

Four kinds of case, each one pass through the public entry points of mlfma_pmchwt_amd.api:

* "apply":   y = A x on device vectors (Operator.apply_device), for one or many right-hand sides: the
             operation that every Krylov iteration of a user's own or of the built-in solver runs.
* "solve":   a fixed number of GMRES iterations (Operator.solve / solve_batch) from host right-hand
             sides to host solutions, preconditioner and true residuals included.
* "member":  one training problem of the learned preconditioner: operator set-up, one excitation,
             the spectral features and the Krylov statistics of its coefficients.
* "scatter": the incident field of many plane waves and the scattered field of solved currents
             (Operator.excitation_batch, Operator.rcs), before and after a solve.

Lengths are in free-space wavelengths (299,792,458 Hz).  A program builds its operator once and then
applies it to many vectors, so prepare() keeps the operator of the last case and makes only the
vectors anew from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mlfma_pmchwt_amd import api, configs, geometry

EFIE, CFIE, PMCHWT = api.EFIE, api.CFIE, api.PMCHWT
FP64, FP32, BF16 = api.FP64, api.FP32, api.BF16
DEGREE = 6                      # of the near-field polynomial, as learned.DEGREE
ALPHA = np.array([1.0, 0.5, 0.25, 0.1, 0.05, 0.02, 0.01], dtype=complex)   # and coefficients for it
STEPS = 30                      # Krylov pairs per training problem


def _case(name, kind, shape, size, density, ie, **more):
    c = {"kind": kind, "shape": shape, "a": 0.0, "b": 0.0, "c": 0.0, "density": density, "ie": ie, "eps_re": 1.0,
         "eps_im": 0.0, "alpha": 0.2, "far": FP64, "near": FP64, "pre": FP64, "nrhs": 1, "tuned": False, "precond": 0,
         "iterations": 0, "restart": 0, "batched": False, "angles": 0}
    c.update(zip(("a", "b", "c"), size))
    c.update(more)
    if name is not None:
        c["name"] = name
    return c


def listed():
    mixed = dict(far=FP32, near=BF16, pre=BF16)
    return [
        # a small PEC sphere, one vector: the call that a program makes while it is being written,
        # and an iterative solver's on a small target; launches and latency count
        _case("apply_efie_480", "apply", "sphere", (0.5,), 4, EFIE),
        # the dielectric sphere r = 0.5 (15,360 unknowns), one vector, FP64: the reference's own size
        _case("apply_pmchwt_15k", "apply", "sphere", (0.5,), 16, PMCHWT, eps_re=4.0),
        # the PEC sphere r = 4 (300,000 unknowns), one vector, FP64: the largest single product
        _case("apply_cfie_300k", "apply", "sphere", (4.0,), 100, CFIE, alpha=0.5),
        # the same sphere meshed coarser, single precision throughout, an odd block of vectors
        _case("apply_cfie_fp32_x19", "apply", "sphere", (4.0,), 53, CFIE, alpha=0.5, far=FP32, near=FP32, nrhs=19,
              tuned=True),
        # the lossy sphere r = 2 at half density in FP64, a block of 13: true residuals of a batch
        _case("apply_lossy_fp64_x13", "apply", "sphere", (2.0,), 25, PMCHWT, eps_re=2.5, eps_im=-0.1, nrhs=13),
        # a small cylinder of the object mix, its 8 incidences, mixed precision: uneven leaves
        _case("apply_cylinder_mixed_x8", "apply", "cylinder", (0.37, 1.13), 0.1, PMCHWT, eps_re=3.3, nrhs=8, tuned=True,
              **mixed),
        # the ellipsoid (3, 2, 1) at full size (302,460 unknowns), 64 incidences, mixed precision,
        # recorded and tuned: the product that the headline solve repeats
        _case("apply_ellipsoid_mixed_x64", "apply", "ellipsoid", configs.C5_AXES, 71, PMCHWT,
              eps_re=configs.c5_eps(1000), nrhs=64, tuned=True, **mixed),
        # one incidence on the dielectric sphere, the reference's method: FP64 GMRES(30)
        _case("solve_sphere_gmres30", "solve", "sphere", (0.5,), 16, PMCHWT, eps_re=4.0, iterations=30, restart=30),
        # the lossy sphere r = 2 at full size (150,000 unknowns), 64 incidences in lockstep, mixed
        # precision, polynomial preconditioner: ten iterations of the production solve
        _case("solve_lossy_poly_x64", "solve", "sphere", (2.0,), 50, PMCHWT, eps_re=2.5, eps_im=-0.1, nrhs=64,
              tuned=True, batched=True, precond=api.PRECOND_POLY, iterations=10, restart=50, **mixed),
        # an ellipsoid of the object mix, 8 incidences, the inner near-field solve
        _case("solve_ellipsoid_inner_x8", "solve", "ellipsoid", (1.5, 1.0, 0.7), 23, PMCHWT, eps_re=5.1, nrhs=8,
              tuned=True, batched=True, precond=api.PRECOND_INNER, iterations=12, restart=50, **mixed),
        # one of the 200 problems that the coefficient network is trained on (9,720 RWG): set-up
        _case("member_ellipsoid_9720", "member", "ellipsoid", tuple(0.25 * a for a in configs.C5_AXES), 18, PMCHWT,
              eps_re=configs.c5_eps(0)),
        # excitations of 8 incidences and the 181-angle bistatic pattern of solved currents
        _case("scatter_lossy_181", "scatter", "sphere", (2.0,), 50, PMCHWT, eps_re=2.5, eps_im=-0.1, nrhs=8, angles=181),
    ]


def draw(rng):
    """A case of the same ranges: meshes from 480 to about 90,000 RWG at edges of 0.03 to 0.1, each
    equation, precision mode and kind, 1 to 64 right-hand sides."""
    kind = rng.choice(["apply"] * 7 + ["solve"] * 3 + ["member", "scatter"])
    most = {"apply": 55, "solve": 40, "member": 20, "scatter": 55}[kind]
    density = int(round(math.exp(rng.uniform(math.log(5), math.log(most)))))
    edge = rng.uniform(0.03, 0.1)
    radius = round(max(0.4, min(4.0, density * edge / 1.1)), 3)
    shape = rng.choice(["sphere", "ellipsoid", "cylinder"])
    size = {"sphere": (radius,), "ellipsoid": (radius, round(radius * rng.uniform(0.4, 0.9), 3),
                                               round(radius * rng.uniform(0.3, 0.7), 3)),
            "cylinder": (round(max(0.25, radius * rng.uniform(0.3, 0.5)), 3),
                         round(max(0.7, radius * rng.uniform(0.8, 1.6)), 3))}[shape]
    dens = density if shape != "cylinder" else round(max(1.1 * radius / density, 0.03), 4)
    ie = rng.choice([EFIE, CFIE, PMCHWT, PMCHWT])
    eps = {}
    if ie == PMCHWT:
        eps = {"eps_re": round(rng.uniform(1.5, 8.0), 3), "eps_im": rng.choice([0.0, 0.0, -0.1])}
    nrhs = int(round(math.exp(rng.uniform(0.0, math.log(64)))))
    mode = rng.choice(["fp64", "fp32", "mixed", "mixed"])
    prec = {"fp64": {}, "fp32": dict(far=FP32, near=FP32), "mixed": dict(far=FP32, near=BF16, pre=BF16)}[mode]
    if kind == "apply":
        return _case(None, kind, shape, size, dens, ie, nrhs=min(nrhs, 12) if mode == "fp64" else nrhs,
                     tuned=rng.random() < 0.5, **eps, **prec)
    if kind == "solve":
        nrhs = min(nrhs, 32)
        if mode == "fp64":
            return _case(None, kind, shape, size, dens, ie, iterations=rng.randint(5, 15), restart=30, **eps)
        return _case(None, kind, shape, size, dens, ie, nrhs=max(2, nrhs), batched=True, tuned=rng.random() < 0.5,
                     precond=rng.choice([api.PRECOND_POLY, api.PRECOND_INNER]), iterations=rng.randint(3, 8), restart=50,
                     **eps, **prec)
    if kind == "member":
        return _case(None, kind, shape, size, dens, PMCHWT, eps_re=round(rng.uniform(2.0, 8.0), 3))
    return _case(None, kind, shape, size, dens, ie, nrhs=max(2, nrhs // 4), angles=rng.choice([37, 91, 181, 361]), **eps)


# ---------------------------------------------------------------- operators
def _mesh(case):
    n = case["density"]
    if case["shape"] == "sphere":
        return geometry.geodesic_sphere(int(n), case["a"])
    if case["shape"] == "ellipsoid":
        return geometry.ellipsoid((case["a"], case["b"], case["c"]), frequency=int(n))
    r, h = case["a"], case["b"]
    return geometry.cylinder(r, h, max(8, math.ceil(2 * math.pi * r / n)), max(2, math.ceil(h / n)),
                             max(2, math.ceil(r / n)))


def _params(case):
    return dict(integral_equation=case["ie"], eps_r_re=case["eps_re"], eps_r_im=case["eps_im"],
                cfie_alpha=case["alpha"], far_precision=case["far"], near_precision=case["near"],
                precond_precision=case["pre"], max_rhs=case["nrhs"])


_last = {"key": None, "op": None}
_sizes = {}


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "kind", "angles", "iterations")))


def _operator(case):
    """The operator of this case, set up as its program would: the last one is kept."""
    key = _key(case)
    if _last["key"] != key:
        _last.update(key=None, op=None)   # freed before the next one is built
        op = api.Operator(_mesh(case), **_params(case))
        if case["far"] == FP32:
            op.set_apply_precision(FP32)
        if case["precond"] == api.PRECOND_POLY:
            op.set_precond_poly(ALPHA)
        if case["tuned"]:
            if case["nrhs"] > 1:
                op.autotune(case["nrhs"], case["far"])
            op.set_graphs(True)
        _last.update(key=key, op=op)
    _measure(case, _last["op"])
    return _last["op"]


def _measure(case, op):
    """Counts of the operator that work() needs, kept apart from the operator itself."""
    key = _key(case)
    if key in _sizes:
        return _sizes[key]
    nw = 2 if case["ie"] == PMCHWT else 1
    s = {"n": op.n, "rwg": op.n_rwg, "near": op.near_entries, "k0": 0, "samples": 0, "pairs": 0, "interp": 0}
    for wn in range(1, nw + 1):
        for lvl in range(2, op.max_level + 1):
            k = 2 * op.grid(wn, lvl)[0] ** 2
            boxes = op.level(lvl)[0].size
            s["pairs"] += k * op.level_list(lvl, 1)[1].size
            s["samples"] += k * boxes
            if lvl < op.max_level:
                s["interp"] += k * op.level(lvl + 1)[0].size   # parent samples x children
        s["k0"] += 2 * op.grid(wn, op.max_level)[0] ** 2
    _sizes[key] = s
    return s


def _waves(case, rng, count):
    """Directions and polarisations of incident plane waves."""
    return rng.integers(0, 2, count) * 90.0, rng.uniform(5.0, 175.0, count), rng.uniform(0.0, 360.0, count)


def prepare(case, seed):
    rng = np.random.default_rng([7, seed])
    if case["kind"] == "member":
        pol, th, ph = _waves(case, rng, 1)
        return {"case": case, "mesh": _mesh(case), "params": _params(case), "wave": (pol[0], th[0], ph[0])}
    op = _operator(case)
    state = {"case": case, "op": op}
    if case["kind"] == "apply":
        # Krylov vectors: complex noise
        gen = torch.Generator(device="cuda")
        gen.manual_seed(1_000_003 * seed + 17)
        x = torch.randn(case["nrhs"], op.n, dtype=torch.complex128, device="cuda", generator=gen)
        state.update(x=x, y=torch.empty_like(x))
        torch.cuda.synchronize()
    elif case["kind"] == "solve":
        state["b"] = np.asfortranarray(op.excitation_batch(*_waves(case, rng, case["nrhs"])))
    else:
        state["waves"] = _waves(case, rng, case["nrhs"])
        state["theta"] = np.linspace(0.0, 180.0, case["angles"]) + rng.uniform(0.0, 0.3)
        state["phi"] = float(rng.uniform(0.0, 360.0))
        state["i"] = rng.standard_normal(op.n) + 1j * rng.standard_normal(op.n)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "apply":
        state["op"].apply_device(state["x"].data_ptr(), state["y"].data_ptr(), case["nrhs"])
        return state["y"]
    if case["kind"] == "solve":
        op, b = state["op"], state["b"]
        how = dict(itr_max=case["iterations"], restart=case["restart"], tol_rel=0.0, precond=case["precond"])
        if case["batched"]:
            x, st = op.solve_batch(b, **how)
            return {"x": x, "residual": np.array([s["rel_residual"] for s in st])}
        x, st = op.solve(b[:, 0], **how)
        return {"x": x, "residual": np.array([st["rel_residual"]])}
    if case["kind"] == "member":
        op = api.Operator(state["mesh"], **state["params"])
        b = op.excitation(*state["wave"])
        f = op.precond_features()
        g, h, c = op.precond_statistics(b, steps=STEPS, degree=DEGREE)
        op.close()
        return {"b": b, "features": f, "g": g, "h": h, "c": c}
    op = state["op"]
    v = op.excitation_batch(*state["waves"])
    return {"v": v, "rcs": op.rcs(state["i"], state["theta"], state["phi"])}


# ---------------------------------------------------------------- work
def _matvec(s, case, nrhs, mode):
    """Bytes and flops of one product with nrhs vectors: every stored near entry and pattern sample
    read once, x and y once; each multiply-add of the method."""
    cur = 2 if case["ie"] == PMCHWT else 1
    entry = 16 if mode == "fp64" else 8        # FP32 complex, or a split pair of BF16 complex
    b = s["near"] * entry + 2 * s["rwg"] * 3 * s["k0"] * entry + 2 * s["n"] * nrhs * 16
    f = 8 * nrhs * s["near"] * (4.0 / 3.0 if cur == 2 else 1.0)              # PMCHWT: 3 planes, 4 products
    f += 8 * nrhs * 3 * cur * (2 * s["rwg"] * s["k0"] + s["pairs"] + 2 * (6 / 4.0 + 1) * s["interp"])
    return b, f


def work(case):
    if case["kind"] == "member":
        op = None
        if _key(case) not in _sizes:
            op = api.Operator(_mesh(case), **_params(case))
            _measure(case, op)
            op.close()
        s = _sizes[_key(case)]
        # set-up: 4 triangle pairs x 49 points x 2 media x about 60 flops per near entry (3 planes share
        # them), 14 points x about 40 flops per pattern sample; then the products
        b, f = _matvec(s, case, 1, "fp64")
        near_f = 8 * s["near"] * 4.0 / 3.0
        return {"bytes": b * (STEPS + 1) + s["near"] * 16 * (8 + DEGREE),
                "flops": s["near"] / 3.0 * 4 * 49 * 2 * 60 + 2 * s["rwg"] * s["k0"] * 14 * 40 + STEPS * f
                + 8 * near_f + DEGREE * STEPS * near_f}
    if _key(case) not in _sizes:
        _operator(case)
    s = _sizes[_key(case)]
    mode = "fp64" if case["far"] == FP64 else "mixed"
    if case["kind"] == "apply":
        b, f = _matvec(s, case, case["nrhs"], mode)
    elif case["kind"] == "solve":
        b, f = 0.0, 0.0
        its, r, vec = case["iterations"], case["nrhs"], s["n"] * case["nrhs"] * (16 if mode == "fp64" else 8)
        for steps, m in ((its, mode), (1, "fp64")):         # the start's residual is of x = 0
            mb, mf = _matvec(s, case, r, m)
            b, f = b + steps * mb, f + steps * mf
        inner = {0: 0, api.PRECOND_POLY: DEGREE, api.PRECOND_INNER: 10}[case["precond"]]
        b += its * inner * s["near"] * (4 if case["pre"] == BF16 else 16)
        f += its * inner * 8 * r * s["near"] * 4.0 / 3.0
        b += vec * 2 * its * (its + 1)                      # Gram-Schmidt: the basis read twice per pass
        f += 16 * 2 * s["n"] * r * its * (its + 1)
    else:
        b = 16 * s["n"] * (case["nrhs"] + 1) + s["rwg"] * 320
        f = s["rwg"] * 14 * 60 * (case["nrhs"] + case["angles"])
    return {"bytes": b, "flops": f}


def tolerance(case):
    # measured against the 64-bit evaluation (FP64 products 3e-16 to 7e-16, FP32 5e-7, split pairs of
    # BF16 4e-6, scatter 6e-15) and, for solves, between two summation orders of the near field and
    # the disaggregation (3e-4 in mixed precision after ten iterations)
    if case["kind"] == "apply":
        if case["far"] == FP64:
            return {"rel": 1e-14}
        return {"rel": 2e-5} if case["near"] == BF16 else {"rel": 2e-6}
    if case["kind"] == "solve":
        return {"rel": 1e-10} if case["far"] == FP64 else {"rel": 1e-3}
    if case["kind"] == "member":
        return {"rel": 5e-7}       # the features come back in 32 bits
    return {"rel": 5e-14}


# ---------------------------------------------------------------- the same in 64 bits
def _exact_apply(case, seed):
    """The method's stages in complex128 on the tables that the operator was given at set-up, read
    back through the inspection calls: near rows, then aggregation, interpolation, translation,
    anterpolation and disaggregation, one sum after another."""
    state = prepare(case, seed)
    op, n = state["op"], state["op"].n_rwg
    x = state["x"].cpu().numpy().T
    r = x.shape[1]
    y = np.zeros_like(x)
    for row in range(op.n):
        cols, vals = op.near_row(row)
        y[row] = vals @ x[cols]
    pm, top = case["ie"] == PMCHWT, op.max_level
    ptr, rwgs = op.level_list(top, 4)
    box = np.empty(n, dtype=np.int64)
    for t in range(len(ptr) - 1):
        box[rwgs[ptr[t]:ptr[t + 1]]] = t
    cur = [x[:n], x[n:]] if pm else [x]
    er = complex(case["eps_re"], case["eps_im"])
    ks = [2 * np.pi, 2 * np.pi * np.sqrt(er)] if pm else [2 * np.pi]
    etai = np.sqrt(1.0 / er)
    for wn, k in enumerate(ks, 1):
        lvl = {}
        for l in range(2, top + 1):
            n_theta, th, ph, w, dphi = op.grid(wn, l)
            T, P = np.meshgrid(th, ph, indexing="ij")
            kp = np.stack([np.sin(T) * np.cos(P), np.sin(T) * np.sin(P), np.cos(T)], -1).reshape(-1, 3)
            _, centre, _, parent = op.level(l)
            lvl[l] = dict(kp=kp, w=np.repeat(w, 2 * n_theta) * dphi, centre=centre, parent=parent)
        vs = np.stack([op.pattern(wn, 0, i) for i in range(n)])         # n x K x 3
        vf = np.stack([op.pattern(wn, 1, i) for i in range(n)])
        S = {top: np.zeros((len(cur), len(lvl[top]["parent"])) + vs.shape[1:] + (r,), complex)}
        for c, xc in enumerate(cur):
            np.add.at(S[top][c], box, vs[..., None] * xc[:, None, None, :])
        for l in range(top - 1, 1, -1):
            taps, wt = op.interp(wn, l)
            S[l] = np.zeros((len(cur), len(lvl[l]["centre"]), len(taps), 3, r), complex)
            ch = lvl[l + 1]
            for b, p in enumerate(ch["parent"]):
                e = np.exp(-1j * k * (lvl[l]["kp"] @ (lvl[l]["centre"][p] - ch["centre"][b])))
                S[l][:, p] += e[:, None, None] * np.einsum("qt,cqtxr->cqxr", wt, S[l + 1][:, b][:, taps])
        B = {}
        for l in range(2, top + 1):
            B[l] = np.zeros_like(S[l])
            dp, di = op.level_list(l, 1)
            dv = op.level_list(l, 2)[1]
            tf = op.tf(wn, l) * lvl[l]["w"]
            for b in range(len(dp) - 1):
                for j in range(dp[b], dp[b + 1]):
                    B[l][:, b] += tf[dv[j]][:, None, None] * S[l][:, di[j]]
            if l > 2:
                taps, wt = op.interp(wn, l - 1)
                up = lvl[l - 1]
                for b, p in enumerate(lvl[l]["parent"]):
                    e = np.exp(-1j * k * (up["kp"] @ (lvl[l]["centre"][b] - up["centre"][p])))
                    v = e[:, None, None] * B[l - 1][:, p]
                    for t in range(9):
                        for c in range(len(cur)):
                            np.add.at(B[l][c, b], taps[:, t], wt[:, t, None, None] * v[c])
        leaf = B[top][:, box]                                            # cur x n x K x 3 x r
        lin = np.einsum("nqx,cnqxr->cnr", vf, leaf)
        if not pm:
            y += (k * _ETA0 / (4 * np.pi)) * (k / (4 * np.pi)) * lin[0]
            continue
        kx = lvl[top]["kp"][None, None, :, :, None]
        curl = np.einsum("nqx,cnqxr->cnr", vf, np.cross(np.broadcast_to(kx, leaf.shape), leaf, axis=3))
        c = k * k / (16 * np.pi * np.pi)
        z = 1.0 if wn == 1 else etai
        y[:n] += c * (z * lin[0] - curl[1])
        y[n:] += c * (curl[0] + lin[1] / z)
    return torch.from_numpy(np.ascontiguousarray(y.T))


_ETA0 = 119.9169832 * np.pi      # the impedance of free space as the method states it


def _rwg(mesh):
    """RWG functions in the interface's order: edges by (smaller, larger) point id, the first face in
    file order positive; free vertices, lengths."""
    f = np.asarray(mesh.faces).reshape(-1, 3) - 1
    e = np.concatenate([f[:, [1, 2]], f[:, [2, 0]], f[:, [0, 1]]])
    free = np.concatenate([f[:, 0], f[:, 1], f[:, 2]])
    face = np.tile(np.arange(len(f)), 3)
    e = np.sort(e, axis=1)
    order = np.lexsort((face, e[:, 1], e[:, 0]))
    e, free, face = e[order], free[order], face[order]
    first = np.flatnonzero((e[:-1] == e[1:]).all(axis=1))
    p = mesh.xyz
    return dict(tri=(p[f[face[first]]], p[f[face[first + 1]]]), free=(p[free[first]], p[free[first + 1]]),
                length=np.linalg.norm(p[e[first, 0]] - p[e[first, 1]], axis=1))


_RULE = [(1 / 3, 1 / 3, 1 / 3, 0.1125)]      # the 7-point triangle rule, weights of half the unit triangle
for _a, _b, _w in ((0.059715871789770, 0.470142064105115, 0.066197076394253),
                   (0.797426985353087, 0.101286507323456, 0.0629695902724135)):
    _RULE += [(_a, _b, _b, _w), (_b, _a, _b, _w), (_b, _b, _a, _w)]


def _plane_wave(pol, th, ph):
    t, p = math.radians(th), math.radians(ph)
    r = np.array([math.sin(t) * math.cos(p), math.sin(t) * math.sin(p), math.cos(t)])
    v = -np.array([math.cos(t) * math.cos(p), math.cos(t) * math.sin(p), -math.sin(t)])
    h = np.array([-math.sin(p), math.cos(p), 0.0])
    e = v if pol == 0.0 else h
    return r, v, h, -r, e, np.cross(-r, e)


def _exact_scatter(case, seed):
    """Testing integrals of plane waves and the far field by the quadrature rule, in numpy / torch."""
    state = prepare(case, seed)
    g = _rwg(_mesh(case))
    n, k = len(g["length"]), 2 * np.pi
    dev = "cuda"
    pts, rho, nrm, wl = [], [], [], []
    for side, sign in ((0, 1.0), (1, -1.0)):
        tri, free = g["tri"][side], g["free"][side]
        nv = np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
        nv /= np.linalg.norm(nv, axis=1, keepdims=True)
        for a, b, c, w in _RULE:
            q = a * tri[:, 0] + b * tri[:, 1] + c * tri[:, 2]
            pts.append(q), rho.append(sign * (q - free)), nrm.append(nv), wl.append(w * g["length"])
    pts, rho, nrm = (torch.from_numpy(np.stack(z)).to(dev) for z in (pts, rho, nrm))     # 14 x n x 3
    wl = torch.from_numpy(np.stack(wl)).to(dev)

    def t(z):
        return torch.as_tensor(z, dtype=torch.float64, device=dev)
    out = torch.zeros(state["op"].n, case["nrhs"], dtype=torch.complex128, device=dev)
    for j, (pol, th, ph) in enumerate(zip(*state["waves"])):
        _, _, _, kin, e, h = _plane_wave(pol, th, ph)
        ex = torch.exp(-1j * k * (pts @ t(kin))) * wl
        ve = (ex * (rho @ t(e))).sum(0)
        vh = (ex * ((torch.linalg.cross(nrm, t(h).expand_as(nrm)) if case["ie"] == CFIE else t(h)) * rho).sum(-1)).sum(0)
        if case["ie"] == PMCHWT:
            out[:n, j], out[n:, j] = ve, vh
        else:
            out[:, j] = ve if case["ie"] == EFIE else case["alpha"] * ve + (1 - case["alpha"]) * vh
    i = torch.from_numpy(state["i"]).to(dev)
    rcs = np.empty((len(state["theta"]), 3))
    for a, th in enumerate(state["theta"]):
        r, v, h, *_ = _plane_wave(0.0, th, state["phi"])
        ex = torch.exp(1j * k * (pts @ t(r))) * wl
        tang = rho - (rho @ t(r))[..., None] * t(r)
        f = (ex[..., None] * tang).sum(0)
        if case["ie"] == PMCHWT:
            fm = (ex[..., None] * torch.linalg.cross(t(r).expand_as(rho), rho)).sum(0)
            tot = 1j * k * (f * i[:n, None] - fm * i[n:, None]).sum(0)
        else:
            tot = 1j * k * _ETA0 * (f * i[:, None]).sum(0)
        tot = tot.cpu().numpy()
        s = np.array([abs(v @ tot) ** 2, abs(h @ tot) ** 2]) / (4 * np.pi)
        rcs[a] = 10 * np.log10([s.sum(), s[0], s[1]])
    return {"v": out.cpu().numpy(), "rcs": rcs}


def exact(case, seed):
    if case["kind"] == "scatter":
        return _exact_scatter(case, seed)
    if case["kind"] == "apply":
        op = _operator(case)
        # reading the tables back takes a copy for each block of each row, the stages run on the host
        if op.n <= 6000 and op.n * case["nrhs"] <= 40000:
            return _exact_apply(case, seed)
    return None
