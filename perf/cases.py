"""Performance cases of rapt_amd: the work that a user of the framework has it do.

``listed()`` names the cases that are timed, ``draw(rng)`` gives further ones of
the same ranges, ``prepare``/``run`` set one up and perform one pass through
the public entry points, ``work`` counts what a pass cannot do without, and
``exact`` restates the outputs in 64-bit numpy/torch where a closed form or a
plain formula gives them.

The kinds of case, each over the sizes it is used at:

- ``particle``: ``batch.advance_particles``, full-orbit protons of 1 MeV in the
  Earth's dipole (the ``dipole_protons_1mev`` workload), from one particle (what
  a single ``Particle.advance`` does) to a few thousand.
- ``gc``: a resident guiding-centre batch advanced with a fixed output step:
  electrons in the double dipole (``doubledipole_electrons_gc``), state restored
  on the device, rows and final state brought back.
- ``gc_bounce``: guiding centres whose output step is a fraction of their bounce
  period, the library's default: ``gc_bounce_dt``, then ``advance_gcs``.
- ``adaptive``: ``batch.advance_adaptive``, protons in a tanh current sheet
  (``current_sheet_protons``), switching between the two descriptions.
- ``bounce_step``: ``batch.gc_bounce_dt`` alone, the half-bounce path of every
  guiding centre of a batch.
- ``labels``: ``surrogate.traced_labels``, bounce period, drift rate and mirror
  latitude by field-line tracing: the surrogate's training labels and the
  fallback of its flagged queries.
- ``drift``: bounce centres advanced by the bounce-averaged drift, the entry
  point behind ``BounceCenter.advance``.
- ``train``: ``Surrogate.train_steps``, Adam steps of the ensemble.
- ``infer``: ``Surrogate.infer``, ensemble inference on host queries.
- ``mu``: guiding centre and first invariant of trajectory rows, the entry
  point behind ``Particle.guidingcenter`` and ``Particle.mu``.
"""
import math

import numpy as np
import torch

import rapt_amd as rapt
from rapt_amd import _native as N
from rapt_amd import batch as BT
from rapt_amd import surrogate as SG
from rapt_amd import workloads as W

RES = 20  # rows per gyration of the full-orbit cases, as in the proton workload


def listed():
    return [
        # one proton: the smallest call, launches and the step's latency
        {"name": "particle_one", "kind": "particle", "n": 1, "delta": 3.0},
        # the full-orbit workload of 1,024 protons over its 10 s
        {"name": "particle_1024", "kind": "particle", "n": 1024, "delta": 10.0},
        # a handful of guiding centres with the default output step
        {"name": "gc_bounce_16", "kind": "gc_bounce", "n": 16, "delta": 10.0},
        # the double-dipole electron batch at its full size, a row a second
        {"name": "gc_65536", "kind": "gc", "n": 65536, "delta": 30.0, "dt": 1.0},
        # current-sheet protons, a part of the workload's 262,144 and 120 s
        {"name": "adaptive_4096", "kind": "adaptive", "n": 4096, "delta": 30.0},
        # the output steps of the whole electron batch
        {"name": "bounce_step_65536", "kind": "bounce_step", "n": 65536, "field": "double"},
        # the traced fallback of a few hundred flagged queries
        {"name": "labels_300", "kind": "labels", "n": 300, "field": "dipole"},
        # training labels in the perturbed dipole
        {"name": "labels_16384", "kind": "labels", "n": 16384, "field": "uniform"},
        # a few bounce centres, four output rows each
        {"name": "drift_5", "kind": "drift", "n": 5, "rows": 4, "field": "dipole"},
        # an epoch's part of the default two-member ensemble's training
        {"name": "train_4096", "kind": "train", "members": 2, "batch": 4096, "steps": 16},
        # half a million queries
        {"name": "infer_512k", "kind": "infer", "members": 2, "n": 1 << 19},
        # the rows of a Particle sub-batch
        {"name": "mu_200k", "kind": "mu", "n": 200003},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["particle", "gc", "gc_bounce", "adaptive", "bounce_step", "labels", "drift",
                       "train", "infer", "mu"])
    if kind == "particle":
        return {"kind": kind, "n": _log_int(rng, 1, 3000), "delta": round(rng.uniform(1, 8), 2)}
    if kind == "gc":
        return {"kind": kind, "n": _log_int(rng, 100, 65536), "delta": float(rng.randint(3, 30)),
                "dt": rng.choice([0.5, 1.0])}
    if kind == "gc_bounce":
        return {"kind": kind, "n": _log_int(rng, 1, 2000), "delta": round(rng.uniform(2, 10), 2)}
    if kind == "adaptive":
        return {"kind": kind, "n": _log_int(rng, 50, 4096), "delta": round(rng.uniform(10, 30), 1)}
    if kind == "bounce_step":
        return {"kind": kind, "n": _log_int(rng, 1, 65536),
                "field": rng.choice(["dipole", "double", "uniform"])}
    if kind == "labels":
        return {"kind": kind, "n": _log_int(rng, 20, 16384),
                "field": rng.choice(["dipole", "uniform"])}
    if kind == "drift":
        return {"kind": kind, "n": _log_int(rng, 1, 500), "rows": rng.randint(1, 4),
                "field": rng.choice(["dipole", "uniform"])}
    if kind == "train":
        return {"kind": kind, "members": rng.randint(1, 4), "batch": 64 * _log_int(rng, 2, 64),
                "steps": rng.randint(1, 8)}
    if kind == "infer":
        return {"kind": kind, "members": rng.randint(1, 4), "n": _log_int(rng, 100, (1 << 20) // 4)}
    return {"kind": kind, "n": _log_int(rng, 10, 200003)}


def _field(name):
    if name == "double":
        return rapt.fields.DoubleDipole()
    if name == "uniform":
        return rapt.fields.DipolePlusUniform(Bu=(0.0, 0.0, -10e-9))
    return rapt.fields.EarthDipole()


# ---- inputs -----------------------------------------------------------------------

def _protons(n, seed):
    """Rows (t, x, y, z, px, py, pz) of the 1 MeV proton workload."""
    w = W.dipole_protons_1mev(n=n, seed=seed)
    g = 1 / np.sqrt(1 - np.sum(w["vel"] ** 2, axis=1) / rapt.c ** 2)
    return np.c_[np.zeros(n), w["pos"], (rapt.m_pr * g)[:, None] * w["vel"]]


def _electrons(field, n, seed):
    """Rows (t, x, y, z, ppar), mu and v of the electron guiding-centre workload."""
    w = W.doubledipole_electrons_gc(n=n, seed=seed)
    m, v = rapt.m_el, w["v"]
    g = 1 / np.sqrt(1 - (v / rapt.c) ** 2)
    ppar = g * m * v * np.cos(np.radians(w["pa"]))
    tpos = np.c_[np.zeros(n), w["pos"]]
    B = N.context().field_eval(field.descriptor(), "magB", tpos)[:, 0]
    vpar = ppar / (m * g)
    mu = g ** 2 * m * (v - vpar) * (v + vpar) / (2 * B)
    return np.c_[tpos, ppar], mu, v


def _queries(n, seed):
    """(L, equatorial pitch angle [deg], log10 K [eV]) over the surrogate's domain."""
    rng = np.random.default_rng([seed, 7])
    return np.c_[rng.uniform(2, 8, n), rng.uniform(10, 89, n), rng.uniform(4, 7, n)]


def _drift_inputs(n, seed):
    """Start points, mirror fields, drift coefficients and output steps of 1 MeV proton
    bounce centres (L U[3,7], equatorial pitch angle U[20,80] deg), a row every tenth of
    a bounce period (BCtimestep's default)."""
    rng = np.random.default_rng([seed, 8])
    L, ph = rng.uniform(3, 7, n), rng.uniform(0, 2 * np.pi, n)
    sa = np.sin(np.radians(rng.uniform(20, 80, n)))
    v = float(W.speedfromKE(1e6, rapt.m_pr))
    g = 1 / math.sqrt(1 - (v / rapt.c) ** 2)
    r = L * rapt.Re
    tpos = np.c_[np.zeros(n), r * np.cos(ph), r * np.sin(ph), np.zeros(n)]
    tb = 4 * r / v * (1.30 - 0.56 * sa)  # Hamlin's bounce period in a dipole
    return tpos, rapt.B0 / L ** 3 / sa ** 2, g * rapt.m_pr * v * v / rapt.e, 0.1 * tb


def _train_inputs(case, seed):
    """Features in [-1, 1] and smooth normalised targets, the members' starting weights
    and the order of the samples."""
    rng = np.random.default_rng([seed, 9])
    n = max(4 * case["batch"], 16384)
    X = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    A = rng.normal(0, 1.5, (3, 6))
    T = np.sin(X @ A + rng.uniform(0, 6.28, 6)) @ rng.normal(0, 0.6, (6, 3))
    order = np.concatenate([rng.permutation(n) for _ in range(
        1 + case["batch"] * case["steps"] // n)])[:case["batch"] * case["steps"]]
    return X, T.astype(np.float32), SG.init_params(seed, case["members"]), order


def _infer_weights(case, seed):
    """An ensemble whose members nearly agree, as trained ones do, with biases."""
    rng = np.random.default_rng([seed, 10])
    th = SG.init_params(seed, 1)
    th = th + rng.normal(0, 0.02, th.shape)
    th = np.repeat(th, case["members"], axis=0)
    return (th * (1 + 0.01 * rng.normal(0, 1, th.shape))).astype(np.float32)


_SHIFT, _SCALE = np.array([0.01, -0.02, 0.005]), np.array([0.02, 0.03, 0.01])


def _mu_inputs(n, seed):
    """Rows of 1 MeV protons anywhere in the dipole between L = 4 and 7."""
    rows = _protons(n, seed)
    lat = W.uniform(seed, 9, n, -0.6, 0.6)
    rows[:, 1:3] *= np.cos(lat)[:, None] ** 3
    rows[:, 3] = W.uniform(seed, 0, n, 4.0, 7.0) * rapt.Re * np.cos(lat) ** 2 * np.sin(lat)
    return rows


def prepare(case, seed):
    k, s = case["kind"], {"case": case}
    ctx = N.context()
    s["ctx"] = ctx
    if k == "particle":
        s.update(field=_field("dipole"), last=_protons(case["n"], seed),
                 params=dict(rapt.params, cyclotronresolution=RES))
    elif k == "gc":
        f, n = _field("double"), case["n"]
        last, mu, v = _electrons(f, n, seed)
        S = BT.gc_state(last, rapt.m_el, -rapt.e, mu, v, case["dt"])
        s["cap"] = int(round(case["delta"] / case["dt"])) + 3
        b = N.Batch(ctx, n)
        b.upload(S, np.zeros(n, np.int32))
        b.set_rows(5, np.full(n, s["cap"], np.int64))
        desc = N.make_desc(N.MODE_GC, dict(rapt.params, solvertolerances=(1e-8, 1e-8)),
                           case["delta"])
        s.update(field=f.descriptor(), batch=b, desc=desc)
    elif k == "gc_bounce":
        f = _field("double")
        last, mu, v = _electrons(f, case["n"], seed)
        s.update(field=f, last=last, mu=mu, v=v)
    elif k == "adaptive":
        s.update(field=rapt.fields.CurrentSheet(), w=W.current_sheet_protons(case["n"], seed),
                 params=dict(rapt.params, GCtimestep=0.5))
    elif k == "bounce_step":
        f = _field(case["field"])
        last, mu, _ = _electrons(f, case["n"], seed)
        s.update(field=f, last=last, mu=mu)
    elif k == "labels":
        s.update(field=_field(case["field"]), query=_queries(case["n"], seed))
    elif k == "drift":
        s.update(field=_field(case["field"]).descriptor(), inputs=_drift_inputs(case["n"], seed))
    elif k == "train":
        X, T, th, order = _train_inputs(case, seed)
        s.update(X=X, T=T, order=order,
                 net=SG.Surrogate(_field("uniform"), members=case["members"], theta0=th))
    elif k == "infer":
        net = SG.Surrogate(_field("uniform"), members=case["members"],
                           theta0=_infer_weights(case, seed))
        net.set_norm(_SHIFT, _SCALE)
        s.update(net=net, query=_queries(case["n"], seed))
    else:
        s.update(field=_field("dipole").descriptor(), rows=_mu_inputs(case["n"], seed))
    return s


# ---- one pass -----------------------------------------------------------------------

# rows a second that a case's tracers write: the mean, its spread from tracer to tracer and
# the most that any of them can (the strongest field, the shortest bounce period of the draw)
_ROWS = {"particle": (67.0, 36.0, 150.0, 4), "gc_bounce": (19.0, 15.0, 60.0, 4),
         "adaptive": (3.1, 0.0, 3.1, 40)}


def _traced(case, res):
    """All trajectories one after the other, then zeros up to a length that is the same for
    every draw of the inputs; the final state."""
    n, (mean, spread, most, more) = case["n"], _ROWS[case["kind"]]
    per = min(most, mean + 6 * spread / math.sqrt(n)) * case["delta"] + more
    rows = np.zeros((int(n * per), res.rows[0].shape[1]))
    np.concatenate(res.rows, out=rows[:sum(map(len, res.rows))])
    return {"rows": rows, "state": res.state, "status": res.status, "naccpt": res.naccpt}


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "particle":
        return _traced(case, BT.advance_particles(s["field"], s["last"], rapt.m_pr, rapt.e,
                                            case["delta"], params=s["params"]))
    if k == "gc":
        b = s["batch"]
        s["ctx"].set_field(s["field"])
        b.reset()
        b.run(s["desc"])
        out = b.download()
        rows = out["rows"].reshape(case["n"], s["cap"], 5)
        rows[np.arange(s["cap"]) >= out["nrows"][:, None]] = 0.0  # rows that were not written
        return {"rows": rows, "state": out["state"], "status": out["status"],
                "naccpt": out["naccpt"]}
    if k == "gc_bounce":
        dt, _ = BT.gc_bounce_dt(s["field"], s["last"], rapt.m_el, s["mu"])
        return _traced(case, BT.advance_gcs(s["field"], s["last"], rapt.m_el, -rapt.e, s["mu"], s["v"],
                                      dt, case["delta"]))
    if k == "adaptive":
        w = s["w"]
        return _traced(case, BT.advance_adaptive(s["field"], w["pos"], w["vel"], 0.0, rapt.m_pr,
                                           rapt.e, case["delta"], params=s["params"]))
    if k == "bounce_step":
        return BT.gc_bounce_dt(s["field"], s["last"], rapt.m_el, s["mu"])
    if k == "labels":
        return SG.traced_labels(s["field"], s["query"])
    if k == "drift":
        tpos, Bm, coef, dt = s["inputs"]
        rtol, atol = rapt.params["solvertolerances"]
        rows, end, st, acc = s["ctx"].bounce_center_advance(
            s["field"], tpos, Bm, coef, dt, 0.0, case["rows"], rtol, atol,
            rapt.params["eyegradientstep"], rapt.params["fieldlineresolution"])
        return np.concatenate(rows), end, st, acc
    if k == "train":
        loss, grad = s["net"].train_steps(s["X"], s["T"], s["order"], case["batch"], 1e-3, 5e-4,
                                          want_grad=True)
        return loss, grad, s["net"].params()
    if k == "infer":
        vals, flag, _, _ = s["net"].infer(s["query"], 1e-3)
        return vals, flag
    return s["ctx"].particle_gc(s["field"], s["rows"], rapt.m_pr, rapt.e)


# ---- what a pass cannot do without -----------------------------------------------------
# Floating-point operations: a Lorentz right-hand side in the dipole 34 and a DOP853
# attempt 988 beside its right-hand sides (1,396 an accepted step); a guiding-centre
# right-hand side 484 and a DOPRI5 attempt 282 (3,238 an accepted step); a point of a traced
# field line 6 field directions of about 40. Steps and points a second are those that the
# workloads take on average.
_STEP_P, _STEP_G = 1396.0, 3238.0
_LINE = 2 * 100 * 6 * 40.0 + 512 * 8.0  # both halves at 50 points a curvature radius, one integral


def work(case):
    k, n = case["kind"], case.get("n", 1)
    if k == "particle":
        rows = 67.0 * n * case["delta"]
        return {"bytes": 56.0 * n + 56.0 * rows, "flops": 2.6 * rows * _STEP_P}
    if k == "gc":
        rows = n * (case["delta"] / case["dt"])
        return {"bytes": 2 * 128.0 * n + 40.0 * rows, "flops": 100.0 * n * case["delta"] * _STEP_G}
    if k == "gc_bounce":
        rows = 18.0 * n * case["delta"]
        return {"bytes": 2 * 128.0 * n + 40.0 * rows,
                "flops": n * _LINE + 143.0 * n * case["delta"] * _STEP_G}
    if k == "adaptive":
        rows = 3.0 * n * case["delta"]
        return {"bytes": 2 * 128.0 * n + 64.0 * rows, "flops": 4.3 * n * case["delta"] * _STEP_P}
    if k == "bounce_step":
        return {"bytes": (48.0 + 16.0) * n, "flops": n * _LINE}
    if k == "labels":
        return {"bytes": (24.0 + 28.0) * n, "flops": 5 * n * _LINE}
    if k == "drift":
        return {"bytes": (64.0 + 44.0 + 32.0 * case["rows"]) * n,
                "flops": 5 * 7 * n * case["rows"] * _LINE}
    if k == "train":
        p, m, bt, st = SG.NPARAM, case["members"], case["batch"], case["steps"]
        return {"bytes": 24.0 * bt * st + 32.0 * p * m, "flops": 6.0 * p * m * bt * st}
    if k == "infer":
        return {"bytes": (12.0 + 16.0) * n, "flops": 2.0 * SG.NPARAM * case["members"] * n}
    return {"bytes": (56.0 + 52.0) * n, "flops": 5 * 60.0 * n}


# ---- the same in 64 bits -----------------------------------------------------------------

def _dipole_line(L, Bm, nodes=200):
    """S_b and I between the mirror points of the dipole line of equatorial distance L [Re]
    at mirror field Bm, and the mirror latitude [rad]; Gauss-Legendre in a variable that
    removes the end-point singularities. Zero I where the line has no mirror point."""
    beq = rapt.B0 / L ** 3
    s2 = np.minimum(beq / Bm, 1.0)
    lo, hi = np.zeros_like(s2), np.ones_like(s2)  # (1 - x)^3 = s2 sqrt(1 + 3 x), x = sin^2 lat
    for _ in range(200):
        x = 0.5 * (lo + hi)
        up = (1 - x) ** 3 - s2 * np.sqrt(1 + 3 * x) > 0
        lo, hi = np.where(up, x, lo), np.where(up, hi, x)
    lat = np.arcsin(np.sqrt(0.5 * (lo + hi)))
    u, w = np.polynomial.legendre.leggauss(nodes)
    u, w = 0.5 * np.pi * (u + 1), 0.5 * np.pi * w
    S, I = np.zeros_like(s2), np.zeros_like(s2)
    for uk, wk in zip(u, w):
        la = -lat * np.cos(uk)
        c2 = np.cos(la) ** 2
        q = np.sqrt(4 - 3 * c2)
        ds = L * rapt.Re * np.cos(la) * q * lat * np.sin(uk) * wk
        val = np.maximum(1 - s2 * q / c2 ** 3, 1e-300)
        S += ds / np.sqrt(val)
        I += ds * np.sqrt(val)
    return S, np.where(beq < Bm, I, 0.0), lat


def _exact_labels(query):
    q = np.asarray(query, np.float64)
    L, K = q[:, 0], 10.0 ** q[:, 2] * rapt.e
    g = 1 + K / (rapt.m_pr * rapt.c ** 2)
    v = rapt.c * np.sqrt(1 - 1 / g ** 2)
    beq, d = rapt.B0 / L ** 3, rapt.params["eyegradientstep"] / rapt.Re
    Bm = beq / np.sin(np.radians(q[:, 1])) ** 2
    S, I, lat = _dipole_line(L, Bm)
    Ip, Im = _dipole_line(L + d, Bm)[1], _dipole_line(L - d, Bm)[1]
    dI = np.where(Im == 0.0, (Ip - I) / d, (Ip - Im) / (2 * d)) / rapt.Re
    wd = -g * rapt.m_pr * v * v / (rapt.e * S * beq) * dI / (L * rapt.Re)
    return np.c_[2 * S / v, wd, np.degrees(lat)]


def _exact_mu(rows):
    p, m, q, c = rows[:, 4:7], rapt.m_pr, rapt.e, rapt.c

    def B(r):
        r2 = np.sum(r * r, axis=1)[:, None]
        return -rapt.B0 * rapt.Re ** 3 / r2 ** 2.5 * (3 * r[:, 2:3] * r - r2 * [[0.0, 0.0, 1.0]])

    gm = np.sqrt(m * m + np.sum(p * p, axis=1) / c ** 2)[:, None]
    v, r = p / gm, rows[:, 1:4]

    def rho(at):
        b = B(at)
        return gm / (q * np.sum(b * b, axis=1)[:, None]) * np.cross(b, v)

    old, done = r - rho(r), np.zeros(len(r), bool)
    out = old.copy()
    for _ in range(20):
        new = r - rho(old)
        out[~done] = new[~done]
        done |= np.linalg.norm(new - old, axis=1) < 1e-3 * np.linalg.norm(new, axis=1)
        old = new
    b = B(out)
    bn, vsq = np.linalg.norm(b, axis=1), np.sum(v * v, axis=1)
    vp, sp = np.sum(v * b, axis=1) / bn, np.sqrt(vsq)
    mu = m / (1 - vsq / c ** 2) * (sp - vp) * (sp + vp) / (2 * bn)
    res = np.c_[out, vp, sp, mu]
    res[~done] = np.nan
    return res


_PARTS = (("W1", (256, 3)), ("b1", (256,)), ("W2", (256, 256)), ("b2", (256,)),
          ("W3", (256, 256)), ("b3", (256,)), ("W4", (3, 256)), ("b4", (3,)))


def _net(th, X):
    """The network in base-2 units: hidden units a / (1 + 2^-a)."""
    at, ps = 0, []
    for _, shape in _PARTS:
        size = int(np.prod(shape))
        ps.append(th[at:at + size].reshape(shape))
        at += size
    h = X
    for W_, b in zip(ps[0:6:2], ps[1:6:2]):
        a = h @ W_.T + b
        h = a * torch.sigmoid(a * math.log(2.0))
    return h @ ps[6].T + ps[7]


def _exact_train(case, seed):
    X, T, th0, order = _train_inputs(case, seed)
    X, T = torch.from_numpy(X).double(), torch.from_numpy(T).double()
    loss, grad, theta = [], [], []
    for k in range(case["members"]):
        th = torch.from_numpy(th0[k]).double()
        m1, m2 = torch.zeros_like(th), torch.zeros_like(th)
        for st in range(case["steps"]):
            idx = torch.from_numpy(order[st * case["batch"]:(st + 1) * case["batch"]])
            th.requires_grad_(True)
            ls = ((_net(th, X[idx]) - T[idx]) ** 2).mean()
            g, = torch.autograd.grad(ls, th)
            th = th.detach()
            f = st / (case["steps"] - 1) if case["steps"] > 1 else 0.0
            lr = 5e-4 + 0.5 * 5e-4 * (1 + math.cos(math.pi * f))
            m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
            th = th - lr * (m1 / (1 - 0.9 ** (st + 1))) / (
                torch.sqrt(m2 / (1 - 0.999 ** (st + 1))) + 1e-8)
        loss.append(float(ls.detach()))
        grad.append(g.numpy())
        theta.append(th.numpy())
    return np.array(loss), np.array(grad), np.array(theta)


def _exact_infer(case, seed):
    q = _queries(case["n"], seed).astype(np.float32).astype(np.float64)
    L, al, K = q[:, 0], q[:, 1], 10.0 ** q[:, 2] * rapt.e
    d = rapt.params["eyegradientstep"]

    def beq(x):  # equatorial field of the dipole and the uniform field along z
        return np.abs(rapt.B0 * (rapt.Re / x) ** 3 - 10e-9)

    sa = np.sin(np.radians(al))
    Bm = beq(L * rapt.Re) / sa ** 2
    side = (beq(L * rapt.Re - d) > Bm) | (np.abs(beq(L * rapt.Re - d) - Bm) / Bm < 1e-12)
    X = np.c_[(L - 5) / 3, (al - 49.5) / 39.5 + 2.5 * side, (q[:, 2] - 5.5) / 1.5]
    Xt = torch.from_numpy(X)
    th = torch.from_numpy(_infer_weights(case, seed)).double()
    y = sum(_net(t, Xt) for t in th).numpy() / len(th)
    g = 1 + K / (rapt.m_pr * rapt.c ** 2)
    beta = np.sqrt(1 - 1 / g ** 2)
    base = np.c_[0.117 * L / beta * (1 - 0.4635 * sa ** 0.75),
                 2 * np.pi * L * g * beta ** 2 / (8.481 * (1 - sa ** 0.62 / 3)
                                                  * (rapt.m_pr / 1.672621777e-27)),
                 np.degrees(_dipole_line(L, rapt.B0 / L ** 3 / sa ** 2, 2)[2])]
    out = base * np.exp(_SHIFT + _SCALE * y)
    out[:, 1] *= -1
    return out, None


def exact(case, seed):
    k = case["kind"]
    if k == "bounce_step" and case["field"] == "dipole":
        last, mu, v = _electrons(_field("dipole"), case["n"], seed)
        L = np.linalg.norm(last[:, 1:4], axis=1) / rapt.Re
        g = 1 / np.sqrt(1 - (v / rapt.c) ** 2)
        S = _dipole_line(L, rapt.m_el * g ** 2 * v ** 2 / (2 * mu))[0]
        return 2 / v * S / rapt.params["bounceresolution"], S
    if k == "labels" and case["field"] == "dipole":
        return _exact_labels(_queries(case["n"], seed)), None
    if k == "train" and case["members"] * case["batch"] * case["steps"] <= 200000:
        return _exact_train(case, seed)
    if k == "infer" and case["members"] * case["n"] <= 1 << 20:
        return _exact_infer(case, seed)
    if k == "mu":
        return _exact_mu(_mu_inputs(case["n"], seed)), None
    return None
