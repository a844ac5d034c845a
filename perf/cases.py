"""Performance cases of the MI355X evolution library: what its users run.

Each case is one pass through the public entry points of the oaxis package,
from a state a user's program holds to the arrays it reads back.  The kinds:

  evolve     a spacetime alone: Spacetime.evolve(steps), then its evolved
             arrays are read back on every level
  drop_in    the same step driven piece by piece (saveold, substep,
             finebound, auxiliary, restrict), as a Fortran main loop does
  batch      many uneven spacetimes advanced together (Batch.evolve)
  analysis   an output step: constraints, 0D norms and 2D arrays of all levels
  horizon    an apparent-horizon search of a state (shooting, then the flow)
  monitor    an evolution that searches its horizon every few coarse steps
  elliptic   initial data with the Hamiltonian constraint's elliptic solve
  serving    a request stream through the continuous-batching loop

Sizes are those of the library's benchmark and serving configurations and
tests (16 to 512 points along rho, 1 to 6 levels) and lie between them;
masses, amplitudes and widths come from the seed, drawn from the ranges the
workload generator uses.
"""
import os
import sys
from concurrent.futures import ThreadPoolExecutor

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(ROOT, "ollinaxis-bib_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import oaxis  # noqa: E402
from oaxis import serve, workloads  # noqa: E402


def listed():
    return [
        # the smallest evolution in use: one member of the reduced amplitude
        # bisection (equatorial symmetry, a handful of steps between checks);
        # launches and the host path count
        dict(name="collapse_32x32_2lev", kind="evolve", physics="collapse", Nr=32, Nz=32, levels=2, steps=4),
        # the plain configuration: one puncture, one level, vacuum RK4
        dict(name="puncture_128x256", kind="evolve", physics="puncture", Nr=128, Nz=256, levels=1, steps=100),
        # the largest grid the serving mix admits: one level fills the device
        dict(name="puncture_512x1024", kind="evolve", physics="puncture", Nr=512, Nz=1024, levels=1, steps=200),
        # the Brill-wave configuration: 5 box-in-box levels, ICN, Gamma-driver
        dict(name="brill_5x256x512_icn", kind="evolve", physics="brill", Nr=256, Nz=512, levels=5, steps=16),
        # one scalar pulse with shift and matter, subcycled over 3 levels
        dict(name="pulse_3x128x256_rk4", kind="evolve", physics="pulse", Nr=128, Nz=256, levels=3, steps=16),
        # a Fortran main loop keeps the recursion and calls the pieces: odd
        # sizes, ICN, advected Gamma-driver
        dict(name="drop_in_odd_93x210", kind="drop_in", physics="brill_adv", Nr=93, Nz=210, levels=2, steps=2),
        # the batched scalar-collapse family: uneven grids and level counts
        dict(name="batch_16_pulses", kind="batch", members=16, Nr=256, Nz=512, levels=4, steps=10),
        # what a run writes every so many steps: constraints, norms, arrays
        dict(name="analysis_2x256x512", kind="analysis", physics="brill", Nr=256, Nz=512, levels=2),
        # a horizon search on its own: many shots, then the spectral flow
        dict(name="horizon_both_2x128x256", kind="horizon", Nr=128, Nz=256, levels=2, method="both"),
        # horizon monitoring: a search every 16 coarse steps
        dict(name="monitor_2x128x256", kind="monitor", Nr=128, Nz=256, levels=2, steps=16, method="spectral"),
        # initial data of one request: thousands of small relaxation sweeps
        dict(name="elliptic_pulse_2x128x256", kind="elliptic", physics="pulse", Nr=128, Nz=256, levels=2),
        # the serving loop end to end: admission, preparation, batched steps,
        # searches, retirement
        dict(name="serving_6_requests", kind="serving", requests=6, Nr=128, Nz=256, levels=3, steps=48),
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case of the same kinds and ranges."""
    kind = rng.choice(["evolve", "evolve", "evolve", "evolve", "drop_in", "batch", "analysis", "horizon", "monitor",
                       "elliptic", "serving"])
    if kind == "evolve":
        physics = rng.choice(["puncture", "puncture_eq", "brill", "brill_adv", "pulse", "collapse"])
        Nr = _log_int(rng, 24, 480 if physics.startswith("puncture") else 256)
        Nz = max(24, int(Nr * rng.uniform(1.0, 2.0)))
        top = 1 if Nr > 256 else (4 if Nr > 96 else 3)
        steps = _log_int(rng, 4, 32)
        return dict(kind=kind, physics=physics, Nr=Nr, Nz=Nz, levels=rng.randint(1, top), steps=steps)
    if kind == "drop_in":
        Nr = _log_int(rng, 24, 200)
        return dict(kind=kind, physics=rng.choice(["brill_adv", "puncture_eq", "pulse"]), Nr=Nr,
                    Nz=max(24, int(Nr * rng.uniform(1.0, 2.0))), levels=rng.randint(1, 3), steps=rng.randint(1, 3))
    if kind == "batch":
        Nr = _log_int(rng, 48, 200)
        return dict(kind=kind, members=rng.randint(3, 12), Nr=Nr, Nz=2 * Nr + rng.randint(-9, 9),
                    levels=rng.randint(1, 4), steps=_log_int(rng, 2, 10))
    if kind == "analysis":
        Nr = _log_int(rng, 24, 250)
        return dict(kind=kind, physics=rng.choice(["brill", "brill_adv"]), Nr=Nr,
                    Nz=max(24, int(Nr * rng.uniform(1.0, 2.0))), levels=rng.randint(1, 2))
    if kind in ("horizon", "monitor"):
        Nr = _log_int(rng, 96, 200)
        case = dict(kind=kind, Nr=Nr, Nz=2 * Nr + rng.randint(-9, 9), levels=rng.randint(1, 2),
                    method="both" if kind == "horizon" else "spectral")
        if kind == "horizon":
            case["method"] = rng.choice(["both", "shoot"])
        else:
            case["steps"] = rng.randint(8, 24)
        return case
    if kind == "elliptic":
        Nr = _log_int(rng, 24, 120)
        return dict(kind=kind, physics=rng.choice(["brill", "pulse"]), Nr=Nr,
                    Nz=max(24, int(Nr * rng.uniform(1.0, 2.0))), levels=rng.randint(1, 2))
    Nr = _log_int(rng, 48, 100)
    return dict(kind="serving", requests=rng.randint(3, 6), Nr=Nr, Nz=2 * Nr + rng.randint(-5, 5),
                levels=rng.randint(1, 2), steps=rng.randint(16, 40))


# ------------------------------------------------------------------ inputs
def _text(physics, rng, Nr, Nz, levels):
    """Par-file text of one spacetime; the physical size of the coarsest
    level does not depend on its resolution."""
    size = "\nNrtotal = %d\nNztotal = %d\nNl0 = %d\n" % (Nr, Nz, levels - 1)
    if physics in ("puncture", "puncture_eq"):
        text = workloads.schwarzschild(float(rng.uniform(0.5, 2.0)), Nr, Nz, levels - 1)
        if physics == "puncture_eq":          # equatorial symmetry, harmonic slicing, ICN
            text += "eqsym = .true.\nslicing = harmonic\ngauge_f = 1.0\nintegrator = icn\n"
        return text
    if physics in ("brill", "brill_adv"):
        text = workloads.brill(int(rng.integers(0, 2 ** 31)), Nr, Nz, levels - 1, dr0=25.6 / Nr)
        if physics == "brill_adv":            # advected Gamma-driver with damping
            text += "driveradv = .true.\ndrivereta = 0.5\n"
        return text
    if physics == "collapse":
        return workloads.collapse_pulse(float(rng.uniform(0.1, 0.4)), Nr, Nz, levels - 1, dr0=4.0 / Nr)
    text = workloads.scalar_pulse(int(rng.integers(0, 2 ** 31)), 0)
    return text + size + "dr0 = %.17g\ndz0 = %.17g\n" % (12.0 / Nr, 12.0 / Nr)


def _horizon_text(case, rng):
    text = workloads.schwarzschild(float(rng.uniform(1.5, 2.0)), case["Nr"], case["Nz"], case["levels"] - 1)
    return text + "ahfind = .true.\nahmethod = %s\n" % case["method"]


def _spacetime(text, warm=0):
    """A spacetime with its initial data, ready to step; ``warm`` steps taken."""
    st = oaxis.Spacetime(oaxis.params_from_text(text))
    st.initial_data()
    st.initial_aux()
    if warm:
        st.evolve(warm)
    return st


def _warm(case):
    """Coarse steps before the pass: an eighth of the coarsest level's
    light-crossing of its points, so that every level's clock is past 0 and
    the curvature and the gauge have left their initial values, as in nearly
    all of a run."""
    return max(2, case["Nr"] // 8)


# grids of the batched family relative to its largest, and its level counts
_UNEVEN = ((4, 2), (2, 4), (1, 2), (2, 3), (4, 4), (1, 3), (2, 2), (4, 3))


def _batch_sizes(case):
    out = []
    for k in range(case["members"]):
        div, lev = _UNEVEN[k % len(_UNEVEN)]
        out.append((max(24, case["Nr"] // div), max(24, case["Nz"] // div), min(lev, case["levels"])))
    return out


def _serving_sizes(case):
    """(physics, Nr, Nz, levels, steps) of each request: 40 % punctures, 30 %
    Brill waves, 30 % scalar pulses, small ones and the case's largest."""
    kinds = ("puncture", "pulse", "brill", "puncture", "pulse")
    out = []
    for k in range(case["requests"]):
        div = 2 if k % 2 else 1
        lev = 1 + (k + 1) % case["levels"]
        kind = kinds[k % len(kinds)]
        out.append((kind, max(24, case["Nr"] // (div if kind == "puncture" else 2)),
                    max(24, case["Nz"] // (div if kind == "puncture" else 2)), lev,
                    max(4, case["steps"] * (k + 3) // (case["requests"] + 2))))
    return out


def prepare(case, seed):
    rng = np.random.default_rng([seed, 20])
    kind = case["kind"]
    state = {"case": dict(case)}
    if kind in ("evolve", "drop_in"):
        state["st"] = _spacetime(_text(case["physics"], rng, case["Nr"], case["Nz"], case["levels"]),
                                 warm=_warm(case))
    elif kind == "batch":
        texts = [_text("pulse", rng, nr, nz, lev) for nr, nz, lev in _batch_sizes(case)]
        with ThreadPoolExecutor(max_workers=8) as pool:
            state["members"] = list(pool.map(_spacetime, texts))
        state["batch"] = oaxis.Batch(state["members"])
        state["batch"].evolve(_warm(case) // 2)
    elif kind == "analysis":
        state["st"] = _spacetime(_text(case["physics"], rng, case["Nr"], case["Nz"], case["levels"]),
                                 warm=_warm(case))
    elif kind in ("horizon", "monitor"):
        state["st"] = _spacetime(_horizon_text(case, rng))
    elif kind == "elliptic":
        text = _text(case["physics"], rng, case["Nr"], case["Nz"], case["levels"])
        state["st"] = oaxis.Spacetime(oaxis.params_from_text(text))
    elif kind == "serving":
        state["requests"] = []
        for k, (phys, nr, nz, lev, steps) in enumerate(_serving_sizes(case)):
            text = _text(phys, rng, nr, nz, lev)
            text += "ahfind = .true.\nahfind_every = 16\n"
            state["requests"].append(serve.Request(k, text, steps, 0.01 * k, phys))
    else:
        raise ValueError("unknown kind %r" % (kind,))
    return state


# ------------------------------------------------------------------ one pass
def _evolved(params):
    """The evolved arrays (with chimethod phi follows from chi)."""
    return [n for n in oaxis.state_fields(params) if n != "phi"]


def _read(st, names):
    """{name: the array on every level, level 0 first}."""
    return {n: np.concatenate([st.download(n, lev).ravel(order="F") for lev in range(st.nlevels)]) for n in names}


# the components of one vector or tensor go together: those that a symmetry
# or a weak field keeps small are read beside the large ones
_TENSORS = {"A": "metric", "B": "metric", "H": "metric", "C": "metric", "KTA": "KT", "KTB": "KT", "KTC": "KT",
            "Delta_r": "Delta", "Delta_z": "Delta", "beta_r": "beta", "beta_z": "beta", "dtbeta_r": "dtbeta",
            "dtbeta_z": "dtbeta", "scalar_xi_r": "scalar_xi", "scalar_xi_z": "scalar_xi"}


def _read_state(st):
    """Every evolved array of every level, by tensor."""
    parts = {}
    for name, a in _read(st, _evolved(st.params)).items():
        parts.setdefault(_TENSORS.get(name, name), []).append(a)
    return {k: np.concatenate(v) for k, v in parts.items()}


def _onestep(st, level):
    """onestep(level) of the reference from the library's pieces."""
    p = st.params
    rk4 = p.integrator == oaxis.ENUMS["OA_RK4"]
    niter = 4 if rk4 else p.icniter
    dt = st.level_info(level)["dt"]
    st.saveold(level)
    for it in range(1, niter + 1):
        if rk4:
            dtw, w = ((0.5 * dt, 1 / 6), (0.5 * dt, 1 / 3), (dt, 1 / 3), (dt, 1 / 6))[it - 1]
        else:
            dtw, w = (0.5 * dt if it < niter else dt), 0.0
        st.substep(level, it, niter, dtw, w)
        if level > 0:
            st.finebound(level, dtw)
        st.auxiliary(level)
    st.advance_time(level)
    if level < st.nlevels - 1:
        _onestep(st, level + 1)
        _onestep(st, level + 1)
    if level > 0 and st.time(level)[3] % 2 == 0:
        st.restrict(level)
        st.auxiliary(level - 1)


_CONSTRAINTS = ("ham", "mom_r", "mom_z", "CDelta_r", "CDelta_z")


def _horizon_out(h):
    # dradlast and the iteration residual are what the search drives to zero,
    # and the step counts follow from rounding at its thresholds
    return {k: h[k] for k in ("found", "zcenter", "area", "radius", "mass", "theta", "rad") if k in h}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "evolve":
        st = state["st"]
        st.evolve(case["steps"])
        return _read_state(st)
    if kind == "drop_in":
        st = state["st"]
        for _ in range(case["steps"]):
            _onestep(st, 0)
        return _read_state(st)
    if kind == "batch":
        state["batch"].evolve(case["steps"])
        # what a scan looks at after a stretch of steps
        out = {}
        for name in ("alpha", "chi", "trK", "scalar_phi"):
            out[name] = np.concatenate([_read(st, [name])[name] for st in state["members"]])
        return out
    if kind == "analysis":
        st = state["st"]
        names = _evolved(st.params)
        norms, arrays = {}, {n: [] for n in _CONSTRAINTS + ("alpha", "chi")}
        for lev in range(st.nlevels):
            st.constraints(lev)
            norms[lev] = np.array([[st.norms0d(n, lev)[k] for k in ("max", "min", "nm1", "nm2")]
                                   for n in names + list(_CONSTRAINTS)])
            for n in arrays:
                arrays[n].append(st.download(n, lev).ravel(order="F"))
        # the constraints are residuals at truncation level; CDelta, nearly at
        # rounding, goes with ham and mom
        cons = np.concatenate([np.concatenate(arrays[n]) for n in _CONSTRAINTS])
        return {"norms": norms, "constraints": cons, "alpha": np.concatenate(arrays["alpha"]),
                "chi": np.concatenate(arrays["chi"])}
    if kind == "horizon":
        # a shooting search's surface has one point per accepted step, a number
        # that depends on the mass; the flow's has 10 ahNmodes + 1
        return _horizon_out(state["st"].ahfind(0, shape=case["method"] == "both"))
    if kind == "monitor":
        st = state["st"]
        st.evolve(case["steps"])
        out = _horizon_out(st.ahfind(0, shape=True))
        out.update(_read(st, ["alpha", "chi"]))
        return out
    if kind == "elliptic":
        st = state["st"]
        st.initial_data()
        st.initial_aux()
        return _read(st, ["alpha", "chi", "A", "H"] + (["scalar_phi"] if case["physics"] == "pulse" else []))
    # serving
    got = {}

    def retired(req, st, rec):
        got[req.rid] = dict(_read(st, ["alpha", "chi", "trK"]), steps=rec.steps)

    server = serve.Server(memory_budget=64e9, on_retire=retired)
    server.run(state["requests"])
    return got


# ------------------------------------------------------------------ work
_FIELDS = {"puncture": 12, "puncture_eq": 12, "brill": 16, "brill_adv": 16, "pulse": 20, "collapse": 20}
# FP64 operations of one right-hand side at a point (counted from hardware
# counters in vacuum and with shift and scalar field; between them with shift)
_RHS_FLOPS = {12: 2489.0, 16: 2950.0, 20: 3574.0}


def _step_work(physics, Nr, Nz, levels, steps):
    """Bytes and operations of ``steps`` coarse steps: each substep of a level
    reads its input, the step's start and the accumulator once and writes the
    accumulator and its output once."""
    nf = _FIELDS[physics]
    updates = float(Nr) * Nz * (2 ** levels - 1) * steps
    icn = physics in ("brill", "brill_adv", "puncture_eq")
    return updates * (64.0 if icn else 136.0) * nf, updates * (3 if icn else 4) * _RHS_FLOPS[nf]


def _solve_work(Nr, Nz, levels, sweeps):
    """An elliptic solve: ``sweeps`` coarse steps of two fields and one
    coefficient, three iterations each."""
    pts = float(Nr) * Nz * (2 ** levels - 1)
    return pts * sweeps * 3 * 7 * 8.0, pts * sweeps * 3 * 90.0


def work(case):
    kind = case["kind"]
    if kind == "serving":
        b = f = 0.0
        for phys, nr, nz, lev, steps in _serving_sizes(case):
            w = _step_work(phys, nr, nz, lev, steps)
            b, f = b + w[0], f + w[1]
            if phys != "puncture":
                w = _solve_work(nr, nz, lev, 500)
                b, f = b + w[0], f + w[1]
            b += 3 * lev * nr * nz * 16.0
        return {"bytes": b, "flops": f}
    if kind == "batch":
        b = f = 0.0
        for nr, nz, lev in _batch_sizes(case):
            w = _step_work("pulse", nr, nz, lev, case["steps"])
            b, f = b + w[0] + 4 * lev * nr * nz * 16.0, f + w[1]
        return {"bytes": b, "flops": f}
    Nr, Nz, lev = case["Nr"], case["Nz"], case["levels"]
    pts = float(Nr) * Nz * lev
    if kind in ("evolve", "drop_in"):
        b, f = _step_work(case["physics"], Nr, Nz, lev, case["steps"])
        return {"bytes": b + 16.0 * _FIELDS[case["physics"]] * pts, "flops": f}
    if kind == "analysis":
        nf = _FIELDS[case["physics"]]
        return {"bytes": pts * (nf * 8.0 + 5 * 8.0 + 7 * 16.0), "flops": pts * 1600.0}
    # a search reads the metric and curvature once (13 arrays); a shot is
    # some 100 steps of 11 source evaluations of about 1500 operations, and
    # the flow some 150 iterations of 2 x 101 evaluations
    search_b = pts * 13 * 8.0
    shots = 275.0 * Nr / 128.0
    if kind == "horizon":
        f = shots * 100 * 11 * 1500.0 + (150 * 202 * 1500.0 if case["method"] == "both" else 0.0)
        return {"bytes": search_b, "flops": f}
    if kind == "monitor":
        b, f = _step_work("puncture", Nr, Nz, lev, case["steps"])
        return {"bytes": b + search_b + 2 * 16.0 * pts, "flops": f + 20 * 202 * 1500.0}
    b, f = _solve_work(Nr, Nz, lev, 500)
    return {"bytes": b + 4 * 16.0 * pts, "flops": f}


# ------------------------------------------------------------------ exact
def exact(case, seed):
    """What run returns, where a closed form gives it: the scalar pulse's
    profile in the initial data.  The evolved arrays of the full equations
    have no closed form, and a restatement of them in numpy would be another
    FP64 program with rounding of its own, no more exact than the library."""
    if case["kind"] != "elliptic" or case["physics"] != "pulse":
        return None
    rng = np.random.default_rng([seed, 20])
    text = _text(case["physics"], rng, case["Nr"], case["Nz"], case["levels"])
    par = dict((k.strip(), v.strip()) for k, v in (line.split("=", 1) for line in text.splitlines() if "=" in line))
    dr0, dz0 = float(par["dr0"]), float(par["dz0"])
    a0, r0, s0 = float(par["scalar_a0"]), float(par["scalar_r0"]), float(par["scalar_sr0"])
    Nr, g = case["Nr"], 3
    Nz = case["Nz"] + (1 if (case["Nz"] + g) % 2 == 0 else 0)   # the forced odd z size
    arrays = []
    for lev in range(case["levels"]):
        dr, dz = dr0 / 2 ** lev, dz0 / 2 ** lev
        r = (np.arange(1 - g, Nr + 1) - 0.5)[:, None] * dr
        z = (np.arange(1 - g, Nz + 1) - 0.5 * (Nz - g + 1))[None, :] * dz
        R = np.sqrt(r * r + z * z)
        phi = a0 * (np.exp(-((R - r0) / s0) ** 2) + np.exp(-((R + r0) / s0) ** 2))
        arrays.append(phi.ravel(order="F"))
    return {"alpha": None, "chi": None, "A": None, "H": None, "scalar_phi": np.concatenate(arrays)}
