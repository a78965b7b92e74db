"""The work users have the growth machine do, as cases that can be timed.

Every case is one or more whole domains, from host arrays to host results, as
the host application hands them over (caHdl::solve_RXGROWTH,
SCORE_Kernel.cpp:6497-6792): create the handle, grow to completion, read back
what the application reads, release.  Sizes and settings are those of this
repository's workloads (`synth.WORKLOADS`, the ensemble, served-stream and
rolled-sheet sections of `bench.py`) and of its GPU tests.

Fields of a case:
  nx, ny, nz, grains, nuclei   the Voronoi domain
  model      "rh" Rollett-Holm or "sg" Sebald-Gottstein mobility
  T0, T1     temperature at the start and after 3.6e5 s (equal: isothermal)
  sheet      1: pancake grains, sites biased to boundaries, half the nuclei
             arriving over steps 1..70, rho recovering as exp(-t/100 s)
  regions    OMP_NUM_THREADS of the SCORE run to reproduce (0: one region)
  logs       1: defragmentation and grain-evolution log at seven fractions of X
  watch      n > 0: stepped n at a time with a status vector after each chunk
  domains    > 0: that many domains of edges lo..hi in one batch, `inflight` at a time;
             `mix` settles their edges, densities and temperatures
"""
from __future__ import annotations

import math
import random

import numpy as np

from score_amd import abi, synth
from score_amd.growth import GrowthMachine, batch_run

FRACTIONS = (0.05, 0.2, 0.4, 0.6, 0.8, 0.9, 0.95)
# trajectory columns a user plots or writes to SCORE's kinetics and front files
COLUMNS = ("t", "dt", "X", "rhomax", "sv", "nfull_inside", "nfull_border", "ninfected")
# rows a program sets aside for them: a run's steps depend on its inputs
ROWS = 8192


def _case(name, nx, ny, nz, grains, nuclei, model="rh", T0=1000.0, T1=1000.0, sheet=0, regions=0, logs=0, watch=0):
    return dict(name=name, nx=nx, ny=ny, nz=nz, grains=grains, nuclei=nuclei, model=model, T0=T0, T1=T1, sheet=sheet,
                regions=regions, logs=logs, watch=watch, domains=0)


def listed():
    return [
        # the smallest domains of the tests: a few hundred steps of a few hundred
        # cells each, all launches and round trips
        _case("tiny", 24, 20, 18, 6, 10),
        # the 100^3 workload, the size of SCORE's own single-core example decks
        _case("voronoi100", 100, 100, 100, 50, 500),
        # ragged edges, with the on-the-fly defragmentation and the grain log that
        # SCORE's decks switch on through their X log points
        _case("ragged_logs", 131, 77, 59, 75, 600, logs=1),
        # the other mobility model: its time step depends on the weights
        _case("sebald", 72, 64, 81, 45, 300, model="sg", T0=900.0, T1=900.0),
        # annealing with a heating ramp: every scalar changes in every step
        _case("ramp", 90, 66, 75, 50, 250, T0=900.0, T1=1100.0),
        # the rolled sheet at a quarter of its edges: arrivals and recovery
        _case("sheet", 256, 256, 64, 3125, 15625, sheet=1),
        # a SCORE run with eight OpenMP threads
        _case("regions8", 160, 160, 160, 244, 3052, regions=8),
        # growth watched from outside: the front's status vector every 20 steps
        _case("watched", 192, 160, 144, 264, 3300, watch=20),
        # an ensemble, as the rank's loop over its domains runs it
        dict(name="ensemble", domains=24, inflight=12, lo=64, hi=192, mix=1),
        # the largest requests of the served stream
        _case("cube320", 320, 320, 320, 1953, 24414),
        # the 512^3 workload
        _case("voronoi512", 512, 512, 512, 8000, 100000),
    ]


def draw(rng):
    """A domain of log-uniform volume between the tests' and the 512^3
    workload's, of odd edges within a factor of two or so of each other, grain
    and nucleus densities of the workloads and of the ensemble, options as they
    come; or a small ensemble."""
    if rng.random() < 0.12:
        lo = rng.randint(32, 96)
        return dict(domains=rng.randint(3, 24), inflight=rng.randint(2, 16), lo=lo, hi=lo + rng.randint(8, 96),
                    mix=rng.randint(0, 1 << 30))
    kind = rng.choice(("plain", "plain", "plain", "plain", "logs", "sg", "ramp", "sheet", "regions", "watch"))
    # the stepwise settings stay at the sizes they are used at
    top = 512 ** 3 if kind == "plain" else 200 ** 3
    v = math.exp(rng.uniform(math.log(8000.0), math.log(top)))
    a, b = math.exp(rng.uniform(-0.35, 0.35)), math.exp(rng.uniform(-0.35, 0.35))
    if kind == "sheet":
        a, b = 2.0, 2.0
    e = v ** (1.0 / 3.0) / (a * b) ** (1.0 / 3.0)
    least = 48 if kind == "regions" else 16
    nx, ny, nz = (max(least, min(640, int(round(f * e)))) for f in (a, b, 1.0))
    N = nx * ny * nz
    T = float(rng.randint(900, 1100))
    c = _case(None, nx, ny, nz, max(1, int(N / rng.choice((2000, 16777, 20000)))), max(2, int(N * 10.0 ** rng.uniform(-4.0, -3.0))),
              T0=T, T1=T)
    del c["name"]
    if kind == "logs":
        c["logs"] = 1
    elif kind == "sg":
        c["model"] = "sg"
    elif kind == "ramp":
        c["T0"], c["T1"] = 900.0, 1100.0
    elif kind == "sheet":
        c["sheet"], c["T0"], c["T1"] = 1, 1000.0, 1000.0
    elif kind == "regions":
        c["regions"] = rng.choice((2, 3, 4, 6, 8))
    elif kind == "watch":
        c["watch"] = rng.randint(5, 60)
    return c


def _domain(c, seed):
    if c["sheet"]:
        return synth.make_rolled_sheet_domain(c["nx"], c["ny"], c["nz"], n_grains=c["grains"], n_nuclei=c["nuclei"],
                                              arrival_steps=70, gb_bias=3.0, seed=seed)
    return synth.make_voronoi_domain(c["nx"], c["ny"], c["nz"], n_grains=c["grains"], n_nuclei=c["nuclei"], seed=seed)


def _params(c, N):
    kw = dict(mobility_model=abi.MOB_SEBALDGOTTSTEIN if c["model"] == "sg" else abi.MOB_ROLLETTHOLM,
              sched_temp=(c["T0"], c["T1"]), n_regions=c["regions"])
    if c["sheet"]:
        kw.update(recovery_mode=4, rec_tau=100.0, rh_hagb_m0=100.0)
    if c["logs"]:
        kw.update(defrag_at=tuple(f * N for f in FRACTIONS), grainlog_at=tuple(f * N for f in FRACTIONS))
    return synth.ParamsSpec(**kw)


def prepare(case, seed):
    """Host arrays, as SCORE holds its domains before solve_RXGROWTH."""
    if case["domains"]:
        rng = random.Random(case["mix"])
        doms, prms = [], []
        for i in range(case["domains"]):
            e = rng.randint(case["lo"], case["hi"])
            T = rng.uniform(900.0, 1100.0)
            doms.append(synth.make_voronoi_domain(e, e, e, n_grains=max(1, e ** 3 // 2000),
                                                  n_nuclei=max(1, round(10.0 ** rng.uniform(-5.0, -3.0) * e ** 3)),
                                                  seed=seed * 100003 + i))
            prms.append(synth.ParamsSpec(sched_temp=(T, T)))
        return dict(case=case, doms=doms, prms=prms)
    dom = _domain(case, seed)
    return dict(case=case, dom=dom, prm=_params(case, dom.N))


def _rows(a, n):
    """The rows of a log in the n that are set aside for it."""
    out = np.zeros((n,) + a.shape[1:], a.dtype)
    out[:len(a)] = a[:n]
    return out


def run(state):
    c = state["case"]
    if c["domains"]:
        outs = batch_run(state["doms"], state["prms"], max_inflight=c["inflight"])
        return dict(defg=np.concatenate([o["defg_counts"] for o in outs]),
                    rxg=np.concatenate([o["rxg_counts"] for o in outs]),
                    t=np.array([o["result"]["t"] for o in outs]), X=np.array([o["result"]["X"] for o in outs]),
                    step=np.array([o["result"]["step"] for o in outs]),
                    sum_sv=np.array([o["result"]["sum_sv"] for o in outs]))
    out = {}
    with GrowthMachine(state["dom"], state["prm"]) as gm:
        if c["watch"]:
            # the grain each cell of the front was last seen with
            out["seen"] = np.zeros(state["dom"].N, np.uint32)
            while not gm.step(c["watch"]):
                ixyz, gid = gm.status()
                out["seen"][ixyz] = gid
        else:
            gm.solve_rxgrowth()
        out["defg"], out["rxg"] = gm.counts()
        out["map"] = gm.grainmap()
        tr = gm.trajectory()
        for k in COLUMNS:
            out[k] = _rows(tr[k], ROWS)
        if c["logs"]:
            rows, counts = gm.grainlog()
            n = len(FRACTIONS)
            out["log_t"], out["log_X"], out["log_counts"] = _rows(rows["t"], n), _rows(rows["X"], n), _rows(counts, n)
    return out


def work(case):
    """Each input read once, each output written once (the trajectory is a few
    hundred rows and not counted): the cell grid in and the grain map out, or the
    counts alone for a batch; orientations, densities and sites; the counts."""
    if case["domains"]:
        e = 0.5 * (case["lo"] + case["hi"])
        N = case["domains"] * e ** 3
        return {"bytes": 4.0 * N + (N / 2000.0) * 52.0 + N * 2e-4 * 48.0, "flops": 0.0}
    N = case["nx"] * case["ny"] * case["nz"]
    return {"bytes": 8.0 * N + case["grains"] * 52.0 + case["nuclei"] * 48.0, "flops": 0.0}


# The 26 infection attempts in SCORE's call order (SCORE_Kernel.cpp:4611-4638)
# with their distance class (1 face, 2 edge, 3 corner) and the carry and velocity
# factors of the classes (:4051-4053, :4568-4599).
_OFFS = ([(-1, -1, 0), (0, -1, 0), (1, -1, 0), (-1, 0, 0), (1, 0, 0), (-1, 1, 0), (0, 1, 0), (1, 1, 0)]
         + [(-1, 1, -1), (0, 1, -1), (1, 1, -1), (-1, -1, -1), (0, -1, -1), (1, -1, -1), (-1, 0, -1), (0, 0, -1), (1, 0, -1)]
         + [(x, y, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)])
_CARRY = np.array([0.0, 0.0682, 0.0542, 0.0484])
_SHAPE = np.array([1.0, 1.0, 0.7957, 0.6494])


def _weight(p, q, prm):
    """Rollett-Holm weight of the cubic disorientation between rows of p and q."""
    q = q * np.array([1.0, -1.0, -1.0, -1.0])
    a = q[:, 0] * p[:, 0] - q[:, 1] * p[:, 1] - q[:, 2] * p[:, 2] - q[:, 3] * p[:, 3]
    b = p[:, 0] * q[:, 1] + q[:, 0] * p[:, 1] + (q[:, 2] * p[:, 3] - q[:, 3] * p[:, 2])
    c = p[:, 0] * q[:, 2] + q[:, 0] * p[:, 2] + (q[:, 3] * p[:, 1] - q[:, 1] * p[:, 3])
    d = p[:, 0] * q[:, 3] + q[:, 0] * p[:, 3] + (q[:, 1] * p[:, 2] - q[:, 2] * p[:, 1])
    s = -np.sort(-np.abs(np.stack([a, b, c, d], 1)), axis=1)
    om = np.maximum(np.maximum(s[:, 0], (s[:, 0] + s[:, 1]) * math.sqrt(0.5)), s.sum(1) * 0.5)
    th = np.where(om < 1.0 - 5e-16, 2.0 * np.arccos(np.minimum(om, 1.0)), 0.0)
    return 1.0 - prm.rh_cut * np.exp(-prm.rh_trans * (th / math.radians(15.0)) ** prm.rh_exponent)


def _grow(dom, prm):
    """SCORE's growth loop in plain numpy: one region, isothermal, Rollett-Holm,
    site-saturated nuclei.  Returns the trajectory's floating columns."""
    nx, ny, nz, N, nd = dom.nx, dom.ny, dom.nz, dom.N, dom.n_defg
    xyz = lambda c: (c % nx, (c // nx) % ny, c // (nx * ny))  # noqa: E731
    grid = dom.cellgrid.astype(np.int64).copy()
    qd, qr = dom.ori_quat[dom.defg_ori], dom.ori_quat[dom.rxg_ori]
    T = prm.sched_temp[0]
    Gb = 0.5 * prm.G0 * (-1.38e-9 * T ** 3 + 1.21e-6 * T ** 2 - 4.58e-4 * T + 1.0) * prm.b0 ** 2
    m = prm.rh_hagb_m0 * math.exp(-prm.rh_hagb_hact_ev * synth.ECHARGE / (1.3806488e-23 * T))
    press = Gb * (dom.defg_rho - 1.0e11)
    count = np.bincount(dom.cellgrid, minlength=nd)

    def shell(x, y, z):
        return ~((x > 0) & (x < nx - 1) & (y > 0) & (y < ny - 1) & (z > 0) & (z < nz - 1))

    # lists as columns over slots: act, frac, P, cell, defg, rxg, shape
    cap = [N, 2 * (nx * ny + nx * nz + ny * nz)]
    reuse = [int(prm.rel_cell_caching * N * prm.maxfill * 3.0), int(cap[1] * prm.maxfill * 3.0)]
    L = [dict(n=0, act=np.zeros(k, bool), frac=np.zeros(k), P=np.zeros(k), cell=np.zeros(k, np.int64),
              defg=np.zeros(k, np.int64), rxg=np.zeros(k, np.int64), shape=np.ones(k)) for k in cap]

    def put(l, slots, frac, P, cell, defg, rxg, shape):
        q = L[l]
        q["act"][slots], q["frac"][slots], q["P"][slots], q["cell"][slots] = True, frac, P, cell
        q["defg"][slots], q["rxg"][slots], q["shape"][slots] = defg, rxg, shape

    sites, first = np.unique(dom.rxg_site.astype(np.int64), return_index=True)
    k = np.sort(first)
    w = dom.rxg_site[k].astype(np.int64)
    g = grid[w]
    out = shell(*xyz(w))
    for l in (0, 1):
        s = out == bool(l)
        n = int(s.sum())
        put(l, np.arange(n), 1.0, _weight(qr[k[s]], qd[g[s]], prm), w[s], g[s], k[s], 1.0)
        L[l]["n"] = n
    grid[w] = -1
    offs = np.array(_OFFS, np.int64)
    cls = np.abs(offs).sum(1)
    t, X, xc, step, tr = 0.0, 0.0, 0, 0, dict(t=[], dt=[], X=[], rhomax=[])
    dt = 1e-6
    while not (xc >= N or X > prm.xmax or step > prm.nmax or t > prm.sched_time[-1] or t > prm.tmax):
        full, free = [], []
        for q, r in zip(L, reuse):
            n, a = q["n"], q["act"][:q["n"]]
            p = press[q["defg"][:n]]
            q["frac"][:n] += np.where(a & (p > 5e-16), q["P"][:n] * m * p * q["shape"][:n] * dt / dom.cellsize, 0.0)
            full.append(np.nonzero(a & (q["frac"][:n] >= 1.0))[0])
            free.append(np.nonzero(~a)[0][:r])
        col = {f: np.concatenate([q[f][s] for q, s in zip(L, full)]) for f in ("frac", "P", "cell", "defg", "rxg")}
        par = len(col["cell"])
        if par:
            border = np.arange(par) >= len(full[0])
            x, y, z = xyz(col["cell"])
            tx, ty, tz = ((v[:, None] + offs[None, :, i]) for i, v in enumerate((x, y, z)))
            ok = (tz >= 0) & (tz < nz)
            tx, ty = tx % nx, ty % ny
            tc = np.where(ok, tx + nx * (ty + ny * np.clip(tz, 0, nz - 1)), 0)
            near = ~((x > 1) & (x < nx - 2) & (y > 1) & (y < ny - 2) & (z > 1) & (z < nz - 2))
            toB = np.where(border[:, None], shell(tx, ty, tz), near[:, None])
            a = np.nonzero((ok & (grid[tc] >= 0) & (grid[tc] < nd)).ravel())[0]
            # the first attempt in serial order takes a cell
            _, f = np.unique(tc.ravel()[a], return_index=True)
            a = a[np.sort(f)]
            pp, r = a // 26, a % 26
            c, into = tc.ravel()[a], toB.ravel()[a]
            g = grid[c]
            P = col["P"][pp].copy()
            new = col["defg"][pp] != g
            P[new] = _weight(qr[col["rxg"][pp[new]]], qd[g[new]], prm)
            carry = (col["frac"][pp] - 1.0) * _CARRY[cls[r]]
            grid[c] = -1
            grid[col["cell"]] = nd + col["rxg"]
            np.subtract.at(count, col["defg"], 1)
            for q, s in zip(L, full):
                q["act"][s], q["frac"][s] = False, 0.0
            for l in (0, 1):
                s = into == bool(l)
                n = int(s.sum())
                k = min(n, len(free[l]))
                slots = np.concatenate([free[l][:k], np.arange(L[l]["n"], L[l]["n"] + n - k)])
                L[l]["n"] += n - k
                put(l, slots, carry[s], P[s], c[s], g[s], col["rxg"][pp[s]], _SHAPE[cls[r[s]]])
        xc += par
        X = xc / N
        left = dom.defg_rho[count > 0]
        rhomax = max(1e8, float(left.max())) if len(left) else 1e8
        for f, v in (("t", t), ("dt", dt), ("X", X), ("rhomax", rhomax)):
            tr[f].append(v)
        t += dt
        step += 1
        dt = min(3600.0, prm.sched_time[-1], prm.maxfill * dom.cellsize / (m * Gb * rhomax))
    return {f: _rows(np.array(v), ROWS) for f, v in tr.items()}


def exact(case, seed):
    """The trajectory's floating columns from a plain numpy run of the automaton,
    for single isothermal Rollett-Holm domains up to the 100^3 workload's size;
    everything else a run returns is whole numbers, and larger domains or other
    settings take minutes this way."""
    if case["domains"] or case["nx"] * case["ny"] * case["nz"] > 1000000:
        return None
    if case["model"] != "rh" or case["T0"] != case["T1"] or case["sheet"] or case["regions"] or case["logs"] or case["watch"]:
        return None
    dom = _domain(case, seed)
    tr = _grow(dom, _params(case, dom.N))
    return {k: tr.get(k) for k in ("defg", "rxg", "map") + COLUMNS}
