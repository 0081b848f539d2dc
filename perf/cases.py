"""Performance cases of the level update: what a driver has this library do,
through the entry points of amrclaw_amd.capi / capi3 (the C ABI of
include/amrgpu.h and include/amrgpu3.h).

Kinds of cases
  patch2   amrgpu_stepgrid_noalloc: one 2-D patch on device arrays.
  grid3    amrgpu3_stepgrid: one 3-D grid from and to host arrays, with the six
           flux arrays the driver's register code reads.
  amr2     a 2-D run configuration (config_hierarchy: advection, acoustics,
           Euler quadrants; three levels): the grids are handed over from the
           host heap, advanced `steps` coarse Berger-Oliger steps with the
           Courant numbers read after every level step, and the frame is read
           back.  `pull` reads every level back after each of its steps, as
           the Fortran driver's shim does; `flag` ends with the gradient flags
           of the levels below the finest, as a regrid begins.
  level2   the two-level batched Euler hierarchy (n uneven patches on level 2)
           through the same cycle.
  batch3   a batch of uneven 3-D grids, `steps` steps in place.
  amr3     the 3-D radial-bump hierarchy through Berger-Oliger steps.

The library holds one run per process (like the reference's amr_module), so a
state keeps the run's host heap, and a pass hands it over, advances it and
reads it back into the state's own arrays; the layout (grids, plans) stays
installed for as long as passes use the same one.

exact() advances the same data in 64 bits with plain numpy, written from the
wave-propagation formulas: grids as padded arrays, each level also as a dense
array over its index space, so that ghost cells, refluxing and averaging are
array expressions.
"""
import functools

import numpy as np
import torch

from amrclaw_amd import capi, capi3, workload

SOLVERS = {"advection": capi.ADVECTION, "acoustics": capi.ACOUSTICS, "euler": capi.EULER}
NVAR = {"advection": 1, "acoustics": 3, "euler": 4}
PRECISION = {"f64": capi.FP64, "f32": capi.FP32, "mixed": capi.MIXED}
LAUNCH = {"default": capi.LAUNCH_BATCHED, "march": capi.LAUNCH_MARCH}
CONFIG = {"advection": "C1", "acoustics": "C2", "euler": "C3"}
GAMMA = 1.4


def listed():
    return [
        # the smallest call: one little patch, all latency
        dict(name="patch2-acoustics-16x12-f64", kind="patch2", solver="acoustics", mx=16, my=12,
             precision="f64"),
        # one odd-sized 3-D grid through the reference's stepgrid interface
        dict(name="grid3-euler-21x18x13-f64", kind="grid3", mx=21, my=18, mz=13, precision="f64"),
        # the run configuration of periodic advection between two frames
        dict(name="amr2-advection-f64", kind="amr2", solver="advection", tile=8, ibuff=3,
             steps=20, precision="f64", pull=False, flag=False),
        # acoustics as the Fortran driver runs it: every level read back after each step
        dict(name="amr2-acoustics-pull-f64", kind="amr2", solver="acoustics", tile=8, ibuff=3,
             steps=2, precision="f64", pull=True, flag=False),
        # the Euler quadrants between two regrids and frames, flags at the end
        dict(name="amr2-euler-flag-f64", kind="amr2", solver="euler", tile=8, ibuff=3, steps=10,
             precision="f64", pull=False, flag=True),
        # a small batched level, mixed precision
        dict(name="level2-mixed-24", kind="level2", n=24, layout=7, steps=6, precision="mixed",
             launch="march"),
        # the batched benchmark's level at half its patch count
        dict(name="level2-mixed-2048", kind="level2", n=2048, layout=20261202, steps=20,
             precision="mixed", launch="march"),
        # an ordinary batched level in the reference's precision
        dict(name="level2-f64-256", kind="level2", n=256, layout=11, steps=20, precision="f64",
             launch="default"),
        # 3-D batches: a small FP32 one, half the 3-D benchmark's grids, and FP64
        dict(name="batch3-f32-6", kind="batch3", n=6, layout=5, steps=4, precision="f32"),
        dict(name="batch3-f32-256", kind="batch3", n=256, layout=20261203, steps=40,
             precision="f32"),
        dict(name="batch3-f64-32", kind="batch3", n=32, layout=9, steps=10, precision="f64"),
        # the 3-D run configuration
        dict(name="amr3-euler-f32", kind="amr3", n=64, nlev=3, tile=8, ibuff=3, steps=4,
             precision="f32"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["patch2", "grid3", "amr2", "level2", "level2", "batch3", "batch3", "amr3"])
    if kind == "patch2":
        return dict(kind=kind, solver=rng.choice(list(SOLVERS)), mx=_log(rng, 4, 400),
                    my=_log(rng, 4, 400), precision=rng.choice(["f64", "f32", "mixed"]))
    if kind == "grid3":
        return dict(kind=kind, mx=_log(rng, 4, 40), my=_log(rng, 4, 40), mz=_log(rng, 4, 40),
                    precision=rng.choice(["f64", "f32"]))
    if kind == "amr2":
        pull = rng.random() < 0.25
        return dict(kind=kind, solver=rng.choice(list(SOLVERS)), tile=rng.choice([4, 6, 8, 11, 16]),
                    ibuff=rng.randint(1, 4), steps=rng.randint(1, 4) if pull else rng.randint(2, 16),
                    precision=rng.choice(["f64", "f64", "f32", "mixed"]), pull=pull, flag=False)
    if kind == "level2":
        n = _log(rng, 3, 1200)
        return dict(kind=kind, n=n, layout=rng.randrange(1 << 20), steps=rng.randint(2, 20),
                    precision=rng.choice(["f64", "f32", "mixed"]),
                    launch=rng.choice(["default", "march"]))
    if kind == "batch3":
        precision = rng.choice(["f64", "f32"])
        return dict(kind=kind, n=_log(rng, 1, 200 if precision == "f32" else 48),
                    layout=rng.randrange(1 << 20), steps=rng.randint(2, 20), precision=precision)
    return dict(kind=kind, n=rng.choice([16, 24, 32, 40, 48]), nlev=rng.choice([2, 3]),
                tile=rng.choice([4, 6, 8]), ibuff=rng.randint(1, 3), steps=rng.randint(1, 4),
                precision=rng.choice(["f64", "f32", "f32"]))


# ------------------------------------------------------------- layouts ---
def _key(case):
    """What the installed run depends on: everything but the data."""
    return tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "steps", "pull", "flag")))


@functools.lru_cache(maxsize=2)
def _layout(key):
    """The hierarchy or batch of a case, with its unperturbed initial data."""
    c = dict(key)
    if c["kind"] == "amr2":
        return workload.config_hierarchy(CONFIG[c["solver"]], tile=c["tile"], ibuff=c["ibuff"])
    if c["kind"] == "level2":
        # Courant 0.6 on level 2, whose steps are halves of level 1's
        H, _ = workload.batched_euler_hierarchy(c["n"], c["layout"], courant=0.6)
        return H
    if c["kind"] == "amr3":
        return workload.radial_euler3_hierarchy(c["n"], c["nlev"], tile=c["tile"], ibuff=c["ibuff"],
                                                nsteps=26 * c["n"] // 64)
    if c["kind"] == "batch3":
        sizes, _, h, qs = workload.batched_euler3_level(c["n"], c["layout"])
        flat = np.concatenate([q.ravel() for q in qs])
        return sizes, h, 0.4 * h / max(workload.max_wave_speed3(q) for q in qs), flat, \
            [q.shape for q in qs]
    return None


def _perturbed(flat, nvar, seed):
    """The data times 1 +- 1e-3, one factor a cell, from the seed."""
    rng = np.random.default_rng(seed)
    f = rng.random(flat.size // nvar)
    f *= 2e-3
    f += 1.0 - 1e-3
    return (flat.reshape(-1, nvar) * f[:, None]).reshape(-1)


_held = [None]


def _hold(state):
    """Install the state's run in the library unless it is the one it holds."""
    case, key = state["case"], state["key"]
    if _held[0] == key:
        return
    _held[0] = None
    kind = case["kind"]
    if kind in ("patch2", "amr2", "level2"):
        H = _layout(key)
        if kind == "patch2":
            cfg = capi.make_config(SOLVERS[case["solver"]], precision=PRECISION[case["precision"]])
        else:
            cfg = capi.make_config(SOLVERS[case.get("solver", "euler")], mthbc=H.mthbc,
                                   domain=H.domain, precision=PRECISION[case["precision"]])
        capi.init(cfg)
        if kind != "patch2":
            capi.set_launch_mode(LAUNCH[case.get("launch", "default")])
            lv = H.levels
            capi.set_geometry([L["iregsz"] for L in lv], [L["jregsz"] for L in lv],
                              [L["ratx"] for L in lv], [L["raty"] for L in lv],
                              [L["hx"] for L in lv], [L["hy"] for L in lv])
            for l, L in enumerate(lv, start=1):
                capi.set_level(l, L["boxes"], L["hx"], L["hy"])
    else:
        capi3.init3(capi3.make_config3(capi.EULER, precision=PRECISION[case["precision"]]))
        if kind == "batch3":
            capi3.set_patches3(_layout(key)[0])
        elif kind == "amr3":
            capi3.load_hierarchy3(_layout(key))
    _held[0] = key


def prepare(case, seed):
    state = dict(case=case, key=_key(case))
    kind = case["kind"]
    if kind == "patch2":
        q = _patch2(case, seed)
        state["q"] = torch.from_numpy(q).cuda()
        state["out"] = torch.empty_like(state["q"])
        state["h"], state["dt"] = 1.0 / 256, _patch2_dt(case)
    elif kind == "grid3":
        state["q"] = _grid3(case, seed)
        state["h"], state["dt"] = 1.0 / 64, 0.2 / 64
    elif kind == "batch3":
        sizes, h, dt, flat, shapes = _layout(state["key"])
        q = _perturbed(flat, 5, seed)
        out = np.zeros_like(q)
        state.update(h=h, dt=dt, q=_views(q, shapes), outs=_views(out, shapes), out=out)
    else:
        H = _layout(state["key"])
        state["levels"] = [dict(q=_perturbed(L["qnew"], H.nvar, seed + l), new=np.zeros_like(L["qnew"]),
                                old=np.zeros_like(L["qold"]) if case.get("pull") else None,
                                off=L["off"], possk=p)
                           for l, (L, p) in enumerate(zip(H.levels, _possk(case, H)))]
        state["ratio"] = [L["ratx"] for L in H.levels]
        state["shapes"] = [L["shapes"] for L in H.levels]
    _hold(state)
    return state


def _views(flat, shapes):
    out, pos = [], 0
    for s in shapes:
        n = int(np.prod(s))
        out.append(flat[pos:pos + n].reshape(s))
        pos += n
    return out


def _possk(case, H):
    if case["kind"] == "level2":
        dt2 = H.levels[1]["possk"]
        return [2.0 * dt2, dt2]
    return [L["possk"] for L in H.levels]


def _patch2(case, seed):
    """A rough patch: random states of the solver about a mean flow."""
    rng = np.random.default_rng(seed)
    shape = (case["my"] + 4, case["mx"] + 4)
    if case["solver"] == "advection":
        return rng.random(shape + (1,))
    if case["solver"] == "acoustics":
        return np.stack([1.0 + 0.1 * rng.random(shape), 0.1 * rng.normal(size=shape),
                         0.1 * rng.normal(size=shape)], -1)
    rho, p = 0.8 + 0.4 * rng.random(shape), 0.8 + 0.4 * rng.random(shape)
    u, v = 0.3 * rng.normal(size=shape), 0.3 * rng.normal(size=shape)
    return np.stack([rho, rho * u, rho * v, p / (GAMMA - 1) + 0.5 * rho * (u * u + v * v)], -1)


def _patch2_dt(case):
    return {"advection": 0.8, "acoustics": 0.4, "euler": 0.2}[case["solver"]] / 256


def _grid3(case, seed):
    rng = np.random.default_rng(seed)
    shape = (case["mz"] + 4, case["my"] + 4, case["mx"] + 4)
    rho, p = 0.8 + 0.4 * rng.random(shape), 0.8 + 0.4 * rng.random(shape)
    u = [0.3 * rng.normal(size=shape) for _ in range(3)]
    return np.stack([rho, rho * u[0], rho * u[1], rho * u[2],
                     p / (GAMMA - 1) + 0.5 * rho * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)], -1)


# ---------------------------------------------------------------- passes ---
def run(state):
    _hold(state)
    case = state["case"]
    return {"patch2": _run_patch2, "grid3": _run_grid3, "amr2": _run_amr, "level2": _run_amr,
            "batch3": _run_batch3, "amr3": _run_amr3}[case["kind"]](case, state)


def _run_patch2(case, s):
    cfl, dtnew = capi.stepgrid_noalloc(case["mx"], case["my"], s["q"].data_ptr(),
                                       s["out"].data_ptr(), s["h"], s["h"], s["dt"])
    return [s["out"], cfl, dtnew]


def _run_grid3(case, s):
    q, flux, cfl, dtnew = capi3.stepgrid3(s["q"], s["h"], s["h"], s["h"], s["dt"],
                                          want_fluxes=case["precision"] == "f64")
    return [q, flux or [], cfl, dtnew]


def _run_batch3(case, s):
    L = capi3.lib()
    for p, q in enumerate(s["q"]):
        capi3._check(L.amrgpu3_put_patch(p, q))
    for _ in range(case["steps"]):
        cfl = capi3.step_patches3(s["h"], s["h"], s["h"], s["dt"], npatch=len(s["q"]))
    for p, q in enumerate(s["outs"]):
        capi3._check(L.amrgpu3_get_patch(p, q))
    return [s["out"], cfl]


def _run_amr(case, s):
    L, levels, nlev = capi.lib(), s["levels"], len(s["levels"])
    for l, v in enumerate(levels, start=1):
        capi._check(L.amrgpu_put_level(l, 0, v["q"], v["off"]))
        capi.set_time(l, 0.0, v["possk"])
    pull, seen = case.get("pull"), [0.0] * nlev

    def tick(l):
        dt, cfl = capi.advance_level(l)
        seen[l - 1] = max(seen[l - 1], cfl)
        v = levels[l - 1]
        if pull:
            capi._check(L.amrgpu_get_level(l, 0, v["new"], v["off"]))
            if l < nlev:
                capi._check(L.amrgpu_get_level(l, 1, v["old"], v["off"]))
        if l < nlev:
            for _ in range(s["ratio"][l - 1]):
                tick(l + 1)
            capi.update_level(l)
            if pull:
                capi._check(L.amrgpu_get_level(l, 0, v["new"], v["off"]))

    for _ in range(case["steps"]):
        tick(1)
    out = []
    for l, v in enumerate(levels, start=1):
        if not pull:
            capi._check(L.amrgpu_get_level(l, 0, v["new"], v["off"]))
        out.append(v["new"])
        if pull and l < nlev:
            out.append(v["old"])
    out.append(np.array(seen))
    if case.get("flag"):
        for l in range(1, nlev):
            flags, n = capi.flag_level(l, 0.1, 0.0, mbuff=4,
                                       shapes=[(sh[1] - 4, sh[0] - 4) for sh in s["shapes"][l - 1]])
            out += [np.concatenate([f.ravel() for f in flags]).astype(np.int8), n]
    return out


def _run_amr3(case, s):
    L, levels, nlev = capi3.lib(), s["levels"], len(s["levels"])
    for l, v in enumerate(levels, start=1):
        capi3._check(L.amrgpu3_put_level(l, 0, v["q"], v["off"]))
        capi3.set_time3(l, 0.0, v["possk"])
    seen = [0.0] * nlev

    def tick(l):
        dt, cfl = capi3.advance_level3(l)
        seen[l - 1] = max(seen[l - 1], cfl)
        if l < nlev:
            for _ in range(2):
                tick(l + 1)
            capi3.update_level3(l)

    for _ in range(case["steps"]):
        tick(1)
    for l, v in enumerate(levels, start=1):
        capi3._check(L.amrgpu3_get_level(l, 0, v["new"], v["off"]))
    return [v["new"] for v in levels] + [np.array(seen)]


# ------------------------------------------------------------------ work ---
#: floating-point operations of one cell update (normal solves, limiter,
#: corrections, transverse solves), counted from the formulas below
FLOPS = {"advection": 60, "acoustics": 220, "euler": 1400, "euler3": 9000}


def _updates(case):
    """(cell updates of a pass, values handed over and read back, nvar)."""
    kind = case["kind"]
    if kind == "patch2":
        return case["mx"] * case["my"], 0, NVAR[case["solver"]]
    if kind == "grid3":
        cells = case["mx"] * case["my"] * case["mz"]
        ghosted = (case["mx"] + 4) * (case["my"] + 4) * (case["mz"] + 4)
        return cells, ghosted * 5 * (8 if case["precision"] == "f64" else 2), 5
    H = _layout(_key(case))
    if kind == "batch3":
        return case["steps"] * int(H[0].prod(axis=1).sum()), 2 * H[3].size, 5
    total, values, sub = 0, 0, 1
    for l, L in enumerate(H.levels):
        cells = sum(int(np.prod([n - 4 for n in s[:-1]])) for s in L["shapes"])
        total += case["steps"] * sub * cells
        reads = 1
        if case.get("pull"):   # new and old times after a step, new after an update
            reads = case["steps"] * sub * (3 if l + 1 < H.nlev else 1)
        values += L["qnew"].size * (1 + reads)
        sub *= L["ratx"]
    return total, values, H.nvar


def work(case):
    updates, values, nvar = _updates(case)
    size = 4 if case["precision"] == "f32" else 8
    if case["kind"] == "patch2":
        size = 8           # the caller's arrays are FP64 in every precision
    per = FLOPS["euler3"] if nvar == 5 else FLOPS[case.get("solver", "euler")]
    return {"bytes": updates * 2 * nvar * size + values * 8, "flops": updates * per}


def tolerance(case):
    # FP64 is the reference's arithmetic in the reference's order
    if case["precision"] == "f64":
        return "exact"
    # about four times what the launch forms (tile, march; fused, per-direction)
    # differ by among themselves and from the FP64 run over up to 40 steps
    # (FP32 storage 3e-7 and 5e-6 at single cells, mixed 1.5e-7 and 5e-7; a
    # limiter that switches in one cell moves the second)
    if case["precision"] == "mixed":
        return {"rel": 6e-7, "max": 1e-5}
    return {"rel": 1.2e-6, "max": 2e-5}


# ----------------------------------------------------------------- exact ---
# 64-bit wave propagation on numpy arrays.  States are (nvar, ...) arrays; a
# sweep works along the last axis; `mu` is the component of the momentum (or
# velocity) along the sweep.

def _euler_roe(gl, ql, qr, mom):
    """Roe averages of the conserved states: velocities by component, the
    enthalpy and the sound speed."""
    def h(q):
        p = gl * (q[-1] - 0.5 * sum(q[m] ** 2 for m in mom) / q[0])
        return q[-1] + p
    wl, wr = np.sqrt(ql[0]), np.sqrt(qr[0])
    u = {m: (ql[m] / wl + qr[m] / wr) / (wl + wr) for m in mom}
    H = (h(ql) / wl + h(qr) / wr) / (wl + wr)
    u2 = sum(u[m] ** 2 for m in mom)
    return dict(u=u, H=H, u2=u2, a=np.sqrt(gl * (H - 0.5 * u2)), gl=gl, mom=mom)


def _euler_waves(r, d, mu, separate):
    """Waves and speeds of a jump d along component mu; `separate` keeps the
    shear wave apart from the entropy wave (2-D)."""
    u, H, a, mom = r["u"], r["H"], r["a"], r["mom"]
    others = [m for m in mom if m != mu]
    a3 = r["gl"] / a ** 2 * ((H - r["u2"]) * d[0] + sum(u[m] * d[m] for m in mom) - d[-1])
    shear = {m: d[m] - u[m] * d[0] for m in others}
    ar = (d[mu] + (a - u[mu]) * d[0] - a * a3) / (2.0 * a)
    al = d[0] - a3 - ar
    wl, w0, ws, wr = (np.zeros_like(d) for _ in range(4))
    for w, x, sgn in ((wl, al, -1.0), (wr, ar, 1.0)):
        w[0], w[mu], w[-1] = x, x * (u[mu] + sgn * a), x * (H + sgn * u[mu] * a)
        for m in others:
            w[m] = x * u[m]
    w0[0], w0[-1] = a3, a3 * 0.5 * r["u2"]
    for m in mom:
        w0[m] = a3 * u[m]
    for m in others:
        ws[m] = shear[m]
        ws[-1] += shear[m] * u[m]
    if separate:
        return [wl, ws, w0, wr], [u[mu] - a, u[mu], u[mu], u[mu] + a]
    return [wl, w0 + ws, wr], [u[mu] - a, u[mu], u[mu] + a]


def _sound(gl, q, mom):
    return np.sqrt((gl + 1.0) * gl * (q[-1] - 0.5 * sum(q[m] ** 2 for m in mom) / q[0]) / q[0])


class _Euler:
    """Roe solver with the Harten-Hyman fix of the acoustic waves."""

    def __init__(self, dim):
        self.mom, self.dim, self.nvar = list(range(1, dim + 1)), dim, dim + 2

    def normal(self, ql, qr, mu):
        gl = GAMMA - 1.0
        r = _euler_roe(gl, ql, qr, self.mom)
        waves, s = _euler_waves(r, qr - ql, mu, self.dim == 2)
        first, last, mid = waves[0], waves[-1], waves[1:-1]
        with np.errstate(invalid="ignore", divide="ignore"):
            s0 = ql[mu] / ql[0] - _sound(gl, ql, self.mom)
            q1 = ql + first
            s1 = q1[mu] / q1[0] - _sound(gl, q1, self.mom)
            f1 = np.where((s0 < 0) & (s1 > 0), s0 * (s1 - s[0]) / np.where(s1 == s0, 1.0, s1 - s0),
                          np.minimum(s[0], 0.0))
            s3 = qr[mu] / qr[0] + _sound(gl, qr, self.mom)
            q2 = qr - last
            s2 = q2[mu] / q2[0] + _sound(gl, q2, self.mom)
            f3 = np.where((s2 < 0) & (s3 > 0), s2 * (s3 - s[-1]) / np.where(s3 == s2, 1.0, s3 - s2),
                          np.minimum(s[-1], 0.0))
        left = (s[1] < 0).astype(float)
        am = f1 * first + left * (sum(min_s * w for min_s, w in zip(s[1:-1], mid)) + f3 * last)
        am = np.where((s0 >= 0) & (s[0] > 0), 0.0, am)
        return waves, s, am, sum(x * w for x, w in zip(s, waves)) - am, r

    def split(self, r, d, mv):
        waves, s = _euler_waves(r, d, mv, self.dim == 2)
        return (sum(np.minimum(x, 0.0) * w for x, w in zip(s, waves)),
                sum(np.maximum(x, 0.0) * w for x, w in zip(s, waves)))

    def flux(self, q, mu):
        p = (GAMMA - 1.0) * (q[-1] - 0.5 * sum(q[m] ** 2 for m in self.mom) / q[0])
        f = q * (q[mu] / q[0])
        f[mu] += p
        f[-1] += p * (q[mu] / q[0])
        return f


class _Acoustics:
    nvar, rho, bulk = 3, 1.0, 4.0
    c, z = 2.0, 2.0

    def _pair(self, d, mu):
        z = self.z
        a1, a2 = (-d[0] + z * d[mu]) / (2 * z), (d[0] + z * d[mu]) / (2 * z)
        w1, w2 = np.zeros_like(d), np.zeros_like(d)
        w1[0], w1[mu], w2[0], w2[mu] = -a1 * z, a1, a2 * z, a2
        return w1, w2

    def normal(self, ql, qr, mu):
        w1, w2 = self._pair(qr - ql, mu)
        s = np.full(w1.shape[1:], self.c)
        return [w1, w2], [-s, s], -self.c * w1, self.c * w2, None

    def split(self, r, d, mv):
        w1, w2 = self._pair(d, mv)
        return -self.c * w1, self.c * w2

    def flux(self, q, mu):
        f = np.zeros_like(q)
        f[0], f[mu] = self.bulk * q[mu], q[0] / self.rho
        return f


class _Advection:
    nvar = 1
    speed = {1: 0.5, 2: 1.0}

    def normal(self, ql, qr, mu):
        w, s = qr - ql, self.speed[mu]
        return [w], [np.full(w.shape[1:], s)], min(s, 0.0) * w, max(s, 0.0) * w, None

    def split(self, r, d, mv):
        s = self.speed[mv]
        return min(s, 0.0) * d, max(s, 0.0) * d

    def flux(self, q, mu):
        return self.speed[mu] * q


def _solver(case):
    name = case.get("solver", "euler")
    return {"advection": _Advection, "acoustics": _Acoustics}[name]() if name != "euler" else \
        _Euler(3 if case["kind"] in ("grid3", "batch3", "amr3") else 2)


def _normal_sweep(sol, q, mu, dtdx):
    """Along the last axis (two ghost cells a side, n cells): at the n + 1
    interior interfaces the fluctuations, the limited second-order term and
    the solver's averages; and the largest Courant number."""
    waves, s, am, ap, r = sol.normal(q[..., :-1], q[..., 1:], mu)
    i = slice(1, -1)
    cq, cfl = 0.0, 0.0
    for w, x in zip(waves, s):
        cfl = max(cfl, float((dtdx * np.abs(x[..., i])).max()))
        dot = (w[..., :-1] * w[..., 1:]).sum(axis=0)
        norm = (w[..., i] ** 2).sum(axis=0)
        up = np.where(x[..., i] > 0, dot[..., :-1], dot[..., 1:])
        t = up / np.where(norm == 0, 1.0, norm)
        phi = np.maximum(0.0, np.minimum(np.minimum((1 + t) / 2, 2.0), 2 * t))
        phi = np.where(norm == 0, 1.0, phi)
        ax = np.abs(x[..., i])
        cq = cq + 0.5 * ax * (1 - ax * dtdx) * phi * w[..., i]
    if r is not None:
        r = dict(r, u={m: v[..., i] for m, v in r["u"].items()}, H=r["H"][..., i],
                 u2=r["u2"][..., i], a=r["a"][..., i])
    return am[..., i], ap[..., i], cq, r, cfl


def _step2(sol, q, dx, dy, dt):
    """One step of 2-D grids q (nvar, ..., my+4, mx+4): (new interior, x-fluxes
    (fm, fp) at mx+1 faces, y-fluxes (gm, gp) at my+1 faces, Courant)."""
    faces, cross, top = [], [], 0.0
    for axis in (0, 1):
        p = q if axis == 0 else np.swapaxes(q, -1, -2)
        dtd = dt / (dx if axis == 0 else dy)
        am, ap, cq, r, cfl = _normal_sweep(sol, p[..., 1:-1, :], axis + 1, dtd)
        top = max(top, cfl)
        amt, apt = am + 2 * cq, ap - 2 * cq
        # transverse: the left-going part enters the cell left of the interface
        lm, lp = sol.split(r, amt, 2 - axis)
        rm, rp = sol.split(r, apt, 2 - axis)
        low = -0.5 * dtd * (rm[..., :-1] + lm[..., 1:])   # at the mx interior cells
        upp = -0.5 * dtd * (rp[..., :-1] + lp[..., 1:])
        faces.append((am + cq, -ap + cq))
        # face between rows j and j+1 of the m + 2 rows: upper of j, lower of j+1
        cross.append(upp[..., :-1, :] + low[..., 1:, :])
    fm, fp = (f[..., 1:-1, :] + np.swapaxes(cross[1], -1, -2) for f in faces[0])
    gm, gp = (np.swapaxes(f[..., 1:-1, :], -1, -2) + cross[0] for f in faces[1])
    new = q[..., 2:-2, 2:-2] - dt / dx * (fm[..., 1:] - fp[..., :-1]) \
        - dt / dy * (gm[..., 1:, :] - gp[..., :-1, :])
    return new, (fm, fp), (gm, gp), top


def _step3(sol, q, h, dt):
    """One step of a 3-D grid q (5, mz+4, my+4, mx+4): (new interior, the six
    face arrays padded like q, Courant), with both transverse corrections and
    the double-transverse terms."""
    t, top = dt / h, 0.0
    low = [np.zeros_like(q) for _ in range(3)]   # transverse terms at each cell's low face
    normal = [None] * 3
    for ax in range(3):
        # arrays permuted to (component, w, v, u): u = ax, then cyclic
        perm = (0, 3 - (ax + 2) % 3, 3 - (ax + 1) % 3, 3 - ax)
        p = np.transpose(q, perm)[:, 1:-1, 1:-1, :]
        mu, mv, mw = ax + 1, (ax + 1) % 3 + 1, (ax + 2) % 3 + 1
        am, ap, cq, r, cfl = _normal_sweep(sol, p, mu, t)
        top = max(top, cfl)
        normal[ax] = (am + cq, -ap + cq)
        sp = {(m, k): sol.split(r, d, m) for m in (mv, mw)
              for k, d in (("am", am), ("ap", ap), ("cq", cq))}
        for m, o, av in ((mv, mw, (ax + 1) % 3), (mw, mv, (ax + 2) % 3)):
            acc = np.transpose(low[av], perm)
            # faces normal to m, shifted along o by the double-transverse terms
            for side in (0, 1):          # 0: part entering the left cell, 1: the right cell
                sign, part = (1.0, "am") if side == 0 else (-1.0, "ap")
                om, op = (sp[o, part][k] + sign * 3.0 * sp[o, "cq"][k] for k in (0, 1))
                dm, dp = sol.split(r, om, m), sol.split(r, op, m)
                for face in (0, 1):      # lower, upper face of the cell along m
                    base = -0.5 * t * sp[m, part][face] - sign * t * sp[m, "cq"][face]
                    base = base + t * t / 6.0 * (dp[face] - dm[face])
                    # interfaces 1..n+1 -> interior cells: left cells i - 1, right cells i
                    cells = slice(1, None) if side == 0 else slice(0, -1)
                    for shift, val in ((0, base), (1, -t * t / 6.0 * dp[face]),
                                       (-1, t * t / 6.0 * dm[face])):
                        _add(acc, val[..., cells], m == mv, face, shift)
    out = q[:, 2:-2, 2:-2, 2:-2].copy()
    flux = []
    for ax in range(3):
        perm = (0, 3 - (ax + 2) % 3, 3 - (ax + 1) % 3, 3 - ax)
        add = np.transpose(low[ax], perm)[:, 2:-2, 2:-2, 2:-1]
        m_, p_ = (f[:, 1:-1, 1:-1, :] + add for f in normal[ax])
        np.transpose(out, perm)[...] -= t * (m_[..., 1:] - p_[..., :-1])
        for f in (m_, p_):
            full = np.zeros_like(q)
            np.transpose(full, perm)[:, 2:-2, 2:-2, 2:-1] = f
            flux.append(full)
    return out, flux, top


def _add(acc, val, along_v, face, shift):
    """Add val (w and v from 0 to n + 1, u interior) to the faces of
    acc (padded): `face` along the face's own direction, `shift` across."""
    nw, nv = acc.shape[1] - 4, acc.shape[2] - 4
    w0, v0 = (shift, face) if along_v else (face, shift)
    # clip what falls outside the padded array
    w = slice(max(0, -1 - w0), min(nw + 2, nw + 3 - w0))
    v = slice(max(0, -1 - v0), min(nv + 2, nv + 3 - v0))
    acc[:, 1 + w0 + w.start:1 + w0 + w.stop, 1 + v0 + v.start:1 + v0 + v.stop, 2:-2] += val[:, w, v, :]


class _Dense:
    """A hierarchy in 2 or 3 dimensions: each level a dense (nvar, [nz,] ny, nx)
    array over its index space with the mask of the cells its grids cover."""

    def __init__(self, H, sol, flats, possk):
        self.sol, self.H, self.nlev = sol, H, H.nlev
        self.dim = len(H.levels[0]["boxes"][0]) // 2
        self.dt, self.time = possk, [0.0] * H.nlev
        self.periodic = H.mthbc[0] == 2
        self.q, self.old, self.mask, self.pads, self.seen = [], [], [], [], [0.0] * H.nlev
        self.ghost = (slice(None),) + (slice(2, -2),) * self.dim
        for L, flat in zip(H.levels, flats):
            size = [L[k] for k in ("kregsz", "jregsz", "iregsz")[3 - self.dim:]]
            q, mask, pads = np.zeros([H.nvar] + size), np.zeros(size, bool), []
            for b, g in zip(L["boxes"], _views(flat, L["shapes"])):
                g = np.moveaxis(g, -1, 0).copy()
                q[self._at(b)] = g[self.ghost]
                mask[self._at(b)[1:]] = True
                pads.append(g)
            self.q.append(q)
            self.old.append(q.copy())
            self.mask.append(mask)
            self.pads.append(pads)
        # fluxes through the faces of each level: its last step's, and the sum of
        # dt * flux of the finer level's steps since
        self.face = [None] * H.nlev
        self.fine = [None] * H.nlev

    def _at(self, b, grow=0, face=None):
        """The box b (x first) as an index; its faces normal to array axis `face`."""
        return (slice(None),) + tuple(
            slice(int(b[2 * d]), int(b[2 * d + 1]) + 1 + 2 * grow + (self.dim - d == face))
            for d in range(self.dim - 1, -1, -1))

    def _outside(self, a, n):
        return np.pad(a, [(0, 0)] + [(n, n)] * self.dim, mode="wrap" if self.periodic else "edge")

    def filled(self, l, t):
        """The level's values at time t, cells outside its grids interpolated
        from the next coarser level with limited linear slopes."""
        a = 1.0 - (self.time[l] - t) / self.dt[l]
        if abs(a - 1.0) < 1e-4:
            own = self.q[l]
        elif abs(a) < 1e-4:
            own = self.old[l]
        else:
            own = a * self.q[l] + (1.0 - a) * self.old[l]
        if l == 0 or self.mask[l].all():
            return own
        r = self.H.levels[l - 1]["ratx"]
        c = self._outside(self.filled(l - 1, t), 1)
        core = [slice(None)] + [slice(1, -1)] * self.dim
        mid = c[tuple(core)]

        def finer(x):
            for ax in range(1, self.dim + 1):
                x = np.repeat(x, r, ax)
            return x
        interp = finer(mid)
        for ax in range(self.dim, 0, -1):
            lo, hi = list(core), list(core)
            lo[ax], hi[ax] = slice(None, -2), slice(2, None)
            m, p = c[tuple(lo)], c[tuple(hi)]
            dm, dp, dc = mid - m, p - mid, p - m
            d = np.minimum(2.0 * np.minimum(np.abs(dm), np.abs(dp)), 0.5 * np.abs(dc))
            eta = np.tile((np.arange(r) + 0.5) / r - 0.5, mid.shape[ax])
            eta = eta.reshape([-1 if k == ax else 1 for k in range(self.dim + 1)])
            interp = interp + eta * finer(np.where(dm * dp >= 0, d * np.copysign(1.0, dc), 0.0))
        return np.where(self.mask[l], own, interp)

    def _grids(self, L, f, dt):
        """Every grid's (index, padded array, new interior, {array axis: its
        conservative face fluxes}, Courant): the step of the level from f."""
        sol = self.sol
        if self.dim == 3:
            for k, b in enumerate(L["boxes"]):
                g = f[self._at(b, 2)]
                out, fl, cfl = _step3(sol, g, L["hx"], dt)
                face = {}
                for ax in (1, 2, 3):
                    left = [slice(None)] + [slice(2, -2)] * 3
                    at = list(left)
                    left[ax], at[ax] = slice(1, -2), slice(2, -1)
                    face[ax] = fl[2 * (3 - ax)][tuple(at)] + sol.flux(g[tuple(left)], 4 - ax)
                yield k, g, out, face, cfl
            return
        shapes = {}
        for k, b in enumerate(L["boxes"]):
            shapes.setdefault((b[3] - b[2], b[1] - b[0]), []).append(k)
        for ks in shapes.values():
            g = np.stack([f[self._at(L["boxes"][k], 2)] for k in ks], 1)
            out, (fm, _), (gm, _), cfl = _step2(sol, g, L["hx"], L["hy"], dt)
            fm = fm + sol.flux(g[..., 2:-2, 1:-2], 1)
            gm = gm + sol.flux(g[..., 1:-2, 2:-2], 2)
            for i, k in enumerate(ks):
                yield k, g[:, i], out[:, i], {2: fm[:, i], 1: gm[:, i]}, cfl

    def advance(self, l):
        L, dt = self.H.levels[l], self.dt[l]
        f = self._outside(self.filled(l, self.time[l]), 2)
        new = self.q[l].copy()
        face = {ax: np.zeros([n + (k == ax) for k, n in enumerate(new.shape)])
                for ax in range(1, self.dim + 1)}
        for k, g, out, through, cfl in self._grids(L, f, dt):
            self.seen[l] = max(self.seen[l], cfl)
            self.pads[l][k] = g.copy()
            new[self._at(L["boxes"][k])] = out
            for ax, v in through.items():
                face[ax][self._at(L["boxes"][k], 0, ax)] = v
        self.old[l], self.q[l], self.face[l] = self.q[l], new, face
        self.time[l] += dt
        if l + 1 < self.nlev:
            self.fine[l] = {ax: 0.0 for ax in face}
        if l > 0:
            for ax in face:
                self.fine[l - 1][ax] = self.fine[l - 1][ax] + dt * face[ax]

    def _mean(self, x, r, skip=None):
        """Means over r cells along every axis but `skip` (whose every r-th face
        is kept)."""
        for ax in range(1, self.dim + 1):
            if ax == skip:
                x = x[tuple(slice(None, None, r) if k == ax else slice(None) for k in range(x.ndim))]
            else:
                x = x.reshape(x.shape[:ax] + (-1, r) + x.shape[ax + 1:]).mean(axis=ax + 1)
        return x

    def update(self, l):
        """Reflux into the cells of level l next to level l + 1, then average.
        Finer grids lie inside the domain or end at an open side, so no face of
        theirs is shared across a periodic one."""
        L, r, q = self.H.levels[l], self.H.levels[l]["ratx"], self.q[l]
        cover = self.mask[l + 1][(slice(None, None, r),) * self.dim]
        near, free = np.pad(cover, 1), self.mask[l] & ~cover
        for ax in range(1, self.dim + 1):
            d = (self.dt[l] * self.face[l][ax] - self._mean(self.fine[l][ax], r, ax)) \
                / L[("hx", "hy", "hz")[self.dim - ax]]
            for off, sign in ((1, 1.0), (-1, -1.0)):
                # the cell below a covered one along the axis: its upper face, and so on
                nb = near[tuple(slice(1 + off, near.shape[k - 1] - 1 + off) if k == ax else
                                slice(1, -1) for k in range(1, self.dim + 1))]
                side = d[tuple((slice(1, None) if off == 1 else slice(None, -1)) if k == ax else
                               slice(None) for k in range(self.dim + 1))]
                q += sign * np.where(free & nb, side, 0.0)
        q[:, cover] = self._mean(self.q[l + 1], r)[:, cover]

    def tick(self, l=0):
        self.advance(l)
        if l + 1 < self.nlev:
            for _ in range(self.H.levels[l]["ratx"]):
                self.tick(l + 1)
            self.update(l)

    def packed(self, l, old=False):
        out = []
        for b, g in zip(self.H.levels[l]["boxes"], self.pads[l]):
            g = g.copy()
            if not old:
                g[self.ghost] = self.q[l][self._at(b)]
            out.append(np.moveaxis(g, 0, -1).ravel())
        return np.concatenate(out)


#: seconds that a numpy cell update takes (2-D Euler, 3-D Euler), to leave out
#: the cases that would run past about 20 s
_COST = {2: 5e-6, 3: 4e-5}


def exact(case, seed):
    kind = case["kind"]
    three = kind in ("grid3", "batch3", "amr3")
    cells, _, _ = _updates(case)
    if cells * _COST[3 if three else 2] > 18.0:
        return None
    sol = _solver(case)
    if kind == "patch2":
        q = _patch2(case, seed)
        new, _, _, cfl = _step2(sol, np.moveaxis(q, -1, 0), 1 / 256, 1 / 256, _patch2_dt(case))
        out = q.copy()
        out[2:-2, 2:-2] = np.moveaxis(new, 0, -1)
        return [out, cfl, _patch2_dt(case) * 0.9 / cfl]
    if kind == "grid3":
        q, h, dt = _grid3(case, seed), 1.0 / 64, 0.2 / 64
        new, flux, cfl = _step3(sol, np.moveaxis(q, -1, 0), h, dt)
        out = q.copy()
        out[2:-2, 2:-2, 2:-2] = np.moveaxis(new, 0, -1)
        flux = [np.ascontiguousarray(np.moveaxis(f, 0, -1)) for f in flux]
        return [out, flux if case["precision"] == "f64" else [], cfl, dt * 0.9 / cfl]
    key = _key(case)
    if kind == "batch3":
        sizes, h, dt, flat, shapes = _layout(key)
        q = _perturbed(flat, 5, seed)
        cfl = np.zeros(len(shapes))
        for p, g in enumerate(_views(q, shapes)):
            for _ in range(case["steps"]):
                new, _, cfl[p] = _step3(sol, np.moveaxis(g, -1, 0), h, dt)
                g[2:-2, 2:-2, 2:-2] = np.moveaxis(new, 0, -1)
        return [q, cfl]
    H = _layout(key)
    flats = [_perturbed(L["qnew"], H.nvar, seed + l) for l, L in enumerate(H.levels)]
    D = _Dense(H, sol, flats, _possk(case, H))
    for _ in range(case["steps"]):
        D.tick()
    out = []
    for l in range(H.nlev):
        out.append(D.packed(l))
        if case.get("pull") and l + 1 < H.nlev:
            out.append(D.packed(l, old=True))
    out.append(np.array(D.seen))
    if case.get("flag"):
        out += [None, None] * (H.nlev - 1)   # whole numbers, compared as they are
    return out
