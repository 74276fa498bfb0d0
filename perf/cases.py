"""Cases by which this framework's speed is measured: the reaction step, the
warm start, the operator-split and global-implicit steps and constraint
speciation, each through the package's public entry points.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a program holds before the call, on the GPU
  run(state)           one pass, and its outputs
  work(case)           bytes and flops that one pass cannot do without
  exact(case, seed)    the outputs in 64 bits from plain torch

The cells of a case are drawn from the seed by the plain torch chemistry
below (class Chemistry): constraint speciation of log-uniform totals and a
uniform pH, as the benchmark's and the tests' cells are drawn, then the
totals of every cell moved by up to 2 %, as one transport step moves them.
Cells that this plain Newton does not bring to convergence in 100 iterations,
or whose iterates still wander after a dozen, are replaced, so a case holds no
cell whose outcome is left to rounding.
The iteration counts, which describe the path and not the result, are not
among the outputs.
"""
import math
import os

import numpy as np
import torch

from pflotran_amd import abi, column, runtime, surrogate, synth, workload
from pflotran_amd.database import MineralKinetics, build_tables, read_database

DEV = "cuda"
F64 = torch.float64
DATABASE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tests", "golden", "db",
                        "hanford_subset.dat")
LN10 = 2.30258509299          # the reference's truncated constant (pflotran_constants.F90:48)
POROSITY, VOLUME, DT = 0.25, 1.0, synth.STEP_DT
QK_CAP = 6.90776              # ln(Q/K) above which Q/K is held at 1e3 (reaction_mineral.F90:699)
CHUNK = 1 << 18               # cells per piece of the plain chemistry


# --------------------------------------------------------------------------
# cases
def listed():
    n15 = dict(N=15, M=50, K=3, ionx=True, net=synth.SEED)
    return [
        # the 100-cell column of the operator-split examples: one reaction call of a host program, where the
        # launches and the wait count
        dict(name="react_column_100", kind="react", N=5, cells=100, net=0, capped=False),
        # the same column's whole step (transport, reaction, mineral update) as the captured graph that a time
        # loop replays
        dict(name="os_step_column_100", kind="os_step", cells=100),
        # one rank's slab of a mid-size run, an odd number of cells
        dict(n15, name="react_50021", kind="react", cells=50021, capped=False),
        # the million-cell batched reaction step, the headline configuration
        dict(n15, name="react_1m", kind="react", cells=1000000, capped=False),
        # the same step from the learned warm start: network inference, then the Newton with its fallback
        dict(n15, name="warm_1m", kind="warm", cells=1000000, width=256),
        # eight minibatches of the warm start's training
        dict(name="train_4096", kind="train", batch=4096, inputs=40, width=256, outputs=15, steps=8),
        # four chemistry zones of unequal networks in one launch, replayed as a graph
        dict(name="zones_800k", kind="zones", n8=400000, n12=200000, n20=120000, n30=80000),
        # initial condition of a field: every cell's constraint speciated
        dict(name="equilibrate_200k", kind="equilibrate", cells=200000),
        # residual and block Jacobian of the global-implicit step, 128^3 grid
        dict(n15, name="gi_assembly_128", kind="gi_assembly", nx=128, ny=128, nz=128),
        # the same on a small ragged grid of another network
        dict(name="gi_assembly_ragged", kind="gi_assembly", N=8, M=24, K=3, ionx=False, net=7, nx=29, ny=17, nz=23),
        # one global-implicit time step, predictor and Newton with its linear solves
        dict(n15, name="gi_step_63k", kind="gi_step", nx=44, ny=40, nz=36),
        # the implicit transport half of an operator-split step, 15 components
        dict(name="os_transport_128", kind="os_transport", nx=128, ny=128, nz=128, comps=15),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["react", "os_step", "warm", "train", "zones", "equilibrate", "gi_assembly", "gi_step",
                        "os_transport"], [5, 1, 2, 1, 2, 1, 2, 1, 2])[0]
    net = rng.randrange(1, 1000)
    if kind == "react":
        N = rng.choice([5, 6, 7, 8, 9, 11, 12, 13, 14, 15, 16, 17, 20, 24, 27, 30])
        hi = 400000 if N <= 16 else 60000
        return dict(kind=kind, N=N, M=rng.randrange(N, 3 * N + 1), K=rng.randrange(1, 5), ionx=rng.random() < 0.5,
                    net=net, cells=_log_int(rng, 60, hi), capped=rng.random() < 0.3)
    if kind == "os_step":
        return dict(kind=kind, cells=_log_int(rng, 20, 3000))
    if kind == "warm":
        N = rng.randrange(8, 16)
        return dict(kind=kind, N=N, M=rng.randrange(2 * N, 3 * N + 1), K=rng.randrange(1, 4), ionx=rng.random() < 0.5,
                    net=net, cells=_log_int(rng, 1000, 400000), width=rng.choice([64, 128, 256]))
    if kind == "train":
        return dict(kind=kind, batch=_log_int(rng, 200, 8192), inputs=rng.choice([24, 33, 40, 64]),
                    width=rng.choice([64, 128, 256]), outputs=rng.randrange(8, 17), steps=rng.randrange(2, 9))
    if kind == "zones":
        return dict(kind=kind, n8=_log_int(rng, 500, 200000), n12=_log_int(rng, 500, 100000),
                    n20=_log_int(rng, 500, 60000), n30=_log_int(rng, 500, 40000))
    if kind == "equilibrate":
        return dict(kind=kind, cells=_log_int(rng, 500, 200000))
    if kind == "gi_assembly":
        N = rng.choice([5, 8, 9, 12, 15, 16, 18, 21])
        side = 56 if N <= 16 else 36
        return dict(kind=kind, N=N, M=rng.randrange(N, 3 * N + 1), K=rng.randrange(1, 4), ionx=rng.random() < 0.5,
                    net=net, nx=_log_int(rng, 3, side), ny=_log_int(rng, 3, side), nz=_log_int(rng, 3, side))
    if kind == "gi_step":
        return dict(kind=kind, N=15, M=50, K=3, ionx=True, net=synth.SEED, nx=_log_int(rng, 6, 36),
                    ny=_log_int(rng, 6, 36), nz=_log_int(rng, 4, 30))
    return dict(kind="os_transport", nx=_log_int(rng, 5, 110), ny=_log_int(rng, 5, 110), nz=_log_int(rng, 3, 110),
                comps=rng.randrange(2, 21))


# --------------------------------------------------------------------------
# networks
def carbonate():
    """The calcite column's chemistry (hanford database, 25 C)."""
    return build_tables(read_database(DATABASE), ["H+", "HCO3-", "Ca++", "Mg++", "Cl-"],
                        ["OH-", "CO2(aq)", "CO3--", "CaHCO3+", "CaCO3(aq)", "MgHCO3+", "MgCO3(aq)", "CaCl+"],
                        {"Calcite": MineralKinetics(1e-9)}, act_freq=abi.PFX_ACT_TIMESTEP)


def network(case):
    if case.get("net", 0) == 0:
        return carbonate()
    return synth.random_network(case["N"], case["M"], case["K"], ionx=case["ionx"], seed=case["net"])


# --------------------------------------------------------------------------
# plain chemistry in torch, species first: vectors are [species][cells]
def solve_inplace(J, b):
    """J x = b per cell by elimination without pivoting (the Jacobians in ln m
    are diagonally strong); J [N][N][n] and b [N][n] are overwritten."""
    N = b.shape[0]
    for j in range(N - 1):
        f = J[j + 1:, j] / J[j, j]
        J[j + 1:, j + 1:].addcmul_(f[:, None], J[j, None, j + 1:], value=-1.0)
        b[j + 1:].addcmul_(f, b[j][None], value=-1.0)
    for j in reversed(range(N)):
        if j + 1 < N:
            b[j] -= (J[j, j + 1:] * b[j + 1:]).sum(0)
        b[j] /= J[j, j]
    return b


class Chemistry:
    """A network's equations for cells at `temp` (C, or None for 25 C)."""

    def __init__(self, t, temp, n):
        T = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device=DEV)  # noqa: E731
        self.t, self.N, self.M, self.K = t, t.N, t.M, t.K
        dense = lambda ids, st: np.stack([  # noqa: E731
            np.bincount(i[1:1 + i[0]], weights=s[:i[0]], minlength=t.N) for i, s in zip(ids, st)])
        self.nu, self.mnu = T(dense(t.cplx_specid, t.cplx_stoich)), T(dense(t.mnrl_specid, t.mnrl_stoich))
        self.outer = (self.nu[:, :, None] * self.nu[:, None, :]).reshape(t.M, -1).t().contiguous()
        self.mouter = (self.mnu[:, :, None] * self.mnu[:, None, :]).reshape(t.K, -1).t().contiguous()
        self.Z, self.a0, self.cZ, self.ca0 = T(t.Z), T(t.a0), T(t.cplx_Z), T(t.cplx_a0)
        self.k = T(t.mnrl_rate_constant)
        self.lnK = self._lnK(T(t.cplx_logK), t.cplx_logKcoef, temp, n)
        self.mlnK = self._lnK(T(t.mnrl_logK), t.mnrl_logKcoef, temp, n)
        self.dl = synth.DEN_25C * 1.0e-3
        self.cats = [int(j) for j in t.ionx_cationid[0, 1:1 + t.ionx_cationid[0, 0]]] if t.R else []
        if self.cats:
            self.xk, self.cec = T(t.ionx_k[0, :len(self.cats)]), float(t.ionx_CEC[0])
            self.uneven = any(t.Z[j] != t.Z[self.cats[0]] for j in self.cats)

    def _lnK(self, ref, coef, temp, n):
        if temp is None or coef is None:
            return (-ref * LN10)[:, None].expand(-1, n)
        c, tk = torch.as_tensor(np.asarray(coef), device=DEV), temp + 273.15
        return -(torch.outer(c[:, 0], tk.log()) + c[:, 1:2] + torch.outer(c[:, 2], tk) + torch.outer(c[:, 3], 1 / tk)
                 + torch.outer(c[:, 4], 1 / (tk * tk))) * LN10

    def part(self, idx):
        """The equations of some of the cells."""
        p = object.__new__(Chemistry)
        p.__dict__.update(self.__dict__)
        p.lnK, p.mlnK = self.lnK[:, idx], self.mlnK[:, idx]
        return p

    def activity(self, m, C):
        """ln activity coefficients of primaries and complexes (Debye-Hueckel at the ionic strength of m, C)."""
        A, B, Bd = self.t.debye
        I = 0.5 * ((self.Z ** 2) @ m + (self.cZ ** 2) @ C)
        s = I.sqrt()

        def lng(z, a0):
            v = (-(z * z)[:, None] * s * A / (1.0 + (a0 * B)[:, None] * s) + Bd * I) * LN10
            return torch.where((z.abs() > 1e-10)[:, None], v, torch.zeros_like(v))
        return lng(self.Z, self.a0), lng(self.cZ, self.ca0)

    def complexes(self, x, lng, lngc):
        return (self.lnK + self.nu @ (x + lng) - lngc).exp()

    def totals(self, x, C):
        return (x.exp() + self.nu.t() @ C) * self.dl

    def total_jacobian(self, x, C):
        """dT / d ln m, [N][N][n]"""
        J = (self.outer @ C).reshape(self.N, self.N, -1)
        J.diagonal().add_(x.exp().t())
        return J.mul_(self.dl)

    def exchange(self, la):
        """Sorbed totals [N][n] (mol/m^3 bulk), exchange fractions of the cations, the reference cation's sorbed
        concentration: sum_j k_j a_j D^(z_j / z_ref) = 1 solved in ln D."""
        S = torch.zeros_like(la)
        if not self.cats:
            return S, None, None
        z = self.Z[self.cats]
        ratio, lk = (z / z[0])[:, None], la[self.cats] + self.xk.log()[:, None]
        y = -lk.amax(0)
        for _ in range(40):
            X = (lk + ratio * y).exp()
            tot = X.sum(0)
            d = tot.log() * tot / (X * ratio).sum(0)
            y = y - d
            if d.numel() == 0 or float(d.abs().max()) < 1e-15 * max(1.0, float(y.abs().max())):
                break
        X = (lk + ratio * y).exp()
        X = X / X.sum(0)
        S[self.cats] = X * self.cec / z[:, None]
        return S, X, X[0] * self.cec / z[0]

    def speciate(self, total, ph, lng, lngc, x, its=80):
        """ln m of H+ at its pH and every other total (mol/L): Newton on a convex problem.  Returns the cells'
        convergence."""
        x = x.clone()
        x[0] = -ph * LN10 - lng[0]
        conv = torch.zeros(x.shape[1], dtype=torch.bool, device=DEV)
        live = torch.arange(x.shape[1], device=DEV)
        p, xs, lg, lc, tt = self, x.clone(), lng, lngc, total
        for _ in range(its):
            C = p.complexes(xs, lg, lc)
            r = (p.totals(xs, C) - tt)[1:]
            d = solve_inplace(p.total_jacobian(xs, C)[1:, 1:], r).clamp_(-4.0, 4.0)
            xs[1:] -= d
            step = d.abs().amax(0)
            done = step < 1e-12
            x[:, live] = xs
            conv[live[done]] = True
            if bool(done.any()) and int((~done).sum()) < 0.7 * done.numel():
                keep = torch.nonzero(~done).flatten()
                if keep.numel() == 0:
                    break
                live, p, xs, tt = live[keep], p.part(keep), xs[:, keep], tt[:, keep]
                lg, lc = lg[:, keep], lc[:, keep]
        return x, conv & torch.isfinite(x).all(0)

    def reaction_system(self, x, lng, lngc, fixed, vf, dt, capped):
        """Residual (mol/s) and d/d ln m of one cell's reaction step; capped: no mineral derivative above the Q/K
        cap."""
        psv = POROSITY * 1000.0 * VOLUME
        la = x + lng
        C = self.complexes(x, lng, lngc)
        J = self.total_jacobian(x, C).mul_(psv / dt)
        R = psv * self.totals(x, C) / dt - fixed / dt
        if self.cats:
            S, X, _ = self.exchange(la)
            R += S * (VOLUME / dt)
            w = (VOLUME / dt) * self.cec
            z = self.Z[self.cats]
            zx = (z[:, None] * X).sum(0)
            for a, ja in enumerate(self.cats):
                for b, jb in enumerate(self.cats):
                    J[ja, jb] -= w * X[a] * X[b] / zx
                J[ja, ja] += w * X[a] / z[a]
        I, QK, over = self.rates(la, vf)
        R += self.mnu.t() @ (I * VOLUME)
        g = self.k[:, None] * VOLUME * QK * self.dl * (vf > 0)
        if capped:
            g = torch.where(over, torch.zeros_like(g), g)
        J += (self.mouter @ g).reshape(J.shape)
        return R, J

    def rates(self, la, vf):
        """Mineral rates (mol/s/m^3, unit area), the held Q/K, and where it is held."""
        lnQK = self.mlnK + self.mnu @ la
        over = lnQK > QK_CAP
        QK = torch.where(over, torch.full_like(lnQK, 1.0e3), lnQK.exp())
        aff = 1.0 - QK
        return -self.k[:, None] * torch.where((vf > 0) | (aff < 0), aff, torch.zeros_like(aff)), QK, over

    def react(self, x, lng, lngc, fixed, vf, dt, capped, its=100, tol=1e-11):
        """Newton of the reaction step at fixed activity coefficients from ln m = x.  Returns ln m and which cells
        converged without still taking long steps after a dozen (whose path, and root, hang on the rounding)."""
        x = x.clone()
        conv = torch.zeros(x.shape[1], dtype=torch.bool, device=DEV)
        steady = torch.ones_like(conv)
        live = torch.arange(x.shape[1], device=DEV)
        p, s = self, [x.clone(), lng, lngc, fixed, vf]
        for k in range(its):
            R, J = p.reaction_system(*s, dt, capped)
            d = solve_inplace(J, R).clamp_(-5.0, 5.0)
            s[0] = s[0] - d
            step = d.abs().amax(0)
            done = step < tol
            if k >= 12:
                steady[live[step > 0.3]] = False
            x[:, live] = s[0]
            conv[live[done]] = True
            if bool(done.any()) and int((~done).sum()) < 0.7 * done.numel():
                keep = torch.nonzero(~done).flatten()
                if keep.numel() == 0:
                    break
                live, p, s = live[keep], p.part(keep), [v[:, keep] for v in s]
        return x, conv & steady & torch.isfinite(x).all(0)

    def react_root(self, x, lng, lngc, fixed, vf, dt):
        """The step's solution: the consistent derivative first, the reference's where that does not settle."""
        a, ca = self.react(x, lng, lngc, fixed, vf, dt, True, its=50, tol=1e-13)
        rest = torch.nonzero(~ca).flatten()
        if rest.numel():
            b, cb = self.part(rest).react(x[:, rest], lng[:, rest], lngc[:, rest], fixed[:, rest], vf[:, rest], dt,
                                          False, its=300, tol=1e-13)
            a[:, rest] = b
        return a


# --------------------------------------------------------------------------
# cells
def rows(v):
    """[species][cells] -> the cell-major array of the interface"""
    return v.t().contiguous()


def _generator(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) % (1 << 62))
    return g


def _piece(t, n, g, with_temp, total_range, ph_range, step):
    """n drawn cells, and which of them are usable."""
    u = lambda lo, hi, *s: torch.rand(*s, generator=g, device=DEV, dtype=F64) * (hi - lo) + lo  # noqa: E731
    lo, hi = math.log(total_range[0]), math.log(total_range[1])
    total = u(lo, hi, t.N, n).exp()
    ph = u(*ph_range, n)
    temp = u(10.0, 60.0, n) if with_temp else None
    vf = u(0.01, 0.1, max(t.K, 1), n)
    moved = 1.0 + 0.02 * u(-1.0, 1.0, t.N, n)
    ch = Chemistry(t, temp, n)
    one, onec = torch.zeros(t.N, n, device=DEV, dtype=F64), torch.zeros(t.M, n, device=DEV, dtype=F64)
    x, ok = ch.speciate(total, ph, one, onec, total.log().clamp_(max=math.log(1e-2)))
    x = torch.where(ok, x, torch.full_like(x, math.log(1e-6)))
    lng, lngc = one, onec
    for _ in range(2):      # the same totals and pH with the activity coefficients switched on
        lng, lngc = ch.activity(x.exp(), ch.complexes(x, lng, lngc))
        y, again = ch.speciate(total, ph, lng, lngc, x)
        ok = ok & again
        x = torch.where(ok, y, x)
    for _ in range(2):      # the initial refresh: two activity passes (condition_control.F90:929-935)
        lng, lngc = ch.activity(x.exp(), ch.complexes(x, lng, lngc))
    C = ch.complexes(x, lng, lngc)
    T = ch.totals(x, C)
    S, _, ref = ch.exchange(x + lng)
    s = dict(x=x, lng=lng, lngc=lngc, T=T, S=S, ref=ref if ref is not None else T.new_full((n,), 1e-9), vf=vf,
             moved=T * moved)
    if temp is not None:
        s["temp"] = temp
    if step:
        a, ac = ch.activity(x.exp(), C)
        _, c2 = ch.react(x, a, ac, POROSITY * 1000.0 * VOLUME * s["moved"] + S * VOLUME, vf[:t.K], DT, False)
        ok = ok & c2
    return s, ok


def draw_cells(t, n, seed, salt=0, with_temp=True, total_range=(1e-6, 1e-2), ph_range=(5.0, 9.0), step=True):
    """n cells at the start of a reaction step, as a dict of [species][n] (x = ln m, lng, lngc, T, S, ref, vf,
    moved = the transported totals, temp)."""
    g = _generator(seed, salt)
    got, have = [], 0
    while have < n:
        k = min(CHUNK, max(256, int((n - have) * 1.08) + 64))
        s, ok = _piece(t, k, g, with_temp, total_range, ph_range, step)
        idx = torch.nonzero(ok).flatten()[:n - have]
        if 4 * idx.numel() < min(k, n - have):
            raise ValueError("too few usable cells in this network")
        got.append({key: v[..., idx] for key, v in s.items()})
        have += int(idx.numel())
    return {key: torch.cat([p[key] for p in got], dim=-1) for key in got[0]}


RESTORED = ("total", "total_sorb", "pri_molal", "pri_act_coef", "sec_act_coef", "ionx_ref_sorbed")


def device_cells(t, s, n, total):
    """The interface's arrays.  The fields that a reaction step overwrites lie in one buffer, so that a program
    hands over the next step's inputs with one copy."""
    mol = lambda v: rows(v.exp())  # noqa: E731
    src = dict(total=rows(total), total_sorb=rows(s["S"]), pri_molal=mol(s["x"]), pri_act_coef=mol(s["lng"]),
               sec_act_coef=mol(s["lngc"]), ionx_ref_sorbed=s["ref"].reshape(n, 1).clone())
    if not t.has_sorption:
        src["total_sorb"] = None
    flat = torch.cat([src[k].reshape(-1) for k in RESTORED if src[k] is not None])
    work, at, arr = flat.clone(), 0, {}
    for k in RESTORED:
        v = src[k]
        if v is not None:
            arr[k] = work[at:at + v.numel()].view(v.shape)
            at += v.numel()
    z = lambda *sh: torch.zeros(*sh, device=DEV, dtype=F64)  # noqa: E731
    K = max(t.K, 1)
    arr.update(sec_molal=z(n, max(t.M, 1)), mnrl_volfrac=rows(s["vf"]), mnrl_area=z(n, K) + 1.0, mnrl_rate=z(n, K),
               temperature=s.get("temp"), porosity=None, saturation=None, volume=None, den_kg=None, guess=z(n, t.N),
               num_iterations=torch.zeros(n, dtype=torch.int32, device=DEV),
               status=torch.zeros(n, dtype=torch.int32, device=DEV), rel_res=z(n))
    if "total_sorb" not in arr:
        arr["total_sorb"] = None
    return runtime.DeviceCells(arr, n), work, flat


def cell_outputs(dc):
    keys = ("total", "total_sorb", "pri_molal", "pri_act_coef", "sec_act_coef", "sec_molal", "ionx_ref_sorbed",
            "mnrl_rate", "status")
    return {k: dc.t[k] for k in keys if dc.t.get(k) is not None}


def exact_reaction(t, s, total, vf, dt=DT):
    """The reaction step's outputs from plain torch."""
    n = total.shape[1]
    parts = []
    for i in range(0, n, CHUNK):
        c = slice(i, min(n, i + CHUNK))
        ch = Chemistry(t, s["temp"][c] if "temp" in s else None, total[:, c].shape[1])
        x, lng, lngc, S0 = (s[k][:, c].contiguous() for k in ("x", "lng", "lngc", "S"))
        lng, lngc = ch.activity(x.exp(), ch.complexes(x, lng, lngc))
        fixed = POROSITY * 1000.0 * VOLUME * total[:, c] + S0 * VOLUME
        x = ch.react_root(x, lng, lngc, fixed, vf[:t.K, c], dt)
        C = ch.complexes(x, lng, lngc)
        S, _, ref = ch.exchange(x + lng)
        if ref is None or not ch.uneven:      # the equal-valence form keeps the state it was given
            ref = s["ref"][c]
        parts.append(dict(total=rows(ch.totals(x, C)), total_sorb=rows(S), pri_molal=rows(x.exp()),
                          pri_act_coef=rows(lng.exp()), sec_act_coef=rows(lngc.exp()), sec_molal=rows(C),
                          ionx_ref_sorbed=ref.reshape(-1, 1), mnrl_rate=rows(ch.rates(x + lng, vf[:t.K, c])[0])))
    out = {k: torch.cat([p[k] for p in parts]) for k in parts[0]}
    if not t.has_sorption:
        out["total_sorb"] = None
    out["status"] = None
    return out


# --------------------------------------------------------------------------
# one reaction step, plain or from the warm start
def reaction_cells(case, seed):
    t = network(case)
    if case.get("net", 0) == 0:
        return t, draw_cells(t, case["cells"], seed, with_temp=False, total_range=(1e-5, 1e-2), ph_range=(6.0, 9.0))
    return t, draw_cells(t, case["cells"], seed)


def prepare_react(case, seed):
    t, s = reaction_cells(case, seed)
    dc, work, flat = device_cells(t, s, case["cells"], s["moved"])
    opts = synth.react_opts(guess_mode=abi.PFX_GUESS_PREVIOUS,
                            jacobian_flags=abi.PFX_JAC_CAPPED_QK if case.get("capped") else 0)
    return dict(kind="react", tab=runtime.Tables(t), dc=dc, work=work, flat=flat, opts=opts)


def run_react(s):
    s["work"].copy_(s["flat"])
    runtime.react_batch(s["tab"], s["dc"], s["opts"])
    return cell_outputs(s["dc"])


def exact_react(case, seed):
    t, s = reaction_cells(case, seed)
    return exact_reaction(t, s, s["moved"], s["vf"])


def warm_network(case, t, dc, seed):
    """A network of the warm start's shape whose prediction is off by about 0.01 in ln m, as a trained one's is."""
    ni = 2 * t.N + 1 + t.K
    ni += (-ni) % 8
    mlp = surrogate.MLP((ni, case["width"], case["width"], case["width"], t.N), batch_max=1024, seed=seed + 1)
    X = surrogate.features(runtime.Tables(t), mlp, runtime.DeviceCells(
        {k: (None if v is None else v[:20000]) for k, v in dc.t.items()}, min(dc.ncells, 20000)))
    sd = X.double().std(0)
    mlp.set_norm(X.double().mean(0).cpu().numpy(), torch.where(sd > 1e-6, 1.0 / sd, torch.ones_like(sd)).cpu().numpy(),
                 np.zeros(t.N), np.full(t.N, 50.0))
    return mlp


def prepare_warm(case, seed):
    t, s = reaction_cells(case, seed)
    dc, work, flat = device_cells(t, s, case["cells"], s["moved"])
    opts = synth.react_opts(guess_mode=abi.PFX_GUESS_ARRAY_FALLBACK, fallback_after=100, fallback_previous=1)
    return dict(kind="warm", tab=runtime.Tables(t), dc=dc, work=work, flat=flat, opts=opts,
                mlp=warm_network(case, t, dc, seed))


def run_warm(s):
    s["work"].copy_(s["flat"])
    surrogate.guess(s["tab"], s["mlp"], s["dc"])
    runtime.react_batch(s["tab"], s["dc"], s["opts"])
    return cell_outputs(s["dc"])


# --------------------------------------------------------------------------
# training of the warm start
def training_batches(case, seed):
    g = _generator(seed, 3)
    n = case["batch"] * case["steps"]
    X = torch.randn(n, case["inputs"], generator=g, device=DEV)
    X[:, -max(1, case["inputs"] // 8):] = 0.0                  # the features' empty slots
    A = torch.randn(case["inputs"], case["outputs"], generator=g, device=DEV) / math.sqrt(case["inputs"])
    T = torch.tanh(X @ A) + 0.05 * torch.randn(n, case["outputs"], generator=g, device=DEV)
    return list(X.split(case["batch"])), list(T.split(case["batch"]))


def training_network(case, seed):
    w = case["width"]
    return surrogate.MLP((case["inputs"], w, w, w, case["outputs"]), batch_max=case["batch"], seed=seed + 5)


# the first steps' rate of the warm start's schedule; the last step's gradients are the outputs (Adam's first
# updates follow the sign of a gradient however small, so weights repeat only to the rate itself)
LR = 1e-5


def prepare_train(case, seed):
    X, T = training_batches(case, seed)
    return dict(kind="train", mlp=training_network(case, seed), X=X, T=T)


def run_train(s):
    for x, y in zip(s["X"], s["T"]):
        s["mlp"].train_step(x, y, LR)
    return s["mlp"].gradients_host()


def exact_train(case, seed):
    X, T = training_batches(case, seed)
    W = [torch.as_tensor(a, device=DEV).double() for wb in training_network(case, seed).weights() for a in wb]
    m, v = [torch.zeros_like(w) for w in W], [torch.zeros_like(w) for w in W]
    for k, (x, y) in enumerate(zip(X, T), 1):
        p = [w.clone().requires_grad_(True) for w in W]
        h = x.double()
        for i in range(0, len(p), 2):
            h = h @ p[i].t() + p[i + 1]
            if i + 2 < len(p):
                h = torch.nn.functional.gelu(h)
        g = torch.autograd.grad(((h - y.double()) ** 2).mean(), p)
        if k == len(X):
            g = [w.cpu().numpy() for w in g]
            return [(g[i], g[i + 1]) for i in range(0, len(g), 2)]
        for i in range(len(W)):
            m[i] = 0.9 * m[i] + 0.1 * g[i]
            v[i] = 0.999 * v[i] + 0.001 * g[i] ** 2
            W[i] = W[i] - LR * (m[i] / (1 - 0.9 ** k)) / ((v[i] / (1 - 0.999 ** k)).sqrt() + 1e-8)


# --------------------------------------------------------------------------
# chemistry zones
def zone_parts(case, seed):
    for N, t in zip(workload.ZONE_N, workload.zone_networks()):
        yield N, t, draw_cells(t, case["n%d" % N], seed, salt=N)


def prepare_zones(case, seed):
    tabs, dcs, moves = [], [], []
    for N, t, s in zone_parts(case, seed):
        dc, work, flat = device_cells(t, s, case["n%d" % N], s["moved"])
        tabs.append(runtime.Tables(t))
        dcs.append(dc)
        moves.append((work, flat))
    opts = synth.react_opts(guess_mode=abi.PFX_GUESS_PREVIOUS)
    # the split that a time loop settles on after its first steps, then the graph it replays
    plan = abi.ZonePlan()
    plan.nzones, plan.variant = len(tabs), 1
    for k in range(3):
        _, _, plan = runtime.react_zones(tabs, dcs, opts, plan)
        for work, flat in moves:
            work.copy_(flat)
        runtime.rebalance(plan)
    return dict(kind="zones", tabs=tabs, dcs=dcs, moves=moves, graph=runtime.ZonesGraph(tabs, dcs, opts, plan))


def run_zones(s):
    for work, flat in s["moves"]:
        work.copy_(flat)
    s["graph"].launch()
    return [cell_outputs(dc) for dc in s["dcs"]]


def exact_zones(case, seed):
    return [exact_reaction(t, s, s["moved"], s["vf"]) for _, t, s in zone_parts(case, seed)]


# --------------------------------------------------------------------------
# constraint speciation
def constraints(case, seed):
    t = carbonate()
    s = draw_cells(t, case["cells"], seed, with_temp=False, total_range=(1e-5, 1e-2), ph_range=(6.0, 9.0))
    conc = rows(s["T"])
    conc[:, 0] = -(s["x"][0] + s["lng"][0]) / LN10
    return t, s, conc


def prepare_equilibrate(case, seed):
    t, s, conc = constraints(case, seed)
    dc, _, _ = device_cells(t, s, case["cells"], s["T"])
    return dict(kind="equilibrate", tab=runtime.Tables(t), dc=dc, conc=conc,
                ctype=[abi.PFX_CONSTRAINT_PH] + [abi.PFX_CONSTRAINT_TOTAL] * (t.N - 1),
                opts=synth.react_opts(max_iterations=300))


def run_equilibrate(s):
    runtime.equilibrate(s["tab"], s["dc"], s["ctype"], s["conc"], s["opts"])
    return {k: s["dc"].t[k] for k in ("total", "pri_molal", "pri_act_coef", "sec_act_coef", "sec_molal", "status")}


def exact_equilibrate(case, seed):
    t, s, conc = constraints(case, seed)
    n = case["cells"]
    ch = Chemistry(t, None, n)
    total, ph = conc.t().contiguous(), conc[:, 0].contiguous()
    lng, lngc, x = s["lng"], s["lngc"], s["x"]
    for _ in range(40):                       # the activity coefficients' fixed point
        x, _ = ch.speciate(total, ph, lng, lngc, x, its=30)
        lng, lngc = ch.activity(x.exp(), ch.complexes(x, lng, lngc))
    C = ch.complexes(x, lng, lngc)
    return dict(total=rows(ch.totals(x, C)), pri_molal=rows(x.exp()), pri_act_coef=rows(lng.exp()),
                sec_act_coef=rows(lngc.exp()), sec_molal=rows(C), status=None)


# --------------------------------------------------------------------------
# the operator-split step of a column, and its transport half on a grid
def column_parts(case, seed):
    t, n = carbonate(), case["cells"]
    s = draw_cells(t, n + 1, seed, with_temp=False, total_range=(1e-5, 1e-2), ph_range=(6.0, 9.0))
    inflow = s["T"][:, n].cpu().numpy()
    return t, {k: v[..., :n].contiguous() for k, v in s.items()}, column.Column(ncells=n), inflow


def prepare_os_step(case, seed):
    t, s, col, inflow = column_parts(case, seed)
    dc, _, _ = device_cells(t, s, case["cells"], s["T"])
    f = column.grid_faces(col, inflow)
    grid = runtime.DeviceGrid(f["nx"], f["ny"], f["nz"], f["q"], f["dd"], area=f["area"], bc_q=f["bc_q"],
                              bc_dd=f["bc_dd"], bc_total=f["bc_total"])
    tr, tab = runtime.OsTransport(grid), runtime.Tables(t)
    o_t = abi.default_opts(dt=DT, porosity=col.porosity, saturation=col.saturation, volume=col.volume)
    o_r = synth.react_opts(dt=DT, guess_mode=abi.PFX_GUESS_PREVIOUS, max_iterations=100)
    graph = runtime.OsStepGraph(tr, grid, tab, dc, t.N, o_t, o_r, rtol=1e-12, max_iterations=12)
    return dict(kind="os_step", tab=tab, dc=dc, grid=grid, transport=tr, graph=graph)


def run_os_step(s):
    s["graph"].launch()
    return dict(cell_outputs(s["dc"]), mnrl_volfrac=s["dc"].t["mnrl_volfrac"])


def exact_os_step(case, seed):
    t, s, col, inflow = column_parts(case, seed)
    n = case["cells"]
    (tu, td), (bu, bd), (ou, od) = col.coefficients()
    A = torch.zeros(n, n, device=DEV, dtype=F64)
    i = torch.arange(n, device=DEV)
    A[i, i] += col.porosity * col.saturation * 1000.0 * col.volume / DT
    A[i[:-1], i[:-1]] += tu
    A[i[:-1], i[1:]] += td
    A[i[1:], i[1:]] -= td
    A[i[1:], i[:-1]] -= tu
    A[0, 0] -= bd
    A[n - 1, n - 1] -= ou + od
    b = s["T"].t() * (col.porosity * col.saturation * 1000.0 * col.volume / DT)
    b[0] += bu * torch.as_tensor(inflow, device=DEV)
    total = torch.linalg.solve(A.cpu(), b.cpu()).to(DEV).t().contiguous()
    out = exact_reaction(t, s, total, s["vf"])
    mv = torch.as_tensor(t.mnrl_molar_vol, device=DEV)
    out["mnrl_volfrac"] = (rows(s["vf"]) + out["mnrl_rate"] * mv * DT).clamp_(min=0.0)
    return out


def prepare_os_transport(case, seed):
    n, N = case["nx"] * case["ny"] * case["nz"], case["comps"]
    g = _generator(seed, 11)
    total = (torch.rand(n, N, generator=g, device=DEV, dtype=F64) * math.log(1e4) + math.log(1e-6)).exp()
    f = workload.gi_grid(case["nx"], case["ny"], case["nz"], bc_total=np.full(N, 1e-4))
    grid = runtime.DeviceGrid(**f)
    dc = runtime.DeviceCells({"total": total.clone()}, n)
    return dict(kind="os_transport", dc=dc, flat=total, grid=grid, comps=N, transport=runtime.OsTransport(grid),
                opts=abi.default_opts(dt=10.0 * DT, porosity=POROSITY, saturation=1.0, volume=VOLUME))


def run_os_transport(s):
    s["dc"].t["total"].copy_(s["flat"])
    s["transport"].step(s["dc"], s["grid"], s["comps"], s["opts"], rtol=1e-8)
    return s["dc"].t["total"]


class Stencil:
    """Upwind fluxes of a grid's faces: coefficients of a cell's own value and of its neighbours', [nz][ny][nx]."""

    def __init__(self, f, true_outflow):
        T = lambda a: torch.as_tensor(a, device=DEV)  # noqa: E731
        nx, ny, nz = f["nx"], f["ny"], f["nz"]
        self.shape = (nz, ny, nx)
        self.diag = torch.zeros(nz, ny, nx, device=DEV, dtype=F64)
        self.lo, self.hi = [None] * 3, [None] * 3          # per direction x, y, z
        for d in range(3):
            dim = 2 - d
            q, dd, a = T(f["q"][d]), T(f["dd"][d]), f["area"][d] * 1000.0
            up = torch.where(q > 0, dd + q, dd) * a
            dn = torch.where(q > 0, -dd, q - dd) * a
            self.lo[d], self.hi[d] = -up, dn
            m = self.shape[dim]
            self.diag.narrow(dim, 1, m - 1).sub_(dn)
            self.diag.narrow(dim, 0, m - 1).add_(up)
        self.inflow = torch.zeros(nz, ny, nx, device=DEV, dtype=F64)   # coefficient of the boundary's value
        self.own = torch.zeros(nz, ny, nx, device=DEV, dtype=F64)      # of the cell's own value on an open face
        for side, i in ((0, 0), (1, nx - 1)):
            q, dd, a = T(f["bc_q"][side]), T(f["bc_dd"][side]), f["area"][0] * 1000.0
            up = torch.where(q > 0, dd + q, dd) * a
            dn = torch.where(q > 0, -dd, q - dd) * a
            self.diag[:, :, i] -= dn
            if f["bc_total"][side] is not None:
                self.inflow[:, :, i] += up
            else:
                self.own[:, :, i] -= up
        if true_outflow:
            self.diag = self.diag + self.own

    def apply(self, v):
        """the faces' net flux out of each cell, v [..][nz][ny][nx]"""
        r = self.diag * v
        for d in range(3):
            dim = 2 - d
            ax, m = v.dim() - 1 - d, self.shape[dim]
            if m > 1:
                r.narrow(ax, 1, m - 1).addcmul_(self.lo[d], v.narrow(ax, 0, m - 1))
                r.narrow(ax, 0, m - 1).addcmul_(self.hi[d], v.narrow(ax, 1, m - 1))
        return r


def bicgstab(apply, precondition, b, tol, its=200):
    """BiCGStab on the whole of b, for the plain solutions."""
    x, r = torch.zeros_like(b), b.clone()
    h, p, v = r.clone(), torch.zeros_like(b), torch.zeros_like(b)
    rho = alpha = omega = 1.0
    stop = tol * float(b.norm())
    for _ in range(its):
        if float(r.norm()) <= stop:
            break
        new = float((h * r).sum())
        if new == 0.0:
            break
        p = r + (new / rho) * (alpha / omega) * (p - omega * v)
        rho = new
        ph = precondition(p)
        v = apply(ph)
        alpha = rho / float((h * v).sum())
        s = r - alpha * v
        sh = precondition(s)
        t = apply(sh)
        omega = float((t * s).sum()) / max(float((t * t).sum()), 1e-300)
        x = x + alpha * ph + omega * sh
        r = s - omega * t
    return x


def exact_os_transport(case, seed):
    n, N = case["nx"] * case["ny"] * case["nz"], case["comps"]
    g = _generator(seed, 11)
    total = (torch.rand(n, N, generator=g, device=DEV, dtype=F64) * math.log(1e4) + math.log(1e-6)).exp()
    f = workload.gi_grid(case["nx"], case["ny"], case["nz"], bc_total=np.full(N, 1e-4))
    st = Stencil(f, True)
    acc = POROSITY * 1000.0 * VOLUME / (10.0 * DT)
    d = st.diag + acc
    out = torch.empty_like(total)
    for c in range(N):
        b = total[:, c].reshape(st.shape) * acc + st.inflow * 1e-4
        x = bicgstab(lambda v: st.apply(v) + acc * v, lambda v: v / d, b, 1e-15)
        x = x + bicgstab(lambda v: st.apply(v) + acc * v, lambda v: v / d, b - st.apply(x) - acc * x, 1e-8)
        out[:, c] = x.reshape(-1)
    return out


# --------------------------------------------------------------------------
# global-implicit assembly and time step
def case_range(case):
    return GI_RANGE if case["kind"] == "gi_step" else {}


GI_RANGE = dict(total_range=(1e-6, 1e-3), ph_range=(6.0, 8.0))


def gi_parts(case, seed, moved):
    """Cells on a grid: a base of speciated cells, each grid cell's free ions a Newton iterate's distance off."""
    t = network(case)
    n = case["nx"] * case["ny"] * case["nz"]
    nb = min(n, CHUNK)
    s = draw_cells(t, nb, seed, step=not moved, **case_range(case))
    if n > nb or moved:
        g = _generator(seed, 17)
        idx = torch.arange(n, device=DEV) % nb
        s = {k: v[..., idx] for k, v in s.items()}
        if moved:
            s["x"] = s["x"] + 0.01 * torch.randn(t.N, n, generator=g, device=DEV, dtype=F64)
    f = workload.gi_grid(case["nx"], case["ny"], case["nz"], bc_total=s["T"].mean(1).cpu().numpy())
    return t, s, f, n


def prepare_gi_assembly(case, seed):
    t, s, f, n = gi_parts(case, seed, True)
    dc, _, _ = device_cells(t, s, n, s["T"])
    grid = runtime.DeviceGrid(**f)
    row_ptr, col_idx = runtime.gi_structure(grid)
    return dict(kind="gi_assembly", tab=runtime.Tables(t), dc=dc, grid=grid, row_ptr=row_ptr, opts=synth.react_opts(),
                residual=torch.empty((n, t.N), dtype=F64, device=DEV),
                values=torch.empty((int(col_idx.numel()), t.N, t.N), dtype=F64, device=DEV))


def run_gi_assembly(s):
    res, vals = runtime.gi_residual_jacobian(s["tab"], s["dc"], s["grid"], s["opts"], s["row_ptr"], s["residual"],
                                             s["values"])
    return dict(residual=res, values=vals, mnrl_rate=s["dc"].t["mnrl_rate"])


def gi_cells_system(t, s, x, n, capped):
    """Per cell: residual and Jacobian (in ln m) without fluxes, totals, dT/d ln m, rates, cells first."""
    R, J, T, D, I = [], [], [], [], []
    for i in range(0, n, CHUNK):
        c = slice(i, min(n, i + CHUNK))
        ch = Chemistry(t, s["temp"][c], x[:, c].shape[1])
        a = [v[:, c].contiguous() for v in (x, s["lng"], s["lngc"])]
        fixed = POROSITY * 1000.0 * VOLUME * s["T"][:, c] + s["S"][:, c] * VOLUME
        r, j = ch.reaction_system(*a, fixed, s["vf"][:t.K, c], DT, capped)
        C = ch.complexes(*a)
        R.append(r)
        J.append(j.permute(2, 0, 1).contiguous())
        T.append(ch.totals(a[0], C))
        D.append(ch.total_jacobian(a[0], C).permute(2, 0, 1).contiguous())
        I.append(rows(ch.rates(a[0] + a[1], s["vf"][:t.K, c])[0]))
    return torch.cat(R, 1), torch.cat(J), torch.cat(T, 1), torch.cat(D), torch.cat(I)


def gi_residual(st, R, T, f):
    """The global residual: the cells' own and the faces' fluxes, [N][n]."""
    v = T.reshape((-1,) + st.shape)
    open_faces = 0.0 if st.diag_has_outflow else st.own * v
    bt = torch.as_tensor(f["bc_total"][0], device=DEV)
    return R + (st.apply(v) + open_faces - st.inflow * bt[:, None, None, None]).reshape(R.shape)


def exact_gi_assembly(case, seed):
    t, s, f, n = gi_parts(case, seed, True)
    st = Stencil(f, False)
    st.diag_has_outflow = False
    R, J, T, D, I = gi_cells_system(t, s, s["x"], n, False)
    res = rows(gi_residual(st, R, T, f))
    nz, ny, nx = st.shape
    cell = torch.arange(n, device=DEV).reshape(st.shape)
    has, coef, nb = [], [], []
    for d, side in ((2, 0), (1, 0), (0, 0), (None, 0), (0, 1), (1, 1), (2, 1)):     # a row's blocks in column order
        h = torch.ones(st.shape, dtype=torch.bool, device=DEV)
        w, other = st.diag.clone(), cell.clone()
        if d is not None:
            dim = 2 - d
            m = st.shape[dim]
            h.narrow(dim, 0 if side == 0 else m - 1, 1).fill_(False)
            w.zero_()
            if m > 1:
                w.narrow(dim, 1 if side == 0 else 0, m - 1).copy_(st.lo[d] if side == 0 else st.hi[d])
                other.narrow(dim, 1 if side == 0 else 0, m - 1).copy_(cell.narrow(dim, 0 if side == 0 else 1, m - 1))
        has.append(h.reshape(-1))
        coef.append(w.reshape(-1))
        nb.append(other.reshape(-1))
    count = torch.stack(has).long()
    row_ptr = torch.cat([torch.zeros(1, dtype=torch.long, device=DEV), count.sum(0).cumsum(0)])
    at = row_ptr[:-1] + count.cumsum(0) - count
    vals = torch.empty((int(row_ptr[-1]), t.N, t.N), dtype=F64, device=DEV)
    for i in range(0, n, CHUNK):
        c = slice(i, min(n, i + CHUNK))
        for k in range(7):
            on = torch.nonzero(has[k][c]).flatten() + i
            if on.numel() == 0:
                continue
            b = coef[k][on][:, None, None] * D[nb[k][on]]
            if k == 3:
                b += J[on]
            vals[at[k][on]] = b.transpose(1, 2)
    return dict(residual=res, values=vals, mnrl_rate=I)


def prepare_gi_step(case, seed):
    t, s, f, n = gi_parts(case, seed, False)
    dc, work, flat = device_cells(t, s, n, s["T"])
    grid, tab = runtime.DeviceGrid(**f), runtime.Tables(t)
    return dict(kind="gi_step", tab=tab, dc=dc, work=work, flat=flat, grid=grid, solver=runtime.GiSolver(tab, grid),
                opts=synth.react_opts())


def run_gi_step(s):
    s["work"].copy_(s["flat"])
    runtime.gi_initial_iterate(s["tab"], s["dc"], s["opts"])
    st = s["solver"].timestep(s["dc"], s["grid"], s["opts"])
    return dict(pri_molal=s["dc"].t["pri_molal"], mnrl_rate=s["dc"].t["mnrl_rate"], dt=float(st.dt),
                converged=int(st.reason > 0))


def exact_gi_step(case, seed):
    """Newton on the whole grid with the consistent derivative, every linear system to 1e-13."""
    t, s, f, n = gi_parts(case, seed, False)
    st = Stencil(f, True)
    st.diag_has_outflow = True
    N = t.N
    x = s["x"].clone()
    for i in range(0, n, CHUNK):
        c = slice(i, min(n, i + CHUNK))
        ch = Chemistry(t, s["temp"][c], x[:, c].shape[1])
        fixed = POROSITY * 1000.0 * VOLUME * s["T"][:, c] + s["S"][:, c] * VOLUME
        lng, lngc = s["lng"][:, c].contiguous(), s["lngc"][:, c].contiguous()
        x[:, c], _ = ch.react(x[:, c].contiguous(), lng, lngc, fixed, s["vf"][:t.K, c], DT, True, its=40)
    for k in range(80):
        R, J, T, D, I = gi_cells_system(t, s, x, n, k < 40)
        F = gi_residual(st, R, T, f)
        P = torch.linalg.inv(J + st.diag.reshape(-1, 1, 1) * D)
        block = lambda B, v: (B * v.t()[:, None, :]).sum(2).t().contiguous()  # noqa: E731
        flux = lambda w: st.apply(w.reshape((N,) + st.shape)).reshape(N, n)   # noqa: E731
        y = bicgstab(lambda v: block(J, v) + flux(block(D, v)), lambda v: block(P, v), F, 1e-13, its=60)
        x = x - y.clamp(-5.0, 5.0)
        if float(y.abs().max()) < 1e-12:
            break
    return dict(pri_molal=rows(x.exp()), mnrl_rate=I, dt=DT, converged=None)


# --------------------------------------------------------------------------
PREPARE = dict(react=prepare_react, warm=prepare_warm, train=prepare_train, zones=prepare_zones,
               equilibrate=prepare_equilibrate, os_step=prepare_os_step, os_transport=prepare_os_transport,
               gi_assembly=prepare_gi_assembly, gi_step=prepare_gi_step)
RUN = dict(react=run_react, warm=run_warm, train=run_train, zones=run_zones, equilibrate=run_equilibrate,
           os_step=run_os_step, os_transport=run_os_transport, gi_assembly=run_gi_assembly, gi_step=run_gi_step)
EXACT = dict(react=exact_react, warm=exact_react, train=exact_train, zones=exact_zones, equilibrate=exact_equilibrate,
             os_step=exact_os_step, os_transport=exact_os_transport, gi_assembly=exact_gi_assembly,
             gi_step=exact_gi_step)


def prepare(case, seed):
    return PREPARE[case["kind"]](case, seed)


def run(state):
    return RUN[state["kind"]](state)


def exact(case, seed):
    return EXACT[case["kind"]](case, seed)


# Newton iterations of a cell's reaction step, the step test's pass among them, as the cells above need them on
# average: the arithmetic a pass cannot do without is counted from it
ITERATIONS = 6


def _reaction_work(N, M, K, R, cells, t):
    byts = 8 * ((5 * N + M + 2 * K + 1 + R) + (4 * N + 2 * M + K + R + 1)) + 8
    fl = t.flops_per_iteration()
    return byts * cells, ITERATIONS * (fl["flops"] + fl["transcendentals"]) * cells


def work(case):
    kind = case["kind"]
    if kind == "train":
        d = [case["inputs"]] + [case["width"]] * 3 + [case["outputs"]]
        weights = sum(a * b for a, b in zip(d, d[1:]))
        n = case["batch"] * case["steps"]
        return {"bytes": 4 * n * (d[0] + d[-1]) + case["steps"] * 24 * weights, "flops": 6 * weights * n}
    if kind == "os_transport":
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 8 * (2 * n * case["comps"] + 6 * n), "flops": 60 * n * case["comps"]}
    if kind == "zones":
        b = f = 0.0
        for N, t in zip(workload.ZONE_N, workload.zone_networks()):
            p, q = _reaction_work(N, t.M, t.K, 0, case["n%d" % N], t)
            b, f = b + p, f + q
        return {"bytes": b, "flops": f}
    t = network(case) if kind not in ("os_step", "equilibrate") else carbonate()
    if kind in ("gi_assembly", "gi_step"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        n = nx * ny * nz
        nnzb = 7 * n - 2 * (ny * nz + nx * nz + nx * ny)
        fl = t.flops_per_iteration()
        if kind == "gi_assembly":
            return {"bytes": 8 * (nnzb * t.N ** 2 + n * (5 * t.N + t.M + 3 * t.K + 4)), "flops": n * fl["flops"]}
        # at least the Newton iterations of the coupled step, each an assembly and a linear iteration: the block
        # matrix written once and read twice
        return {"bytes": ITERATIONS * 3 * 8 * nnzb * t.N ** 2, "flops": ITERATIONS * n * (fl["flops"] + 28 * t.N ** 2)}
    b, f = _reaction_work(t.N, t.M, t.K, t.R, case["cells"], t)
    if kind == "warm":
        ni = 2 * t.N + 1 + t.K
        d = [ni + (-ni) % 8] + [case["width"]] * 3 + [t.N]
        f += 2 * sum(p * q for p, q in zip(d, d[1:])) * case["cells"]
    return {"bytes": b, "flops": f}
