"""The work a user of this framework has it do, as cases that can be timed.

A pass is what one round of a user's program does between two frames of its
output: some motion steps, then the state and the observables read back (the
reference copies its arrays to the host after every `loopsPerPrint` steps and
goes on), a loop of single calls, a start from given atoms, or the data
primitives on caller-owned device memory.

A case is a dict of plain values:
  work    "steps"      step(n) on one context, then a frame
          "group"      the same on a batch split over two contexts
          "calls"      the FP64 loop body call by call, a temperature per step
          "restart"    set_state, step(n), a frame and observe()
          "sample"     init_distribution, step(n), a frame and observe()
          "primitives" sort_by_key, exclusive_scan and remove_if
  form    "fp64" or "fp32"
  trap    "quadrupole", "ip" (the reference's Ioffe-Pritchard run), "box"
  n, nc, traps, steps, spin, cut, bits: sizes and options of that work

`exact` restates the step in 64 bits with torch: Philox draws, NTC collisions,
velocity Verlet, spins, losses.  It has no value for the outputs that are whole
numbers, and none for long runs of the FP32 form, whose accept decisions part
from the 64-bit ones now and then (one trial in some 1e7).
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from cudadsmc_amd import Simulation, SimulationGroup, _abi, configs

MASK = 0xFFFFFFFF


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the named FP64 workload of N = 1e4: every launch counts
        dict(name="plain_1e4", work="steps", form="fp64", trap="quadrupole", n=10000, nc=35, traps=1,
             steps=200, spin=0, cut=0),
        # the reference's own run (Nc 50, N 10000): spinors, losses, spin flips
        dict(name="plain_reference", work="steps", form="fp64", trap="ip", n=10000, nc=50, traps=1,
             steps=500, spin=1, cut=0),
        # the precision workload in the FP64 form
        dict(name="plain_1e6", work="steps", form="fp64", trap="quadrupole", n=1000000, nc=100, traps=1,
             steps=200, spin=0, cut=0),
        # the reference's main loop, bound call by call, with an energy cut
        dict(name="plain_calls", work="calls", form="fp64", trap="quadrupole", n=30011, nc=41, traps=1,
             steps=20, spin=0, cut=1),
        # a small FP32 trap, where latency counts
        dict(name="kahan_2e4", work="steps", form="fp32", trap="quadrupole", n=20011, nc=41, traps=1,
             steps=200, spin=0, cut=0),
        # the precision workload in the FP32 form
        dict(name="kahan_1e6", work="steps", form="fp32", trap="quadrupole", n=1000000, nc=100, traps=1,
             steps=1000, spin=0, cut=0),
        # thermalisation of a dense gas in a periodic box, N = 2^22
        dict(name="kahan_box", work="steps", form="fp32", trap="box", n=1 << 22, nc=128, traps=1,
             steps=1000, spin=0, cut=0),
        # spin precession (20 substeps) and evaporation, N = 4e6
        dict(name="kahan_spin", work="steps", form="fp32", trap="quadrupole", n=4000000, nc=100, traps=1,
             steps=500, spin=20, cut=1),
        # the batched headline workload: 256 traps, 5.2 M atoms, two groups
        dict(name="batch_256", work="group", form="fp32", trap="quadrupole", n=0, nc=0, traps=256,
             steps=1000, spin=0, cut=1),
        # a scan of a few dozen traps in one context
        dict(name="batch_24", work="steps", form="fp32", trap="quadrupole", n=0, nc=0, traps=24,
             steps=200, spin=0, cut=1),
        # a run taken up from saved atoms
        dict(name="restart_3e5", work="restart", form="fp32", trap="quadrupole", n=300007, nc=67, traps=1,
             steps=100, spin=0, cut=0),
        # the reference's Thrust calls on caller-owned memory
        dict(name="primitives_1m", work="primitives", n=1000003, bits=20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Sizes are spread over the logarithm of their range; grids give the
    central cell between 4 and 16 test particles, as tune.py's do."""
    work = rng.choice(["steps"] * 6 + ["batch"] * 3 + ["calls", "restart", "sample", "primitives"])
    if work == "primitives":
        return dict(work=work, n=_log(rng, 1000, 16000000), bits=rng.randint(8, 31))
    if work == "batch":
        traps = _log(rng, 2, 220)
        return dict(work=rng.choice(["steps", "group"]), form="fp32", trap="quadrupole", n=0, nc=0,
                    traps=traps, steps=rng.choice([100, 200, 500]), spin=0, cut=rng.randint(0, 1))
    if work == "calls":
        return dict(work=work, form="fp64", trap="quadrupole", n=_log(rng, 3000, 300000),
                    nc=rng.randint(20, 60), traps=1, steps=rng.choice([5, 10, 20]), spin=0,
                    cut=rng.randint(0, 1))
    form = "fp32" if work != "steps" else rng.choice(["fp32", "fp32", "fp64"])
    trap = rng.choice(["quadrupole", "quadrupole", "ip", "box"])
    if form == "fp32" and trap == "ip":
        trap = "quadrupole"
    n = _log(rng, 2000, 4000000 if form == "fp32" else 1000000)
    if trap == "ip":
        n = min(n, 200000)
    nc = max(8, min(160, round((1000.0 * n / (4.0 * math.pi * rng.uniform(4, 16))) ** (1.0 / 3.0))))
    spin = 0
    if trap == "ip":
        spin = rng.randint(0, 1)
    elif trap == "quadrupole" and form == "fp32" and work == "steps":
        spin = rng.choice([0, 0, 0, 1, 10, 20])
    cut = rng.randint(0, 1) if trap == "quadrupole" else 0
    return dict(work=work, form=form, trap=trap, n=n, nc=nc, traps=1,
                steps=rng.choice([50, 100, 200] if n > 300000 else [100, 200, 400]), spin=spin, cut=cut)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _run_of(case, seed):
    """The configuration that a user's program writes for this case."""
    steps, spin, cut = case["steps"], case["spin"], bool(case["cut"])
    if case["traps"] > 1:
        r = configs.batched_traps(n_traps=case["traps"])
        r = r.with_(energy_cut=cut)
    elif case["trap"] == "ip":
        r = configs.reference(case["nc"], case["n"])
        if not spin:
            r = r.with_(spin=False, spin_loss=False, mcwf=False)
    elif case["trap"] == "box":
        r = configs.box_thermalise(case["form"], case["n"], case["nc"])
    elif spin:
        r = configs.spin_evaporation(case["form"], case["n"], case["nc"])
        r = r.with_(spin_substeps=spin, energy_cut=cut)
    else:
        t = configs.quadrupole_trap(case["n"], case["nc"])
        if cut:
            t.eta_start, t.eta_end, t.T_cut, t.eta_steps = 8.0, 6.0, t.T, 20000
        r = configs.Run(traps=[t], dt=1e-6, energy_cut=cut)
    return r.with_(precision=case["form"], seed=int(seed) + 1, obs_capacity=steps)


def _atoms_given(case, seed):
    """Saved atoms of a run that is taken up again (host arrays, FP64)."""
    r = _run_of(case, seed)
    x, v = _sample(r, "cpu")[:2]
    return x.numpy(), v.numpy()


def prepare(case, seed):
    if case["work"] == "primitives":
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        n, hi = case["n"], 1 << case["bits"]
        keys = torch.randint(0, hi, (n,), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
        return dict(case=case, lib=_abi.load_library(), keys=keys,
                    vals=torch.randperm(n, generator=g, device="cuda").to(torch.int32),
                    counts=torch.randint(0, 12, (n,), generator=g, device="cuda", dtype=torch.int32),
                    out=torch.empty(n, device="cuda", dtype=torch.int32),
                    # one value in fifty is removed
                    lost=(torch.randperm(n, generator=g, device="cuda") < n // 50).to(torch.int32))
    r = _run_of(case, seed)
    if case["work"] == "group":
        sim = SimulationGroup(configs.split_traps(r, 2))
    else:
        sim = Simulation(r)
    state = dict(case=case, sim=sim)
    state["frames"] = [_frame_buffers(s.run) for s in (sim.sims if case["work"] == "group" else [sim])]
    if case["work"] == "restart":
        state["pos"], state["vel"] = _atoms_given(case, seed)
    elif case["work"] != "sample":
        sim.init_distribution()
        sim.sync()
    return state


# ---------------------------------------------------------------------------
# A pass
# ---------------------------------------------------------------------------
def _frame_buffers(run_):
    """Host arrays for a frame, as a driver allocates them once: a row for
    every atom of the capacity (rows past the alive atoms stay as they are)."""
    n = run_.n_atoms
    out = dict(pos=np.zeros((n, 3)), vel=np.zeros((n, 3)), label=np.zeros(n, dtype=np.int32))
    if run_.spin:
        out["spin"] = np.zeros((n, 4 if run_.precision == "fp64" else 3))
    if run_.mcwf:   # the rest of the reference's thirteen datasets
        cells = int(np.prod(run_.traps[0].nc)) + 1
        out.update(up=np.zeros(n, dtype=np.int32), cell=np.zeros(n, dtype=np.int32),
                   cell_count=np.zeros(cells, dtype=np.int32), cell_collisions=np.zeros(cells, dtype=np.int32),
                   lost_pos=np.zeros((n, 3)), lost_vel=np.zeros((n, 3)))
    return out


_FIELDS = dict(pos=_abi.FIELD_POS, vel=_abi.FIELD_VEL, label=_abi.FIELD_ATOM_ID, spin=_abi.FIELD_SPIN,
               up=_abi.FIELD_SPIN_UP, cell=_abi.FIELD_CELL_ID, cell_count=_abi.FIELD_CELL_COUNT,
               cell_collisions=_abi.FIELD_COLLISION_COUNT, lost_pos=_abi.FIELD_EVAP_POS,
               lost_vel=_abi.FIELD_EVAP_VEL)


def _frame(sim, frame):
    for k, a in frame.items():
        _abi.check(sim.lib, sim.lib.dsmc_copy_out(sim.h, _FIELDS[k], a.ctypes.data, a.nbytes), sim.h)
    return frame


def _log_fields(lg):
    return {k: lg[k] for k in ("ek", "ep", "v2", "n_alive", "n_evap", "collisions")}


def run(state):
    case = state["case"]
    work = case["work"]
    if work == "primitives":
        return _primitives(state)
    sim, frame = state["sim"], state["frames"][0]
    if work == "group":
        sim.step(case["steps"])
        out = dict(log=_log_fields(sim.obs_log()))
        for i, s in enumerate(sim.sims):
            out["group%d" % i] = _frame(s, state["frames"][i])
        return out
    if work == "calls":
        temps, flips = [], []
        for _ in range(case["steps"]):
            sim.index_atoms()
            sim.sort_arrays()
            sim.build_cell_table()
            sim.collide()
            sim.move_atoms()
            temps.append(sim.calculate_temp())
            if case["cut"]:
                sim.evaporation_tag()
                flips.append(sim.compact())
        return dict(temperature=np.array(temps), alive=np.array(flips, dtype=np.int64), **_frame(sim, frame))
    if work == "restart":
        sim.set_state(state["pos"], state["vel"])
    elif work == "sample":
        sim.init_distribution()
    sim.step(case["steps"])
    out = dict(_frame(sim, frame), log=_log_fields(sim.obs_log()))
    if work in ("restart", "sample"):
        o = sim.observe()[0]
        out["now"] = dict(ek=o.ek, ep=o.ep, v2=np.array(o.v2), n_alive=int(o.n_alive))
    return out


def _primitives(state):
    lib, n = state["lib"], state["case"]["n"]
    keys, vals, kept = state["keys"].clone(), state["vals"].clone(), state["vals"].clone()
    _abi.check(lib, lib.dsmc_sort_by_key(keys.data_ptr(), vals.data_ptr(), n, state["case"]["bits"], None))
    _abi.check(lib, lib.dsmc_exclusive_scan(state["counts"].data_ptr(), state["out"].data_ptr(), n, None))
    m = ctypes.c_int()
    _abi.check(lib, lib.dsmc_remove_if(kept.data_ptr(), state["lost"].data_ptr(), n, ctypes.byref(m), None))
    return keys, vals, state["out"], kept[:m.value]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    if case["work"] == "primitives":
        n = case["n"]
        # pairs in and out; counts in, sums out; values and stencil in, values out
        return {"bytes": 16.0 * n + 8.0 * n + 12.0 * n, "flops": 0.0}
    r = _run_of(case, 0)
    n = r.n_atoms
    # each step reads and writes every atom's position and velocity (with
    # their remainders in the FP32 form), spins too; the frame writes them once
    # more in 64 bits, with a label
    spin = 0 if not r.spin else 64 if case["form"] == "fp64" else 24
    per_step = 96.0 + spin
    subs = r.spin_substeps if r.spin else 0
    frame = 52.0 + (0 if not r.spin else 32 if case["form"] == "fp64" else 24)
    given = 48.0 if case["work"] == "restart" else 0.0
    return {"bytes": n * (per_step * case["steps"] + frame + given),
            "flops": float(n) * case["steps"] * (90.0 + 50.0 * subs)}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _philox(a, b, c, d, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors or numbers."""
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & MASK, (k1 + 0xBB67AE85) & MASK
        p0, p1 = a * 0xD2511F53, c * 0xCD9E8D57   # the product's 64 bits (two's complement)
        a, b, c, d = ((p1 >> 32) & MASK) ^ b ^ k0, p1 & MASK, ((p0 >> 32) & MASK) ^ d ^ k1, p0 & MASK
    return a, b, c, d


def _u01(hi, lo):
    return (((hi << 20) | (lo >> 12)).double() + 0.5) * 2.0 ** -52


def _u23(r):
    return ((r >> 9).double() + 0.5) * 2.0 ** -23


class _Model:
    """One or more traps in 64 bits; every per-trap number is a tensor."""

    def __init__(self, r, dev):
        self.r, self.dev = r, dev
        T = r.traps
        f = lambda v: torch.tensor(v, dtype=torch.float64, device=dev)   # noqa: E731
        self.kind = T[0].kind
        self.T = len(T)
        self.cells = torch.tensor([t.nc[0] * t.nc[1] * t.nc[2] for t in T], device=dev)
        self.base = torch.cumsum(self.cells + 1, 0) - self.cells - 1
        self.n_keys = int((self.cells + 1).sum())
        self.nc = torch.tensor([list(t.nc) for t in T], device=dev)
        self.hw = f([list(t.half_width) for t in T])
        self.len = 2.0 * self.hw / self.nc
        self.vol = self.len.prod(1)
        self.mu, self.dB = f([t.mu for t in T]), f([t.dBdz for t in T])
        self.alpha = f([t.n_real / t.n_atoms for t in T])
        self.stream = torch.tensor([i + t.philox_stream for i, t in enumerate(T)], device=dev)
        t0 = T[0]
        self.B0, self.g, self.c = t0.B0, t0.dBdx, t0.d2Bdx2
        self.eta = f([[t.eta_start, t.eta_end, t.T_cut * configs.KB if t.eta_start > 0 else 0.0, t.eta_steps]
                      for t in T])
        tax = [[a if a > 0 else t.T for a in t.T_axis] for t in T]
        self.smax0 = f([math.sqrt(16. * configs.KB * (sum(a) / 3 if max(t.T_axis) > 0 else t.T) /
                                  (configs.PI_REF * r.mass)) * r.sigma for t, a in zip(T, tax)])

    def draws(self, t, a, b, c, purpose, d):
        seed = self.r.seed
        return _philox(a, b, c, (purpose << 24) | d, seed & MASK, ((seed >> 32) + self.stream[t]) & MASK)

    def ip_field(self, x):
        X, Y, Z = x.unbind(1)
        c = 0.5 * self.c
        return torch.stack([self.g * X - c * X * Z, -self.g * Y - c * Y * Z,
                            self.B0 + c * (Z * Z - 0.5 * (X * X + Y * Y))], 1)

    def field(self, x, t):
        """|B| and its direction."""
        if self.kind == "ip":
            B = self.ip_field(x)
            m = B.square().sum(1).sqrt()
            return m, B / m[:, None]
        s = x * torch.tensor([1.0, 1.0, -2.0], dtype=torch.float64, device=self.dev)
        rho = s.square().sum(1).sqrt()
        return self.dB[t] * rho, s / rho[:, None]

    def accel(self, x, t, up):
        if self.kind == "box":
            return torch.zeros_like(x)
        k = -self.mu[t] / self.r.mass
        if self.kind == "quadrupole":
            s = x * torch.tensor([1.0, 1.0, 4.0], dtype=torch.float64, device=self.dev)
            rho = (x[:, 0] ** 2 + x[:, 1] ** 2 + 4 * x[:, 2] ** 2).sqrt()
            return s * (k * self.dB[t] / rho)[:, None]
        n = self.field(x, t)[1]
        X, Y, Z = x.unbind(1)
        h = 0.5 * self.c
        g = torch.stack([(self.g - h * Z) * n[:, 0] - h * X * n[:, 2],
                         (-self.g - h * Z) * n[:, 1] - h * Y * n[:, 2],
                         -h * X * n[:, 0] - h * Y * n[:, 1] + self.c * Z * n[:, 2]], 1)
        return g * torch.where(up, k, -k)[:, None]

    def potential(self, x, t):
        if self.kind == "box":
            return torch.zeros_like(x[:, 0])
        return self.mu[t] * (self.field(x, t)[0] - (self.B0 if self.kind == "ip" else 0.0))

    def key(self, x, t):
        q = torch.floor((x + self.hw[t]) / self.len[t])
        nc = self.nc[t]
        ok = ((q > -1) & (q < nc)).all(1)
        i = q.long()
        return self.base[t] + torch.where(ok, (i[:, 2] * nc[:, 1] + i[:, 1]) * nc[:, 0] + i[:, 0], self.cells[t])

    def directions(self, t, cell, step, tr, fp32):
        """Marsaglia (1972): points on the sphere, draws 2, 3, ..."""
        out = torch.zeros((len(cell), 3), dtype=torch.float64, device=self.dev)
        left = torch.arange(len(cell), device=self.dev)
        for k in range(16):
            if not len(left):
                break
            o = self.draws(t[left], cell[left], step, tr, 1, 2 + k)
            pairs = [(_u23(o[0]), _u23(o[1])), (_u23(o[2]), _u23(o[3]))] if fp32 else \
                [(_u01(o[0], o[1]), _u01(o[2], o[3]))]
            for u, w in pairs:
                u, w = 2 * u - 1, 2 * w - 1
                s = u * u + w * w
                ok = (s < 1) & (out[left].square().sum(1) == 0)
                q = 2 * (1 - s).clamp(min=0).sqrt()
                out[left[ok]] = torch.stack([u * q, w * q, 1 - 2 * s], 1)[ok]
            left = left[out[left].square().sum(1) == 0]
        return out

    def collide(self, key, v, smax, step):
        """NTC trials of every cell, one trial of all cells at a time; returns
        the accepted collisions per cell."""
        r, fp32 = self.r, self.r.precision == "fp32"
        count = torch.bincount(key, minlength=self.n_keys)
        first = torch.cumsum(count, 0) - count
        K = torch.nonzero(count > 1)[:, 0]
        t = torch.searchsorted(self.base, K, right=True) - 1
        cell = K - self.base[t]
        keep = cell < self.cells[t]
        K, t, cell = K[keep], t[keep], cell[keep]
        n, done = count[K], torch.zeros_like(count)
        Mc = 0.5 * n * (n - 1)
        X = Mc * self.alpha[t] * r.lpc * r.dt * smax[K] / self.vol[t]
        lam = X.ceil() / Mc
        trials = (Mc * lam).long() if r.pair_mode == "reference" else X.ceil().long()
        pc = self.alpha[t] * r.lpc * r.dt / self.vol[t] * r.sigma / lam
        for tr in range(int(trials.max()) if len(K) else 0):
            s = torch.nonzero(trials > tr)[:, 0]
            ns, ts, cs = n[s], t[s], cell[s]
            if r.pair_mode == "reference":
                i, j = torch.zeros_like(ns), torch.zeros_like(ns)
                for q in range(64):
                    same = torch.nonzero((i == j) & (ns > 2))[:, 0]
                    if not len(same):
                        break
                    o = self.draws(ts[same], cs[same], step, tr, 1, 16 + q)
                    i[same] = torch.floor(_u01(o[0], o[1]) * (ns[same] - 1)).long()
                    j[same] = torch.floor(_u01(o[2], o[3]) * (ns[same] - 1)).long()
                j = torch.where(i == j, torch.ones_like(j), j)
                i = torch.where(ns == 2, torch.zeros_like(i), i)
                o = self.draws(ts, cs, step, tr, 1, 1)
                u = _u01(o[0], o[1])
            else:
                o = self.draws(ts, cs, step, tr, 1, 0)
                i, j = (o[0] * ns) >> 32, (o[1] * (ns - 1)) >> 32
                j = j + (j >= i)
                u = _u23(o[2]) if fp32 else _u01(o[2], o[3])
            a, b = first[K[s]] + i, first[K[s]] + j
            vr = (v[a] - v[b]).square().sum(1).sqrt()
            smax[K[s]] = torch.maximum(smax[K[s]], vr * r.sigma)
            hit = torch.nonzero(pc[s] * vr > u)[:, 0]
            a, b = a[hit], b[hit]
            w = 0.5 * vr[hit][:, None] * self.directions(ts[hit], cs[hit], step, tr, fp32)
            mid = 0.5 * (v[a] + v[b])
            v[a], v[b] = mid - w, mid + w
            done[K[s[hit]]] += 1
        return done

    def cut_at(self, step):
        e = self.eta
        f = torch.where(e[:, 3] > 0, (step / e[:, 3].clamp(min=1)).clamp(max=1.0), torch.ones_like(e[:, 3]))
        return torch.where(e[:, 2] > 0, (e[:, 0] + (e[:, 1] - e[:, 0]) * f) * e[:, 2], math.inf)


def _sample(r, dev):
    """init_distribution: positions, velocities, traps."""
    m = _Model(r, dev)
    out = []
    for ti, tr in enumerate(r.traps):
        n = int(tr.n_atoms)
        a = torch.arange(n, device=dev)
        t = torch.full((n,), ti, dtype=torch.long, device=dev)
        gauss = lambda o: ((-2.0 * torch.log(_u01(o[0], o[1]))).sqrt(), 2 * math.pi * _u01(o[2], o[3]))   # noqa: E731
        if tr.kind == "quadrupole":
            o, p = m.draws(t, a, 0, 0, 2, 2), m.draws(t, a, 0, 0, 2, 3)
            rad = -tr.thermal_radius() * (_u01(o[0], o[1]).log() + _u01(o[2], o[3]).log() + _u01(p[0], p[1]).log())
            x = torch.zeros((n, 3), dtype=torch.float64, device=dev)
            left = a
            for k in range(32):
                if not len(left):
                    break
                o = m.draws(t[left], left, 0, 0, 2, 4 + k)
                u, w = 2 * _u01(o[0], o[1]) - 1, 2 * _u01(o[2], o[3]) - 1
                s = u * u + w * w
                ok = s < 1
                q = 2 * (1 - s).clamp(min=0).sqrt()
                x[left[ok]] = (rad[left][:, None] * torch.stack([u * q, w * q, 0.5 * (1 - 2 * s)], 1))[ok]
                left = left[~ok]
        elif tr.kind == "box":
            o, p = m.draws(t, a, 0, 0, 2, 2), m.draws(t, a, 0, 0, 2, 3)
            u = torch.stack([_u01(o[0], o[1]), _u01(o[2], o[3]), _u01(p[0], p[1])], 1)
            x = -m.hw[ti] + 2.0 * m.hw[ti] * u
        else:   # the reference's rejection sampler, 32 proposals at a time
            x = torch.zeros((n, 3), dtype=torch.float64, device=dev)
            left, k0 = a, 0
            while len(left):
                A, k = left[:, None], torch.arange(k0, k0 + 32, device=dev)[None, :]
                z, w = gauss(m.draws(ti, A, 0, k, 2, 8)), gauss(m.draws(ti, A, 0, k, 2, 9))
                p = torch.stack([z[0] * z[1].cos(), z[0] * z[1].sin(), w[0] * w[1].cos()], 2) * m.hw[ti] / 3.
                B = m.ip_field(p.reshape(-1, 3)).square().sum(1).sqrt().reshape(p.shape[:2])
                o = m.draws(ti, A, 0, k, 2, 10)
                ok = _u01(o[0], o[1]) < torch.exp(-0.5 * (B - m.B0) * r.gs * configs.MUB / configs.KB / tr.T)
                any_, at = ok.any(1), ok.int().argmax(1)
                x[left[any_]] = p[any_, at[any_]]
                left, k0 = left[~any_], k0 + 32
        z, w = gauss(m.draws(t, a, 0, 0, 2, 0)), gauss(m.draws(t, a, 0, 0, 2, 1))
        tax = torch.tensor([b if b > 0 else tr.T for b in tr.T_axis], dtype=torch.float64, device=dev)
        v = torch.stack([z[0] * z[1].cos(), z[0] * z[1].sin(), w[0] * w[1].cos()], 1) * \
            (configs.KB * tax / r.mass).sqrt()
        out.append((x, v, t))
    return tuple(torch.cat(c) for c in zip(*out))


def _spinor_step(m, st, r, dt):
    """SU(2) rotation at the pre-move position (FP64 form)."""
    B, n = m.field(st["x"], st["t"])
    th = 0.5 * r.gs * configs.MUB * B * dt / configs.HBAR
    s, c = th.sin(), th.cos()
    (nx, ny, nz), (ur, ui, dr, di) = n.unbind(1), st["psi"].unbind(1)
    st["psi"] = torch.stack([ur * c + (nx * di - ny * dr + nz * ui) * s, ui * c - (nx * dr + ny * di + nz * ur) * s,
                             dr * c + (nx * ui + ny * ur - nz * di) * s, di * c + (-nx * ur + ny * ui + nz * dr) * s], 1)


def _bloch_step(m, st, r):
    """Rotations of the Bloch vector along the drift (FP32 form)."""
    dts = r.dt / r.spin_substeps
    for k in range(r.spin_substeps):
        tau = (k + 0.5) * dts if r.spin_interp else 0.0
        B, n = m.field(st["x"] + st["v"] * tau, st["t"])
        phi = (r.gs * configs.MUB * B * dts / configs.HBAR)[:, None]
        s = st["psi"]
        st["psi"] = s * phi.cos() + torch.cross(n, s, dim=1) * phi.sin() + n * (n * s).sum(1, True) * (1 - phi.cos())
    st["psi"] = st["psi"] / st["psi"].square().sum(1, True).sqrt()


def _pops(m, st):
    n = m.field(st["x"], st["t"])[1]
    ur, ui, dr, di = st["psi"].unbind(1)
    d = n[:, 0] * (ur * dr + ui * di) - n[:, 1] * (ui * dr - ur * di) - n[:, 2] * (0.5 - ur * ur - ui * ui)
    return torch.stack([0.5 + d, 0.5 - d], 1)


def _flip_and_decay(m, st, r, coll_steps):
    x, v, t, up = st["x"], st["v"], st["t"], st["up"]
    old, new = st["pops"][st["id"]], _pops(m, st)
    B, n = m.field(x, t)
    p = torch.where(up, (new[:, 1] - old[:, 1]) / old[:, 0], (new[:, 0] - old[:, 0]) / old[:, 1])
    de = torch.where(up, 1.0, -1.0) * 2.0 * m.mu[t] * B
    ek = 0.5 * r.mass * v.square().sum(1)
    o = m.draws(t, st["id"], coll_steps, 0, 3, 0)
    flip = (p > _u01(o[0], o[1])) & (ek + de > 0)
    scale = torch.where(flip, ((ek + de).clamp(min=0) / ek).sqrt(), torch.ones_like(ek))
    st["v"], st["up"] = v * scale[:, None], up ^ flip
    rel = 2.0 * m.accel(x, t, torch.ones_like(up)).square().sum(1).sqrt()
    tp = 1.163 * (r.sigma / rel).sqrt()
    tv = math.sqrt(2. / configs.PI_REF) * configs.HBAR / (r.mass * r.sigma * rel)
    e = torch.exp(-r.lpc * r.dt * (tp ** -3 + tv ** -3) ** (1. / 3.))
    om, op = 1 - e, 1 + e
    (nx, ny, nz), (ur, ui, dr, di) = n.unbind(1), st["psi"].unbind(1)
    st["psi"] = 0.5 * torch.stack([(nx * dr + ny * di + nz * ur) * om + ur * op, (nx * di - ny * dr + nz * ui) * om + ui * op,
                                   (nx * ur - ny * ui - nz * dr) * om + dr * op, (nx * ui + ny * ur - nz * di) * om + di * op], 1)


def _sums(m, st, r):
    """ek, ep and sum v^2 per axis, per trap."""
    v2 = st["v"].square()
    u = m.potential(st["x"], st["t"])
    if r.mcwf:
        u = torch.where(st["up"], u, -u - 2.0 * m.mu[st["t"]] * m.B0)
    add = lambda w: torch.zeros(m.T, dtype=torch.float64, device=m.dev).index_add(0, st["t"], w)   # noqa: E731
    per = torch.stack([add(v2[:, k]) for k in range(3)], 1)
    return 0.5 * r.mass * per.sum(1), add(u), per


def exact(case, seed):
    if case["work"] in ("primitives", "group"):
        return None   # whole numbers; two groups hold too many atoms and steps
    r = _run_of(case, seed)
    trials = float(r.n_atoms) * case["steps"]
    if trials > (6e6 if case["form"] == "fp32" else 3e8) or trials * max(1, case["spin"]) > 3e8:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    m = _Model(r, dev)
    x, v, t = (c.to(dev) for c in (_sample(r, "cpu") if case["work"] == "restart" else _sample(r, dev)))
    n, fp64, calls = len(x), r.precision == "fp64", case["work"] == "calls"
    st = dict(x=x, v=v, t=t, id=torch.arange(n, device=dev), up=torch.ones(n, dtype=torch.bool, device=dev))
    st["a"] = m.accel(x, t, st["up"])
    if r.spin:
        b = m.field(x, t)[1]
        rs = 0.5 / (1 + b[:, :1]).sqrt()
        st["psi"] = b if not fp64 else rs * torch.stack([1 + b[:, 0] + b[:, 2], -b[:, 1], 1 + b[:, 0] - b[:, 2], b[:, 1]], 1)
        st["pops"] = torch.zeros((n, 2), dtype=torch.float64, device=dev)
    smax = torch.repeat_interleave(m.smax0, m.cells + 1)
    lost_pos, lost_vel = torch.zeros_like(x), torch.zeros_like(v)
    logs, temps = [], []

    def keep(at):
        for k in ("x", "v", "t", "id", "up", "a", "psi"):
            if k in st:
                st[k] = st[k][at]

    for step in range(case["steps"]):
        if step % r.lpc == 0:
            key, at = torch.sort(m.key(st["x"], st["t"]), stable=True)
            keep(at)
            m.collide(key, st["v"], smax, step)
            if r.mcwf:
                st["pops"][st["id"]] = _pops(m, st)
        if r.spin and fp64:
            _spinor_step(m, st, r, r.dt)
        st["v"] = st["v"] + 0.5 * st["a"] * r.dt
        if r.spin and not fp64:
            _bloch_step(m, st, r)
        st["x"] = st["x"] + st["v"] * r.dt
        if m.kind == "box":
            hw = m.hw[st["t"]]
            st["x"] = torch.where(st["x"] >= hw, st["x"] - 2 * hw, torch.where(st["x"] < -hw, st["x"] + 2 * hw, st["x"]))
        st["a"] = m.accel(st["x"], st["t"], st["up"])
        st["v"] = st["v"] + 0.5 * st["a"] * r.dt
        if calls:
            temps.append(float(r.mass / 3. / configs.KB * st["v"].square().sum() / len(st["v"])))
        lost = torch.zeros(len(st["x"]), dtype=torch.bool, device=dev)
        if r.spin_loss:
            b = m.field(st["x"], st["t"])[1]
            if fp64:
                ur, ui, dr, di = st["psi"].unbind(1)
                s = torch.stack([ur * dr + ui * di, ur * di - ui * dr, ur * ur + ui * ui - 0.5], 1)
            else:
                s = st["psi"]
            lost = (b * s).sum(1) < 0
        if r.energy_cut:
            e = 0.5 * r.mass * st["v"].square().sum(1) + m.potential(st["x"], st["t"])
            lost = lost | (e > m.cut_at(step + 1 if calls else step)[st["t"]])
        if r.spin_loss or r.energy_cut:
            lost_pos[st["id"][lost]], lost_vel[st["id"][lost]] = st["x"][lost], st["v"][lost]
            keep(~lost)
        if r.mcwf and (step + 1) % r.lpc == 0:
            _flip_and_decay(m, st, r, step // r.lpc + 1)
        if r.spin and fp64 and (step + 1) % r.lpc == 0:
            st["psi"] = st["psi"] / st["psi"].square().sum(1, True).sqrt()
        if not calls:
            logs.append(_sums(m, st, r))
    host = lambda c: c.cpu().numpy()   # noqa: E731
    now = _sums(m, st, r)
    if len(st["x"]) < n:   # rows past the alive atoms
        for k in ("x", "v", "psi"):
            if k in st:
                st[k] = torch.cat([st[k], torch.zeros((n - len(st[k]), st[k].shape[1]), dtype=torch.float64, device=dev)])
    out = dict(pos=host(st["x"]), vel=host(st["v"]), label=None)
    if r.spin:
        out["spin"] = host(st["psi"])
    if r.mcwf:
        out.update(up=None, cell=None, cell_count=None, cell_collisions=None,
                   lost_pos=host(lost_pos), lost_vel=host(lost_vel))
    if calls:
        return dict(temperature=np.array(temps), alive=None, **out)
    out["log"] = dict(ek=host(torch.stack([g[0] for g in logs])), ep=host(torch.stack([g[1] for g in logs])),
                      v2=host(torch.stack([g[2] for g in logs])), n_alive=None, n_evap=None, collisions=None)
    if case["work"] in ("restart", "sample"):
        ek, ep, v2 = now
        out["now"] = dict(ek=float(ek), ep=float(ep), v2=host(v2[0]), n_alive=None)
    return out
