"""Learned chemistry step: a BF16 MFMA perceptron (include/nrg_mlp.h) trained
on split-step increments generated by the FP64 integrator, gated by element
and energy conservation and backed by FP64 fallback (include/nrg_surrogate.h).

Network: 12 inputs (T, ln p, ln(Y_s + y_floor) for the 9 species, ln dt) ->
4 x 256 GELU -> 10 outputs (dT, dY_1..dY_9) of one split step (chemistry +
closure).  The features are computed exactly as the device's featurize
kernel computes them, so training and inference see the same inputs.

Nothing here falls back to the CPU: every array lives on the GPU and every
kernel is the library's own (training included).
"""
from __future__ import annotations

import ctypes as C
import math
import time

import numpy as np

from . import capi
from .capi import check, load_library
from .mechanism import P_ATM, element_matrix

N_HIDDEN = 256
N_LAYERS = 4
Y_FLOOR = 1.0e-12


def _torch():
    import torch
    return torch


# ---- the network handle -----------------------------------------------------------

class MLP:
    """One nrg_mlp handle (BF16 MFMA forward/backward/Adam on the GPU)."""

    def __init__(self, n_in, n_out, hidden=N_HIDDEN, layers=N_LAYERS, device_index=0):
        self.lib = load_library()
        h = C.c_void_p()
        check(self.lib, self.lib.nrg_mlp_create(n_in, hidden, layers, n_out, device_index,
                                                C.byref(h)))
        self.h = h
        self.n_in, self.n_out, self.hidden, self.layers = n_in, n_out, hidden, layers

    def close(self):
        if self.h:
            self.lib.nrg_mlp_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    @property
    def num_params(self):
        return int(self.lib.nrg_mlp_num_params(self.h))

    def set_params(self, p):
        p = np.ascontiguousarray(p, dtype=np.float32)
        assert p.size == self.num_params
        check(self.lib, self.lib.nrg_mlp_set_params(self.h, p.ctypes.data))

    def get_params(self):
        p = np.empty(self.num_params, dtype=np.float32)
        check(self.lib, self.lib.nrg_mlp_get_params(self.h, p.ctypes.data))
        return p

    def forward(self, x):
        """Fused inference kernel; x: cuda float32 (n, n_in)."""
        torch = _torch()
        x = x.contiguous()
        y = torch.empty((x.shape[0], self.n_out), dtype=torch.float32, device=x.device)
        torch.cuda.synchronize()
        check(self.lib, self.lib.nrg_mlp_forward_dev(self.h, x.shape[0], x.data_ptr(), y.data_ptr()))
        return y

    def grad(self, x, t, w=None):
        """(gradient vector, loss, training-path forward) of the weighted MSE."""
        torch = _torch()
        x, t = x.contiguous(), t.contiguous()
        g = torch.empty(self.num_params, dtype=torch.float32, device=x.device)
        loss = torch.empty(1, dtype=torch.float32, device=x.device)   # written, not added to
        y = torch.empty((x.shape[0], self.n_out), dtype=torch.float32, device=x.device)
        torch.cuda.synchronize()
        check(self.lib, self.lib.nrg_mlp_grad_dev(self.h, x.shape[0], x.data_ptr(), t.data_ptr(),
                                                  w.data_ptr() if w is not None else None,
                                                  g.data_ptr(), loss.data_ptr(), y.data_ptr()))
        return g, loss, y

    def train_step(self, x, t, lr, w=None, loss=None):
        check(self.lib, self.lib.nrg_mlp_train_step_dev(
            self.h, x.shape[0], x.data_ptr(), t.data_ptr(),
            w.data_ptr() if w is not None else None, float(lr),
            loss.data_ptr() if loss is not None else None))


def init_params(n_in, n_out, hidden=N_HIDDEN, layers=N_LAYERS, seed=0):
    """He-normal hidden weights, small output weights, zero biases (packed order)."""
    rng = np.random.default_rng(seed)
    parts = []
    fan = [n_in] + [hidden] * layers + [n_out]
    for i in range(layers + 1):
        std = math.sqrt(2.0 / fan[i]) if i < layers else 0.1 / math.sqrt(fan[i])
        parts.append(rng.normal(0.0, std, size=(fan[i], fan[i + 1])).astype(np.float32).ravel())
        parts.append(np.zeros(fan[i + 1], dtype=np.float32))
    return np.concatenate(parts)


# ---- features and normalisation ----------------------------------------------------

def raw_features(T, p, Y, dt, y_floor=Y_FLOOR):
    """f = (T, ln p, ln(Y_s + y_floor), ln dt) as float32, as featurize_kernel computes it.
    T, p: (n,) float64; Y: (S, n) float64; dt: float or (n,) float64.  Returns (n, S+3)."""
    torch = _torch()
    n = T.shape[0]
    S = Y.shape[0]
    f = torch.empty((n, S + 3), dtype=torch.float32, device=T.device)
    f[:, 0] = T.float()
    f[:, 1] = torch.log(p).float()
    f[:, 2:2 + S] = torch.log(Y.float().t() + y_floor)
    if isinstance(dt, (float, int)):
        f[:, S + 2] = float(np.float32(math.log(dt)))
    else:
        f[:, S + 2] = torch.log(dt).float()
    return f


class Normalizer:
    """x = (f - in_shift) * in_scale; increment = y * out_scale + out_shift."""

    def __init__(self, in_shift, in_scale, out_shift, out_scale, y_floor=Y_FLOOR):
        self.in_shift = np.asarray(in_shift, dtype=np.float32)
        self.in_scale = np.asarray(in_scale, dtype=np.float32)
        self.out_shift = np.asarray(out_shift, dtype=np.float32)
        self.out_scale = np.asarray(out_scale, dtype=np.float32)
        self.y_floor = float(y_floor)

    @classmethod
    def fit(cls, feats, incr, y_floor=Y_FLOOR):
        f = feats.double()
        d = incr.double()
        fs = f.std(0).clamp_min(1e-6)
        ds = d.std(0).clamp_min(1e-12)
        return cls(f.mean(0).cpu().numpy(), (1.0 / fs).cpu().numpy(),
                   d.mean(0).cpu().numpy(), ds.cpu().numpy(), y_floor)

    def x(self, feats):
        torch = _torch()
        sh = torch.as_tensor(self.in_shift, device=feats.device)
        sc = torch.as_tensor(self.in_scale, device=feats.device)
        return ((feats - sh) * sc).contiguous()

    def y(self, incr):
        torch = _torch()
        sh = torch.as_tensor(self.out_shift, device=incr.device, dtype=torch.float64)
        sc = torch.as_tensor(self.out_scale, device=incr.device, dtype=torch.float64)
        return ((incr.double() - sh) / sc).float().contiguous()

    def incr(self, y):
        torch = _torch()
        sh = torch.as_tensor(self.out_shift, device=y.device, dtype=torch.float64)
        sc = torch.as_tensor(self.out_scale, device=y.device, dtype=torch.float64)
        return y.double() * sc + sh

    def struct(self):
        s = capi.NrgSurrogateNorm()
        for i, v in enumerate(self.in_shift):
            s.in_shift[i] = float(v)
        for i, v in enumerate(self.in_scale):
            s.in_scale[i] = float(v)
        for i, v in enumerate(self.out_shift):
            s.out_shift[i] = float(v)
        for i, v in enumerate(self.out_scale):
            s.out_scale[i] = float(v)
        s.y_floor = self.y_floor
        return s


def gate_struct(mech, t_range=(300.0, 2800.0), p_range=(0.5 * P_ATM, 5.0 * P_ATM),
                dt_range=(1e-8, 1e-6), elem_tol=0.05, elem_floor=1e-3, y_neg_tol=1e-5,
                energy_tol=5.0, dT_max=1e9, dT_freeze=0.0, dY_freeze=0.0, rate_tol=0.0,
                screen=capi.NRG_SUR_SCREEN_NONE, screen_fp64=False):
    g = capi.NrgSurrogateGate()
    g.screen = int(screen)
    g.screen_fp64 = 1 if screen_fp64 else 0
    g.t_min, g.t_max = t_range
    g.p_min, g.p_max = p_range
    g.dt_min, g.dt_max = dt_range[0] * (1 - 1e-9), dt_range[1] * (1 + 1e-9)
    g.elem_tol, g.elem_floor, g.y_neg_tol, g.energy_tol = elem_tol, elem_floor, y_neg_tol, energy_tol
    g.dT_max = dT_max
    g.dT_freeze, g.dY_freeze = dT_freeze, dY_freeze
    g.rate_tol = rate_tol
    E = element_matrix(mech.species_names)
    g.n_elements = E.shape[0]
    for e in range(E.shape[0]):
        for s in range(E.shape[1]):
            g.elements[e][s] = float(E[e, s])
    return g


# ---- training data from the FP64 integrator ----------------------------------------

def generate_pairs(engine, mech, n_traj, n_steps, seed=11, device="cuda:0", groups=16,
                   dt_range=(1e-8, 1e-6), log=None, **state_kw):
    """Split-step pairs (state, dt) -> (dT, dY) from FP64 trajectories.

    n_traj cells in `groups` groups, each group with its own dt drawn
    log-uniformly from dt_range, are advanced n_steps split steps (chemistry
    step + source application + e->T) by the library's FP64 kernels; every
    non-gated cell-step is one pair.  Returns dict of cuda tensors: T, p (n,),
    Y (S, n), dt (n,), dT (n,), dY (S, n), all float64."""
    torch = _torch()
    from . import inputs
    S = mech.species_number
    rng = np.random.default_rng(seed)
    out = {k: [] for k in ("T", "p", "Y", "dt", "dT", "dY")}
    per = n_traj // groups
    t0 = time.time()
    for gi in range(groups):
        dt = float(math.exp(rng.uniform(math.log(dt_range[0]), math.log(dt_range[1]))))
        st = inputs.training_states(mech, per, seed=seed * 1000 + gi, device=device, **state_kw)
        T, p, rho, Y = st["T"].clone(), st["p"].clone(), st["rho"], st["Y"].clone()
        grid = capi.flat_grid(per)
        E = torch.empty(per, dtype=torch.float64, device=device)
        engine.energy_from_temperature_dev(grid, T.data_ptr(), [Y[s].data_ptr() for s in range(S)],
                                           E.data_ptr())
        Yp = torch.zeros((S, per), dtype=torch.float64, device=device)
        Yp2 = torch.zeros_like(Yp)
        Ef = torch.zeros(per, dtype=torch.float64, device=device)
        for _ in range(n_steps):
            live = T >= engine.opts.t_gate
            T0, p0, Y0 = T.clone(), p.clone(), Y.clone()
            engine.step_dev(grid, dt, T.data_ptr(), rho.data_ptr(), [Y[s].data_ptr() for s in range(S)],
                            [Yp[s].data_ptr() for s in range(S)], [Yp2[s].data_ptr() for s in range(S)],
                            Ef.data_ptr())
            engine.closure_dev(grid, dt, rho.data_ptr(), Ef.data_ptr(),
                               [Yp[s].data_ptr() for s in range(S)], E.data_ptr(),
                               [Y[s].data_ptr() for s in range(S)], T.data_ptr(), p=p.data_ptr())
            torch.cuda.synchronize()
            out["T"].append(T0[live])
            out["p"].append(p0[live])
            out["Y"].append(Y0[:, live])
            out["dt"].append(torch.full((int(live.sum()),), dt, dtype=torch.float64, device=device))
            out["dT"].append((T - T0)[live])
            out["dY"].append((Y - Y0)[:, live])
        if log:
            log("pairs: group %d/%d dt=%.3g done (%.1f s)" % (gi + 1, groups, dt, time.time() - t0))
    cat = {k: torch.cat(v, dim=-1) for k, v in out.items()}
    return cat


def pair_tensors(pairs, norm=None):
    """Network inputs/targets of a pair set: (features, increments (n, 1+S))."""
    torch = _torch()
    f = raw_features(pairs["T"], pairs["p"], pairs["Y"], pairs["dt"], Y_FLOOR)
    d = torch.cat([pairs["dT"].view(-1, 1), pairs["dY"].t()], dim=1)
    return f, d


def train(mlp, x, y, epochs=10, batch=4096, lr=1e-3, lr_min=2e-5, seed=0, log=None,
          log_every=2000, w=None):
    """Adam with cosine learning-rate decay on normalised (x, y), all on the GPU."""
    torch = _torch()
    n = x.shape[0]
    steps_per = n // batch
    total = epochs * steps_per
    g = torch.Generator(device=x.device)
    g.manual_seed(seed)
    loss = torch.zeros(1, dtype=torch.float32, device=x.device)
    hist = []
    k = 0
    t0 = time.time()
    for ep in range(epochs):
        perm = torch.randperm(n, generator=g, device=x.device)
        run = 0.0
        for i in range(steps_per):
            idx = perm[i * batch:(i + 1) * batch]
            xb = x[idx].contiguous()
            yb = y[idx].contiguous()
            lr_k = lr_min + 0.5 * (lr - lr_min) * (1.0 + math.cos(math.pi * k / max(1, total)))
            loss.zero_()
            torch.cuda.synchronize()
            mlp.train_step(xb, yb, lr_k, w=w, loss=loss)
            k += 1
            if (k % log_every == 0) or i == steps_per - 1:
                lv = float(loss.item())
                hist.append((k, lv))
                if log:
                    log("train: epoch %d step %d/%d loss %.4e lr %.2e (%.1f s)"
                        % (ep, k, total, lv, lr_k, time.time() - t0))
    return hist


def evaluate(mlp, norm, feats, incr, major=(0, 1, 6)):
    """Errors of the network's increments against the FP64 ones (physical units)."""
    torch = _torch()
    pred = norm.incr(mlp.forward(norm.x(feats)))
    err = (pred - incr).abs()
    base = incr.abs()
    maj = [1 + s for s in major]
    return {
        "n": int(feats.shape[0]),
        "max_abs_dT": float(err[:, 0].max()),
        "p99_abs_dT": float(torch.quantile(err[:, 0].float()[:1_000_000], 0.99)),
        "max_abs_dY_major": float(err[:, maj].max()),
        "p99_abs_dY_major": float(torch.quantile(err[:, maj].float().max(dim=1).values[:1_000_000], 0.99)),
        "zero_model_max_abs_dY_major": float(base[:, maj].max()),
        "zero_model_max_abs_dT": float(base[:, 0].max()),
        "rmse_dY_major": float(err[:, maj].pow(2).mean().sqrt()),
        "zero_model_rmse_dY_major": float(base[:, maj].pow(2).mean().sqrt()),
    }


# ---- persistence ---------------------------------------------------------------------

def save(path, mlp, norm, meta=None):
    np.savez(path, params=mlp.get_params(), in_shift=norm.in_shift, in_scale=norm.in_scale,
             out_shift=norm.out_shift, out_scale=norm.out_scale,
             y_floor=np.float64(norm.y_floor),
             dims=np.array([mlp.n_in, mlp.hidden, mlp.layers, mlp.n_out], dtype=np.int64),
             meta=np.array(repr(meta or {})))


def load(path, device_index=0):
    z = np.load(path, allow_pickle=False)
    n_in, hidden, layers, n_out = (int(v) for v in z["dims"])
    mlp = MLP(n_in, n_out, hidden, layers, device_index)
    mlp.set_params(z["params"])
    norm = Normalizer(z["in_shift"], z["in_scale"], z["out_shift"], z["out_scale"],
                      float(z["y_floor"]))
    return mlp, norm


# ---- the solver with the learned step ------------------------------------------------

class SurrogateChemistry:
    """chemical_kinetics_solver with the learned step: same fields, same outputs,
    FP64 fallback for every cell the gate rejects.

    `engine`: the handle the learned step runs on (default: the solver's).  A
    handle created with other integrator options (a looser eps, the analytic
    Jacobian) gives the fallback those options; the screen and the gate do
    not depend on them."""

    def __init__(self, solver, mlp, norm, gate, engine=None):
        self.solver = solver
        self.engine = engine if engine is not None else solver.engine
        self.mlp, self.norm, self.gate = mlp, norm, gate
        self.norm_s = norm.struct() if norm is not None else None
        self.last = None

    def solve_chemical_kinetics(self, time_step):
        from .solver import _order_after_torch
        s = self.solver
        m = s.manager
        eng = self.engine
        _order_after_torch()
        st = capi.NrgSurrogateStats()
        rc = eng.lib.nrg_chem_surrogate_step_dev(
            eng.h, self.mlp.h if self.mlp is not None else None,
            C.byref(self.norm_s) if self.norm_s is not None else None, C.byref(self.gate),
            C.byref(m.grid),
            float(time_step), s.T.ptr(), s.p.ptr(), s.rho.ptr(), capi.ptr_array(s.Y.ptrs()),
            s.boundary.ptr(), capi.ptr_array(s.Y_prod.ptrs()), capi.ptr_array(s.Y_prod2.ptrs()),
            s.E_f_prod.ptr(), s.cell_status.ptr(), C.byref(st))
        self.last = st
        check(eng.lib, rc)
        return st

    def apply_split_sources(self, time_step):
        self.solver.apply_split_sources(time_step)


# ---- gate calibration -------------------------------------------------------------------

def _flat_outputs(n, S, device):
    torch = _torch()
    return dict(Yp=torch.zeros((S, n), dtype=torch.float64, device=device),
                Yp2=torch.zeros((S, n), dtype=torch.float64, device=device),
                Ef=torch.zeros(n, dtype=torch.float64, device=device),
                status=torch.zeros(n, dtype=torch.int32, device=device))


def surrogate_step_flat(engine, mlp, norm_s, gate, T, p, rho, Y, dt, out):
    """nrg_chem_surrogate_step_dev on a flat list of cells (device tensors)."""
    from .solver import _order_after_torch
    S = Y.shape[0]
    n = T.shape[0]
    _order_after_torch()
    st = capi.NrgSurrogateStats()
    rc = engine.lib.nrg_chem_surrogate_step_dev(
        engine.h, mlp.h if mlp is not None else None,
        C.byref(norm_s) if norm_s is not None else None, C.byref(gate),
        C.byref(capi.flat_grid(n)), float(dt),
        T.data_ptr(), p.data_ptr(), rho.data_ptr(), capi.ptr_array([Y[s].data_ptr() for s in range(S)]),
        None, capi.ptr_array([out["Yp"][s].data_ptr() for s in range(S)]),
        capi.ptr_array([out["Yp2"][s].data_ptr() for s in range(S)]), out["Ef"].data_ptr(),
        out["status"].data_ptr(), C.byref(st))
    check(engine.lib, rc)
    return st


def calibration_states(engine, mech, n, dts=(1e-8, 1e-7, 1e-6), snap_steps=(0, 3, 8), seed=99,
                       device="cuda:0", **state_kw):
    """States met along FP64 split-step trajectories: [(dt, T, p, rho, Y)]."""
    torch = _torch()
    from . import inputs
    S = mech.species_number
    out = []
    for di, dt in enumerate(dts):
        st = inputs.training_states(mech, n, seed=seed + di, device=device, **state_kw)
        T, p, rho, Y = st["T"].clone(), st["p"].clone(), st["rho"].clone(), st["Y"].clone()
        grid = capi.flat_grid(n)
        E = torch.empty(n, dtype=torch.float64, device=device)
        engine.energy_from_temperature_dev(grid, T.data_ptr(), [Y[s].data_ptr() for s in range(S)],
                                           E.data_ptr())
        o = _flat_outputs(n, S, device)
        for k in range(max(snap_steps) + 1):
            if k in snap_steps:
                out.append((dt, T.clone(), p.clone(), rho.clone(), Y.clone()))
            engine.step_dev(grid, dt, T.data_ptr(), rho.data_ptr(), [Y[s].data_ptr() for s in range(S)],
                            [o["Yp"][s].data_ptr() for s in range(S)],
                            [o["Yp2"][s].data_ptr() for s in range(S)], o["Ef"].data_ptr())
            engine.closure_dev(grid, dt, rho.data_ptr(), o["Ef"].data_ptr(),
                               [o["Yp"][s].data_ptr() for s in range(S)], E.data_ptr(),
                               [Y[s].data_ptr() for s in range(S)], T.data_ptr(), p=p.data_ptr())
        torch.cuda.synchronize()
    return out


def calibrate_gate(engine, mech, mlp, norm, states, target_dY=1e-4, major=(0, 1, 6),
                   dT_maxes=(0.25, 0.5, 1.0, 2.0, 5.0, 10.0, 20.0, 50.0, 1e9),
                   energy_tols=(0.1, 0.25, 0.5, 1.0, 2.0, 5.0), elem_tol=0.05, elem_floor=1e-2,
                   log=None):
    """Gate thresholds that leave the FP64 fallback the least work (its NFE)
    while every accepted cell of every calibration state set stays within
    target_dY (max abs one-step error of the major species against the FP64
    step on the same state)."""
    torch = _torch()
    S = mech.species_number
    norm_s = norm.struct()
    refs = []
    for dt, T, p, rho, Y in states:
        n = T.shape[0]
        o = _flat_outputs(n, S, T.device)
        st = engine.step_dev(capi.flat_grid(n), dt, T.data_ptr(), rho.data_ptr(),
                             [Y[s].data_ptr() for s in range(S)],
                             [o["Yp"][s].data_ptr() for s in range(S)],
                             [o["Yp2"][s].data_ptr() for s in range(S)], o["Ef"].data_ptr())
        refs.append((o["Yp"].clone(), int(st.nfe_sum)))
    results = []
    for dm in dT_maxes:
        for et in energy_tols:
            gate = gate_struct(mech, energy_tol=et, elem_tol=elem_tol, elem_floor=elem_floor,
                               dT_max=dm)
            worst, acc, tot, nfe, nfe_all = 0.0, 0, 0, 0, 0
            per_dt = {}
            for (dt, T, p, rho, Y), (ref, ref_nfe) in zip(states, refs):
                n = T.shape[0]
                o = _flat_outputs(n, S, T.device)
                st = surrogate_step_flat(engine, mlp, norm_s, gate, T, p, rho, Y, dt, o)
                torch.cuda.synchronize()
                a = o["status"] == capi.NRG_CELL_SURROGATE
                w = 0.0
                if bool(a.any()):
                    w = float(((o["Yp"][list(major)][:, a] - ref[list(major)][:, a]).abs() * dt
                               / rho[a]).max())
                worst = max(worst, w)
                live = int((T >= engine.opts.t_gate).sum())
                acc += int(a.sum())
                tot += live
                nfe += int(st.fallback.nfe_sum)
                nfe_all += ref_nfe
                d = per_dt.setdefault("%.0e" % dt, [0.0, 0, 0])
                d[0] = max(d[0], w)
                d[1] += int(a.sum())
                d[2] += live
            r = dict(dT_max=dm, energy_tol=et, elem_tol=elem_tol, elem_floor=elem_floor,
                     worst_dY=worst, accepted=acc / max(1, tot),
                     fallback_nfe_frac=nfe / max(1, nfe_all),
                     per_dt={k: {"worst_dY": v[0], "accepted": v[1] / max(1, v[2])}
                             for k, v in per_dt.items()})
            results.append(r)
            if log:
                log("calibrate: dT_max %.3g energy_tol %.2f -> accepted %.4f fallback NFE %.4f "
                    "worst %.2e" % (dm, et, r["accepted"], r["fallback_nfe_frac"], worst))
    ok = [r for r in results if r["worst_dY"] <= target_dY]
    best = (min(ok, key=lambda r: r["fallback_nfe_frac"]) if ok
            else min(results, key=lambda r: r["worst_dY"]))
    return best, results


GATE_KEYS = ("dT_max", "dT_freeze", "dY_freeze", "energy_tol", "elem_tol", "elem_floor",
             "rate_tol")


def set_gate(path_in, path_out, **gate_kw):
    """Rewrite (or add) the gate thresholds stored with a trained network
    (GATE_KEYS), keeping the network, normalizer and metadata."""
    with np.load(path_in, allow_pickle=False) as z:
        arrays = {k: z[k] for k in z.files}
    for k, v in gate_kw.items():
        if k not in GATE_KEYS:
            raise KeyError("no gate threshold %r (known: %s)" % (k, ", ".join(GATE_KEYS)))
        arrays["gate_" + k] = np.float64(v)
    np.savez(path_out, **arrays)


def save_with_gate(path, mlp, norm, gate_kw, meta=None):
    np.savez(path, params=mlp.get_params(), in_shift=norm.in_shift, in_scale=norm.in_scale,
             out_shift=norm.out_shift, out_scale=norm.out_scale,
             y_floor=np.float64(norm.y_floor),
             dims=np.array([mlp.n_in, mlp.hidden, mlp.layers, mlp.n_out], dtype=np.int64),
             gate_dT_max=np.float64(gate_kw["dT_max"]),
             gate_dT_freeze=np.float64(gate_kw.get("dT_freeze", 0.0)),
             gate_dY_freeze=np.float64(gate_kw.get("dY_freeze", 0.0)),
             gate_energy_tol=np.float64(gate_kw["energy_tol"]),
             gate_elem_tol=np.float64(gate_kw["elem_tol"]),
             gate_elem_floor=np.float64(gate_kw["elem_floor"]),
             meta=np.array(repr(meta or {})))
