"""Field passes on either side of the sizes at which they change their way: above
them the per-cell passes store past the caches, and the host-pointer step copies
field by field instead of through pinned memory.  A cell's result does not depend
on its neighbours, so each large pass has to give, bit for bit, what its cells give
in passes small enough for the other way."""
import ctypes as C

import numpy as np
import pytest

from nrg_amd import capi, inputs

pytestmark = pytest.mark.gpu

# just above: 320 MiB of 29 fields, of 37 fields, 128 MiB of 23 to 29 fields
ABOVE = {"table": 1446400 + 333, "closure": 1133600 + 333, "low_mach": 729500 + 333}


def _fields(mech, n, seed):
    import torch
    st = inputs.ignition_mix(mech, n, seed=seed, device="cuda:0", frac_window=0.5)
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    bc = (torch.rand(n, generator=g, device="cuda:0") < 0.05).to(torch.int8)
    rnd = lambda scale: scale * (torch.rand(n, generator=g, device="cuda:0", dtype=torch.float64) - 0.5)  # noqa: E731
    return st["T"], st["rho"], [y.contiguous() for y in st["Y"]], bc, rnd


def _run(engine, kind, T, rho, Y, bc, src, lo, hi):
    import torch
    S, n = len(Y), hi - lo
    cut = lambda v: v[lo:hi].clone()  # noqa: E731
    T, rho, Y, bc = cut(T), cut(rho), [cut(y) for y in Y], cut(bc)
    E, W = [cut(v) for v in src[:S]], cut(src[S])
    new = lambda: torch.full((n,), -7.0, dtype=torch.float64, device="cuda:0")  # noqa: E731
    p = lambda v: [x.data_ptr() for x in v] if isinstance(v, list) else v.data_ptr()  # noqa: E731
    grid = capi.flat_grid(n)
    if kind == "table":
        Yp, Yp2, Ef = [new() for _ in Y], [new() for _ in Y], new()
        st = torch.full((n,), -1, dtype=torch.int32, device="cuda:0")
        engine.table_step_dev(grid, 1e-7, p(T), p(rho), p(Y), p(Yp), p(Yp2), p(Ef), bc=p(bc), status=p(st))
        out = Yp + Yp2 + [Ef, st]
    elif kind == "closure":
        Ef, pr = new(), new()
        engine.energy_from_temperature_dev(grid, p(T), p(Y), p(Ef))
        engine.closure_dev(grid, 1e-7, p(rho), p(W), p(E), p(Ef), p(Y), p(T), p(pr), bc=p(bc))
        out = Y + [Ef, T, pr]
    else:
        ps, po, mmm, div, ro = [new() for _ in range(5)]
        ps.fill_(101325.0)
        opt = {k: new() for k in ("p", "mixture_cp", "gamma", "h_s", "v_s", "e_i", "E_f")}
        Yo = [new() for _ in Y]
        engine.low_mach_state_equation_dev(grid, 1e-5, True, p(rho), p(Y), p(W), p(ps), p(po), p(T), p(mmm),
                                           v=[p(W)], bc=p(bc), **{k: p(v) for k, v in opt.items()})
        engine.low_mach_species_dev(grid, 1e-5, False, p(rho), p(Y), p(ro), p(Yo), Y_prod_chem=p(E), bc=p(bc))
        mmm = torch.where(bc != 0, torch.ones_like(mmm), mmm)
        engine.low_mach_chem_divergence_dev(grid, p(rho), p(T), p(Y), p(mmm), p(W), p(E), p(div), bc=p(bc))
        out = [ps, po, T, mmm, div, ro] + Yo + list(opt.values())
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("kind", sorted(ABOVE))
def test_a_large_pass_equals_its_parts(engine, mech, kind):
    import torch
    n = ABOVE[kind]
    T, rho, Y, bc, rnd = _fields(mech, n, 11)
    src = [rnd(1e3) for _ in Y] + [rnd(1e8)]
    engine.set_table(np.linspace(320.0, 2600.0, 60), np.random.default_rng(1).normal(size=(len(Y), 60)) * 1e-3)
    whole = _run(engine, kind, T, rho, Y, bc, src, 0, n)
    cut = n // 2 + 17
    parts = [_run(engine, kind, T, rho, Y, bc, src, a, b) for a, b in ((0, cut), (cut, n))]
    for k, w in enumerate(whole):
        assert torch.equal(w.view(torch.int64 if w.dtype == torch.float64 else w.dtype),
                           torch.cat([q[k] for q in parts]).view(torch.int64 if w.dtype == torch.float64 else w.dtype)), k


@pytest.mark.parametrize("n,with_bc,with_status", [(1, True, True), (4099, False, True), (4099, True, False),
                                                   (138000, True, True)])
def test_host_fields_equal_device_fields(engine, mech, n, with_bc, with_status):
    """One cell, and either side of 32 MiB of fields; without markers or status too."""
    import torch
    T, rho, Y, bc, _ = _fields(mech, max(n, 64), 5)
    T, rho, Y, bc = T[:n], rho[:n], [y[:n].contiguous() for y in Y], bc[:n].contiguous()
    S, grid = len(Y), capi.flat_grid(n)
    dev = [torch.full((n,), 3.0 + k, dtype=torch.float64, device="cuda:0") for k in range(2 * S + 1)]
    st = torch.full((n,), -1, dtype=torch.int32, device="cuda:0")
    ptr = lambda v: [x.data_ptr() for x in v]  # noqa: E731
    engine.step_dev(grid, 1e-7, T.data_ptr(), rho.data_ptr(), ptr(Y), ptr(dev[:S]), ptr(dev[S:2 * S]),
                    dev[2 * S].data_ptr(), bc=bc.data_ptr() if with_bc else None, status=st.data_ptr())
    torch.cuda.synchronize()
    host = [np.full(n, 3.0 + k) for k in range(2 * S + 1)]
    sth = np.full(n, -1, np.int32)
    Th, rh, Yh, bh = T.cpu().numpy(), rho.cpu().numpy(), [y.cpu().numpy() for y in Y], bc.cpu().numpy()
    at = lambda v: [x.ctypes.data for x in v]  # noqa: E731
    stats = capi.NrgChemStats()
    capi.check(engine.lib, engine.lib.nrg_chem_step(
        engine.h, C.byref(grid), 1e-7, Th.ctypes.data, None, rh.ctypes.data, capi.ptr_array(at(Yh)),
        bh.ctypes.data if with_bc else None, capi.ptr_array(at(host[:S])), capi.ptr_array(at(host[S:2 * S])),
        host[2 * S].ctypes.data, sth.ctypes.data if with_status else None, C.byref(stats)))
    for a, b in zip(dev, host):
        assert np.array_equal(a.cpu().numpy().view(np.int64), b.view(np.int64))
    assert np.array_equal(sth, st.cpu().numpy() if with_status else np.full(n, -1))
