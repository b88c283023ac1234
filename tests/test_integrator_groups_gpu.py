"""The integrator's lane groups at the edges of their layout: cell counts around
one cell to a wave, a full wave and the resident grid (the waves then hold 1 to
64/G cells), lone cells in a wave, and cells whose vectors leave the ordinary
range of the norm and of the pivot search (single species, zeros, values at the
ends of the exponent range, NaN and infinity).  Against the oracle: the same
status and work counters in every cell, and outputs to the parity bars, which
the device's exp/log/pow (1 ulp from glibc's) stay far below.  (A cell that
fails on non-finite values counts its right-hand sides in another way than the
oracle, which meets other NaN; its status is the same.)"""
import numpy as np
import pytest

from gpu_util import TOL_Y_ABS, compare_step, gpu_flat_step
from nrg_amd import capi, inputs
from nrg_amd import mechanism as M

pytestmark = pytest.mark.gpu

MECHS = {"KEROMNES": (), "KONNOV": ("KONNOV.txt", "KONNOV_THERMO.txt"),
         "TEREZA": ("TEREZA.txt", "TEREZA_THERMO.txt"), "ZHANG": ("ZHANG.txt", "ZHANG_THERMO.txt")}


def _same(eng, mech, st, dt):
    from oracle import Oracle
    stn = inputs.to_numpy(st)
    o = Oracle(mech).chem_cells(dt, stn["T"], stn["rho"], stn["Y"], nthreads=8)
    g = gpu_flat_step(eng, {k: v.to("cuda:0") for k, v in st.items()}, dt)
    assert np.array_equal(g["status"], o["status"])
    for k in ("nstep", "nfe", "nje"):
        assert np.array_equal(g[k], o[k]), k
    on = o["status"] == capi.NRG_CELL_OK
    assert compare_step({k: g[k][..., on] for k in ("Y_prod",)}, {k: o[k][..., on] for k in ("Y_prod",)},
                        stn["T"][on], stn["rho"][on], dt).max(initial=0.0) <= TOL_Y_ABS
    return g, o


@pytest.mark.parametrize("name,n", [("KEROMNES", n) for n in (1, 7, 1023, 1025, 3500, 8193)] +
                         [("KONNOV", 3), ("KONNOV", 1030), ("TEREZA", 2051)])
def test_cell_counts(name, n):
    from nrg_amd.solver import ChemistryStep
    mech = M.load_mechanism(*MECHS[name])
    st = inputs.flame_front_2d(mech, max(n, 64), 1, seed=n, width=max(n, 64) / 8.0)
    half = (max(n, 64) - n) // 2
    st = {k: v[..., half:half + n].contiguous() for k, v in st.items()}
    eng = ChemistryStep(mech)
    try:
        _same(eng, mech, st, 1e-7)
    finally:
        eng.close()


@pytest.mark.parametrize("name,analytic,n", [("KEROMNES", 0, (5 << 17) - 1), ("KEROMNES", 0, (5 << 17) + 37),
                                             ("KEROMNES", 1, (3 << 16) + 37), ("ZHANG", 0, 5 << 17),
                                             ("ZHANG", 1, 3 << 16), ("TEREZA", 1, (3 << 16) + 37),
                                             ("TEREZA", 0, (1 << 22) + 37)])
def test_one_cell_per_lane_equals_the_lane_groups(name, analytic, n):
    """Grids in stiffness order around the size from which a cell has a lane, bit
    for bit against the lane groups that the natural order takes at every size:
    fresh, burnt and igniting gas, gated cells, and cells with negative, tiny and
    missing species, at densities far from the ordinary."""
    import torch
    from nrg_amd.solver import ChemistryStep
    mech = M.load_mechanism(*MECHS[name])
    st = inputs.flame_front_2d(mech, n, 1, seed=5, width=n / 6.0, device="cuda:0")
    g = torch.Generator().manual_seed(n)
    pick = lambda k: torch.randint(0, n, (k,), generator=g).to("cuda:0")  # noqa: E731
    for s in range(mech.species_number):
        st["Y"][s, pick(64)] = 0.0
        st["Y"][s, pick(64)] = 1e-300
        st["Y"][s, pick(64)] *= -1.0
    st["rho"][pick(256)] *= 1e-6
    st["rho"][pick(256)] *= 1e-40
    bc = np.zeros(n, np.int8)
    bc[::97] = 1
    import nrg_amd.solver as solver_module
    real, codes, got = solver_module.check, [], []
    solver_module.check = lambda lib, rc: codes.append(rc)   # failed cells: the return codes are compared too
    try:
        for order in (capi.NRG_ORDER_NATURAL, capi.NRG_ORDER_STIFFNESS):
            eng = ChemistryStep(mech, capi.default_opts(cell_order=order, jacobian=analytic))
            try:
                got.append(gpu_flat_step(eng, st, 1e-7, bc=bc))
            finally:
                eng.close()
    finally:
        solver_module.check = real
    a, b = got
    half = len(codes) // 2                                   # each engine's calls, its set-up first
    assert codes[:half] == codes[half:] and set(codes) <= {capi.NRG_CHEM_OK, capi.NRG_CHEM_E_REPEATED_FAIL}
    for k in ("Y_prod", "Y_prod2", "E_f_prod", "status", "nstep", "nfe", "nje"):
        assert np.array_equal(a[k], b[k], equal_nan=True), k
    for k in ("cells_integrated", "nstep_sum", "nfe_sum", "nje_sum", "ncorr_sum", "nstep_max", "nfe_max"):
        assert getattr(a["stats"], k) == getattr(b["stats"], k), k
    assert (a["status"] == capi.NRG_CELL_OK).sum() > n // 4 and (a["status"] == capi.NRG_CELL_GATED).any()


def test_cells_out_of_the_ordinary_range(mech):
    from nrg_amd.solver import ChemistryStep
    st = inputs.flame_front_2d(mech, 64, 4, seed=9)
    T, rho, Y = st["T"], st["rho"], st["Y"]
    hot = np.where(T.numpy() > 1200.0)[0]
    S = mech.species_number
    i = iter(hot)
    for s in range(S):                         # one species alone
        k = next(i)
        Y[:, k] = 0.0
        Y[s, k] = 1.0
    for v in (0.0, 1e-300, 1e-12):             # next to nothing
        Y[:, next(i)] = v
    for v in (1e20, 1e40, 1e120, 1e-30, 1e-200, 1e-320, 0.0, float("inf"), float("nan")):
        rho[next(i)] = v
    for v in (float("nan"), float("inf"), -1e-3):
        for s in (0, 3, 6):
            Y[s, next(i)] = v
    eng = ChemistryStep(mech)
    from oracle import Oracle
    try:
        stn = inputs.to_numpy(st)
        o = Oracle(mech).chem_cells(1e-7, stn["T"], stn["rho"], stn["Y"], nthreads=8)
        import nrg_amd.solver as solver_module
        real, codes = solver_module.check, []
        solver_module.check = lambda lib, rc: codes.append(rc)
        try:
            g = gpu_flat_step(eng, {k: v.to("cuda:0") for k, v in st.items()}, 1e-7)
        finally:
            solver_module.check = real
        assert codes == [capi.NRG_CHEM_E_REPEATED_FAIL if (o["status"] == capi.NRG_CELL_REPEATED_FAIL).any()
                         else capi.NRG_CHEM_OK]
        assert np.array_equal(g["status"], o["status"])
        ok = o["status"] == capi.NRG_CELL_OK
        for k in ("nstep", "nfe", "nje"):
            assert np.array_equal(g[k][ok], o[k][ok]), k
        on = (o["status"] == capi.NRG_CELL_OK) & np.isfinite(o["Y_prod"]).all(0) & (stn["rho"] > 0)
        assert on.sum() > 100
        assert compare_step({"Y_prod": g["Y_prod"][:, on]}, {"Y_prod": o["Y_prod"][:, on]}, stn["T"][on],
                            stn["rho"][on], 1e-7).max() <= TOL_Y_ABS
    finally:
        eng.close()
