"""Operands over the whole exponent range.  Concentrations, densities, time steps
and table entries come from the caller; wherever the kernels divide without the
scaling steps of an FP64 division they have to know that the operands allow it,
since a numerator under 2^-969 would lose its last bit and an overflowing
quotient its infinity.  Nothing here has a tolerance: the table step and the
output assembly are quotients that the oracle and numpy form as well."""
import numpy as np
import pytest

from gpu_util import gpu_flat_step
from nrg_amd import capi, inputs
from nrg_amd import mechanism as M
from test_chem_table_gpu import _gpu_table_step

pytestmark = pytest.mark.gpu
S = 9


def _same(a, b):
    return np.array_equal(a, b, equal_nan=True) and np.array_equal(np.signbit(a) & (a == a), np.signbit(b) & (b == b))


@pytest.mark.parametrize("dt", [1e-7, 1e-300, 1e300, 5e-324])
@pytest.mark.parametrize("lo,hi", [(-323, -280), (250, 308), (-323, 308)])
def test_table_step(engine, oracle, lo, hi, dt):
    rng = np.random.default_rng(hi - lo)
    n = 5000
    T_t = np.sort(rng.uniform(320.0, 2600.0, 64))
    T_t[10] = np.nextafter(T_t[9], 1e4)                       # an interval of one ulp
    dC = rng.choice([-1.0, 1.0], (S, 64)) * 10.0 ** rng.uniform(lo, hi, (S, 64))
    dC[:, ::7] = 0.0
    T = rng.uniform(300.0, 2700.0, n)
    T[:64] = T_t
    Y = rng.uniform(0.0, 1.0, (S, n))
    engine.set_table(T_t, dC)
    with np.errstate(all="ignore"):
        o = oracle.table_cells(dt, T_t, dC, T, Y, Y_prod2=np.full((S, n), -7.0))
    g = _gpu_table_step(engine, dt, T, np.ones(n), Y, np.zeros(n, np.int8))
    for k in ("Y_prod", "Y_prod2", "E_f_prod"):
        assert _same(g[k], o[k]), k


@pytest.mark.parametrize("order,n", [(capi.NRG_ORDER_NATURAL, 4096), (capi.NRG_ORDER_STIFFNESS, 5 << 17)])
@pytest.mark.parametrize("dt", [1e-7, 1e-200, 1e-290, 1e-300])
def test_output_assembly(mech, dt, order, n):
    """Y_prod and E_f_prod are the quotients by dt of what Y_prod2 holds
    (chemical_kinetics_solver.f90:329-338), in cells with trace species, a cell to
    a group of lanes and a cell to a lane."""
    from nrg_amd.solver import ChemistryStep
    from oracle import Oracle
    o = Oracle(mech)
    st = inputs.flame_front_2d(mech, n, 1, seed=3, width=n / 8.0)
    rng = np.random.default_rng(7)
    trace = rng.random((S, n)) < 0.5
    st["Y"].numpy()[trace] = 10.0 ** rng.uniform(-320.0, -200.0, int(trace.sum()))
    eng = ChemistryStep(mech, capi.default_opts(cell_order=order))
    try:
        dev = {k: v.to("cuda:0") for k, v in st.items()}
        for _ in range(2):                                    # with a history, too
            g = gpu_flat_step(eng, dev, dt)
    finally:
        eng.close()
    on = g["status"] == capi.NRG_CELL_OK
    assert on.sum() > n // 4
    W, dc = np.asarray(mech.molar_masses), g["Y_prod2"][:, on]
    assert _same(g["Y_prod"][:, on], (dc * W[:, None]) / dt)
    ef = np.zeros(dc.shape[1])
    for s in range(S):
        ef = ef - (o.h(298.15, s) * dc[s]) / dt
    assert _same(g["E_f_prod"][on], ef)


@pytest.mark.parametrize("name,analytic,n", [("KEROMNES", 0, 5 << 17), ("ZHANG", 0, 5 << 17), ("TEREZA", 1, 3 << 16)])
def test_lane_groups_equal_one_cell_per_lane(name, analytic, n):
    """The integrator's own quotients, in cells whose densities and trace species
    cover the range: a lane divides, a group looks at its operands first."""
    import torch
    import nrg_amd.solver as solver_module
    from nrg_amd.solver import ChemistryStep
    mech = M.load_mechanism(*(() if name == "KEROMNES" else (name + ".txt", name + "_THERMO.txt")))
    st = inputs.flame_front_2d(mech, n, 1, seed=5, width=n / 6.0, device="cuda:0")
    g = torch.Generator().manual_seed(n)
    rand = lambda *shape: torch.rand(shape, generator=g, dtype=torch.float64).to("cuda:0")  # noqa: E731
    some = rand(n) < 0.02
    st["rho"] = torch.where(some, 10.0 ** (620.0 * rand(n) - 320.0), st["rho"])
    trace = (rand(mech.species_number, n) < 0.5) & (rand(n) < 0.1)
    st["Y"] = torch.where(trace, 10.0 ** (60.0 * rand(mech.species_number, n) - 320.0), st["Y"])
    real, got = solver_module.check, []
    solver_module.check = lambda lib, rc: None                # failed cells: their status is compared
    try:
        for order in (capi.NRG_ORDER_NATURAL, capi.NRG_ORDER_STIFFNESS):
            eng = ChemistryStep(mech, capi.default_opts(cell_order=order, jacobian=analytic))
            for _ in range(2):                                # the second call in stiffness order has a history
                out = gpu_flat_step(eng, st, 1e-7)
            got.append(out)
            eng.close()
    finally:
        solver_module.check = real
    a, b = got
    for k in ("Y_prod", "Y_prod2", "E_f_prod", "status", "nstep", "nfe", "nje"):
        assert np.array_equal(a[k], b[k], equal_nan=True), k
    assert (a["status"] == capi.NRG_CELL_OK).sum() > n // 4 and (a["status"] == capi.NRG_CELL_REPEATED_FAIL).any()
