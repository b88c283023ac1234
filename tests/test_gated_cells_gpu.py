"""Gated cells (T below the gate, or a marked cell): rates_kernel writes their
outputs and leaves them out of the integrator's records, in natural order by
handing out the records as it goes.  Patterns at the edges of its blocks of 128
cells, in both orders: gated cells have the reference's outputs
(chemical_kinetics_solver.f90:341-346), integrated ones the bits that the same
cells have in a field of their own, and the counts add up."""
import numpy as np
import pytest

from gpu_util import gpu_flat_step
from nrg_amd import capi, inputs

pytestmark = pytest.mark.gpu


def _pattern(kind, n):
    i = np.arange(n)
    return {"none": i < 0, "all": i >= 0, "first": i == 0, "last": i == n - 1, "every third": i % 3 == 0,
            "a block": (i >= 128) & (i < 256), "all but a block": (i < 128) | (i >= 256),
            "runs": (i // 77) % 2 == 0}[kind]


@pytest.mark.parametrize("order", [capi.NRG_ORDER_NATURAL, capi.NRG_ORDER_STIFFNESS])
@pytest.mark.parametrize("kind", ["none", "all", "first", "last", "every third", "a block", "all but a block", "runs"])
@pytest.mark.parametrize("n", [1, 127, 128, 129, 1000, 9001])
def test_patterns(mech, n, kind, order):
    import torch
    from nrg_amd.solver import ChemistryStep
    live = _pattern(kind, n)
    st = inputs.flame_front_2d(mech, max(n, 64), 1, seed=n, width=max(n, 64) / 8.0, device="cuda:0")
    st = {k: v[..., :n].contiguous() for k, v in st.items()}
    st["T"] = torch.clamp(st["T"], min=400.0)
    bc = np.zeros(n, np.int8)
    off = np.where(~live)[0]
    bc[off[::2]] = 1                                          # half by marker, half by temperature
    st["T"][torch.as_tensor(off[1::2], device="cuda:0")] = 304.9
    eng = ChemistryStep(mech, capi.default_opts(cell_order=order))
    try:
        for _ in range(2):
            g = gpu_flat_step(eng, st, 1e-8, bc=bc)
        assert np.array_equal(g["status"] == capi.NRG_CELL_GATED, ~live)
        assert (g["Y_prod"][:, ~live] == 0.0).all() and (g["E_f_prod"][~live] == 0.0).all()
        assert (g["Y_prod2"][:, ~live] == -7.0).all()
        for k in ("nstep", "nfe", "nje"):
            assert (g[k][~live] == 0).all()
        s = g["stats"]
        assert s.cells_integrated == live.sum() and s.status_count[capi.NRG_CELL_GATED] == (~live).sum()
        assert s.status_count[capi.NRG_CELL_OK] == live.sum()
        if live.any():
            on = torch.as_tensor(np.where(live)[0], device="cuda:0")
            alone = gpu_flat_step(eng, {k: v[..., on].contiguous() for k, v in st.items()}, 1e-8)
            for k in ("Y_prod", "Y_prod2", "E_f_prod", "nstep", "nfe", "nje"):
                assert np.array_equal(g[k][..., live], alone[k]), k
    finally:
        eng.close()


@pytest.mark.parametrize("order", [capi.NRG_ORDER_NATURAL, capi.NRG_ORDER_STIFFNESS])
def test_gated_grid_costs_a_pass_over_it(mech, order):
    """4.2M gated cells: 0.2 to 0.3 ms of kernels; handed out one by one in
    natural order they took 6.5.  The bar lies far from both."""
    from nrg_amd.solver import ChemistryStep
    st = inputs.flame_front_2d(mech, 1 << 22, 1, seed=3, width=1e5, device="cuda:0")
    st["T"][:] = 300.0
    eng = ChemistryStep(mech, capi.default_opts(cell_order=order))
    try:
        ms = min(gpu_flat_step(eng, st, 1e-7, counters=False)["stats"].kernel_ms for _ in range(4))
    finally:
        eng.close()
    print("[gated] order=%d kernel_ms=%.3f" % (order, ms), flush=True)
    assert ms < 2.0
