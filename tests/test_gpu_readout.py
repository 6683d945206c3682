"""Host read-out of density and velocity: groups of 512 tiles gathered on the device (one group, whole groups, a
remainder) against the device's dense FP32 fields and the dense entry, either array alone, other points untouched."""
import numpy as np
import pytest

from pv_dec_original_amd import Simulation, SubDomain
from pv_dec_original_amd import _native as N
from pv_dec_original_amd.workloads import fluid_box_case, xfaces

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box", [(9, 6, 5), (64, 32, 16), (64, 64, 16), (130, 33, 25), (70, 40, 27)])
def test_readout_groups(box):
    nx, ny, nz = box
    case = fluid_box_case(q=19, box=box, tau=0.8)
    rng = np.random.default_rng(3)
    fluid = (rng.random((nz, ny, nx)) < 0.7).astype(np.uint8)
    case.geometry.fluid = fluid
    sd = SubDomain(case.geometry, xfaces(case.geometry), storage="fp64", tau=case.tau)
    sim = Simulation(sd, case.tau)
    rho0, u0 = 1.0 + 0.01 * rng.standard_normal((nz, ny, nx)), 0.01 * rng.standard_normal((3, nz, ny, nx))
    sim.init_fields(rho0, u0)
    sim.step(2)
    rho, u = sim.macros()
    node = sd.kinds().reshape(nz, ny, nx) != 0
    assert np.array_equal(node, fluid != 0)
    assert not rho[~node].any() and not u[:, ~node].any() and rho[node].all()
    # (the random holes leave nodes whose state is not a number: equal counts them as the same value)
    def equal(a, b):
        return np.array_equal(a, b, equal_nan=True)

    rho_d, u_d = sim.macros_device()
    assert equal(rho.astype(np.float32)[node], rho_d.cpu().numpy()[node])
    assert equal(u.astype(np.float32)[:, node], u_d.cpu().numpy()[:, node])
    # dense entry over what was there before; each array alone
    r, v = np.full_like(rho, 7.0), np.full_like(u, 7.0)
    assert N.lib().pvlbm_get_macros(sim.handle, N.dptr(r), None) == 0
    assert N.lib().pvlbm_get_macros(sim.handle, None, N.dptr(v)) == 0
    assert equal(r, rho) and equal(v, u)
    r, v = np.full_like(rho, 7.0), np.full_like(u, 7.0)
    assert N.lib().pvlbm_fill_macros(sim.handle, N.dptr(r), N.dptr(v)) == 0
    assert equal(r[node], rho[node]) and equal(v[:, node], u[:, node])
    assert (r[~node] == 7.0).all() and (v[:, ~node] == 7.0).all()
