"""A start from a coarse field where rows, tiles and planes end early: the fields against the host restatement of
the expansion, the plane fluxes against their targets, and the count of samples that are not finite, which
covers every point of the box, solid ones too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,coarse,bad", [(61, (5, 3, 7), False), (70, (2, 9, 4), True), (64, (16, 16, 16), False),
                                           (129, (6, 6, 11), True)])
@pytest.mark.parametrize("planes", [False, True])
def test_coarse_start(nx, coarse, bad, planes):
    import torch
    from pv_dec_original_amd import SubDomain, Simulation, native as N
    from pv_dec_original_amd import warmstart as W
    from pv_dec_original_amd.workloads import ybif_case
    case = ybif_case(q=19, box=(nx, 40, 36), tau=0.7, rp=9.0, rd=6.0)
    sd = SubDomain(case.geometry, case.faces, storage="fp64", tau=0.7, triangles=False)
    sim = Simulation(sd, 0.7, 1.0, 8e-6)
    rng = np.random.default_rng(nx)
    rho = (1.0 + 0.01 * rng.standard_normal(coarse)).astype(np.float32)
    u = (0.05 + 0.02 * rng.random((3,) + coarse)).astype(np.float32)
    if bad:
        u[1, 0, 0, 0] = np.nan  # a corner of the box: solid points
        rho[1, 2, 2] = np.inf
    shape = (sd.nz, sd.ny, sd.nx)
    with np.errstate(invalid="ignore"):
        rf = W._trilinear_up(rho.astype(np.float64), shape)
        uf = np.stack([W._trilinear_up(u[c].astype(np.float64), shape) for c in range(3)])
    fin = np.isfinite(rf) & np.isfinite(uf).all(axis=0)
    rf, uf = np.where(fin, np.clip(rf, 0.95, 1.02), 1.0), np.where(fin, uf, 0.0)
    nodes = sd.kinds() != N.SOLID
    flux = drho = None
    if planes:
        flux = 30.0 * (1.0 + 0.2 * np.sin(np.arange(nx)))
        drho = 0.003 * np.cos(np.arange(nx))
        have = np.where(nodes, uf[0], 0.0).sum(axis=(0, 1))
        uf = uf * np.where(have > 1e-12 * flux, np.clip(flux / np.where(have == 0, 1, have), 0.25, 4.0), 1.0)
        rf = np.clip(rf + drho, 0.95, 1.02)
    sp = np.sqrt((uf * uf).sum(axis=0))
    uf = uf * np.where(sp > 0.1, 0.1 / np.maximum(sp, 1e-300), 1.0)
    got = sim.init_fields_coarse(torch.from_numpy(rho).cuda(), torch.from_numpy(u).cuda(), 0.1, (0.95, 1.02), 0.0, flux,
                                 drho)
    assert got == np.count_nonzero(~fin)
    r, v = sim.macros()
    # FP32 interpolation of values up to 1: a few roundings of 2^-24 each
    assert np.abs(r - rf)[nodes].max() < 4e-6 and np.abs(v - uf)[:, nodes].max() < 4e-6
    assert sim.reduce()[3] == 0
    # the FP32 read-out of the same fields: rows of whole and of partial quads
    r32, v32 = (t.cpu().numpy() for t in sim.macros_device())
    assert np.array_equal(r32, np.where(nodes, r, 1.0).astype(np.float32))
    assert np.array_equal(v32, v.astype(np.float32))
