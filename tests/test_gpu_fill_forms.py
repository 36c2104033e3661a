"""Map and force kernels where their lists and workgroups turn over.

A coarse grid over a dense globule gives every tile more atoms than one pass
of the map kernels' LDS tables holds (128 atoms for the charges, 256 for the
spline windows), on a grid whose sides are not multiples of the tile, with
atoms near the faces: maps bitwise, forces per atom, against the oracle.
"""
import numpy as np
import pytest

import orc_driver as od
from apbs_amd import driver, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("srfm,chgm", [("spl2", "spl2"), ("spl4", "spl4"), ("spl3", "spl0")])
@pytest.mark.parametrize("dims,h", [((33, 33, 33), 1.0), ((41, 33, 49), 0.55)])
def test_dense_tiles(srfm, chgm, dims, h):
    atoms = synth.globule(800, (11.0, 9.0, 12.0), 3, min_dist=1.9)[:3]
    pbe = dict(pdie=2.0, sdie=78.54, srfm=srfm, chgm=chgm, swin=0.3, srad=1.4, sdens=10.0,
               temp=298.15, bcfl="sdh", ions=[(1, 0.15, 2.0), (-1, 0.15, 2.0)], etol=1e-12)
    c = od.mol_center(atoms[0])
    mol = driver.Molecule(*atoms)
    _, g = driver.run_manual(mol, list(dims), c, pbe, grid=[h] * 3)
    _, o = od.run_manual(atoms, list(dims), c, pbe, grid=[h] * 3)
    for name in ("epsx", "epsy", "epsz", "kappa", "charge"):
        assert np.array_equal(g.array(name), o.array(name)), name
    big, diff = 0.0, 0.0
    for a in range(0, 800, 7):
        rg, *fg = g.force(a)
        ro, *fo = o.force(a)
        assert bool(rg) == bool(ro), a
        for x, y in zip(fg, fo):
            big, diff = max(big, np.abs(y).max()), max(diff, np.abs(x - y).max())
    print(f"{srfm}/{chgm} {dims}: largest force {big:.3e}, largest difference {diff:.2e}")
    # both potentials are converged to 1e-12 of the residual: the forces agree
    # to that times the operator's conditioning, far inside 1e-8
    assert diff <= 1e-8 * big


@pytest.mark.parametrize("srfm", ["spl2", "spl3", "spl4"])
@pytest.mark.parametrize("swin", [-0.2, 0.0])
def test_windows_of_no_width(srfm, swin):
    """A spline window that is empty (0) or inside out (the core's radius the
    larger, r - swin): every point of an atom's box within the core is zero, so
    no point may be passed over for lying beyond the outer radius.  Maps bitwise
    the oracle's."""
    atoms = synth.globule(40, (5.0,) * 3, 11, net_charge=1)[:3]
    pbe = dict(pdie=2.0, sdie=78.54, srfm=srfm, chgm="spl2", swin=swin, srad=1.4, sdens=10.0,
               temp=298.15, bcfl="zero", ions=[(1, 0.15, 2.0), (-1, 0.15, 2.0)])
    c = od.mol_center(atoms[0])
    mol = driver.Molecule(*atoms)
    g = driver.Calc(mol, driver.manual_mgparm([65, 65, 65], c, grid=[0.25] * 3), pbe)
    g.fillco()
    nlev, dime = od.check_nlev([65, 65, 65])
    o = od.OrcCalc(od.make_params(dime, [0.25] * 3, c, nlev, pbe), atoms)
    o.fillco()
    for name in ("epsx", "epsy", "epsz", "kappa"):
        off = int((~np.isclose(g.array(name), o.array(name), 0, 0, equal_nan=True)).sum())
        assert off == 0, (name, off)


@pytest.mark.parametrize("srfm", ["spl2", "spl3", "spl4"])
@pytest.mark.parametrize("swin", [0.0, 1e-20, 0.5])
def test_nodes_on_the_window_edges(srfm, swin):
    """Nodes and face centres exactly at an atom's radii: atoms on nodes, radii
    and radii with the ion's a multiple of half the spacing.  With a window of no
    width (0, or too little to change the radius) such a point is in the core."""
    xyz = np.array([[0.0, 0.0, 0.0], [5.0, -1.0, 2.0], [-5.5, 4.0, -3.0]])
    atoms = (xyz, np.array([1.0, -0.5, 0.5]), np.array([2.0, 1.5, 1.75]))
    pbe = dict(pdie=2.0, sdie=78.54, srfm=srfm, chgm="spl2", swin=swin, srad=1.4, sdens=10.0,
               temp=298.15, bcfl="zero", ions=[(1, 0.15, 2.0), (-1, 0.15, 2.0)])
    c = np.zeros(3)
    mol = driver.Molecule(*atoms)
    g = driver.Calc(mol, driver.manual_mgparm([65, 65, 65], c, grid=[0.5] * 3), pbe)
    g.fillco()
    nlev, dime = od.check_nlev([65, 65, 65])
    o = od.OrcCalc(od.make_params(dime, [0.5] * 3, c, nlev, pbe), atoms)
    o.fillco()
    for name in ("epsx", "epsy", "epsz", "kappa"):
        off = int((~np.isclose(g.array(name), o.array(name), 0, 0, equal_nan=True)).sum())
        assert off == 0, (name, off)
