"""Solver failure is reported, not hidden (the reference's Vdpbfa leading-minor
test, buildBd.c:106-114, and its loop test, which a NaN norm would pass).

A negative dielectric map makes every level's operator negative definite.
Gauss-Seidel still runs normally on it (it is the same iteration for A and
-A), so every kernel launches and exits as usual.  In lpbe the dense inverse
of the coarsest operator then meets a negative pivot, flags it, and
Vpmg_solve returns 0 with that message.  In npbe the Newton Jacobian adds the
ionic term N'(u) >= 0 to the diagonal; restricted to the coarse levels it
outgrows the (negative) Galerkin stencil, so the coarsest operator can be
positive definite while the fine iteration diverges: the solve then fails on
the residual norm that is not finite.  Either way Vpmg_solve returns 0 with a
message, and the same object and a fresh one stay usable.
"""
import numpy as np
import pytest

from apbs_amd import driver, synth

pytestmark = pytest.mark.gpu

H = 0.5


def calc(diel, precision, npbe, dime):
    atoms = synth.globule(30, (4.0,) * 3, 5, net_charge=1)[:3]
    mol = driver.Molecule(*atoms)
    c = mol.center
    origin = c - 0.25 * (dime - 1) - 2.0  # (the box and 2 A around it)
    shape = (dime + 10,) * 3
    maps = {k: driver.Map(np.full(shape, diel), origin, (0.5,) * 3)
            for k in ("dielx", "diely", "dielz")}
    ions = [(1, 0.0, 2.0), (-1, 0.0, 2.0)]
    if npbe:
        maps["kappa"] = driver.Map(np.ones(shape), origin, (0.5,) * 3)
        ions = [(1, 0.15, 2.0), (-1, 0.15, 2.0)]
    pbe = dict(pdie=2.0, sdie=78.54, srfm="spl2", chgm="spl2", swin=0.3, srad=1.4, sdens=10.0,
               temp=298.15, bcfl="mdh", ions=ions, npbe=npbe, maps=maps)
    g = driver.Calc(mol, driver.manual_mgparm([dime] * 3, c, grid=[H] * 3), pbe,
                    precision=precision)
    g._keep = (mol, maps)
    return g


@pytest.mark.parametrize("precision,npbe,dime", [(0, False, 33), (1, False, 33), (0, True, 33),
                                                 (1, True, 33), (0, False, 57), (1, False, 57)])
def test_negative_dielectric_is_reported(precision, npbe, dime, capfd):
    """33^3: a coarsest grid inverted in registers; 57^3: one of 8^3 (216
    unknowns), inverted by blocks of pivots (in lpbe, where a pivot is what
    reports it: in npbe a diverging iteration may also end at its limit of
    steps with finite norms)."""
    bad = calc(-5.0, precision, npbe, dime)
    bad.fillco()
    with pytest.raises(RuntimeError):
        bad.solve()
    err = capfd.readouterr().err
    if npbe:
        assert "not positive definite" in err or "not finite" in err, err
    else:
        assert "not positive definite" in err, err
    # the device and the library stay usable: the same object solves again
    # after a valid fill is impossible (its maps are fixed), so a fresh one
    good = calc(20.0, precision, npbe, dime)
    good.fillco()
    good.solve()
    st = good.stats()
    assert np.isfinite(good.energy(1)) and st["relres"] <= 1e-6, st
    # the failed object can still be released and its pool memory reused
    bad.release()
