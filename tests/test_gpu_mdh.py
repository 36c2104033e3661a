"""The accuracy of the Debye-Hueckel boundary sum (bcfl mdh).

Every face value against the same sum in extended precision (64-bit mantissa,
the same atoms, nodes and screening length).  Node coordinates are multiples of
the spacing, a power of two times 7 or less, so they are exact.

With u = 2^-53 a term pre1 q exp(kappa r) / (1 + kappa r) exp(-kappa d) / d is
within (16 + 6 kappa d) u of its value: 8 u and kappa r u for the factor, 5 u
for d^2 and half of it with 2 u more for its reciprocal root, 5 kappa d u (6
where the product is rounded) for the exponent, 2 u for the exponential, 1 u for
the product; and adding n terms in c chunks rounds each at most n/c + c times.
"""
import numpy as np
import pytest

from apbs_amd import driver, lib, synth

pytestmark = pytest.mark.gpu

LD = np.longdouble
U = 2.0 ** -53
E_C, K_B, EPS0 = 1.6021773e-19, 1.3806581e-23, 8.8541878e-12


def face_sums(xyz, q, r, nodes, pre1, kappa):
    """The sums on the two faces of each axis, flattened like Calc.boundary(),
    with the sums of the terms' magnitudes and of those times kappa d."""
    out = [[], [], []]
    axes = [n.astype(LD) for n in nodes]
    for axis, (fast, slow) in ((0, (1, 2)), (1, (0, 2)), (2, (0, 1))):
        for f in (axes[axis][0], axes[axis][-1]):
            acc = [np.zeros((axes[slow].size, axes[fast].size), LD) for _ in range(3)]
            for a in range(len(q)):
                p = xyz[a].astype(LD)
                d = np.sqrt((f - p[axis]) ** 2 + (axes[fast][None, :] - p[fast]) ** 2 +
                            (axes[slow][:, None] - p[slow]) ** 2)
                t = LD(pre1) * (LD(E_C) * LD(q[a])) / d
                if kappa > 1e-9:
                    t = t * np.exp(LD(kappa) * (LD(r[a]) - d)) / (1 + LD(kappa) * LD(r[a]))
                acc[0] += t
                acc[1] += np.abs(t)
                acc[2] += np.abs(t) * (LD(kappa) * d)
            for o, v in zip(out, acc):
                o.append(v.reshape(-1))
    return [np.concatenate(o) for o in out]


def boundary(xyz, q, r, dims, h, salt, precision=0):
    """The faces' values, the nodes, and what the exact sums need."""
    mol = driver.Molecule(xyz, q, r)
    pbe = dict(pdie=2.0, sdie=78.5, srfm="spl2", chgm="spl2", swin=0.3, srad=1.4, sdens=10.0,
               temp=298.0, bcfl="mdh", ions=[(1, salt, 2.0), (-1, salt, 2.0)])
    c = driver.Calc(mol, driver.manual_mgparm(list(dims), np.zeros(3), grid=[h] * 3), pbe,
                    precision=precision, mirror=False)
    c.fillco()
    got = np.concatenate([b.reshape(-1) for b in c.boundary()])
    kappa = float(lib().Vpbe_getXkappa(c.pbe))
    c.release()
    assert (kappa > 0) == (salt > 0)
    nodes = [h * (np.arange(n) - (n - 1) / 2) for n in dims]
    # (a factor common to all values: the FP64 number the program forms)
    pre1 = E_C / (4 * np.pi * EPS0 * 78.5 * K_B * 298.0) * 1.0e10
    return got, nodes, pre1, kappa


@pytest.mark.parametrize("salt", [0.15, 0.0])
@pytest.mark.parametrize("natoms,dims,h", [(8, (33, 33, 33), 0.5), (9, (33, 33, 33), 0.5),
                                           (31, (33, 33, 33), 0.5), (63, (41, 33, 41), 0.75),
                                           (64, (41, 33, 41), 0.75), (300, (33, 49, 41), 0.875),
                                           (2000, (49, 49, 49), 1.0), (5000, (17, 17, 17), 4.0)])
def test_sums(natoms, dims, h, salt):
    """Atom counts around the turns from one chunk to two (8) and from chunks of
    8 atoms to chunks of 16 (64), ordinary ones, and many more atoms than
    boundary points: 312 chunks, whose sum is as long as its unrolled loop and
    remainder.  The FP32-term sum within 1e-5 of the largest value."""
    rad = max(2.6, (natoms / 120.0) ** (1.0 / 3.0) * 6.0)
    xyz, q, r, _ = synth.globule(natoms, (rad,) * 3, 5, net_charge=-2)
    got, nodes, pre1, kappa = boundary(xyz, q, r, dims, h, salt)
    exact, mag, far = face_sums(xyz, q, r, nodes, pre1, kappa)
    err = np.abs(got - exact)
    # (n/c + c: up to 18 atoms a chunk, up to 312 chunks)
    bound = U * ((16 + min(natoms + 1, 330)) * mag + 6 * far)
    rms = float(np.linalg.norm(err.astype(float)) / np.linalg.norm(exact.astype(float)))
    print(f"{natoms} atoms, salt {salt}: rms error {rms:.2e}, largest error over its bound "
          f"{float((err / bound).max()):.3f}")
    assert (err <= bound).all()
    fast = boundary(xyz, q, r, dims, h, salt, precision=2)[0]
    assert np.abs(fast - exact).max() <= 1e-5 * np.abs(exact).max()


@pytest.mark.parametrize("salt", [0.05, 0.15, 1.0])
@pytest.mark.parametrize("x", [0.3, 0.7, 1.1])
def test_term(x, salt):
    """One ion: the spread over the faces of the relative error (its mean is the
    factor's error).  Roundings are taken as independent, each with the standard
    deviation u / sqrt(3) of one at a mantissa near 1: five in d^2, halved in the
    reciprocal root, which adds one and half of another; the table, its
    multiply-add, the product with the factor and the addition; and times kappa d
    those of d^2 (halved), the root and d itself.  That is
    sqrt(0.42 + 0.42 + 1.33 + (kappa d)^2 1.17) u, which is also less than the
    spread with a product kappa d that is rounded, 1.5 in the place of 1.17."""
    xyz, q, r = np.array([[x, 0.3, -0.2]]), np.ones(1), np.array([2.1])
    got, nodes, pre1, kappa = boundary(xyz, q, r, (33, 33, 33), 0.5, salt)
    exact, mag, far = face_sums(xyz, q, r, nodes, pre1, kappa)
    spread = float(np.std(((got - exact) / exact).astype(float)))
    kd2 = float(((far / mag) ** 2).mean())
    bar = U * np.sqrt(0.42 + 0.42 + 1.33 + 1.17 * kd2)
    print(f"salt {salt}: spread {spread:.2e}, bar {bar:.2e}, kappa d {np.sqrt(kd2):.2f}")
    assert spread <= bar
