"""Forms of the coarse-level kernels at the sizes where their tiling turns.

The blocked dense inverse (coarsest grids that cannot halve down to 64
unknowns) against numpy, at one unknown past the one-workgroup form, at whole
and partial 64-pivot blocks, and at N = 1000 (the 12^3 coarsest grid under
353^3); and a whole solve whose coarsest grid takes that form, against the
oracle.  The bottom of the cycle, the row and block sweeps, the Galerkin
product and the fine level's norm passes at the edges of their tiles.
"""
import ctypes

import numpy as np
import pytest

import orc_driver as od
from apbs_amd import driver, synth

pytestmark = pytest.mark.gpu

dp = ctypes.POINTER(ctypes.c_double)


def P(a):
    return a.ctypes.data_as(dp)


@pytest.fixture(scope="module")
def L():
    import apbs_amd
    return ctypes.CDLL(apbs_amd.LIB_PATH)


@pytest.mark.parametrize("N", [90, 127, 128, 129, 216, 1000])
def test_blocked_dense_inverse(L, N):
    """Both sides within the backward error of an elimination without
    pivoting of a diagonally dominant matrix, 4 N eps cond(A)."""
    rng = np.random.default_rng(N)
    A = rng.uniform(-1, 0, (N, N))
    A = 0.5 * (A + A.T)
    np.fill_diagonal(A, 0.0)
    A[np.diag_indices(N)] = -A.sum(axis=1) + rng.uniform(0.5, 2.0, N)
    A = np.ascontiguousarray(A)
    out = np.zeros((N, N))
    assert L.pmgtest_dense_invert(N, P(A), P(out), 0) == 1
    ref = np.linalg.inv(A)
    tol = 4 * N * np.finfo(float).eps * np.linalg.cond(A)
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    print(f"N {N}: relative difference {err:.2e}, bound {tol:.2e}")
    assert err <= tol
    assert np.abs(A @ out - np.eye(N)).max() <= tol


@pytest.mark.parametrize("N", [27, 64, 80, 90, 128, 216, 1000])
def test_first_bad_pivot_is_reported(L, N):
    """Matrices inverted in one launch, in the register, LDS and blocked forms:
    positive definite ones are not flagged; one whose leading minors are positive
    up to row p is flagged p + 1, in the first block of pivots, at a block's first
    and last row and in the partial last block; of several bad pivots, in one
    block or in two, the first; a NaN as well."""
    rng = np.random.default_rng(N)
    A = rng.uniform(-1, 0, (N, N))
    A = 0.5 * (A + A.T)
    np.fill_diagonal(A, 0.0)
    A[np.diag_indices(N)] = -A.sum(axis=1) + rng.uniform(0.5, 2.0, N)
    rows = sorted({0, 5, min(63, N - 1), min(64, N - 1), min(127, N - 2), N - 1})
    mats, want = [A], [0]
    for p in rows:
        B = A.copy()
        B[p, p] = -1.0 - np.abs(A[p]).sum()
        mats.append(B)
        want.append(p + 1)
    for first, second in ((3, 9), (min(20, N - 2), N - 1)):
        B = A.copy()
        B[second, second] = -1.0e6
        B[first, first] = -1.0e6
        mats.append(B)
        want.append(first + 1)
    B = A.copy()
    B[N // 2, N // 2] = np.nan
    mats.append(B)
    want.append(N // 2 + 1)
    got = []
    for b in range(0, len(mats), 8):
        m = np.ascontiguousarray(np.stack(mats[b:b + 8]))
        flags = np.full(len(m), -1.0)
        assert L.pmgtest_dense_pivots(N, len(m), P(m), P(flags)) == 1
        got += list(flags)
    assert got == want


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dims", [(57, 57, 57), (49, 57, 57)])
def test_solve_on_a_large_coarsest_grid(dims, precision):
    """Grids that stop halving at 8^3 (216 unknowns) and at 7 x 8 x 8 (180):
    converged energy and potential against the oracle."""
    atoms = synth.globule(60, (6.0,) * 3, 9, net_charge=1)[:3]
    pbe = dict(pdie=2.0, sdie=78.54, srfm="spl2", chgm="spl2", swin=0.3, srad=1.4, sdens=10.0,
               temp=298.15, bcfl="mdh", ions=[(1, 0.15, 2.0), (-1, 0.15, 2.0)], etol=1e-12)
    c = od.mol_center(atoms[0])
    mol = driver.Molecule(*atoms)
    eg, g = driver.run_manual(mol, list(dims), c, pbe, grid=[0.45] * 3, precision=precision)
    eo, o = od.run_manual(atoms, list(dims), c, dict(pbe, coarse_smoother=1, deep_coarse=1),
                          grid=[0.45] * 3)
    ug, uo = g.array("u"), o.array("u")
    rel = abs(eg - eo) / abs(eo)
    l2 = np.linalg.norm(ug - uo) / np.linalg.norm(uo)
    print(f"{dims} precision {precision}: energy {rel:.2e}, potential {l2:.2e}, {g.stats()}")
    assert rel < 1e-9 and l2 < 1e-9


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("npbe", [False, True])
@pytest.mark.parametrize("dims", [(17, 17, 17), (33, 33, 33), (41, 41, 41), (49, 33, 17),
                                  (81, 65, 33), (97, 33, 33)])
def test_bottom_of_the_cycle_bitwise(dims, npbe, precision, monkeypatch):
    """The one-launch bottom of the V-cycle (a level of at most 1,024 interior
    points above a coarsest one of at most 64) against the separate launches:
    the same potential bit for bit and the same iteration counts, cubic and
    ragged levels, both words.  The separate launches run in the colour form
    (APBS_PMG_SMOOTHER27), itself bitwise the oracle's sweep."""
    atoms = synth.globule(40, (5.0,) * 3, 9, net_charge=1)[:3]
    pbe = dict(npbe=npbe, pdie=2.0, sdie=78.54, srfm="spl2", chgm="spl2", swin=0.3, srad=1.4,
               sdens=10.0, temp=298.15, bcfl="mdh", ions=[(1, 0.15, 2.0), (-1, 0.15, 2.0)])
    c = od.mol_center(atoms[0])
    mol = driver.Molecule(*atoms)
    out = []
    for form in (None, "colour"):
        if form:
            monkeypatch.setenv("APBS_PMG_SMOOTHER27", form)
        e, g = driver.run_manual(mol, list(dims), c, pbe, grid=[0.6] * 3, precision=precision)
        out.append((e, g.array("u"), g.stats()))
    (ea, ua, sa), (eb, ub, sb) = out
    assert (sa["iters"], sa["inner"], sa["nlev"]) == (sb["iters"], sb["inner"], sb["nlev"])
    assert ea == eb and np.array_equal(ua, ub)


def _level(n3, seed):
    rng = np.random.default_rng(seed)
    nx, ny, nz = n3
    n = nx * ny * nz
    a = np.zeros((14, nz, ny, nx))
    for s in range(14):
        a[s, 1:-1, 1:-1, 1:-1] = rng.uniform(0.1, 1.0, (nz - 2, ny - 2, nx - 2))
    a[0, 1:-1, 1:-1, 1:-1] = rng.uniform(18.0, 36.0, (nz - 2, ny - 2, nx - 2))
    x = np.zeros((nz, ny, nx))
    x[1:-1, 1:-1, 1:-1] = rng.normal(size=(nz - 2, ny - 2, nx - 2))
    return np.ascontiguousarray(a.reshape(-1)), rng.uniform(0, 1, n), rng.normal(size=n), \
        x.reshape(-1)


def _rows_fit(nx, word, code):
    """A tile of 2m rows in runs of kV points: at most 512 lanes and 64 KB."""
    kv, m = divmod(code, 100)
    runs = -(-(nx - 2) // kv)
    return (2 * m + 1) * runs <= 512 and (2 * m + 4) * nx * word <= 65536 and nx >= kv + 2


def _block_fits(nx, word, code):
    """TY rows of KC planes and their halo: at most 1,024 lanes and 64 KB."""
    ty, kc = divmod(code, 100)
    kv = 16 // word
    runs = -(-(nx - 2) // kv)
    return (runs * ((ty + 2) * kc + 2 * ty) <= 1024 and
            (kc + 2) * (ty + 2) * nx * word <= 65536 and nx >= kv + 2)


def _fitting(shapes, codes, word, fits):
    return [(n3, c) for n3 in shapes for c in codes if fits(n3[0], word, c)]


@pytest.mark.parametrize("n3,code", _fitting(
    [(17, 17, 17), (9, 11, 13), (45, 43, 41), (4, 5, 4), (70, 21, 6), (81, 81, 9), (131, 8, 7),
     (177, 13, 5)], [201, 202, 203, 204, 205, 206, 210], 8, _rows_fit))
def test_row_tiles_bitwise(L, n3, code):
    """The whole-row plane sweep (code 100 kV + m: runs of kV points, 2m rows
    a workgroup) against the oracle's 8-colour sweep, bit for bit: partial
    tiles, rows of 2 to 175 points, odd ends of the last run, both orders and
    odd and even sweep counts."""
    nx, ny, nz = n3
    a, cc, fc, x0 = _level(n3, sum(n3) + code)
    O = od.lib()
    for adj in (0, 1):
        for nu in (2, 3):
            xg, xo = x0.copy(), x0.copy()
            assert L.pmgtest_gsrb27_mode(nx, ny, nz, P(a), P(cc), P(fc), P(xg), nu, adj,
                                         code) == 1
            O.orc_gsrb(nx, ny, nz, 27, P(a), P(cc), P(fc), P(xo), nu, adj, 1)
            assert np.array_equal(xg, xo), (adj, nu)


@pytest.mark.parametrize("n3,code", _fitting(
    [(17, 17, 17), (9, 11, 13), (45, 43, 41), (6, 5, 4), (81, 81, 9), (131, 8, 7), (178, 13, 5)],
    [203, 206, 401, 402, 404, 405, 406, 410], 4, _rows_fit))
def test_row_tiles_fp32_bitwise(L, n3, code):
    """The FP32 rows forms (8- and 16-byte runs) against one launch per colour."""
    fp = ctypes.POINTER(ctypes.c_float)
    nx, ny, nz = n3
    a, cc, fc, x0 = (v.astype(np.float32) for v in _level(n3, sum(n3) + code))
    D = a[:nx * ny * nz] + cc
    for adj in (0, 1):
        for nu in (2, 3):
            out = []
            for mode in (code, 0):
                x = x0.copy()
                assert L.pmgtest_gsrb27_32(nx, ny, nz, a.ctypes.data_as(fp), D.ctypes.data_as(fp),
                                           fc.ctypes.data_as(fp), x.ctypes.data_as(fp), nu, adj,
                                           mode) == 1
                out.append(x)
            assert np.array_equal(out[0], out[1]), (adj, nu)


@pytest.mark.parametrize("n3", [(40, 5, 4), (45, 9, 9), (49, 97, 33), (41, 33, 97), (45, 33, 97),
                                (69, 67, 69), (73, 73, 73), (105, 111, 41), (145, 41, 17)])
def test_row_rule_bitwise(L, n3):
    """The sweep in the form the dispatch takes, on levels for which the rule
    gives 1 to 6 row pairs a workgroup, in FP64 against the oracle and in FP32
    against one launch per colour, bit for bit."""
    fp = ctypes.POINTER(ctypes.c_float)
    nx, ny, nz = n3
    a, cc, fc, x0 = _level(n3, sum(n3))
    af, cf, ff, xf = (v.astype(np.float32) for v in (a, cc, fc, x0))
    D = af[:nx * ny * nz] + cf
    for adj in (0, 1):
        xg, xo = x0.copy(), x0.copy()
        assert L.pmgtest_gsrb27_mode(nx, ny, nz, P(a), P(cc), P(fc), P(xg), 2, adj, 1) == 1
        od.lib().orc_gsrb(nx, ny, nz, 27, P(a), P(cc), P(fc), P(xo), 2, adj, 1)
        assert np.array_equal(xg, xo), adj
        out = []
        for mode in (1, 0):
            x = xf.copy()
            assert L.pmgtest_gsrb27_32(nx, ny, nz, af.ctypes.data_as(fp), D.ctypes.data_as(fp),
                                       ff.ctypes.data_as(fp), x.ctypes.data_as(fp), 2, adj,
                                       mode) == 1
            out.append(x)
        assert np.array_equal(out[0], out[1]), adj


@pytest.mark.parametrize("n3,code", _fitting(
    [(17, 19, 21), (33, 33, 33), (67, 13, 20), (130, 6, 11), (7, 70, 3), (4, 5, 6)],
    [101, 202, 203, 204, 302, 303, 402, 404], 8, _block_fits))
def test_block_sweep_bitwise(L, n3, code):
    """The block form of the fused red-black sweep (100 TY + KC: TY rows of KC
    planes) against the oracle's sweep, bit for bit, boundary values not zero:
    partial blocks in both directions, an odd last run, both colour orders, odd
    and even sweep counts."""
    nx, ny, nz = n3
    n = nx * ny * nz
    rng = np.random.default_rng(sum(n3) + code)
    a = np.zeros((4, nz, ny, nx))
    for s in range(4):
        a[s, 1:-1, 1:-1, 1:-1] = rng.uniform(0.1, 1.0, (nz - 2, ny - 2, nx - 2))
    a[0, 1:-1, 1:-1, 1:-1] = rng.uniform(6.0, 12.0, (nz - 2, ny - 2, nx - 2))
    a = np.ascontiguousarray(a.reshape(-1))
    cc, fc, x0 = rng.uniform(0, 1, n), rng.normal(size=n), rng.normal(size=n)
    O = od.lib()
    for adj in (0, 1):
        for nu in (1, 2, 3):
            xg, xo = x0.copy(), x0.copy()
            assert L.pmgtest_gsrb_tile(nx, ny, nz, P(a), P(cc), P(fc), P(xg), nu, adj,
                                       9000000 + code) == 1
            O.orc_gsrb(nx, ny, nz, 7, P(a), P(cc), P(fc), P(xo), nu, adj, 1)
            assert np.array_equal(xg, xo), (adj, nu)


@pytest.mark.parametrize("n3,code", _fitting(
    [(33, 33, 33), (67, 13, 20), (6, 5, 6), (130, 6, 11)], [101, 202, 203, 204, 305, 402, 404], 4,
    _block_fits))
def test_block_sweep_fp32_bitwise(L, n3, code):
    """The FP32 block form against the scalar march (tile 48), from a given and
    from a zero start (the interior then holds NaN and is not read)."""
    fp = ctypes.POINTER(ctypes.c_float)
    rng = np.random.default_rng(sum(n3) + code)
    nx, ny, nz = n3
    sh = (nz, ny, nx)
    ops = [np.zeros(sh, np.float32) for _ in range(4)]
    for o, (lo, hi) in zip(ops, ((0.1, 1.0),) * 3 + ((6.0, 12.0),)):
        o[1:-1, 1:-1, 1:-1] = rng.uniform(lo, hi, (nz - 2, ny - 2, nx - 2))
    fc = rng.normal(size=sh).astype(np.float32)
    x0 = np.zeros(sh, np.float32)
    x0[1:-1, 1:-1, 1:-1] = rng.normal(size=(nz - 2, ny - 2, nx - 2))
    ptr = lambda v: v.ctypes.data_as(fp)  # noqa: E731
    for zero in (0, 1):
        for adj in (0, 1):
            out = []
            for tile in (9000000 + code, 48):
                x = x0.copy()
                if zero:
                    x[1:-1, 1:-1, 1:-1] = np.nan
                assert L.pmgtest_fused32(nx, ny, nz, *[ptr(o) for o in ops], ptr(fc), ptr(x), 2,
                                         adj, tile, zero) == 1
                out.append(x)
            assert np.array_equal(out[0], out[1]), (zero, adj)


def test_forms_that_do_not_fit_are_refused(L):
    """A forced form that a row does not fit is refused, not replaced by
    another; the largest that fits is taken."""
    fp = ctypes.POINTER(ctypes.c_float)
    for nx, word, code in ((70, 8, 207), (70, 8, 208), (131, 4, 407), (131, 4, 408)):
        n = nx * 4 * 4
        ok = int(_rows_fit(nx, word, code))
        assert ok == (code % 100 == 7)
        one, f32 = np.ones(14 * n), np.ones(14 * n, np.float32)
        if word == 8:
            got = L.pmgtest_gsrb27_mode(nx, 4, 4, P(one), P(one), P(one), P(one.copy()), 1, 0, code)
        else:
            p = f32.ctypes.data_as(fp)
            got = L.pmgtest_gsrb27_32(nx, 4, 4, p, p, p, f32.copy().ctypes.data_as(fp), 1, 0, code)
        assert got == ok, (nx, word, code)
    for nx, code in ((130, 203), (130, 204)):
        one = np.ones(4 * nx * 4 * 4)
        assert _block_fits(nx, 8, code) == (code == 203)
        for f in (lambda t: L.pmgtest_gsrb_tile(nx, 4, 4, P(one), P(one), P(one), P(one.copy()), 2,
                                                0, t),
                  lambda t: L.pmgtest_gsrb_zero(nx, 4, 4, P(one), P(one), P(one), P(one.copy()), 0,
                                                t)):
            assert f(9000000 + code) == int(code == 203)
    one = np.ones(14 * 64)
    assert L.pmgtest_gsrb27_mode(4, 4, 4, P(one), P(one), P(one), P(one.copy()), 1, 0, 32) == 0


@pytest.mark.parametrize("st", [7, 27])
@pytest.mark.parametrize("c3", [(3, 3, 3), (5, 3, 7), (6, 6, 6), (34, 3, 5), (81, 21, 5),
                                (9, 33, 17)])
def test_galerkin_bitwise(L, st, c3):
    """The Galerkin product against the oracle's, bit for bit: one coarse
    point, less and a little more than a wavefront of them, partial last
    wavefronts and workgroups, rows that straddle wavefronts."""
    f3 = tuple(2 * n - 1 for n in c3)
    nf, nc = int(np.prod(f3)), int(np.prod(c3))
    rng = np.random.default_rng(sum(c3) + st)
    na = 4 if st == 7 else 14
    a = np.zeros((na, f3[2], f3[1], f3[0]))
    a[:, 1:-1, 1:-1, 1:-1] = rng.uniform(0.1, 1.0, (na, f3[2] - 2, f3[1] - 2, f3[0] - 2))
    a = np.ascontiguousarray(a.reshape(-1))
    ag, ao = np.zeros(14 * nc), np.zeros(14 * nc)
    assert L.pmgtest_galerkin(*f3, st, P(a), *c3, P(ag)) == 1
    od.lib().orc_galerkin(*f3, st, P(a), *c3, P(ao))
    cut = (slice(None),) + (slice(1, -1),) * 3
    sh = (14, c3[2], c3[1], c3[0])
    assert np.array_equal(ag.reshape(sh)[cut], ao.reshape(sh)[cut])


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("n3", [(3, 3, 3), (17, 19, 21), (33, 9, 130), (66, 67, 35), (130, 131, 5),
                                (517, 515, 4)])
def test_fine_norm_passes(L, n3, f32):
    """The fine level's one-pass forms against the separate passes, bit for
    bit, and each norm against the sum of its array's magnitudes: partial
    tiles of columns, runs of one and of many planes, a short last run, and
    more tiles than blocks.  n eps bounds any order of n non-negative terms."""
    nx, ny, nz = n3
    n = nx * ny * nz
    rng = np.random.default_rng(sum(n3) + f32)
    cut = (slice(None),) + (slice(1, -1),) * 3

    def inside(lo, hi, m=1):
        v = np.zeros((m, nz, ny, nx))
        v[cut] = rng.uniform(lo, hi, (m, nz - 2, ny - 2, nx - 2))
        return np.ascontiguousarray(v.reshape(-1))

    a, cc, fc, fz = inside(0.1, 1.0, 4), inside(0, 1), inside(-1, 1), inside(-1, 1)
    x, z = inside(-3, 3), inside(-1, 1)
    out, norms = np.zeros(10 * n), np.zeros(8)
    assert L.pmgtest_fine_passes(nx, ny, nz, P(a), P(cc), P(fc), P(fz), P(x), P(z), f32, P(out),
                                 P(norms)) == 1
    o = out.reshape(10, nz, ny, nx)[cut]
    for y in (0, 8):
        assert np.array_equal(o[y], o[4])
    for rn in (1, 7, 9):
        assert np.array_equal(o[rn], o[5])
    assert np.array_equal(o[6], o[3])
    assert np.array_equal(o[2], o[3].astype(np.float32).astype(np.float64))
    # inner norms 0, 2, 4; nonlinear ones 1, 3, 5, 6, 7: one order of points
    assert norms[0] == norms[2] == norms[4]
    assert norms[1] == norms[3] == norms[5] == norms[6] == norms[7]
    for got, arr in ((norms[0], o[3]), (norms[1], o[5])):
        ref = np.abs(arr).sum()
        assert abs(got - ref) <= 2 * n * np.finfo(float).eps * ref


@pytest.mark.parametrize("c3", [(3, 3, 3), (9, 33, 17), (17, 16, 16), (41, 5, 11)])
@pytest.mark.parametrize("nb", [1, 3, 8])
def test_restrict_with_diagonal(L, c3, nb):
    """The restricted Helmholtz term with the diagonal it gives, for one and
    for several calculations, against the restriction alone, bit for bit; the
    boundary layer keeps its values and enters the diagonal."""
    f3 = tuple(2 * n - 1 for n in c3)
    nf, nc = int(np.prod(f3)), int(np.prod(c3))
    rng = np.random.default_rng(sum(c3) + nb)
    x, oC, out = rng.normal(size=nb * nf), rng.normal(size=nb * nc), rng.normal(size=nb * nc)
    ref = out.copy()
    for b in range(nb):
        r = ref[b * nc:(b + 1) * nc].copy()
        L.pmgtest_restrict(*f3, *c3, P(np.ascontiguousarray(x[b * nf:(b + 1) * nf])), P(r))
        sh = (c3[2], c3[1], c3[0])
        cut = (slice(1, -1),) * 3
        ref[b * nc:(b + 1) * nc].reshape(sh)[cut] = r.reshape(sh)[cut]
    D, Df = np.zeros(nb * nc), np.zeros(nb * nc, np.float32)
    fp = ctypes.POINTER(ctypes.c_float)
    assert L.pmgtest_restrict_diag(*f3, *c3, nb, P(x), P(oC), P(out), P(D),
                                   Df.ctypes.data_as(fp)) == 1
    assert np.array_equal(out, ref)
    assert np.array_equal(D, oC + ref)
    assert np.array_equal(Df, (oC + ref).astype(np.float32))


@pytest.mark.parametrize("word", [4, 8])
@pytest.mark.parametrize("c3", [(3, 3, 3), (4, 3, 5), (5, 9, 4), (34, 6, 7), (41, 17, 9)])
def test_prolongation_runs(L, c3, word):
    """x_f + damp P x_c in runs of 16 bytes against the terms added one by one
    in their order, bit for bit: rows of 5 points and up, a last run that
    leaves the row, the first run's boundary point, the boundary layer kept."""
    dt = np.float32 if word == 4 else np.float64
    f3 = tuple(2 * n - 1 for n in c3)
    rng = np.random.default_rng(sum(c3) + word)
    xc = np.zeros((c3[2], c3[1], c3[0]), dt)
    xc[1:-1, 1:-1, 1:-1] = rng.normal(size=tuple(n - 2 for n in xc.shape))
    xf = rng.normal(size=(f3[2], f3[1], f3[0])).astype(dt)
    damp = 0.8125 + rng.uniform(0, 0.1)
    k, j, i = np.meshgrid(*(np.arange(1, n - 1) for n in xf.shape), indexing="ij")
    w = (0.5 ** (i % 2 + j % 2 + k % 2)).astype(dt)
    v = np.zeros(i.shape, dt)
    for dz in (0, 1):
        for dy in (0, 1):
            for dx in (0, 1):
                on = (dx <= i % 2) & (dy <= j % 2) & (dz <= k % 2)
                c = xc[np.where(on, k // 2 + dz, 0), np.where(on, j // 2 + dy, 0),
                       np.where(on, i // 2 + dx, 0)]
                v = np.where(on, v + w * c, v)
    ref = xf.copy()
    ref[1:-1, 1:-1, 1:-1] = ref[1:-1, 1:-1, 1:-1] + dt(damp) * v
    got = np.ascontiguousarray(xf)
    ct = ctypes.POINTER(ctypes.c_float if word == 4 else ctypes.c_double)
    f = L.pmgtest_prolong32 if word == 4 else L.pmgtest_prolong
    assert f(*c3, *f3, xc.ctypes.data_as(ct), got.ctypes.data_as(ct), ctypes.c_double(damp)) == 1
    assert np.array_equal(got, ref)
