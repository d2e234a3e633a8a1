"""The wave-number factor of the round-trip matrix (M = FᵀF, log det(1 - FᵀF) =
log det(1 - F Fᵀ)) on the GPU, through the C ABI: the banded Gram matrix
against the matrix M itself and against the Gram matrix run dense through
the LU's kernels, at the edges of its tiles, chunks and windows.

Tolerance.  M comes from the same rows F.  numpy's eigenvalues of M carry an
absolute error of about N eps ||M|| <= N eps tr M, so Σ log1p(-λ) carries N eps
relative to tr M <= |log det|/1, times 1/(1 - λ_max) (below 20 here); the
band's left-out elements, the window and the factorization add less than
1e-13: 20 N eps + 1e-12.  Dense against banded Gram matrix: the same
elements, factored in another order, D <= 600 rows: 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.2e-16


@pytest.fixture(scope="module")
def ca():
    import caps_amd
    caps_amd.lib()
    return caps_amd


def make(ca, rbyl, ldim, metal, detalg=None):
    c = ca.Caps(rbyl * 1e-6, 1e-6, ldim=ldim, detalg=detalg)
    if metal:
        c.set_drude(9.0, 0.035)
    return c


# ldim 1 .. 17: fewer degrees than a chunk of 16, one more than one; 24 more
# than 1.5 chunks; m above ldim and far from the window's start (lmin > m);
# ξ = 900: e^{-ξ} is not a double; ξ = 1e-3: nodes up to x = 1e5; R/L = 0.5
CASES = [(20, 120, 1.0, 0, 0), (20, 120, 1.0, 1, 1), (20, 121, 0.3, 3, 0), (1, 1, 0.1, 0, 0), (2, 2, 0.5, 1, 1),
         (2, 16, 0.5, 0, 1), (2, 17, 0.5, 2, 0), (4, 24, 2.0, 5, 0), (0.5, 20, 0.2, 1, 0), (10, 60, 1e-3, 0, 1),
         (10, 60, 1e-3, 2, 0), (300, 700, 2.0, 90, 0), (500, 300, 1.0, 60, 1), (500, 900, 900.0, 0, 0),
         (500, 900, 900.0, 4, 1), (100, 503, 30.0, 12, 1), (60, 360, 0.01, 7, 0)]


@pytest.mark.parametrize("rbyl,ldim,xi,m,metal", CASES)
def test_band_matches_matrix(ca, rbyl, ldim, xi, m, metal):
    c = make(ca, rbyl, ldim, metal)
    v, tr, fl = c.logdetD_batch([xi], [m], info=True)
    M, _, _ = c.matrix(xi, m)
    assert np.array_equal(M, M.T)
    t = np.trace(M)
    assert abs(tr[0] / t - 1) < 1e-12, (tr[0], t)
    if abs(t) < 1e-8:
        assert (fl[0] & 3) == 1 and v[0] == -tr[0]
        return
    lam = np.linalg.eigvalsh(M)
    assert lam[-1] < 0.95
    ref = float(np.sum(np.log1p(-lam)))
    assert fl[0] == 4 and abs(v[0] / ref - 1) < 20 * len(M) * EPS + 1e-12, (v[0], ref)


def test_band_matches_dense_gram(ca):
    """The same Gram matrix through the LU's kernels: a schedule fixed by
    capsx_lu_config runs the symmetric delta form, CAPS_AMD_LU_SYM=0 the
    general one (the whole matrix); LU mode with its Mercator rule."""
    import os
    from caps_amd import autotune as at
    for rbyl, ldim, metal, detalg in ((20, 120, 0, None), (50, 251, 1, "LU"), (200, 1200, 1, None)):
        c = make(ca, rbyl, ldim, metal, detalg)
        ms = list(range(0, 40, 3))
        xs = [0.8 * rbyl] * len(ms)
        v, tr, fl = c.logdetD_batch(xs, ms, info=True)
        try:
            at.set_config(1, 1, 0, 128)
            w, tw, fw = c.logdetD_batch(xs, ms, info=True)
        finally:
            at.set_config(0)
        os.environ["CAPS_AMD_LU_SYM"] = "0"
        try:
            g, _, fg = c.logdetD_batch(xs, ms, info=True)
        finally:
            os.environ.pop("CAPS_AMD_LU_SYM")
        assert np.array_equal(tr, tw) and np.array_equal(fl, fw) and np.array_equal(fl, fg)
        assert np.max(np.abs(w / v - 1)) < 1e-12 and np.max(np.abs(g / v - 1)) < 1e-12


def test_band_batch_equals_single(ca):
    """Partial sums of a block run alone (its chunks spread over workgroups)
    and of a large batch (one workgroup per strip) are the same bits, and so
    are batches of mixed geometries."""
    a, b = make(ca, 40, 240, 1), make(ca, 90, 470, 0)
    objs = [a, b] * 40
    xs = np.repeat(np.linspace(0.5, 60, 40), 2)
    ms = np.arange(80) % 23
    v = ca.logdetD_multi(objs, xs, ms)
    for i in range(0, 80, 7):
        assert objs[i].logdetD(xs[i], int(ms[i])) == v[i], i


def test_cholesky_mode_takes_the_matrix(ca):
    """CHOLESKY, whose shortcut rule looks at the lower triangle of M, factors
    M itself; the same determinants as the Gram matrix (rounding of an LU of N
    rows: 20 N eps + 1e-12)."""
    c, h = make(ca, 30, 150, 1, "CHOLESKY"), make(ca, 30, 150, 1)
    ms = [0, 1, 2, 5, 9]
    v, w = c.logdetD_batch([1.5] * 5, ms), h.logdetD_batch([1.5] * 5, ms)
    assert np.max(np.abs(v / w - 1)) < 20 * 300 * EPS + 1e-12


@pytest.mark.parametrize("rbyl,ldim", [(0.05, 5), (0.2, 5), (0.5, 8), (1, 12), (2, 20), (5, 40), (12, 80)])
def test_few_tiles(ca, rbyl, ldim):
    """Windows of 1 to some 15 tile columns: the two halves of the band have
    none, one, or one column more than the other before they meet."""
    from caps_amd import autotune as at
    c = make(ca, rbyl, ldim, 1)
    ms = [m for m in range(13) if m <= ldim - 1]
    xs = [0.4] * len(ms)
    v, tr, fl = c.logdetD_batch(xs, ms, info=True)
    try:
        at.set_config(1, 1, 0, 128)
        w, tw, fw = c.logdetD_batch(xs, ms, info=True)
    finally:
        at.set_config(0)
    assert np.array_equal(tr, tw) and np.array_equal(fl, fw)
    assert np.max(np.abs(v / w - 1)) < 1e-12


def test_results_and_times_from_the_kernels(ca):
    """Results and stage times are stored by the kernels: batches of one and
    of many blocks in turn (the buffers grow), factored and not, eager and as
    graphs, give the same bits, and the stages add up to the whole."""
    c = make(ca, 40, 240, 1)
    xs, ms = np.linspace(0.5, 300, 300), np.arange(300) % 60
    one = [c.logdetD(xs[i], int(ms[i])) for i in (0, 7, 59, 150)]
    v, _, fl = c.logdetD_batch(xs, ms, info=True)
    assert {f & 3 for f in fl} == {0, 1}
    assert one == [v[i] for i in (0, 7, 59, 150)]
    t = c.last_timing()
    parts = [t[k] for k in ("mie", "K", "I", "assemble", "lu")]
    assert min(parts) >= 0 and abs(sum(parts) - t["total"]) < 1e-9 and 0.01 < t["total"] < 100
    c.set_graph(1)
    for _ in range(3):
        assert np.array_equal(c.logdetD_batch(xs, ms), v)
        assert c.logdetD(xs[7], 7) == v[7]


@pytest.mark.parametrize("epsm1,rbyl,ldim,xi,m", [(10, 0.1, 10, 0.03, 0), (10, 0.1, 10, 0.03, 1), (10.7, 1, 20, 0.03, 0),
                                                  (10.7, 1, 20, 0.03, 1), (10.7, 5, 40, 0.02, 1)])
def test_grid_dielectrics_small_xi(ca, epsm1, rbyl, ldim, xi, m):
    """Dielectrics at small ξ, whose Fresnel coefficients have singularities
    near the integration path, against the oracle's adaptive quadrature (within
    2e-14 of a grid of step 0.05 on these blocks).  Tolerance: the trapezoidal
    rule of step 0.45 is off by at most 1.1e-12 here (step 0.5: 5.6e-12 to
    2.0e-11), the sums and the Mie coefficients add some 1e-13."""
    import pyoracle as po
    c = ca.Caps(rbyl * 1e-6, 1e-6, ldim=ldim)
    w = xi * 299792458.0 / ((rbyl + 1) * 1e-6)
    wp = (2 * epsm1) ** 0.5 * w   # a Drude metal with γ = ξ: ε - 1 = ωp²/(2 ξ²)
    c.set_drude(wp * ca.HBAR_EV, w * ca.HBAR_EV)
    o = po.caps(rbyl * 1e-6, 1e-6, ldim=ldim, drude=(wp, w))
    v, ref = c.logdetD(xi, m), po.logdetD(o, xi, m)
    print("relative difference %.1e" % (v / ref - 1))
    assert abs(v / ref - 1) < 2e-12, (v, ref)


@pytest.mark.parametrize("detalg", [None, "LU"])
def test_grid_of_the_caller(ca, detalg):
    """CAPS_AMD_QUAD_H and CAPS_AMD_QUAD_V0 reach the determinants.  With step
    0.2 the trapezoidal rule is exact to rounding, what is left against the
    oracle are the sums and the Mie coefficients (3e-13; the default step's own
    error is 6.0e-13 and 1.0e-12 on these blocks).  A grid from v = -4 on leaves
    out part of the integral near x = 1: other values; one from -25.3 on is the
    same rule with its nodes shifted, off by the default's error again."""
    import os
    import pyoracle as po
    c = ca.Caps(0.1e-6, 1e-6, ldim=10, detalg=detalg)
    w = 0.03 * 299792458.0 / 1.1e-6
    wp = 20 ** 0.5 * w
    c.set_drude(wp * ca.HBAR_EV, w * ca.HBAR_EV)
    o = po.caps(0.1e-6, 1e-6, ldim=10, drude=(wp, w), detalg=1 if detalg else 0)
    ref = np.array([po.logdetD(o, 0.03, m) for m in (0, 1)])

    def with_env(name, value):
        os.environ[name] = value
        try:
            return c.logdetD_batch([0.03, 0.03], [0, 1])
        finally:
            os.environ.pop(name)
    v = c.logdetD_batch([0.03, 0.03], [0, 1])
    fine = with_env("CAPS_AMD_QUAD_H", "0.2")
    print("step 0.2: %s" % (fine / ref - 1))
    assert np.max(np.abs(fine / ref - 1)) < 3e-13
    assert not np.any(with_env("CAPS_AMD_QUAD_V0", "-4") == v)
    assert np.max(np.abs(with_env("CAPS_AMD_QUAD_V0", "-25.3") / v - 1)) < 3e-12
    assert np.array_equal(v, c.logdetD_batch([0.03, 0.03], [0, 1]))


def test_fine_grid_matches_default(ca):
    """A step of 0.1 (whose rows of F are wider than the band) on blocks where
    the default step is exact to 2e-14: same values to the rounding of an LU of
    N rows (20 N eps + 1e-12); LU mode with its Mercator rule, and re-run with
    the pivoted LU."""
    import os
    L = ca.lib()
    for rbyl, ldim, metal, detalg in ((20, 120, 1, None), (50, 251, 0, "LU")):
        c = make(ca, rbyl, ldim, metal, detalg)
        ms, xs = list(range(0, 40, 3)), [0.8 * rbyl] * 14
        v, tr, fl = c.logdetD_batch(xs, ms, info=True)
        os.environ["CAPS_AMD_QUAD_H"] = "0.1"
        try:
            w, tw, fw = c.logdetD_batch(xs, ms, info=True)
            old = L.capsx_lu_delta_mode(0)
            try:
                p, _, _ = c.logdetD_batch(xs, ms, info=True)
            finally:
                L.capsx_lu_delta_mode(old)
        finally:
            os.environ.pop("CAPS_AMD_QUAD_H")
        assert np.array_equal(fl, fw) and 0 < np.sum((fl & 3) == 0)
        assert np.max(np.abs(tw / tr - 1)) < 1e-12
        tol = 40 * ldim * EPS + 1e-12
        assert np.max(np.abs(w / v - 1)) < tol and np.max(np.abs(p - v)) < tol * np.abs(v).max()


def test_sequences_keep_the_arena_budget(ca, capfd):
    """A batch of many distinct frequencies and two geometries in launch
    sequences of a small budget: the arena is allocated once, with the budget
    (the Mie tables, 36 bytes per degree, object and frequency, are within it;
    with the pivoted re-run in sequences of its own a second time), and the values are the bits
    of one sequence.  The re-run with the pivoted LU: the rounding of an LU of N
    <= 640 rows in other schedules, 640 eps + 1e-12 of the largest value."""
    import os
    import re
    L = ca.lib()

    def run(budget, pivoted):
        a, b = make(ca, 20, 120, 1), make(ca, 31, 187, 0)
        n = 40 if pivoted else 300
        xs, ms = np.linspace(0.3, 9.3, n), np.arange(n) % 5
        os.environ["CAPS_AMD_PROGRESS"] = "1"
        if budget:
            os.environ["CAPS_AMD_ARENA_GB"] = str(budget)
        old = L.capsx_lu_delta_mode(0 if pivoted else 1)
        try:
            v = ca.logdetD_multi([a, b] * (n // 2), xs, ms)
        finally:
            L.capsx_lu_delta_mode(old)
            os.environ.pop("CAPS_AMD_PROGRESS")
            os.environ.pop("CAPS_AMD_ARENA_GB", None)
        sizes = [float(x) for x in re.findall(r"capsx: arena ([0-9.]+) GB", capfd.readouterr().err)]
        return v, a.stats()["batches"], sizes   # (a runs the batch: objs[0])

    for budget, pivoted in ((0.010, False), (0.017, False), (0.040, True)):
        v, n1, s1 = run(None, pivoted)
        w, n2, s2 = run(budget, pivoted)
        print("budget %g: %d sequences, arenas %s GB; without: %d, %s GB" % (budget, n2, s2, n1, s1))
        assert n1 == 1 + pivoted and n2 >= 4
        assert len(s2) <= 1 + pivoted and max(s2) <= budget + 1e-9, s2
        if pivoted:
            assert np.max(np.abs(w - v)) < (640 * EPS + 1e-12) * np.abs(v).max()
        else:
            assert np.array_equal(v, w)


def test_more_blocks_than_a_grid_takes(ca):
    """66000 blocks: kernels have the block in the grid's y or z (at most 65535),
    so they run in two launch sequences, with the bits of smaller batches."""
    c = ca.Caps(0.2e-6, 1e-6, ldim=3)
    n = 66000
    xs, ms = 0.2 + 1e-5 * (np.arange(n) // 3), np.arange(n) % 3
    v = c.logdetD_batch(xs, ms)
    assert c.stats(reset=True)["batches"] == 2
    # (the library runs a batch's blocks in order of m: the last of m = 2 are the second sequence's)
    for s in (slice(0, 300), slice(32000, 32300), slice(n - 300, n)):
        assert np.array_equal(v[s], c.logdetD_batch(xs[s], ms[s]))
    assert np.all(v < 0)


def test_every_small_number_of_tile_columns(ca):
    """k_band_ldl against the dense Gram matrix with the number of tile columns
    looked at (from the flops that the statistics count for a band): 1 to 6,
    where there is only the middle, 7, where one half has a column, and odd and
    even numbers above.  Fewer than 6 come from coarse grids of the same
    blocks; either side has the same G.  D <= 260 rows: 1e-12."""
    import os
    from caps_amd import autotune as at

    def flops(T):
        N, w = 16.0 * T, min(16.0 * T, 96.0)
        return (N - w) * w * (w + 2) + w ** 3 / 3 + w * w / 2 - 5 * w / 6
    number = {round(flops(T)): T for T in range(1, 30)}
    seen = set()
    try:
        for h in ("0.45", "0.9", "1.5", "2.5", "6"):
            os.environ["CAPS_AMD_QUAD_H"] = h
            for rbyl, ldim in ((1, 12), (5, 40), (20, 120)):
                c = make(ca, rbyl, ldim, 1)
                ms = list(range(7))
                v = []
                for m in ms:
                    c.stats(reset=True)
                    v.append(c.logdetD(0.4, m))
                    s = c.stats()
                    assert s["blocks_factored"] == 1
                    seen.add(number[round(s["lu_flops"])])
                try:
                    at.set_config(1, 1, 0, 128)
                    w = c.logdetD_batch([0.4] * 7, ms)
                finally:
                    at.set_config(0)
                assert np.max(np.abs(np.array(v) / w - 1)) < 1e-12, (h, rbyl)
    finally:
        os.environ.pop("CAPS_AMD_QUAD_H")
    print("tile columns:", sorted(seen))
    assert seen >= set(range(1, 15))
