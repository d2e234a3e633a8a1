"""The pivoted LU's panels on the GPU against numpy, at the edges of the panel
kernel's variants (rows per lane, lanes, leaves of 16 columns, panels of 64),
over the schedules, with equal pivot candidates, and with columns of zeros or NaN.

Tolerance.  The matrices are a permutation times 2 plus a Gaussian one over
√N: singular values within about [1, 3], and elimination has to exchange rows
in nearly every column.  Both sides' log|det| carry N eps times the condition
and the pivots' growth (below 100 together).
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


def mats(n, N, seed):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, N, N)) / np.sqrt(N)
    for a in A:
        a[np.arange(N), rng.permutation(N)] += 2 * rng.choice([-1, 1], N)
    return A


@pytest.mark.parametrize("N", [1, 2, 15, 17, 63, 64, 65, 81, 128, 200, 256, 257, 512, 513, 576, 1024, 1025, 1100])
def test_sizes(ca, N):
    A = mats(2, N, N)
    v = ca.lu_logdet_batch(A)
    assert np.max(np.abs(v - np.linalg.slogdet(A)[1])) < 100 * N * EPS


@pytest.mark.parametrize("N", [2049, 2561, 3073])
def test_tall(ca, N):
    A = mats(1, N, N)
    assert abs(ca.lu_logdet_batch(A)[0] - np.linalg.slogdet(A)[1][0]) < 100 * N * EPS


@pytest.mark.parametrize("levels", [1, 2, 3, 4])
def test_schedules(ca, levels):
    from caps_amd import autotune as at
    A = mats(3, 700, levels)
    try:
        at.set_config(levels, 1, 0, 128)
        v = ca.lu_logdet_batch(A)
    finally:
        at.set_config(0)
    assert np.max(np.abs(v - np.linalg.slogdet(A)[1])) < 100 * 700 * EPS


def test_equal_candidates_and_degenerate_columns(ca):
    H = np.array([[1.0]])
    while len(H) < 256:
        H = np.block([[H, H], [H, -H]])
    Z, Q = mats(2, 256, 5)
    Z[:, 100] = 0
    Q[:, 37] = np.nan
    v = ca.lu_logdet_batch(np.stack([H, Z, Q]))
    assert abs(v[0] - 128 * np.log(256)) < 100 * 256 * EPS
    assert not np.isfinite(v[1])   # a pivot of exactly 0
    assert np.isnan(v[2])


def test_more_matrices_than_a_grid_takes(ca):
    """66000 matrices of one panel: the grid's y and z take 65535, its x more.
    (Some of so many are nearly singular: each by its own condition.)"""
    A = mats(66000, 3, 11)
    v = ca.lu_logdet_batch(A)
    assert np.all(np.abs(v - np.linalg.slogdet(A)[1]) < 100 * 3 * EPS * np.linalg.cond(A))
