"""The k-plane autocorrelation at the edges of its tiles: moduli around the 8
shifts of a thread and the row lengths where the launch shape changes."""
import numpy as np
import pytest

EPS = np.finfo(np.float64).eps


def correlation(a, m1, m2):
    """C and the bound sum |terms|, over the folded plane in 80-bit arithmetic."""
    nf, nkx, nky = a.shape
    e = np.zeros((nf, m1, m2), dtype=np.longdouble)
    for x in range(nkx):
        for y in range(nky):
            e[:, x % m1, y % m2] += a[:, x, y]
    out = np.empty((m1, m2), dtype=np.longdouble)
    corner = a[:, :m1, :m2].astype(np.longdouble)
    for p1 in range(m1):
        r = np.roll(corner, -p1, axis=1)
        for p2 in range(m2):
            out[p1, p2] = (e * np.roll(r, -p2, axis=2)).sum()
    return out[np.ix_(np.arange(nkx) % m1, np.arange(nky) % m2)]


@pytest.mark.gpu
@pytest.mark.parametrize("nkx,nky,m1,m2,nfield", [
    (3, 70, 3, 70, 2), (70, 3, 69, 3, 1), (7, 65, 7, 64, 3), (5, 66, 4, 65, 1), (9, 129, 8, 128, 1),
    (2, 257, 2, 257, 2), (3, 300, 2, 290, 1), (2, 1100, 2, 1030, 1), (1, 2048, 1, 2048, 2),
    (2100, 3, 2049, 2, 1), (8, 8, 1, 1, 1)])
def test_autocorrelation_at_row_edges(gpu, nkx, nky, m1, m2, nfield):
    """All terms positive, so that each order of the n = nfield m1 m2 products
    and of their folds is within (n + folds) eps of the sum."""
    print("row edges", nkx, nky, m1, m2, nfield, flush=True)
    a = np.random.default_rng(nkx * nky + m1).uniform(0.1, 1.0, (nfield, nkx, nky))
    if m1 > 2048:  # longer rows than the library takes
        with pytest.raises(RuntimeError, match="too large"):
            gpu.kplane_autocorrelation(a, m1, m2)
        return
    got = gpu.kplane_autocorrelation(a, m1, m2)
    want = correlation(a, m1, m2)
    tol = (nfield * m1 * m2 + nkx * nky / (m1 * m2)) * EPS
    assert np.abs(got / want - 1).max() <= tol
    # a NaN reaches every sum that has it as a term, an infinity likewise
    a[0, nkx - 1, nky - 1] = np.inf
    assert not np.isfinite(gpu.kplane_autocorrelation(a, m1, m2)).any()
