"""The QPI sums and the H00/H01 download at the edges of their tiles: moduli
around the 8 shifts of a thread and the row lengths where correlate_kernel's
launch shape changes, paths around the 8 shifts of a thread and the lengths
where the path no longer fits the staged layouts, both orders of the jdos
arrays, and more k points than one piece of the download holds."""
import ctypes

import numpy as np
import pytest

from wannier_tools_amd import model as M

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


@pytest.mark.gpu
@pytest.mark.parametrize("nk", [1, 2, 7, 8, 9, 16, 17, 127, 128, 129, 602, 603, 2048, 2049, 5120, 5121])
def test_kpath_jdos_at_path_edges(gpu, nk):
    """Both orders of the arrays against 80-bit sums of positive terms, within
    nk eps; energies on either side of the 16 and 4 staged at once."""
    for nom in (1, 5, 17) if nk <= 603 else (1, 5):
        print("path edges", nk, nom, flush=True)
        a = np.random.default_rng(nk + nom).uniform(0.1, 1.0, (2, nk, nom))
        h = (nk - 1) // 2
        want = np.zeros(a.shape)
        x = a[:, :2 * h + 1].astype(np.longdouble)
        for iq in range(nk) if nk <= 129 else (0, 1, h - 1, h, h + 1, nk - 9, nk - 2, nk - 1):
            s = iq + 1 - h
            lo, hi = max(0, -s), min(2 * h, 2 * h - s)
            if hi >= lo:
                want[:, iq] = (x[:, lo:hi + 1] * x[:, lo + s:hi + s + 1]).sum(axis=1)
        got = gpu.kpath_jdos(a)
        got_k = np.zeros((2, nom, nk))
        src = np.ascontiguousarray(a.transpose(0, 2, 1))
        p = lambda v: v.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        assert gpu.lib.wtsurf_kpath_jdos(gpu.ctx, nk, nom, 2, p(src), p(got_k)) == 0
        assert np.array_equal(got, got_k.transpose(0, 2, 1))
        nz = want > 0
        assert np.all(np.abs(got[nz] / want[nz] - 1) <= nk * EPS)
        if nk <= 129:
            assert np.all(got[~nz] == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("n,nk", [(3, 70), (16, 5), (200, 110)])
def test_ham_of_many_k_points(gpu, n, nk):
    """A whole list of k points (at n = 200 one pair to a piece of the download)
    against the points one by one, bit for bit."""
    print("ham", n, nk, flush=True)
    irvec, hr = M.synthetic_model(n, 1, 0.4, M.decay_l2(1.5), seed=n).surface_cell()
    gpu.set_model_arrays(n, 1, irvec, hr)
    k = np.random.default_rng(n).uniform(-0.5, 0.5, (nk, 2))
    h00, h01 = gpu.ham_qlayer2qlayer(k)
    assert h00.shape == h01.shape == (nk, n, n)
    for i in (0, 1, nk // 2, nk - 7 if nk > 7 else 0, nk - 1):
        a, b = gpu.ham_qlayer2qlayer(k[i])
        assert np.array_equal(a, h00[i]) and np.array_equal(b, h01[i])


@pytest.mark.gpu
def test_kpath_jdos_of_many_fields(gpu):
    """More fields than one launch has workgroups for (2^24 of 256 threads)."""
    nf = (1 << 24) + 5
    a = np.random.default_rng(0).uniform(0.1, 1.0, (nf, 3, 1))
    print("many fields", nf, flush=True)
    got = gpu.kpath_jdos(a)
    # shifts 0, 1, 2 of a path of three points
    want = np.stack([a[:, 0] ** 2 + a[:, 1] ** 2 + a[:, 2] ** 2, a[:, 0] * a[:, 1] + a[:, 1] * a[:, 2],
                     a[:, 0] * a[:, 2]], axis=1)
    assert np.all(np.abs(got / want - 1) <= 3 * EPS)


@pytest.mark.gpu
@pytest.mark.parametrize("nkx,nky,m1,m2,nfield", [(3, 2100, 2, 2060, 2), (2, 2049, 2, 2049, 1)])
def test_autocorrelation_of_long_second_axis(gpu, nkx, nky, m1, m2, nfield):
    """A second modulus beyond the library's row length, which the call then
    takes as columns."""
    print("long columns", nkx, nky, m1, m2, flush=True)
    a = np.random.default_rng(nky).uniform(0.1, 1.0, (nfield, nkx, nky))
    got = gpu.kplane_autocorrelation(a, m1, m2)
    want = correlation(a, m1, m2)
    tol = (nfield * m1 * m2 + nkx * nky / (m1 * m2)) * EPS
    assert np.abs(got / want - 1).max() <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("nk,nom,nfield", [(1, 1, 1), (15, 256, 1), (40, 256, 1), (40, 257, 1), (41, 3, 2),
                                           (5121, 2, 1), (5121, 11, 1), (10240, 2, 1), (10240, 7, 1), (10241, 3, 2),
                                           (10241, 7, 1)])
def test_kpath_jdos_where_the_kernel_changes(gpu, nk, nom, nfield):
    """Short paths of few rows, one workgroup's LDS, and paths beyond it in both
    orders: against 80-bit sums of positive terms, within nk eps."""
    print("jdos kernels", nk, nom, nfield, flush=True)
    a = np.random.default_rng(nk + nom).uniform(0.1, 1.0, (nfield, nk, nom))
    h = (nk - 1) // 2
    x = a[:, :2 * h + 1].astype(np.longdouble)
    got = gpu.kpath_jdos(a)
    src = np.ascontiguousarray(a.transpose(0, 2, 1))
    got_k = np.zeros_like(src)
    p = lambda v: v.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    assert gpu.lib.wtsurf_kpath_jdos(gpu.ctx, nk, nom, nfield, p(src), p(got_k)) == 0
    assert np.array_equal(got, got_k.transpose(0, 2, 1))
    for iq in sorted({0, 1 % nk, h, min(h + 1, nk - 1), max(nk - 2, 0), nk - 1, nk // 3}):
        s = iq + 1 - h
        lo, hi = max(0, -s), min(2 * h, 2 * h - s)
        if hi < lo:
            assert np.all(got[:, iq] == 0)
            continue
        want = (x[:, lo:hi + 1] * x[:, lo + s:hi + s + 1]).sum(axis=1)
        assert np.all(np.abs(got[:, iq] / want - 1) <= nk * EPS)


@pytest.mark.gpu
@pytest.mark.parametrize("nkx,nky,m1,m2,nfield", [(1, 40, 1, 39, 1), (2, 300, 2, 300, 1), (33, 40, 33, 31, 2),
                                                  (40, 33, 31, 33, 2), (200, 5, 129, 5, 3)])
def test_autocorrelation_of_narrow_rows(gpu, nkx, nky, m1, m2, nfield):
    """Narrow planes through the library in both orders of the axes, and the
    Python call, which takes the longer axis as rows."""
    print("narrow rows", nkx, nky, m1, m2, nfield, flush=True)
    a = np.random.default_rng(nkx + nky).uniform(0.1, 1.0, (nfield, nkx, nky))
    want = correlation(a, m1, m2)
    p = lambda v: v.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    lib, ctx = gpu.lib, gpu.ctx
    b = np.ascontiguousarray(a.transpose(0, 2, 1))
    c1, c2 = np.zeros((nkx, nky)), np.zeros((nky, nkx))
    assert lib.wtsurf_kplane_autocorrelation(ctx, nky, nkx, m2, m1, nfield, p(a), p(c1)) == 0
    assert lib.wtsurf_kplane_autocorrelation(ctx, nkx, nky, m1, m2, nfield, p(b), p(c2)) == 0
    tol = (nfield * m1 * m2 + nkx * nky / (m1 * m2)) * EPS
    for got in (gpu.kplane_autocorrelation(a, m1, m2), c1, c2.T):
        assert np.abs(got / want - 1).max() <= tol
