"""Parity of the HIP path (through the C ABI) with the reference and the oracle.

Bar: the Fourier sum to 1e-14 relative (device sincos vs libm); the FP64
decimation on the spectral traces A(k, omega) (dos_l, dos_r, dos_bulk) and on
single diagonal entries of G within a few times the FP64 floor of the case.
The floor is the recursion's own sensitivity: perturbing H(R) by one ulp
moves the oracle's traces by ~1e-12 at Ndim = 12 and 16 but by 1.2e-10 at
Ndim = 72 with eta = 1e-3 eV (test_oracle.py::test_fp64_floor_of_golden_cases
pins these numbers), so no FP64 implementation can promise a closer match
there than that.
"""
import numpy as np
import pytest

from helpers import LARGE_GOLDEN, chain_bulk_g, chain_surface_g, fp64_floor, golden_model, max_rel
from wannier_tools_amd import model as M
from wannier_tools_amd.surface import STATUS_NOT_CONVERGED, STATUS_SINGULAR, WtsurfError

pytestmark = pytest.mark.gpu

CASES = ["ndim16", "np3_ndim12", "ndim72"]
TOL_DIAG = {"ndim16": 1e-11, "np3_ndim12": 1e-11, "ndim72": 5e-10}
TOL_TRACE = {"ndim16": 1e-11, "np3_ndim12": 1e-11, "ndim72": 5e-10}
# Traces against the oracle: within FLOOR_X times the FP64 floor of the same
# inputs (helpers.fp64_floor), and never required below 1e-12.
FLOOR_X = 5.0


def _traces_within_floor(mine, ref, floor):
    errs = [max_rel(m, r) for m, r in zip(mine, ref)]
    _say("  max rel err vs oracle:", errs, "fp64 floor:", floor)
    assert max(errs) < max(FLOOR_X * floor, 1e-12)


def _say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("name", CASES)
def test_fourier_vs_reference_golden(gpu, golden, name):
    _say("fourier", name)
    g = golden(name)
    nw, np_, irvec, hr = golden_model(g, name)
    gpu.set_model_arrays(nw, np_, irvec, hr)
    h00, h01 = gpu.ham_qlayer2qlayer(g["kpts"])
    scale = np.max(np.abs(g["h00"]))
    assert np.max(np.abs(h00 - g["h00"])) < 1e-14 * scale
    assert np.max(np.abs(h01 - g["h01"])) < 1e-14 * scale


@pytest.mark.parametrize("name", CASES)
def test_surfgreen_1985_vs_reference_golden(gpu, golden, name):
    _say("surfgreen_1985", name)
    g = golden(name)
    for ik in range(g["kpts"].shape[0]):
        for iw, w in enumerate(g["omegas"]):
            gll, grr, gb, it = gpu.surfgreen_1985(w, g["h00"][ik], g["h01"][ik], float(g["eta"]))
            assert 1 <= it <= 100
            tol = TOL_DIAG[name]
            assert max_rel(np.diag(gll), g["diag_gll"][ik, iw]) < tol
            assert max_rel(np.diag(grr), g["diag_grr"][ik, iw]) < tol
            assert max_rel(np.diag(gb), g["diag_gb"][ik, iw]) < tol
    if "full_g" in g:
        gll, grr, gb, _ = gpu.surfgreen_1985(g["omegas"][0], g["h00"][0], g["h01"][0], float(g["eta"]))
        for mine, ref in zip((gll, grr, gb), g["full_g"]):
            assert np.max(np.abs(mine - ref)) < 1e-11 * np.max(np.abs(ref))


@pytest.mark.parametrize("name", CASES)
def test_spectral_grid_vs_reference_golden(gpu, golden, oracle_lib, name):
    _say("spectral_grid", name)
    g = golden(name)
    nw, np_, irvec, hr = golden_model(g, name)
    gpu.set_model_arrays(nw, np_, irvec, hr)
    dl, dr, db, its, st = gpu.spectral_grid(g["kpts"], g["omegas"], float(g["eta"]))
    tol = TOL_TRACE[name]
    errs = [max_rel(dl, g["dos_l"]), max_rel(dr, g["dos_r"]), max_rel(db, g["dos_bulk"])]
    _say("  max rel err dos_l, dos_r, dos_bulk vs reference:", errs)
    assert max(errs) < tol
    assert np.all(st == 0)
    top = M.default_top_orbitals(nw)
    *_, oits = oracle_lib.spectral(nw, np_, irvec, hr, g["kpts"], g["omegas"], float(g["eta"]), top, top)
    assert np.array_equal(its, oits)


@pytest.mark.parametrize("name", sorted(LARGE_GOLDEN))
def test_large_orders_vs_reference_golden(gpu, golden, name):
    """Orders beyond 80 (matrix in global memory, panel pairs, blocked GEMMs)
    against the reference's own surfgreen_1985: the spectral traces, and the
    diagonals of GLL, GRR, GB from surfgreen_1985 on the device's H00 / H01."""
    _say("large golden", name)
    g = golden(name)
    nw, np_, irvec, hr = golden_model(g, name)
    tol = LARGE_GOLDEN[name]
    gpu.set_model_arrays(nw, np_, irvec, hr)
    dl, dr, db, its, st = gpu.spectral_grid(g["kpts"], g["omegas"], float(g["eta"]))
    errs = [max_rel(dl, g["dos_l"]), max_rel(dr, g["dos_r"]), max_rel(db, g["dos_bulk"])]
    _say("  max rel err dos_l, dos_r, dos_bulk vs reference:", errs)
    assert max(errs) < tol["trace"]
    assert np.all(st == 0)
    h00, h01 = gpu.ham_qlayer2qlayer(g["kpts"])
    for ik in range(g["kpts"].shape[0]):
        for iw, w in enumerate(g["omegas"]):
            gll, grr, gb, it = gpu.surfgreen_1985(w, h00[ik], h01[ik], float(g["eta"]))
            assert it == its[ik, iw]
            for mine, ref in ((gll, g["diag_gll"]), (grr, g["diag_grr"]), (gb, g["diag_gb"])):
                assert max_rel(np.diag(mine), ref[ik, iw]) < tol["diag"]


def test_spectral_grid_ndim16_subgrid_vs_oracle(gpu, oracle_lib):
    """A 21 k x 41 omega slice of the Ndim = 16 k-path workload."""
    _say("subgrid ndim16")
    mdl = M.model_ndim16()
    irvec, hr = mdl.surface_cell()
    gpu.set_model_arrays(8, 2, irvec, hr)
    kp = M.kpath_slab([((-0.5, 0.0), (0.5, 0.0))], 201)[::10]
    om = M.omega_grid(-1.0, 1.0, 401)[::10] * M.EV2HARTREE
    eta = 1e-3 * M.EV2HARTREE
    dl, dr, db, its, st = gpu.spectral_grid(kp, om, eta)
    top = M.default_top_orbitals(8)
    odl, odr, odb, oits = oracle_lib.spectral(8, 2, irvec, hr, kp, om, eta, top, top)
    floor = fp64_floor(oracle_lib, 8, 2, irvec, hr, kp, om, eta, top, top)
    _traces_within_floor((dl, dr, db), (odl, odr, odb), floor)
    assert np.mean(its == oits) > 0.99


@pytest.mark.parametrize("nw,np_", [(1, 1), (3, 1), (5, 3), (12, 3), (40, 2)])
def test_uneven_orders_vs_oracle(gpu, oracle_lib, nw, np_):
    """Orders that are not multiples of the 16-wide MFMA tile, custom orbital lists,
    and the SurfaceDOSkk trace divisor pi."""
    _say("orders", nw, np_)
    mdl = M.synthetic_model(nw, 2, 0.4, M.decay_l2(1.5), seed=100 + nw)
    irvec, hr = mdl.surface_cell()
    gpu.set_model_arrays(nw, np_, irvec, hr)
    n = nw * np_
    top = np.array(sorted({1, n, (n + 1) // 2}), dtype=np.int32)
    bot = np.array(sorted({1, nw}), dtype=np.int32)
    gpu.set_orbitals(top, bot)
    rng = np.random.default_rng(nw)
    kp = rng.uniform(-0.5, 0.5, (3, 2))
    om = rng.uniform(-1, 1, 4) * M.EV2HARTREE
    eta = 4e-3 * M.EV2HARTREE
    dl, dr, db, its, st = gpu.spectral_grid(kp, om, eta, divisor=M.REF_PI)
    odl, odr, odb, oits = oracle_lib.spectral(nw, np_, irvec, hr, kp, om, eta, top, bot,
                                              divisor=M.REF_PI)
    floor = fp64_floor(oracle_lib, nw, np_, irvec, hr, kp, om, eta, top, bot, divisor=M.REF_PI)
    _traces_within_floor((dl, dr, db), (odl, odr, odb), floor)


@pytest.mark.parametrize("nw,np_", [(12, 2), (13, 3), (20, 2), (11, 5), (28, 2), (33, 2),
                                     (35, 2), (37, 2)])
def test_half_last_tile_row_orders_vs_oracle(gpu, oracle_lib, nw, np_):
    """Round-schedule orders whose last 16-row tile holds at most 8 real rows
    (n = 24, 39, 40, 55, 56, 66, 70; the round GEMMs then stack the last tile
    row of both products into one MFMA tile) and n = 74 just past that bound,
    with the last orbital in the traced lists, against the oracle."""
    n = nw * np_
    _say("orders", nw, np_, "n", n)
    mdl = M.synthetic_model(nw, 2, 0.4, M.decay_l2(1.5), seed=300 + n)
    irvec, hr = mdl.surface_cell()
    gpu.set_model_arrays(nw, np_, irvec, hr)
    top = np.array(sorted({1, n - 1, n}), dtype=np.int32)
    bot = np.array(sorted({1, nw}), dtype=np.int32)
    gpu.set_orbitals(top, bot)
    rng = np.random.default_rng(n)
    kp = rng.uniform(-0.5, 0.5, (3, 2))
    om = rng.uniform(-1, 1, 4) * M.EV2HARTREE
    eta = 2e-3 * M.EV2HARTREE
    gpu.set_schedule("rounds")
    try:
        dl, dr, db, its, st = gpu.spectral_grid(kp, om, eta)
    finally:
        gpu.set_schedule("auto")
    assert not np.any(st)
    odl, odr, odb, oits = oracle_lib.spectral(nw, np_, irvec, hr, kp, om, eta, top, bot)
    floor = fp64_floor(oracle_lib, nw, np_, irvec, hr, kp, om, eta, top, bot)
    _traces_within_floor((dl, dr, db), (odl, odr, odb), floor)
    assert np.array_equal(its, oits)


@pytest.mark.parametrize("nw,np_", [(48, 2), (50, 2), (36, 3), (65, 2), (67, 3), (72, 3),
                                     (125, 2), (144, 2), (152, 2), (160, 2), (168, 2), (192, 2)])
def test_large_orders_vs_oracle(gpu, oracle_lib, nw, np_):
    """Orders beyond 80, where the Gauss-Jordan matrix lives in global memory
    and the GEMMs run in blocks: Ndim 96 (Q 6), 100 (Q 7, 12 pad rows), 108
    (Q 7), 130 (Q 9, 14 pad rows), 201 (Q 13: panel quads, a last panel of one
    column), 216 (Q 14; the largest order of the mixed-model set, a last quad
    of three panels), 250 (Q 16: quads, a last panel of two columns), 288 (Q
    18; the 144-orbital spinful k-plane model), 304 (Q 19, pairs again), 320
    (Q 20, five full row sets in the panel), 336 (Q 21, the first with six) and
    384 (Q 24, the largest order built), with custom orbital lists and the
    trace divisor pi."""
    _say("large orders", nw, np_)
    mdl = M.synthetic_model(nw, 2, 0.5, M.decay_l2(1.5), seed=200 + nw)
    irvec, hr = mdl.surface_cell()
    gpu.set_model_arrays(nw, np_, irvec, hr)
    n = nw * np_
    top = np.array(sorted({1, 2, n // 3, n}), dtype=np.int32)
    bot = np.array(sorted({1, nw // 2, nw}), dtype=np.int32)
    gpu.set_orbitals(top, bot)
    kp = np.array([[0.13, -0.21], [-0.4, 0.05]])
    om = np.array([-0.3, 0.05]) * M.EV2HARTREE
    eta = 2e-2 * M.EV2HARTREE
    dl, dr, db, its, st = gpu.spectral_grid(kp, om, eta, divisor=M.REF_PI)
    odl, odr, odb, oits = oracle_lib.spectral(nw, np_, irvec, hr, kp, om, eta, top, bot,
                                              divisor=M.REF_PI)
    assert np.all(st == 0)
    assert np.array_equal(its, oits)
    floor = fp64_floor(oracle_lib, nw, np_, irvec, hr, kp, om, eta, top, bot, divisor=M.REF_PI,
                       draws=2)
    _traces_within_floor((dl, dr, db), (odl, odr, odb), floor)


def test_large_order_surfgreen_full_g(gpu, oracle_lib):
    """surfgreen_1985 at Ndim 216: the full GLL, GRR, GB from the global-memory
    inverse against the oracle."""
    _say("large surfgreen")
    mdl = M.synthetic_model(72, 2, 0.5, M.decay_l2(1.5), seed=272)
    irvec, hr = mdl.surface_cell()
    gpu.set_model_arrays(72, 3, irvec, hr)
    h00, h01 = gpu.ham_qlayer2qlayer(np.array([[0.2, 0.1]]))
    w, eta = 0.1 * M.EV2HARTREE, 2e-2 * M.EV2HARTREE
    gll, grr, gb, it = gpu.surfgreen_1985(w, h00[0], h01[0], eta)
    ogll, ogrr, ogb, oit, info = oracle_lib.surfgreen_1985(w, eta, h00[0], h01[0])
    assert info == 0 and it == oit
    for mine, ref in zip((gll, grr, gb), (ogll, ogrr, ogb)):
        assert np.max(np.abs(mine - ref)) < 1e-10 * np.max(np.abs(ref))


def test_order_beyond_largest_kernel_fails(gpu):
    from wannier_tools_amd import surface
    nmax = surface.max_ndim()
    assert nmax >= 288
    mdl = M.synthetic_model(nmax // 2 + 1, 1, 0.3, M.decay_l1, seed=5)
    irvec, hr = mdl.surface_cell()
    gpu.set_model_arrays(nmax // 2 + 1, 2, irvec, hr)
    with pytest.raises(WtsurfError):
        gpu.spectral_grid([[0.0, 0.0]], [0.0], 1e-3)


def test_chain_closed_form_on_device(gpu):
    _say("chain")
    e0, t = 0.2 * M.EV2HARTREE, -0.8 * M.EV2HARTREE
    for w_ev in (-1.7, 0.0, 2.5):
        z = w_ev * M.EV2HARTREE + 2e-3j * M.EV2HARTREE
        gll, grr, gb, it = gpu.surfgreen_1985(z.real, np.array([[e0]]), np.array([[t]]), z.imag)
        gs = chain_surface_g(z, e0, t)
        assert abs(gll[0, 0] - gs) < 1e-9 * abs(gs) and abs(grr[0, 0] - gs) < 1e-9 * abs(gs)
        gbk = chain_bulk_g(z, e0, t)
        assert abs(gb[0, 0] - gbk) < 1e-9 * abs(gbk)


def test_block_diagonal_chains_on_device(gpu):
    """72 independent chains (diagonal H00, H01): exact answers at the headline order."""
    _say("diag chains")
    n = 72
    rng = np.random.default_rng(2)
    e0 = rng.uniform(-0.5, 0.5, n) * M.EV2HARTREE
    t = rng.uniform(0.3, 0.9, n) * M.EV2HARTREE * rng.choice([-1, 1], n)
    w, eta = 0.17 * M.EV2HARTREE, 1e-3 * M.EV2HARTREE
    gll, grr, gb, it = gpu.surfgreen_1985(w, np.diag(e0).astype(complex), np.diag(t).astype(complex), eta)
    z = w + 1j * eta
    for i in range(n):
        gs = chain_surface_g(z, e0[i], t[i])
        assert abs(gll[i, i] - gs) < 1e-8 * abs(gs)
        gbk = chain_bulk_g(z, e0[i], t[i])
        assert abs(gb[i, i] - gbk) < 1e-8 * abs(gbk)


def test_singular_in_a_later_panel_quad(gpu):
    """A zero pivot column in the middle of a panel quad (Ndim 200, column 150
    of X = omega - H00 exactly zero with eta = 0): every inverse comes back as
    the identity with the singular bit, as the reference's inv leaves it."""
    _say("singular at order 200")
    n = 200
    rng = np.random.default_rng(5)
    e = rng.uniform(-0.5, 0.5, n) * M.EV2HARTREE
    w = e[150]
    gll, grr, gb, it = gpu.surfgreen_1985(w, np.diag(e).astype(complex), np.zeros((n, n), complex), 0.0)
    for g in (gll, grr, gb):
        assert np.array_equal(g, np.eye(n))


def test_status_singular_and_not_converged(gpu, oracle_lib):
    """eta = 0, H01 = 0 and omega on an eigenvalue of H00: exactly singular
    solve -> identity result and the singular bit.  itermax = 2 on an in-band
    energy -> the not-converged bit."""
    _say("status")
    h00 = np.diag([0.25, -0.5]).astype(complex)
    h01 = np.zeros((2, 2), complex)
    gll, grr, gb, it = gpu.surfgreen_1985(0.25, h00, h01, 0.0)
    assert np.array_equal(gb, np.eye(2))
    mdl = M.model_ndim16()
    irvec, hr = mdl.surface_cell()
    gpu.set_model_arrays(8, 2, irvec, hr)
    gpu.set_stop_rule(2, M.DECIMATION_ACCURACY)
    try:
        dl, dr, db, its, st = gpu.spectral_grid([[0.1, 0.0]], [0.01], 1e-5)
    finally:
        gpu.set_stop_rule()
    assert its[0, 0] == 2 and (st[0, 0] & STATUS_NOT_CONVERGED)


def test_new_model_resets_orbital_lists(gpu, oracle_lib):
    """Orbital lists set for one model must not leak into the next (bottom
    indices past the new Num_wann would read outside the layer)."""
    _say("orbital reset")
    big = M.synthetic_model(8, 1, 0.3, M.decay_l1, seed=3)
    irvec, hr = big.surface_cell()
    gpu.set_model_arrays(8, 2, irvec, hr)
    gpu.set_orbitals([1, 16], [8])
    small = M.synthetic_model(4, 1, 0.3, M.decay_l1, seed=4)
    irvec, hr = small.surface_cell()
    gpu.set_model_arrays(4, 3, irvec, hr)
    kp, om, eta = [[0.1, 0.2]], [0.01, -0.02], 5e-3 * M.EV2HARTREE
    dl, dr, db, its, st = gpu.spectral_grid(kp, om, eta)
    top = M.default_top_orbitals(4)
    odl, odr, odb, _ = oracle_lib.spectral(4, 3, irvec, hr, kp, om, eta, top, top)
    floor = fp64_floor(oracle_lib, 4, 3, irvec, hr, kp, om, eta, top, top)
    _traces_within_floor((dl, dr, db), (odl, odr, odb), floor)


def test_invalid_arguments_raise(gpu):
    _say("invalid")
    mdl = M.model_ndim16()
    irvec, hr = mdl.surface_cell()
    gpu.set_model_arrays(8, 2, irvec, hr)
    with pytest.raises(WtsurfError):
        gpu.set_orbitals([0], [1])
    gpu.set_orbitals(M.default_top_orbitals(8), M.default_top_orbitals(8))
    with pytest.raises(WtsurfError):
        gpu.set_orbitals([1], [9])  # bottom index beyond Num_wann
    gpu.set_orbitals(M.default_top_orbitals(8), M.default_top_orbitals(8))
    with pytest.raises(WtsurfError):
        gpu.set_stop_rule(0, 1e-16)
    big = np.zeros((400, 400), complex)
    with pytest.raises(WtsurfError):
        gpu.surfgreen_1985(0.0, big, big, 1e-3)


@pytest.mark.parametrize("name", CASES)
def test_fp32_measurement_mode_runs(gpu, golden, name):
    """WTSURF_FP32 (FP32 working precision, no refinement) is a speed/accuracy
    measurement mode, not a path offered at the 1e-6 bar: the doubling
    recursion alpha <- alpha g alpha amplifies its rounding far past 1e-6 on
    A(k, omega) at Ndim 72.  This only checks that it runs: every trace
    positive and finite, no status bits, iteration counts within one of the
    FP64 path's."""
    _say("fp32 mode", name)
    g = golden(name)
    nw, np_, irvec, hr = golden_model(g, name)
    gpu.set_model_arrays(nw, np_, irvec, hr)
    d64 = gpu.spectral_grid(g["kpts"], g["omegas"], float(g["eta"]), precision="fp64")
    d32 = gpu.spectral_grid(g["kpts"], g["omegas"], float(g["eta"]), precision="fp32")
    _say("  fp32 max rel err on dos_l, dos_r, dos_bulk:",
         [max_rel(a, b) for a, b in zip(d32[:3], d64[:3])])
    for a in d32[:3]:
        assert np.all(np.isfinite(a)) and np.all(a > 0)
    assert np.all(np.abs(d32[3] - d64[3]) <= 1)
    assert np.all(d32[4] == 0)


def test_fp32_path_refused_beyond_order_80(gpu, golden):
    """FP32 working precision is refused beyond Ndim 80, where the doubling
    recursion in FP32 diverges on some instances (on the Ndim 216 and 288
    golden cases a numpy complex64 emulation overflows, and the device runs hit
    itermax or settle on wrong values); the FP64 path runs as usual."""
    _say("fp32 refused", "ndim216")
    g = golden("ndim216")
    nw, np_, irvec, hr = golden_model(g, "ndim216")
    gpu.set_model_arrays(nw, np_, irvec, hr)
    with pytest.raises(WtsurfError, match="FP32"):
        gpu.spectral_grid(g["kpts"], g["omegas"], float(g["eta"]), precision="fp32")
    d64 = gpu.spectral_grid(g["kpts"], g["omegas"], float(g["eta"]), precision="fp64")
    assert np.all(d64[4] == 0)


def test_surfgreen_1985_during_grid_run_keeps_grid_results(gpu, golden):
    """A per-instance surfgreen_1985 issued while a grid run is still in flight
    waits for it and uses buffers of its own: the grid run's results come out
    as a run alone gives them, and the per-instance result is unchanged."""
    _say("surfgreen_1985 during an async grid run")
    g = golden("ndim16")
    nw, np_, irvec, hr = golden_model(g, "ndim16")
    gpu.set_model_arrays(nw, np_, irvec, hr)
    kp = M.kpath_slab([((-0.5, 0.0), (0.5, 0.0))], 64)
    om = M.omega_grid(-1.0, 1.0, 64) * M.EV2HARTREE
    eta = float(g["eta"])
    alone = gpu.spectral_grid(kp, om, eta)
    one_alone = gpu.surfgreen_1985(float(g["omegas"][0]), g["h00"][0], g["h01"][0], eta)
    gpu.upload_grid(kp, om)
    gpu.run_async(eta)
    one = gpu.surfgreen_1985(float(g["omegas"][0]), g["h00"][0], g["h01"][0], eta)
    gpu.sync()
    after = gpu.download()
    for a, b in zip(after, alone):
        assert np.array_equal(a, b)
    for a, b in zip(one[:3], one_alone[:3]):
        assert np.array_equal(a, b)
    assert one[3] == one_alone[3]


def test_download_after_model_change_fails(gpu, golden):
    """A new model or a ham_qlayer2qlayer call drops the last grid run: its
    download raises instead of returning zeros."""
    _say("stale download")
    g = golden("ndim16")
    nw, np_, irvec, hr = golden_model(g, "ndim16")
    gpu.set_model_arrays(nw, np_, irvec, hr)
    gpu.spectral_grid(g["kpts"], g["omegas"], float(g["eta"]))
    gpu.set_model_arrays(nw, np_, irvec, hr)
    with pytest.raises(WtsurfError, match="no completed run"):
        gpu.lib_download_raw(4096)
    gpu.spectral_grid(g["kpts"], g["omegas"], float(g["eta"]))
    gpu.ham_qlayer2qlayer(g["kpts"])
    with pytest.raises(WtsurfError, match="no completed run"):
        gpu.lib_download_raw(4096)


@pytest.mark.parametrize("name", CASES)
def test_persistent_schedule_vs_rounds_and_oracle(gpu, golden, oracle_lib, name):
    """The persistent schedule (register-resident all-wave inverse, same GEMMs)
    against the round schedule and the oracle: grid traces, spin traces, a
    per-instance batch with uneven eta and surfgreen_1985's full G, each within
    the FP64 floor bar of the case; iteration counts and status equal."""
    _say("persistent vs rounds", name)
    g = golden(name)
    nw, np_, irvec, hr = golden_model(g, name)
    gpu.set_model_arrays(nw, np_, irvec, hr)
    kp = M.kpath_slab([((-0.5, 0.0), (0.5, 0.0))], 40)
    om = M.omega_grid(-1.0, 1.0, 37) * M.EV2HARTREE
    eta = float(g["eta"])
    rng = np.random.default_rng(3)
    nb = 60
    ki = rng.integers(0, kp.shape[0], nb).astype(np.int32)
    wi = rng.uniform(-1.0, 1.0, nb) * M.EV2HARTREE
    ei = 10.0 ** rng.uniform(-4.0, -2.0, nb) * M.EV2HARTREE
    out = {}
    try:
        for sched in ("rounds", "persistent"):
            gpu.set_schedule(sched)
            gpu.set_spin_traces("surfstat")
            grid = gpu.spectral_grid(kp, om, eta)
            spin = gpu.spin_download()
            gpu.set_spin_traces("off")
            batch = gpu.spectral_batch(kp, ki, wi, ei)
            full = gpu.surfgreen_1985(float(g["omegas"][0]), g["h00"][0], g["h01"][0], eta)
            out[sched] = dict(grid=grid, spin=spin, batch=batch, full=full)
    finally:
        gpu.set_schedule("rounds")
        gpu.set_spin_traces("off")
    top = M.default_top_orbitals(nw)
    ref = oracle_lib.spectral(nw, np_, irvec, hr, kp, om, eta, top, top)
    floor = fp64_floor(oracle_lib, nw, np_, irvec, hr, kp, om, eta, top, top)
    bar = max(FLOOR_X * floor, 1e-12)
    r, p = out["rounds"], out["persistent"]
    errs = [max_rel(a, b) for a, b in zip(p["grid"][:3], ref[:3])]
    _say("  persistent vs oracle:", errs, "floor", floor)
    assert max(errs) < bar
    assert max(max_rel(a, b) for a, b in zip(p["grid"][:3], r["grid"][:3])) < bar
    assert np.array_equal(p["grid"][3], ref[3]) and np.all(p["grid"][4] == 0)
    for a, b in zip(p["spin"], r["spin"]):
        assert np.max(np.abs(a - b)) <= bar * max(np.max(np.abs(b)), 1e-300)
    # the batch, instance by instance against the oracle within 5x that
    # instance's floor (eta down to 1e-4 eV: floors up to ~1e-8)
    for t in range(nb):
        one = oracle_lib.spectral(nw, np_, irvec, hr, kp[ki[t]], wi[t:t + 1], ei[t], top, top)
        fl = fp64_floor(oracle_lib, nw, np_, irvec, hr, kp[ki[t]], wi[t:t + 1], ei[t], top, top,
                        draws=6)
        for q in range(3):
            assert abs(p["batch"][q][t] - one[q][0, 0]) <= max(FLOOR_X * fl, 1e-12) * abs(one[q][0, 0])
        assert p["batch"][3][t] == one[3][0, 0]
    assert np.all(p["batch"][4] == 0)
    for a, b in zip(p["full"][:3], r["full"][:3]):
        assert np.max(np.abs(a - b)) <= bar * np.max(np.abs(b))
    assert p["full"][3] == r["full"][3]


@pytest.mark.parametrize("name", CASES)
def test_mixed_precision_vs_reference_golden(gpu, golden, name):
    """WTSURF_MIXED against the reference's own traces: within 1e-6."""
    _say("mixed precision vs golden", name)
    g = golden(name)
    nw, np_, irvec, hr = golden_model(g, name)
    gpu.set_model_arrays(nw, np_, irvec, hr)
    dl, dr, db, its, st = gpu.spectral_grid(g["kpts"], g["omegas"], float(g["eta"]),
                                            precision="mixed")
    errs = [max_rel(dl, g["dos_l"]), max_rel(dr, g["dos_r"]), max_rel(db, g["dos_bulk"])]
    _say("  max rel err on dos_l, dos_r, dos_bulk:", errs)
    assert max(errs) <= 1e-6
    assert np.all(st == 0)


@pytest.mark.parametrize("nw,np_,seed", [(8, 1, 40), (16, 2, 41), (36, 2, 42)])
def test_mixed_precision_low_eta_batch_vs_oracle(gpu, oracle_lib, nw, np_, seed):
    """WTSURF_MIXED on per-instance batches with eta log-uniform in
    [1e-4, 1e-2] eV (the mixed-model set's models at Ndim 8, 32 and 72):
    every instance within 1e-6 of the oracle."""
    _say("mixed precision batch", nw, np_)
    irvec, hr = M.synthetic_model(nw, 2, 0.5, M.decay_l2(1.5), seed=seed).surface_cell()
    gpu.set_model_arrays(nw, np_, irvec, hr)
    rng = np.random.default_rng(seed)
    nb = 64
    kp = rng.uniform(-0.5, 0.5, (16, 2))
    ki = rng.integers(0, 16, nb).astype(np.int32)
    wi = rng.uniform(-1.0, 1.0, nb) * M.EV2HARTREE
    ei = 10.0 ** rng.uniform(-4.0, -2.0, nb) * M.EV2HARTREE
    dl, dr, db, its, st = gpu.spectral_batch(kp, ki, wi, ei, precision="mixed")
    assert np.all(st == 0)
    top = M.default_top_orbitals(nw)
    worst = 0.0
    for t in range(nb):
        one = oracle_lib.spectral(nw, np_, irvec, hr, kp[ki[t]], wi[t:t + 1], ei[t], top, top)
        for q, mine in enumerate((dl, dr, db)):
            worst = max(worst, abs(mine[t] - one[q][0, 0]) / abs(one[q][0, 0]))
    _say("  max rel err vs oracle:", worst)
    assert worst <= 1e-6


@pytest.mark.parametrize("nw,np_", [(4, 2), (24, 1), (36, 2), (40, 2)])
@pytest.mark.parametrize("schedule", ["rounds", "persistent", "auto"])
def test_mixed_precision_is_fp64_on_the_automatic_schedule(gpu, nw, np_, schedule):
    """Whatever schedule is set, a mixed run is the automatic FP64 run."""
    _say("mixed schedule", nw, np_, schedule)
    irvec, hr = M.synthetic_model(nw, 1, 0.4, M.decay_l2(1.5), seed=nw).surface_cell()
    gpu.set_model_arrays(nw, np_, irvec, hr)
    rng = np.random.default_rng(nw)
    kp, om = rng.uniform(-0.5, 0.5, (3, 2)), rng.uniform(-1, 1, 5) * M.EV2HARTREE
    eta = 2e-3 * M.EV2HARTREE
    gpu.set_schedule("auto")
    want = gpu.spectral_grid(kp, om, eta)
    gpu.set_schedule(schedule)
    try:
        got = gpu.spectral_grid(kp, om, eta, precision="mixed")
    finally:
        gpu.set_schedule("auto")
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
