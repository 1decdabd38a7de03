"""The FP64 rounds of orders up to 112 (inverse in registers, wave-strip GEMMs)
against the oracle where their tiling can go wrong: orders on either side of
every multiple of 8, a single instance (whose products are split over the
chip) against the same instance in a grid, more instances than slots, singular
and NaN columns in every panel position."""
import numpy as np
import pytest

from helpers import fp64_floor
from test_gpu_parity import _traces_within_floor
from wannier_tools_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 9, 17, 25, 33, 40, 41, 48, 49, 56, 57, 64, 65, 71, 72, 73,
                               79, 80, 81, 88, 89, 96, 97, 104, 105, 112, 113])
def test_orders_around_multiples_of_8(gpu, oracle_lib, n):
    print("mid order", n, flush=True)
    irvec, hr = M.synthetic_model(n, 1, 0.4, M.decay_l2(1.5), seed=600 + n).surface_cell()
    gpu.set_model_arrays(n, 1, irvec, hr)
    top = np.array(sorted({1, n}), dtype=np.int32)
    gpu.set_orbitals(top, top)
    rng = np.random.default_rng(n)
    kp, om = rng.uniform(-0.5, 0.5, (3, 2)), rng.uniform(-1, 1, 3) * M.EV2HARTREE
    eta = 2e-3 * M.EV2HARTREE
    gpu.set_schedule("rounds")
    try:
        out = gpu.spectral_grid(kp, om, eta)
        one = gpu.spectral_grid(kp[1:2], om[2:3], eta)
    finally:
        gpu.set_schedule("auto")
    assert not np.any(out[4])
    ref = oracle_lib.spectral(n, 1, irvec, hr, kp, om, eta, top, top)
    floor = fp64_floor(oracle_lib, n, 1, irvec, hr, kp, om, eta, top, top)
    _traces_within_floor(out[:3], ref[:3], floor)
    assert np.array_equal(out[3], ref[3])
    # alone on the chip, bit for bit the same
    for a, b in zip(one, out):
        assert a[0, 0] == b[1, 2]


def test_more_instances_than_slots(gpu):
    """9000 instances of order 34 (at most 4096 slots): each energy of the grid
    repeats, and the repeats agree bit for bit whatever slot they ran in."""
    irvec, hr = M.synthetic_model(17, 1, 0.4, M.decay_l2(1.5), seed=9).surface_cell()
    gpu.set_model_arrays(17, 2, irvec, hr)
    kp = np.random.default_rng(1).uniform(-0.5, 0.5, (30, 2))
    om = np.tile(np.linspace(-1.0, 1.0, 60) * M.EV2HARTREE, 5)
    out = gpu.spectral_grid(kp, om, 5e-3 * M.EV2HARTREE)
    assert not np.any(out[4])
    for a in out[:4]:
        for r in range(1, 5):
            assert np.array_equal(a[:, :60], a[:, 60 * r:60 * (r + 1)])


@pytest.mark.parametrize("n,c", [(40, 0), (72, 23), (72, 71), (77, 76), (80, 40), (81, 80),
                                 (108, 50), (112, 111)])
def test_zero_and_nan_pivot_columns(gpu, n, c):
    """Column c of omega - H00 exactly zero (eta = 0), or all NaN: every inverse
    is the identity, as the reference's inv leaves it."""
    print("singular", n, c, flush=True)
    e = np.random.default_rng(n).uniform(-0.5, 0.5, n) * M.EV2HARTREE
    zero = np.zeros((n, n), complex)
    for w, eta, h00 in ((e[c], 0.0, np.diag(e).astype(complex)),
                        (0.1, 1e-3, np.full((n, n), np.nan + 0j))):
        for g in gpu.surfgreen_1985(w, h00, zero, eta)[:3]:
            assert np.array_equal(g, np.eye(n))
