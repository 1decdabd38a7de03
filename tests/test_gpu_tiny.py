"""The wave-resident kernels of orders up to 16 against the oracle where their
layouts can go wrong: every order (tiles of 4 whole and partial, four instances
a wave and one), counts that leave a wave's instances unfilled, instances of one
wave that stop at different iterations, singular and NaN columns."""
import numpy as np
import pytest

from helpers import fp64_floor
from test_gpu_parity import _traces_within_floor
from test_gpu_spin import FLOOR_X, _spin_floor
from wannier_tools_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", range(1, 17))
def test_every_order(gpu, oracle_lib, n):
    """1210 instances (more than one a SIMD: four a wave up to order 8, the
    last wave with two) against the oracle on a part of them, and the same
    instances alone in their waves bit for bit."""
    print("tiny order", n, flush=True)
    irvec, hr = M.synthetic_model(n, 1, 0.4, M.decay_l2(1.5), seed=700 + n).surface_cell()
    gpu.set_model_arrays(n, 1, irvec, hr)
    top = np.array(sorted({1, n}), dtype=np.int32)
    gpu.set_orbitals(top, top)
    rng = np.random.default_rng(n)
    kp, om = rng.uniform(-0.5, 0.5, (2, 2)), rng.uniform(-1, 1, 605) * M.EV2HARTREE
    eta = 2e-3 * M.EV2HARTREE
    gpu.set_schedule("small")
    try:
        out = gpu.spectral_grid(kp, om, eta)
        few = gpu.spectral_grid(kp, om[-5:], eta)
        gpu.set_spin_traces("surfstat" if n > 1 else "off")
        gpu.spectral_grid(kp, om[-5:], eta)
        spin = gpu.spin_download() if n > 1 else None
    finally:
        gpu.set_schedule("auto")
        gpu.set_spin_traces("off")
    assert not np.any(out[4])
    ref = oracle_lib.spectral(n, 1, irvec, hr, kp, om[-5:], eta, top, top)
    floor = fp64_floor(oracle_lib, n, 1, irvec, hr, kp, om[-5:], eta, top, top)
    _traces_within_floor(few[:3], ref[:3], floor)
    assert np.array_equal(few[3], ref[3])
    for a, b in zip(few, out):
        assert np.array_equal(a, b[:, -5:])
    assert len(np.unique(out[3])) > 1  # lanes of one wave stopped at different iterations
    if n > 1:
        want = oracle_lib.spectral_spin(n, 1, irvec, hr, kp, om[-5:], eta, top, top, spin_mode=1)
        floor = _spin_floor(oracle_lib, n, 1, irvec, hr, kp, om[-5:], eta, top, top, 1, 1.0, want)
        for a, b in zip(spin, want[4:6]):
            assert np.abs(a - b).max() <= max(FLOOR_X * floor, 1e-12 * np.abs(b).max())


@pytest.mark.parametrize("n,c", [(1, 0), (3, 2), (4, 0), (5, 4), (8, 7), (9, 3), (12, 11), (16, 4)])
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
