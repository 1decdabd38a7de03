"""Orders beyond 112 with few instances, whose products' row blocks are spread
over the chip, against the same instances among enough others that they are
not: bit for bit, at orders with two, three and five row blocks."""
import numpy as np
import pytest

from wannier_tools_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [113, 130, 150, 257])
def test_spread_rows_bit_for_bit(gpu, n):
    print("spread", n, flush=True)
    irvec, hr = M.synthetic_model(n, 1, 0.4, M.decay_l2(1.5), seed=800 + n).surface_cell()
    gpu.set_model_arrays(n, 1, irvec, hr)
    kp = np.random.default_rng(n).uniform(-0.5, 0.5, (2, 2))
    om = np.linspace(-1.0, 1.0, 110) * M.EV2HARTREE  # 110 a set: not spread
    eta = 5e-3 * M.EV2HARTREE
    out = gpu.spectral_grid(kp, om, eta)
    assert not np.any(out[4])
    for cols in ([3], [0, 50, 109]):
        few = gpu.spectral_grid(kp, om[cols], eta)
        for a, b in zip(few, out):
            assert np.array_equal(a, b[:, cols])
