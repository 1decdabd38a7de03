"""The stop rule's sum |alpha'_ij| does not depend on how many instances a call
has: the sum after the first iteration, found to the last bit as the accuracy
at which the iteration ends, of an instance alone and among enough others that
the call takes the other launch shape (four instances a wave up to order 8;
products not spread beyond order 112)."""
import numpy as np
import pytest

from wannier_tools_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def automatic_schedule(gpu):
    gpu.set_schedule("auto")


def _first_sum(gpu, kp, om, eta):
    """The smallest accuracy with which the first instance takes one iteration."""
    lo, hi = 0, int(np.float64(1e10).view(np.int64))
    while hi - lo > 1:
        mid = (lo + hi) // 2
        gpu.set_stop_rule(2, float(np.int64(mid).view(np.float64)))
        it = gpu.spectral_grid(kp, om, eta)[3]
        assert np.all(it == it[0, 0])
        lo, hi = (lo, mid) if it[0, 0] == 1 else (mid, hi)
    return hi


@pytest.mark.parametrize("n,many", [(1, 1100), (2, 1100), (3, 1100), (4, 1100), (5, 1100), (6, 1100),
                                    (7, 1100), (8, 1100), (40, 70), (113, 206), (130, 206), (200, 206)])
def test_sum_is_the_same_alone_and_among_others(gpu, n, many):
    eta = 5e-3 * M.EV2HARTREE
    try:
        for seed in range(4 if n <= 8 else 2):
            print("stop sum", n, seed, flush=True)
            irvec, hr = M.synthetic_model(n, 1, 0.4, M.decay_l2(1.5), seed=900 + seed).surface_cell()
            gpu.set_model_arrays(n, 1, irvec, hr)
            kp = np.random.default_rng(seed).uniform(-0.5, 0.5, (1, 2))
            om = np.full(many, 0.1 * M.EV2HARTREE)
            assert _first_sum(gpu, kp, om[:1], eta) == _first_sum(gpu, kp, om, eta)
    finally:
        gpu.set_stop_rule()
