"""The pivot of an elimination step is the largest |re| + |im| of the column by
the whole value, the lowest row on ties, on every kernel's inverse.

omega - H00 is i times the identity but for a 2 x 2 block

    [ d           B ]        d = 1e-10, B = 1e300
    [ d (1 + e)   d ]

whose first column has two entries that differ by e.  Elimination with the
second row stays in range; with the first one its B / d overflows and the
result is not finite.  The block's rows are taken in both orders."""
import numpy as np
import pytest

from wannier_tools_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def automatic_schedule(gpu):
    gpu.set_schedule("auto")

# the last bit of a value, the low and the high word of a double
STEPS = [2.0 ** -52, 2.0 ** -40, 2.0 ** -19, 2.0 ** -14]
D, B = 1e-10, 1e300


def _case(n, c, e, low):
    """omega - H00 and its inverse; low: the larger entry in row c."""
    x = np.eye(n, dtype=complex)
    inv = np.eye(n, dtype=complex)
    small, large = (c + 1, c) if low else (c, c + 1)
    f = 1.0 + e
    x[c:c + 2, c:c + 2] = 0
    x[small, c], x[small, c + 1] = D, B
    x[large, c], x[large, c + 1] = D * f, D
    # (D B-scaled determinant: D D is far below the last bit of D B)
    inv[c:c + 2, c:c + 2] = 0
    inv[c, large], inv[c, small] = 1.0 / (D * f), -1.0 / (B * f)
    inv[c + 1, small], inv[c + 1, large] = 1.0 / B, -1.0 / (B * f)
    return 1j * x, -1j * inv


@pytest.mark.parametrize("n,c", [(2, 0), (4, 1), (5, 0), (8, 5), (9, 4), (12, 10), (16, 13), (24, 9),
                                 (32, 30), (33, 25), (40, 0), (72, 69), (80, 34), (81, 72), (112, 110),
                                 (120, 61)])
def test_largest_entry_is_the_pivot(gpu, n, c):
    for e in STEPS:
        for low in (False, True):
            print("pivot", n, c, e, low, flush=True)
            x, want = _case(n, c, e, low)
            out = gpu.surfgreen_1985(0.0, -x, np.zeros((n, n), complex), 0.0)
            for g in out[:3]:
                assert np.abs(g - want).max() <= 1e-13 * np.abs(want).max()
                nz = want != 0
                assert np.abs(g[nz] / want[nz] - 1).max() <= 1e-13
            assert out[3] == 1


@pytest.mark.parametrize("n,c", [(2, 0), (3, 1), (4, 2), (5, 0), (6, 4), (8, 5), (16, 9)])
@pytest.mark.parametrize("low", [False, True])
def test_largest_entry_is_the_pivot_in_a_grid(gpu, n, c, low):
    """1100 instances (orders up to 8 then go four to a wave)."""
    for e in STEPS:
        print("pivot grid", n, c, e, low, flush=True)
        x, want = _case(n, c, e, low)
        gpu.set_model_arrays(n, 1, np.zeros((1, 3), dtype=np.int32), -x[None])
        out = gpu.spectral_grid(np.zeros((1, 2)), np.zeros(1100), 0.0)
        assert np.abs(out[2] / -np.trace(want).imag - 1).max() <= 1e-13
        assert np.all(out[3] == 1) and not np.any(out[4])


@pytest.mark.parametrize("n", [1, 2, 7, 16, 24, 40, 72, 112, 120])
@pytest.mark.parametrize("tiny", [2.0 ** -1074, 2.0 ** -1060, 2.0 ** -1037])
def test_denormal_pivot_is_no_singular_column(gpu, n, tiny):
    """Only a column without a positive entry is singular and gives the
    identity.  A denormal pivot's reciprocal overflows, and the couplings'
    sum is no number from there on: the iterations run to their limit."""
    print("denormal", n, tiny, flush=True)
    x = np.eye(n, dtype=complex)
    x[n - 1, n - 1] = tiny
    gpu.set_model_arrays(n, 1, np.zeros((1, 3), dtype=np.int32), -x[None])
    for count in (1, 1100) if n <= 8 else (1,):
        out = gpu.spectral_grid(np.zeros((1, 2)), np.zeros(count), 0.0)
        assert np.all(out[3] == M.DECIMATION_ITERMAX) and np.all(out[4] & 2)
