"""Runs on a card whose memory other work holds: the rounds up to order 112 take
a workspace for up to sixteen slots a CU, and run with fewer where it does not
fit."""
import ctypes

import numpy as np
import pytest

from hipmem import DeviceBuffer, _hip
from wannier_tools_amd import model as M
from wannier_tools_amd.surface import SurfaceGF

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def automatic_schedule(gpu):
    gpu.set_schedule("auto")

GIB = 1 << 30


def free_memory():
    hip = _hip()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.fixture
def fill():
    """fill(left): hold device memory until about `left` bytes are free."""
    held = []

    def hold(left):
        while free_memory() > left + (64 << 20):
            held.append(DeviceBuffer(min(16 * GIB, free_memory() - left)))
    yield hold
    for b in held:
        b.free()


@pytest.mark.parametrize("left", [3 * GIB, GIB // 2])
def test_rounds_with_little_memory_left(gpu, fill, left):
    """4200 instances of order 112 (7.4 GB of workspace for 4096 slots, a
    quarter of 3 GiB free, and half a GiB, which the smallest plan tried first
    does not fit either): bit for bit the run with all slots."""
    n = 112
    irvec, hr = M.synthetic_model(n, 1, 0.4, M.decay_l2(1.5), seed=112).surface_cell()
    kp = np.random.default_rng(2).uniform(-0.5, 0.5, (30, 2))
    om = np.linspace(-1.0, 1.0, 140) * M.EV2HARTREE
    eta = 5e-3 * M.EV2HARTREE
    ctx = SurfaceGF(0)
    try:
        gpu.set_model_arrays(n, 1, irvec, hr)
        want = gpu.spectral_grid(kp, om, eta)
        ctx.set_model_arrays(n, 1, irvec, hr)
        ctx.upload_grid(kp, om)
        fill(left)
        before = free_memory()
        print("little memory", left, before, flush=True)
        for _ in range(2):
            got = ctx.spectral_grid(kp, om, eta)
            for a, b in zip(got, want):
                assert np.array_equal(a, b)
        if left > GIB:
            assert before - free_memory() < left // 2  # leaves memory to others
    finally:
        ctx.close()


def test_qpi_sums_give_large_buffers_back(gpu):
    """A path whose fields take 0.6 GB on the device, and a plane of 0.5 GB:
    what the calls keep afterwards is bounded."""
    rng = np.random.default_rng(3)
    path, plane = rng.uniform(0.0, 1.0, (1, 21, 1_800_000)), rng.uniform(0.0, 1.0, (1, 2, 16_000_000))
    gpu.kpath_jdos(path[:, :, :100])
    before = free_memory()
    gpu.kpath_jdos(path)
    assert before - free_memory() <= 300 << 20
    gpu.kplane_autocorrelation(plane, 2, 2048)
    assert before - free_memory() <= 300 << 20


def test_hamiltonians_with_little_memory_left(gpu, fill):
    """A list of k points whose H00 and H01 fit the card with little beside them:
    bit for bit as with memory to spare."""
    n, nk = 96, 500
    irvec, hr = M.synthetic_model(n, 1, 0.4, M.decay_l2(1.5), seed=96).surface_cell()
    k = np.random.default_rng(4).uniform(-0.5, 0.5, (nk, 2))
    gpu.set_model_arrays(n, 1, irvec, hr)
    want = gpu.ham_qlayer2qlayer(k)
    ctx = SurfaceGF(0)
    try:
        ctx.set_model_arrays(n, 1, irvec, hr)
        fill(200 << 20)  # 147 MB of H00 and H01
        print("little memory", free_memory(), flush=True)
        got = ctx.ham_qlayer2qlayer(k)
    finally:
        ctx.close()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
