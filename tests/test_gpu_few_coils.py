"""2D gridding of 1 to 16 coils (NC2C waves of 8 coils, C2NC workgroups of 1, 2, 4
and 8): every coil count at which the launch changes or leaves lanes idle, every
kernel width with its own staging, several frames, samples per tile from none to
several blocks and split tiles, each kind of dcw, and accumulation.

Bar: relative L2 <= 1e-5 against the FP32 oracle, as the other 2D tests.
"""
import numpy as np
import pytest

from gadgetron_amd import DeviceArray, NFFT_conv_mode, NFFTPlan
from gadgetron_amd import NFFT_comp_mode as CM
from gadgetron_amd import trajectories as tj
from oracle import pyoracle as po
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-5


def traj_of(N, F, spokes):
    """Radial frames; the first samples of a frame gathered in one cell (a dense
    tile) and the last quarter dropped onto the grid edge, where windows wrap."""
    k = tj.golden_radial_2d(2 * max(N), spokes, frames=F).copy()
    M = k.shape[1]
    rng = np.random.default_rng(3)
    k[:, : M // 4] = 0.11 + 0.004 * rng.standard_normal((F, M // 4, 2))
    k[:, -M // 4:, 0] = np.clip(0.5 - 0.01 * rng.random((F, M // 4)), -0.5, 0.5)
    return k.astype(np.float32)


@pytest.mark.parametrize("C", [1, 2, 3, 4, 5, 8, 9, 13, 16])
@pytest.mark.parametrize("W", [3.5, 5.5, 6.5])
def test_coils_and_widths(C, W):
    print(f"{C} coils, W {W}", flush=True)
    N, F = [50, 44], 2
    k = traj_of(N, F, 24)
    M = k.shape[1]
    rng = np.random.default_rng(C)
    plan = NFFTPlan(N, [76, 66], W=W)
    plan.preprocess(DeviceArray.from_numpy(k))
    op = po.Plan(N, W, Nos=[76, 66], precision="float", cu=True)
    op.preprocess(k)
    shape = (C, F, N[1], N[0])
    smp, img = tj.complex_normal(rng, (C, F, M)), tj.complex_normal(rng, shape)
    for dcw in (None, tj.ramp_dcf(k), rng.random((C, F, M)).astype(np.float32)):
        d_w = None if dcw is None else DeviceArray.from_numpy(dcw)
        oi, os_ = DeviceArray.zeros(shape, np.complex64), DeviceArray.zeros((C, F, M), np.complex64)
        plan.compute(DeviceArray.from_numpy(smp), oi, d_w, CM.BACKWARDS_NC2C)
        plan.compute(DeviceArray.from_numpy(img), os_, d_w, CM.FORWARDS_C2NC)
        e1 = rel_l2(oi.numpy(), op.compute(smp, shape, po.BACKWARDS_NC2C, dcw=dcw))
        e2 = rel_l2(os_.numpy(), op.compute(img, (C, F, M), po.FORWARDS_C2NC, dcw=dcw))
        print(f"  adjoint {e1:.2e}, forward {e2:.2e}", flush=True)
        assert e1 <= TOL and e2 <= TOL


@pytest.mark.parametrize("C", [1, 6, 11])
def test_accumulate_and_repeat(C):
    N, F = [50, 44], 2
    k = traj_of(N, F, 24)
    M = k.shape[1]
    rng = np.random.default_rng(C)
    plan = NFFTPlan(N, [76, 66], W=5.5)
    plan.preprocess(DeviceArray.from_numpy(k))
    grid = tj.complex_normal(rng, (C, F, 66, 76))
    smp = tj.complex_normal(rng, (C, F, M))

    def conv(x, out0, mode, acc):
        out = DeviceArray.from_numpy(out0)
        plan.convolve(DeviceArray.from_numpy(x), out, mode, accumulate=acc)
        return out.numpy()

    for x, o, mode in ((grid, smp, NFFT_conv_mode.C2NC), (smp, grid, NFFT_conv_mode.NC2C)):
        plain = conv(x, np.zeros_like(o), mode, False)
        assert np.array_equal(plain, conv(x, np.full_like(o, 7), mode, False))
        # the sum is rounded once more than the plain result: half an ulp of each term
        assert rel_l2(conv(x, o, mode, True), plain + o) <= 2e-7
