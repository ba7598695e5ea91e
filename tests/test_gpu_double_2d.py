"""Double-precision 2D gridding over 8 x 8 tiles (NC2C) and 16 lanes a sample
(C2NC): grids whose last tile is short, small grids whose windows come back to
their first tile, every window class (windows of 9 cells gather with the general
kernel), coil counts around the register chunks, dense (split) and empty tiles.

Bar: relative L2 <= 1e-10 against the FP64 oracle, as the other double tests.
"""
import numpy as np
import pytest

from gadgetron_amd import DeviceArray, NFFT_conv_mode, NFFTPlan
from gadgetron_amd import NFFT_comp_mode as CM
from oracle import pyoracle as po
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nos,W", [([12, 10], 5.5), ([16, 24], 2.5), ([34, 42], 5.5), ([46, 30], 7.5), ([50, 36], 8.5),
                                   ([34, 42], 3.5), ([46, 30], 4.5), ([50, 36], 6.5)])
@pytest.mark.parametrize("C", [1, 4, 5, 9])
def test_double_2d(Nos, W, C):
    print(f"N_os {Nos}, W {W}, {C} coils", flush=True)
    N, F, M = [n * 2 // 3 // 2 * 2 for n in Nos], 2, 2500
    rng = np.random.default_rng(C)
    k = rng.uniform(-0.5, 0.5, (F, M, 2))
    k[0, :1500] = 0.2 + 0.02 * k[0, :1500]
    k[1, :4] = [[0.5, 0.5], [-0.5, 0.5], [0.5, -0.5], [-0.5, -0.5]]
    plan = NFFTPlan(N, Nos, W=W, precision="double")
    plan.preprocess(DeviceArray.from_numpy(k))
    op = po.Plan(N, W, Nos=Nos, precision="double", cu=True)
    op.preprocess(k)
    shape = (C, F, N[1], N[0])
    smp = rng.standard_normal((C, F, M)) + 1j * rng.standard_normal((C, F, M))
    img = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    for dcw in (None, rng.random((F, M)), rng.random((C, F, M))):
        d_w = None if dcw is None else DeviceArray.from_numpy(dcw)
        oi, os_ = DeviceArray.zeros(shape, np.complex128), DeviceArray.zeros((C, F, M), np.complex128)
        plan.compute(DeviceArray.from_numpy(smp), oi, d_w, CM.BACKWARDS_NC2C)
        plan.compute(DeviceArray.from_numpy(img), os_, d_w, CM.FORWARDS_C2NC)
        e1 = rel_l2(oi.numpy(), op.compute(smp, shape, po.BACKWARDS_NC2C, dcw=dcw))
        e2 = rel_l2(os_.numpy(), op.compute(img, (C, F, M), po.FORWARDS_C2NC, dcw=dcw))
        print(f"  adjoint {e1:.2e}, forward {e2:.2e}", flush=True)
        assert e1 <= 1e-10 and e2 <= 1e-10


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_bad_sample_stays_in_its_window(bad):
    print(f"double 2D 64^2, 5 coils, one sample {bad}", flush=True)
    rng = np.random.default_rng(1)
    nos, C, W, M, j = 96, 5, 5.5, 3000, 11
    k = rng.uniform(-0.5, 0.5, (1, M, 2))
    plan = NFFTPlan([64, 64], None, W=W, os_factor=1.5, precision="double")
    plan.preprocess(DeviceArray.from_numpy(k))
    x = rng.standard_normal((C, 1, M)) + 1j * rng.standard_normal((C, 1, M))
    y = x.copy()
    y[3, 0, j] = bad
    outs = []
    for s in (x, y):
        out = DeviceArray.zeros((C, 1, nos, nos), np.complex128)
        plan.convolve(DeviceArray.from_numpy(s), out, NFFT_conv_mode.NC2C)
        outs.append(out.numpy()[:, 0])
    a, b = outs
    hit = np.zeros((nos, nos), bool)
    win = [np.arange(np.ceil(p - W / 2), np.floor(p + W / 2) + 1).astype(int) % nos for p in (k[0, j] + 0.5) * nos]
    hit[np.ix_(win[1], win[0])] = True
    assert not np.isfinite(b[3][hit]).any()
    assert np.array_equal(a[3][~hit], b[3][~hit])
    assert np.array_equal(np.delete(a, 3, 0), np.delete(b, 3, 0))
