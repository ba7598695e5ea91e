"""Rounding error of the gridding kernels, each coil for itself, against float64 sums
over the same float weights (tests/cpp/kb_weights.cpp) at positions that floats
hold exactly, so that neither the positions nor the weights' own error hide the
sums'.  Coils of one magnitude, and coils down to 1e-7 of the largest: a coil's
error does not depend on the others.

Bars (relative 2-norm of a coil).  FP32 sums: a rounding to nearest is 2^-24 / sqrt(3)
of its binade's top, 2.4e-8 of a value on average; a cell or sample of the sizes
here sees two in each product and, chain by chain, half of the at most 16 terms at
full size: 2.4e-8 sqrt(2 + 8) = 7.6e-8, 1e-7 with some room.  Operands split into
two fp16 halves (3D) lose the last bit of a quarter of the values: 4.4e-8 each of
the sample and the weights, with the sums' 6e-8 8.6e-8: 1.2e-7.
"""
import ctypes
import os

import numpy as np
import pytest

from gadgetron_amd import DeviceArray, NFFT_conv_mode, NFFTPlan

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
FP32, SPLIT = 1e-7, 1.2e-7


def weights(p, nos, W):
    """First cell and float weights (as doubles) of the windows at positions p."""
    lib = ctypes.CDLL(os.path.join(HERE, "cpp", "libkbweights.so"))
    p = np.ascontiguousarray(p, np.float32)
    KW = int(np.floor(W)) + 1
    first, w = np.zeros(len(p), np.int32), np.zeros((len(p), KW), np.float32)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    lib.kb_weights(ptr(p), len(p), ctypes.c_float(nos), ctypes.c_float(W), ctypes.c_float(1.5), KW, ptr(first), ptr(w))
    return first, w.astype(np.float64)


def gridding(D, N, W, M, seed):
    """Trajectory, and functions that grid / gather one coil in float64."""
    rng = np.random.default_rng(seed)
    nos = N * 3 // 2
    k = (rng.integers(-512, 512, (M, D)) / 1024).astype(np.float32)
    per = [weights((k[:, d] + np.float32(0.5)) * np.float32(nos), nos, W) for d in range(D)]
    cells, vals = np.zeros((M, 1), np.int64), np.ones((M, 1))
    for d in reversed(range(D)):  # x runs fastest
        c = (per[d][0][:, None] + np.arange(per[d][1].shape[1])) % nos
        cells = (cells[:, :, None] * nos + c[:, None, :]).reshape(M, -1)
        vals = (vals[:, :, None] * per[d][1][:, None, :]).reshape(M, -1)

    def to_grid(s):
        g = np.zeros(nos ** D, np.complex128)
        np.add.at(g, cells.ravel(), (vals * s.astype(np.complex128)[:, None]).ravel())
        return g

    def to_samples(g):
        return (g.astype(np.complex128)[cells] * vals).sum(axis=1)

    return k, nos, to_grid, to_samples


def errors(D, N, W, C, M, mode, unequal):
    k, nos, to_grid, to_samples = gridding(D, N, W, M, 5)
    rng = np.random.default_rng(C)
    plan = NFFTPlan([N] * D, None, W=W, os_factor=1.5)
    plan.preprocess(DeviceArray.from_numpy(k[None]))
    gain = 10.0 ** -(np.arange(C) % 8) if unequal else np.ones(C)
    n = M if mode == NFFT_conv_mode.NC2C else nos ** D
    x = ((rng.standard_normal((C, n)) + 1j * rng.standard_normal((C, n))) * gain[:, None]).astype(np.complex64)
    shapes = (C, 1, M), (C, 1) + (nos,) * D
    if mode == NFFT_conv_mode.C2NC:
        shapes = shapes[::-1]
    out = DeviceArray.zeros(shapes[1], np.complex64)
    plan.convolve(DeviceArray.from_numpy(x.reshape(shapes[0])), out, mode)
    got = out.numpy().reshape(C, -1)
    ref = to_grid if mode == NFFT_conv_mode.NC2C else to_samples
    e = []
    for c in range(C):
        r = ref(x[c])
        e.append(float(np.linalg.norm(got[c] - r) / np.linalg.norm(r)))
    print(f"{D}D W {W} {C} coils {mode.name} unequal {unequal}: {max(e):.2e}", flush=True)
    return e


@pytest.mark.parametrize("unequal", [False, True])
@pytest.mark.parametrize("C", [1, 3, 8])
def test_3d_nc2c(C, unequal):
    assert max(errors(3, 32, 5.5, C, 3000, NFFT_conv_mode.NC2C, unequal)) <= SPLIT


@pytest.mark.parametrize("unequal", [False, True])
@pytest.mark.parametrize("C", [1, 3, 8])
@pytest.mark.parametrize("W", [3.0, 5.5, 6.5])
def test_2d_nc2c_few_coils(W, C, unequal):
    assert max(errors(2, 64, W, C, 4000, NFFT_conv_mode.NC2C, unequal)) <= FP32


def test_2d_nc2c_few_coils_dense():
    # 2900 entries a tile: items of 512, 110 terms a cell in each, in chains of at most
    # 4 of 16 entries, pairs of those and 16 pairs: 2.4e-8 sqrt(2 + 2 + 1 + 8) = 8.7e-8
    assert max(errors(2, 32, 5.5, 8, 40000, NFFT_conv_mode.NC2C, True)) <= 1.3 * FP32


@pytest.mark.parametrize("M", [300, 9000])  # one chunk a tile; several, and split tiles
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_2d_nc2c_bad_sample_stays_in_its_window(M, bad):
    # cells whose window does not hold the sample, and other coils, are as without it
    print(f"2D 64^2, {M} samples, 8 coils, one sample {bad}", flush=True)
    rng = np.random.default_rng(M)
    nos, C, W, j = 96, 8, 5.5, 17
    k = rng.uniform(-0.5, 0.5, (1, M, 2)).astype(np.float32)
    k[0, : M // 2] *= 0.1
    plan = NFFTPlan([64, 64], None, W=W, os_factor=1.5)
    plan.preprocess(DeviceArray.from_numpy(k))
    x = (rng.standard_normal((C, 1, M)) + 1j * rng.standard_normal((C, 1, M))).astype(np.complex64)
    y = x.copy()
    y[3, 0, j] = bad
    outs = []
    for s in (x, y):
        out = DeviceArray.zeros((C, 1, nos, nos), np.complex64)
        plan.convolve(DeviceArray.from_numpy(s), out, NFFT_conv_mode.NC2C)
        outs.append(out.numpy()[:, 0])
    a, b = outs
    hit = np.zeros((nos, nos), bool)
    win = [np.arange(np.ceil(p - W / 2), np.floor(p + W / 2) + 1).astype(int) % nos
           for p in (k[0, j] + np.float32(0.5)) * np.float32(nos)]
    hit[np.ix_(win[1], win[0])] = True
    assert np.array_equal(np.delete(a, 3, 0), np.delete(b, 3, 0))
    assert not np.isfinite(b[3][hit]).any()
    assert np.isfinite(b[3][~hit]).all()
    # those of the same tiles are summed again, in another order
    assert np.linalg.norm(b[3][~hit] - a[3][~hit]) <= 2 * FP32 * np.linalg.norm(a[3])


@pytest.mark.parametrize("unequal", [False, True])
@pytest.mark.parametrize("C", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("W", [3.0, 5.5, 6.5])
def test_2d_c2nc_few_coils(W, C, unequal):
    assert max(errors(2, 64, W, C, 4000, NFFT_conv_mode.C2NC, unequal)) <= FP32


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_2d_c2nc_bad_cell_stays_in_its_windows(bad):
    # samples whose window's slots do not reach the cell, and other coils, are as without it
    print(f"2D 64^2, 8 coils, one grid cell {bad}", flush=True)
    rng = np.random.default_rng(2)
    nos, C, W, M = 96, 8, 5.5, 5000
    k = rng.uniform(-0.5, 0.5, (1, M, 2)).astype(np.float32)
    plan = NFFTPlan([64, 64], None, W=W, os_factor=1.5)
    plan.preprocess(DeviceArray.from_numpy(k))
    x = (rng.standard_normal((C, 1, nos, nos)) + 1j * rng.standard_normal((C, 1, nos, nos))).astype(np.complex64)
    y = x.copy()
    y[3, 0, 40, 51] = bad
    outs = []
    for g in (x, y):
        out = DeviceArray.zeros((C, 1, M), np.complex64)
        plan.convolve(DeviceArray.from_numpy(g), out, NFFT_conv_mode.C2NC)
        outs.append(out.numpy()[:, 0])
    a, b = outs
    p = (k[0] + np.float32(0.5)) * np.float32(nos)
    d = np.abs((p - np.array([51, 40], np.float32) + nos / 2) % nos - nos / 2)
    inside, near = (d <= W / 2).all(axis=1), (d <= W / 2 + 1).all(axis=1)  # a slot of weight 0 lies next to the window
    assert inside.any() and not np.isfinite(b[3][inside]).any()
    assert np.array_equal(a[3][~near], b[3][~near])
    assert np.array_equal(np.delete(a, 3, 0), np.delete(b, 3, 0))


@pytest.mark.parametrize("mode", [NFFT_conv_mode.NC2C, NFFT_conv_mode.C2NC])
@pytest.mark.parametrize("C", [9, 16, 20, 33])
def test_2d_windows_of_7_cells(C, mode):
    assert max(errors(2, 64, 6.5, C, 4000, mode, True)) <= FP32
