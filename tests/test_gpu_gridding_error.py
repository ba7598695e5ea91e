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
