"""The order in which the denoiser's convolution holds its weights
(raygun_amd/csrc/conv_weights.h), on the CPU: products taken in that order
equal a 3x3 convolution written out, and in the data gradient's order the
gradient of that convolution by its input, for every layer shape."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import unet_oracle as U

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "conv_weights.h"
extern "C" int count(int kin, int nout) { return rgrt::conv_weights(kin, nout); }
extern "C" int at(int e, int cin, int cout, int gradient)
{
    return gradient ? rgrt::conv_gradient_master_index(e, cin, cout) : rgrt::conv_master_index(e, cin, cout);
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("conv_weights")
    (d / "order.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fPIC", "-shared",
                    "-I" + os.path.join(ROOT, "raygun_amd", "csrc"), str(d / "order.cpp"), "-o", str(d / "order.so")], check=True)
    return ctypes.CDLL(str(d / "order.so"))


def packed(order, w, gradient):
    """The weights of a layer in the kernel's order, as (K, outputs)."""
    _, cin, cout = w.shape
    kin, nout = (cout, cin) if gradient else (cin, cout)
    at = np.array([order.at(e, cin, cout, int(gradient)) for e in range(order.count(kin, nout))])
    assert np.array_equal(np.sort(at[at >= 0]), np.arange(w.size))  # each weight once
    p = np.where(at >= 0, w.reshape(-1)[at], 0.0)
    # [K-step][16 outputs][lane = 16 * group + output][8] -> K = (step, group, 8), outputs
    return p.reshape(-1, nout // 16, 4, 16, 8).transpose(0, 2, 4, 1, 3).reshape(-1, nout)


def products(x, k):
    """3x3 products as the kernel takes them: K = (tap, channel), zeros past the last tap."""
    h, w, c = x.shape
    q = np.pad(x, ((1, 1), (1, 1), (0, 0)))
    cols = np.concatenate([q[t // 3:t // 3 + h, t % 3:t % 3 + w] for t in range(9)], -1).reshape(h * w, 9 * c)
    return (np.pad(cols, ((0, 0), (0, len(k) - 9 * c))) @ k).reshape(h, w, -1)


@pytest.mark.parametrize("cin,cout", sorted(set(U.LAYERS)))
def test_products_in_the_kernels_order_are_the_convolution(order, cin, cout):
    rng = np.random.default_rng(cin * 100 + cout)
    w = rng.integers(-8, 9, (9, cin, cout)).astype(float)  # whole numbers: sums are exact in any order
    x = rng.integers(-8, 9, (5, 6, cin)).astype(float)
    dy = rng.integers(-8, 9, (5, 6, cout)).astype(float)
    y, dx = np.zeros_like(dy), np.zeros_like(x)
    for i in range(5):
        for j in range(6):
            for t in range(9):
                a, b = i + t // 3 - 1, j + t % 3 - 1
                if 0 <= a < 5 and 0 <= b < 6:
                    y[i, j] += x[a, b] @ w[t]
                    dx[a, b] += w[t] @ dy[i, j]
    assert np.array_equal(products(x, packed(order, w, False)), y)
    assert np.array_equal(products(dy, packed(order, w, True)), dx)
