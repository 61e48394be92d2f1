"""GPU: convolution layers at the sizes where the kernels' tiles are cut: widths
around 8 and 16, heights around 4 and 8, odd depths, one batch and several, every
number of 16-channel tiles, kernels of 1, 2 and 3 with each padding."""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu

# batch, (D, H, W), cin, cout, k, pad, act
CASES = [
    (1, (1, 1, 1), 8, 8, 3, 1, 0), (1, (2, 4, 8), 16, 16, 3, 1, 1), (3, (3, 5, 9), 16, 16, 3, 1, 1),
    (2, (5, 9, 17), 8, 16, 3, 1, 1), (1, (7, 8, 15), 48, 16, 3, 1, 1), (2, (3, 3, 7), 96, 32, 3, 1, 1),
    (1, (5, 6, 10), 24, 32, 3, 1, 1), (9, (2, 2, 3), 32, 64, 3, 1, 1), (1, (4, 4, 8), 192, 64, 3, 1, 1),
    (2, (1, 5, 11), 64, 128, 3, 1, 0), (1, (3, 4, 9), 128, 128, 3, 1, 1), (2, (4, 7, 12), 16, 8, 2, 1, 0),
    (1, (5, 8, 16), 8, 16, 2, 0, 0), (1, (3, 4, 5), 40, 32, 1, 0, 1), (2, (4, 4, 4), 16, 64, 2, 1, 1),
    # enough positions for the LDS-tile forward, ragged, every tile depth and channel
    # tile count (the input gradient's are the input channels')
    (1, (17, 30, 70), 16, 16, 3, 1, 1), (2, (33, 31, 65), 8, 16, 3, 1, 1),
    (1, (31, 33, 39), 48, 32, 3, 1, 1), (1, (16, 25, 90), 96, 32, 3, 1, 0),
    (1, (14, 31, 40), 192, 64, 3, 1, 1), (1, (13, 20, 50), 24, 128, 3, 1, 1),
    (2, (17, 32, 63), 16, 8, 2, 1, 0), (1, (6, 5, 8), 16, 16, 3, 2, 0), (1, (5, 6, 9), 16, 32, 3, 0, 1), (2, (9, 10, 33), 32, 16, 3, 1, 1),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_conv_tiles(T, gpu, case):
    from oracle import nn_oracle as N
    import topopt_jl_amd.nn as NN
    B, sp, cin, cout, k, pad, act = CASES[case]
    g = np.random.default_rng(100 + case)
    x = g.standard_normal((B, *sp, cin)).astype(np.float32)
    w = (g.standard_normal((cout, k**3, cin)) / np.sqrt(k**3 * cin)).astype(np.float32)
    b = g.standard_normal(cout).astype(np.float32) * 0.1
    osp = tuple(s + 2 * pad - k + 1 for s in sp)
    dy = g.standard_normal((B, *osp, cout)).astype(np.float32)
    y, dx, dw, db = NN.conv_check(x, w, b, dy, k, pad, act)
    ye, dxe, dwe, dbe = N.conv_layer_device_emulation(x, w, b, dy, k, pad, act)
    # FP32 sums of at most 27 x 192 products of the same BF16 operands
    assert relerr(y, ye) < 2e-5
    # a BF16 dZ may round its ties the other way where an activation is applied
    assert relerr(dx, dxe) < 1e-3
    assert relerr(dw, dwe) < 1e-3
    assert relerr(db, dbe) < 1e-3
