"""conv2d on the GPU: the lowering kernels through the C ABI, and op_conv2d / Conv2d through the drop-in module.

Lowering (im2col, col2im, the channel bias add) is index and copy work plus single rounding adds, so it is held to
bit equality with the CPU oracle; the whole convolution is held to the GEMM's tolerances against the oracle's
per-sample chain and against torch.nn.functional.conv2d in float64.  Shapes: the reference's own parity matrix
(tests/stress/stress_torch_parity.py:199-210) and test values (tests/autograd/test_conv2d.py), plus cases that take
the vector store path, several chunks of the batch, and the 1x1 shortcut.
"""
import json
import os

import numpy as np
import pytest

import oracle
import recpulse_cuda as rp
from recpulse.module import Conv2d
from recpulse_amd import capi
from devhelp import ALL, BF16, F16, F32, F64, NAMES, Dev, rand_storage, tol

pytestmark = pytest.mark.gpu
GOLD = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "reference_known_answers.json")))
REF_CASES = [tuple(tuple(v) if isinstance(v, list) else v for v in c) for c in GOLD["conv2d_parity_shapes"]["cases"]]
# (x shape, w shape, stride, pad, dilation, bias): out_H*out_W a multiple of 8 (vector stores), a 1x1 kernel with
# stride, a pointwise kernel (no lowering at all), a wider layer
MORE_CASES = [((3, 4, 16, 16), (6, 4, 3, 3), (1, 1), (1, 1), (1, 1), True),
              ((2, 5, 9, 9), (3, 5, 1, 1), (2, 2), (0, 0), (1, 1), True),
              ((4, 16, 8, 8), (24, 16, 1, 1), (1, 1), (0, 0), (1, 1), True),
              ((2, 32, 14, 14), (64, 32, 3, 3), (1, 1), (1, 1), (1, 1), False),
              # 3 x 3 / stride 1 / padding 1 with whole vectors per row: first, interior and last vectors of a row, and a one-row image
              ((2, 3, 5, 24), (4, 3, 3, 3), (1, 1), (1, 1), (1, 1), True),
              ((1, 2, 1, 8), (2, 2, 3, 3), (1, 1), (1, 1), (1, 1), False),
              # 64 channels in and out: the 16-bit types read the taps from zero-bordered planes, forward and input gradient
              ((2, 64, 8, 8), (64, 64, 3, 3), (1, 1), (1, 1), (1, 1), True)]
CASES = REF_CASES + MORE_CASES
DT_NAME = {F32: "float32", F64: "float64", F16: "float16", BF16: "bfloat16"}


def _geom(xs, ws, s, p, d):
    oH, oW = oracle.conv_out_size(xs[2], ws[2], s[0], p[0], d[0]), oracle.conv_out_size(xs[3], ws[3], s[1], p[1], d[1])
    return (xs[1], xs[2], xs[3], ws[2], ws[3], s[0], s[1], p[0], p[1], d[0], d[1], oH, oW)


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + "_k" + "x".join(map(str, c[1][2:])))
def test_lowering_is_bit_exact(dt, case):
    xs, ws, s, p, d, _ = case
    N, C, H, W = xs
    geom = _geom(xs, ws, s, p, d)
    oH, oW = geom[-2:]
    rows, cols = C * ws[2] * ws[3], oH * oW
    rng = np.random.default_rng(80)
    x = rand_storage(rng, xs, dt)
    L = capi.lib()
    dx, dcol = Dev(x, dt), Dev.empty((N, rows, cols), dt)
    capi.check(L.rp_hip_im2col_batched(dcol.ptr, dx.ptr, N, *geom, dt), "rp_hip_im2col_batched")
    want = np.stack([oracle.im2col(x[n], ws[2:], s, p, d, dt) for n in range(N)])
    assert np.array_equal(dcol.numpy(), want)
    # the adjoint, overwriting and adding
    c2 = rand_storage(rng, (N, rows, cols), dt)
    base = rand_storage(rng, xs, dt)
    dc2, dim = Dev(c2, dt), Dev(base, dt)
    capi.check(L.rp_hip_col2im_batched(dim.ptr, dc2.ptr, N, *geom, 1, dt), "rp_hip_col2im_batched")
    want = np.stack([oracle.col2im(base[n], c2[n], ws[2:], s, p, d, dt) for n in range(N)])
    assert np.array_equal(dim.numpy(), want)
    capi.check(L.rp_hip_col2im_batched(dim.ptr, dc2.ptr, N, *geom, 0, dt), "rp_hip_col2im_batched")
    want = np.stack([oracle.col2im(np.zeros_like(base[n]), c2[n], ws[2:], s, p, d, dt) for n in range(N)])
    assert np.array_equal(dim.numpy(), want)
    # the reference's single-sample entry points on sample 0
    d1, dim1 = Dev.empty((rows, cols), dt), Dev(base[0], dt)
    capi.check(L.im2col_kernel_device(d1.ptr, dx.ptr, *geom, dt), "im2col_kernel_device")
    assert np.array_equal(d1.numpy(), oracle.im2col(x[0], ws[2:], s, p, d, dt))
    capi.check(L.col2im_kernel_device(dim1.ptr, dc2.ptr, *geom, dt), "col2im_kernel_device")
    assert np.array_equal(dim1.numpy(), oracle.col2im(base[0], c2[0], ws[2:], s, p, d, dt))


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_channel_bias_add_and_channel_sums(dt):
    rng = np.random.default_rng(81)
    N, C, HW = 5, 7, 99
    y, b = rand_storage(rng, (N, C, HW), dt), rand_storage(rng, (C,), dt)
    L = capi.lib()
    dy, db = Dev(y, dt), Dev(b, dt)
    capi.check(L.rp_hip_channel_bias_add(dy.ptr, db.ptr, N, C, HW, dt), "rp_hip_channel_bias_add")
    want = oracle.add(y, np.ascontiguousarray(np.broadcast_to(b[None, :, None], y.shape)), dt)
    assert np.array_equal(dy.numpy(), want)
    # sums: a tree of float32 (float64) partial sums here, one running sum in the reference
    ds = Dev(b, dt)
    capi.check(L.rp_hip_channel_sums(ds.ptr, Dev(y, dt).ptr, N, C, HW, 0, dt), "rp_hip_channel_sums")
    exact = oracle.to_f64(y, dt).sum(axis=(0, 2))
    assert oracle.rel_err(oracle.to_f64(ds.numpy(), dt), exact) <= {F32: 1e-6, F64: 1e-14, F16: 2e-3, BF16: 1e-2}[dt]
    got0 = ds.numpy()
    capi.check(L.rp_hip_channel_sums(ds.ptr, Dev(y, dt).ptr, N, C, HW, 1, dt), "rp_hip_channel_sums")
    assert np.array_equal(ds.numpy(), oracle.add(got0, got0, dt))


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("N,C,HW", [(1, 1, 1), (3, 2, 513), (33, 5, 49), (4, 3, 4607), (5, 3, 8001), (5, 2, 18500)])
def test_channel_sums_of_every_size(dt, N, C, HW):
    """Planes that start at any element, channels on either side of what one workgroup sums; small integers, so the sums are exact before they are rounded once."""
    rng = np.random.default_rng(N + HW)
    g = rng.integers(-2, 3, (N, C, HW)).astype(np.float64)
    ds = Dev.empty((C,), dt)
    capi.check(capi.lib().rp_hip_channel_sums(ds.ptr, Dev(oracle.to_storage(g, dt), dt).ptr, N, C, HW, 0, dt), "rp_hip_channel_sums")
    assert np.array_equal(ds.numpy(), oracle.to_storage(g.sum(axis=(0, 2)), dt))


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_channel_sums_over_the_gradient_and_of_very_many_channels(dt):
    """Sums written over values that other channels' sums read, and more channels than workgroups of 1024 threads fit a launch; small integers."""
    rng = np.random.default_rng(82)
    L = capi.lib()
    es = capi.DTYPE_SIZE[dt]
    for N, C, HW in ((5, 600, 49), (1, 3000, 7)):
        g = rng.integers(-2, 3, (N, C, HW)).astype(np.float64)
        want = oracle.to_storage(g.sum(axis=(0, 2)), dt)
        for at in (0, C * HW - C):                       # over the first planes, over the last ones of the first sample
            flat = oracle.to_storage(g, dt).reshape(-1)
            d = capi.DeviceBuffer.from_numpy(flat)
            capi.check(L.rp_hip_channel_sums(d.at(at * es), d.ptr, N, C, HW, 0, dt), "rp_hip_channel_sums")
            assert np.array_equal(d.to_numpy(flat.dtype, (flat.size,))[at:at + C], want)
    C = 1 << 22
    g = oracle.to_storage(rng.integers(-2, 3, (1, C, 2)).astype(np.float64), dt)
    ds = Dev.empty((C,), dt)
    capi.check(L.rp_hip_channel_sums(ds.ptr, Dev(g, dt).ptr, 1, C, 2, 0, dt), "rp_hip_channel_sums")
    assert np.array_equal(ds.numpy(), oracle.to_storage(oracle.to_f64(g, dt).sum(axis=(0, 2)), dt))


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("N,C,HW", [(1035, 2, 14), (300, 5, 21), (1887, 1, 9), (1, 2587, 1024), (3, 2102, 86), (200, 64, 11)])
def test_channel_sums_of_many_samples_or_channels(dt, N, C, HW):
    """Channels that one workgroup could sum, on either side of the line where two launches are the faster; small integers."""
    test_channel_sums_of_every_size(dt, N, C, HW)


def test_lowering_rejects_inconsistent_geometry():
    d = capi.DeviceBuffer(1 << 16)
    L = capi.lib()
    # out_H that the geometry does not imply, zero stride, negative padding
    assert L.rp_hip_im2col_batched(d.ptr, d.ptr, 1, 1, 4, 4, 3, 3, 1, 1, 0, 0, 1, 1, 3, 2, F32) == -1
    assert b"geometry" in L.rp_hip_last_error()
    assert L.rp_hip_im2col_batched(d.ptr, d.ptr, 1, 1, 4, 4, 3, 3, 0, 1, 0, 0, 1, 1, 2, 2, F32) == -1
    assert L.rp_hip_col2im_batched(d.ptr, d.ptr, 1, 1, 4, 4, 3, 3, 1, 1, -1, 0, 1, 1, 2, 2, 0, F32) == -1
    assert L.rp_hip_im2col_batched(None, d.ptr, 1, 1, 4, 4, 3, 3, 1, 1, 0, 0, 1, 1, 2, 2, F32) == -1


SAME_CASES = [  # (batch, C_in, H, W, C_out, kH, kW): whole tiles, ragged columns, several slabs per tap, 5 x 5, one row
    (3, 64, 8, 8, 64, 3, 3), (2, 128, 14, 14, 64, 3, 3), (2, 64, 7, 20, 192, 3, 3), (1, 64, 9, 12, 32, 5, 5),
    (2, 64, 1, 16, 64, 3, 1), (1, 64, 56, 56, 64, 3, 3), (5, 64, 10, 10, 24, 3, 3)]


def _one_rounding(dt, k):
    """Distance from float64 of a sum kept in the accumulate type and rounded once to dt."""
    return {BF16: 2.0 ** -8, F16: 2.0 ** -11}.get(dt, tol(dt, k))


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("case", SAME_CASES, ids=lambda c: "x".join(map(str, c)))
def test_same_convolution_without_lowered_matrix(dt, case):
    """rp_hip_conv2d_same_forward / _backward_input against the oracle's per-sample chain and against float64."""
    import torch
    N, Ci, H, W, Co, kH, kW = case
    L = capi.lib()
    assert L.rp_hip_conv2d_same_supported(Ci, H, W, kH, kW, dt) == 1
    rng = np.random.default_rng(83)
    x, w = rand_storage(rng, (N, Ci, H, W), dt), oracle.to_storage(rng.standard_normal((Co, Ci, kH, kW)) * 0.2, dt)
    b = rand_storage(rng, (Co,), dt)
    s, p, d = (1, 1), (kH // 2, kW // 2), (1, 1)
    dx_, dw_, db_, dy_ = Dev(x, dt), Dev(w, dt), Dev(b, dt), Dev.empty((N, Co, H, W), dt)
    capi.check(L.rp_hip_conv2d_same_forward(dy_.ptr, dx_.ptr, dw_.ptr, db_.ptr, N, Ci, H, W, Co, kH, kW, dt), "same forward")
    y_ref = oracle.conv2d_forward(x, w, b, s, p, d, dt)
    xt, wt = torch.tensor(oracle.to_f64(x, dt)), torch.tensor(oracle.to_f64(w, dt))
    y_exact = torch.nn.functional.conv2d(xt, wt, torch.tensor(oracle.to_f64(b, dt)), padding=p).numpy()
    got = oracle.to_f64(dy_.numpy(), dt)
    assert oracle.rel_err(got, oracle.to_f64(y_ref, dt)) <= tol(dt, Ci * kH * kW)
    assert oracle.rel_err(got, y_exact) <= tol(dt, Ci * kH * kW)
    # without a bias the result is the sum in the accumulate type rounded once: no further from float64 than one rounding of dt
    capi.check(L.rp_hip_conv2d_same_forward(dy_.ptr, dx_.ptr, dw_.ptr, None, N, Ci, H, W, Co, kH, kW, dt), "same forward")
    y_nb = torch.nn.functional.conv2d(xt, wt, None, padding=p).numpy()
    assert oracle.rel_err(oracle.to_f64(dy_.numpy(), dt), y_nb) <= _one_rounding(dt, Ci * kH * kW)
    # gradient with respect to the input (C_out in whole k slabs of the dtype's kernel)
    dx_ok = L.rp_hip_conv2d_same_supported(Co, H, W, kH, kW, dt) == 1
    assert dx_ok == (Co % {BF16: 64, F16: 64, F32: 32, F64: 16}[dt] == 0)
    if dx_ok:
        g = rand_storage(rng, (N, Co, H, W), dt)
        dg_, dgx_ = Dev(g, dt), Dev.empty((N, Ci, H, W), dt)
        capi.check(L.rp_hip_conv2d_same_backward_input(dgx_.ptr, dg_.ptr, dw_.ptr, N, Ci, H, W, Co, kH, kW, dt), "same backward")
        dx_ref, _, _ = oracle.conv2d_backward(x, w, g, s, p, d, dt, with_bias=False)
        dx_exact = torch.nn.grad.conv2d_input((N, Ci, H, W), wt, torch.tensor(oracle.to_f64(g, dt)), padding=p).numpy()
        got = oracle.to_f64(dgx_.numpy(), dt)
        assert oracle.rel_err(got, oracle.to_f64(dx_ref, dt)) <= tol(dt, Co * kH * kW)
        assert oracle.rel_err(got, dx_exact) <= _one_rounding(dt, Co * kH * kW)
    else:
        g = rand_storage(rng, (N, Co, H, W), dt)
        dg_ = Dev(g, dt)
    # gradient with respect to the weights (any channel counts), alone and together with the input gradient
    assert L.rp_hip_conv2d_same_supported(0, H, W, kH, kW, dt) == 1
    dgw_ = Dev.empty((Co, Ci, kH, kW), dt)
    capi.check(L.rp_hip_conv2d_same_backward(None, dgw_.ptr, dg_.ptr, dx_.ptr, None, N, Ci, H, W, Co, kH, kW, dt), "same backward (weights)")
    _, dw_ref, _ = oracle.conv2d_backward(x, w, g, s, p, d, dt, with_bias=False)
    dw_exact = torch.nn.grad.conv2d_weight(xt, (Co, Ci, kH, kW), torch.tensor(oracle.to_f64(g, dt)), padding=p).numpy()
    got_w = oracle.to_f64(dgw_.numpy(), dt)
    assert oracle.rel_err(got_w, oracle.to_f64(dw_ref, dt).reshape(got_w.shape)) <= tol(dt, N * H * W)
    assert oracle.rel_err(got_w, dw_exact) <= tol(dt, N * H * W)
    if dx_ok:
        both_x, both_w = Dev.empty((N, Ci, H, W), dt), Dev.empty((Co, Ci, kH, kW), dt)
        capi.check(L.rp_hip_conv2d_same_backward(both_x.ptr, both_w.ptr, dg_.ptr, dx_.ptr, dw_.ptr, N, Ci, H, W, Co, kH, kW, dt), "same backward (both)")
        assert np.array_equal(both_x.numpy(), dgx_.numpy()) and np.array_equal(both_w.numpy(), dgw_.numpy())


T256, T64, DW, PLANES = "conv_taps16_256x64", "conv_taps16_64x64", "conv_dw16", "conv_planes"
DIRECT_CASES = [  # (batch, C_in, H, W, C_out, kH, kW) and the kernels of forward, dX and dW on 256 CUs: rows of any width (whole eights, fours,
                  # twos, odd), many small samples in a strip, strips that begin inside a row or are shortened to whole rows, 64 and 256
                  # positions a workgroup with three and five taps a row, channels and strips that end inside a tile, shapes refused
    ((11, 64, 7, 7, 64, 3, 3), T64, T64, DW), ((3, 128, 10, 6, 64, 5, 3), T64, T64, DW), ((2, 64, 3, 50, 128, 3, 5), T64, T64, PLANES),
    ((1, 64, 5, 127, 64, 3, 3), PLANES, PLANES, DW), ((2, 64, 2, 130, 64, 1, 3), T64, T64, PLANES), ((64, 64, 32, 32, 64, 3, 3), T256, T256, DW),
    ((70, 64, 31, 31, 64, 3, 3), T256, T256, DW), ((66, 64, 30, 34, 64, 1, 5), T256, T256, PLANES), ((24, 64, 12, 300, 64, 3, 3), PLANES, PLANES, PLANES),
    ((1, 64, 1, 1, 64, 3, 3), PLANES, PLANES, PLANES), ((90, 64, 28, 28, 64, 3, 3), T256, T256, DW), ((64, 64, 56, 56, 64, 3, 3), T256, T256, DW),
    ((90, 64, 28, 28, 64, 5, 5), T256, T256, DW), ((64, 64, 32, 32, 64, 5, 5), T256, T256, DW), ((70, 64, 31, 31, 64, 5, 5), T256, T256, PLANES),
    ((23, 64, 56, 52, 64, 3, 3), PLANES, PLANES, DW), ((29, 64, 48, 48, 64, 5, 5), PLANES, PLANES, DW),
    ((12, 128, 39, 39, 192, 5, 5), PLANES, PLANES, PLANES), ((40, 128, 31, 31, 192, 3, 3), T256, T256, PLANES)]


@pytest.mark.parametrize("dt", [F16, BF16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("case,forward,input_grad,weight_grad", DIRECT_CASES, ids=["x".join(map(str, c[0])) for c in DIRECT_CASES])
def test_same_convolution_from_the_image_is_exact_on_integers(dt, case, forward, input_grad, weight_grad):
    """Small integers: every sum is an integer below 2^24, exact in fp32 (and a sample's share of a weight gradient below 2^8, exact in 16
    bits), so the results are that sum rounded once (the forward's bias: rounded again), bit for bit; each on the kernel that is named."""
    import torch
    N, Ci, H, W, Co, kH, kW = case
    L = capi.lib()
    rng = np.random.default_rng(N + W)
    ints = lambda *shape: rng.integers(-1, 2, shape).astype(np.float64)          # noqa: E731
    x, w, b, g = ints(N, Ci, H, W), ints(Co, Ci, kH, kW), ints(Co), ints(N, Co, H, W)
    dx_, dw_, db_, dg_ = (Dev(oracle.to_storage(v, dt), dt) for v in (x, w, b, g))
    y, gx, gw = Dev.empty((N, Co, H, W), dt), Dev.empty((N, Ci, H, W), dt), Dev.empty((Co, Ci, kH, kW), dt)
    capi.check(L.rp_hip_conv2d_same_forward(y.ptr, dx_.ptr, dw_.ptr, db_.ptr, N, Ci, H, W, Co, kH, kW, dt), "same forward")
    assert capi.last_gemm_kernel() == forward
    capi.check(L.rp_hip_conv2d_same_backward(gx.ptr, None, dg_.ptr, None, dw_.ptr, N, Ci, H, W, Co, kH, kW, dt), "same backward (input)")
    assert capi.last_gemm_kernel() == input_grad
    capi.check(L.rp_hip_conv2d_same_backward(None, gw.ptr, dg_.ptr, dx_.ptr, None, N, Ci, H, W, Co, kH, kW, dt), "same backward (weights)")
    assert capi.last_gemm_kernel() == weight_grad
    alone = gx.numpy(), gw.numpy()
    capi.check(L.rp_hip_conv2d_same_backward(gx.ptr, gw.ptr, dg_.ptr, dx_.ptr, dw_.ptr, N, Ci, H, W, Co, kH, kW, dt), "same backward")
    assert np.array_equal(gx.numpy(), alone[0]) and np.array_equal(gw.numpy(), alone[1])
    xt, wt, gt = (torch.tensor(v, dtype=torch.float32) for v in (x, w, g))       # sums of integers below 2^24: exact in any order
    pad = (kH // 2, kW // 2)
    want = oracle.to_storage(torch.nn.functional.conv2d(xt, wt, None, padding=pad).numpy(), dt)
    want = oracle.to_storage(oracle.to_f64(want, dt) + b[None, :, None, None], dt)
    assert np.array_equal(oracle.to_f64(y.numpy(), dt), oracle.to_f64(want, dt))
    want = oracle.to_storage(torch.nn.grad.conv2d_input((N, Ci, H, W), wt, gt, padding=pad).numpy(), dt)
    assert np.array_equal(oracle.to_f64(gx.numpy(), dt), oracle.to_f64(want, dt))
    want = oracle.to_storage(torch.nn.grad.conv2d_weight(xt, (Co, Ci, kH, kW), gt, padding=pad).numpy(), dt)
    assert np.array_equal(oracle.to_f64(gw.numpy(), dt), oracle.to_f64(want, dt))


SHARED_CASES = [  # fp32 (batch, C_in, H, W, C_out, kH, kW) on 256 CUs.  Forward and input gradient: 16 x 16 tiles, 16 x 32, 64 x 64, the tiles without
                  # shared k; weight gradient: 32 x 32 up to one 64 x 64 tile a CU, 64 x 64, 32 x 32 above; whole and folded rows, ragged channels
    (1, 64, 9, 9, 64, 3, 3), (1, 96, 6, 11, 40, 5, 3), (4, 64, 28, 28, 96, 3, 3), (7, 192, 41, 40, 192, 3, 3), (6, 64, 53, 39, 200, 3, 3),
    (28, 64, 28, 28, 64, 3, 3), (22, 64, 48, 48, 64, 3, 3), (3, 64, 50, 51, 128, 5, 5), (17, 32, 28, 28, 128, 3, 3)]


@pytest.mark.parametrize("case", SHARED_CASES, ids=lambda c: "x".join(map(str, c)))
def test_same_convolution_in_fp32_is_exact_on_integers(case):
    """Small integers: every sum is an integer below 2^24, exact in any order of additions."""
    import torch
    N, Ci, H, W, Co, kH, kW = case
    L = capi.lib()
    rng = np.random.default_rng(H + W)
    ints = lambda *shape: rng.integers(-3, 4, shape).astype(np.float32)          # noqa: E731
    x, w, b, g = ints(N, Ci, H, W), ints(Co, Ci, kH, kW), ints(Co), ints(N, Co, H, W)
    dx_, dw_, db_, dg_ = (Dev(v, F32) for v in (x, w, b, g))
    y, gx, gw = Dev.empty((N, Co, H, W), F32), Dev.empty((N, Ci, H, W), F32), Dev.empty((Co, Ci, kH, kW), F32)
    xt, wt, gt, pad = torch.tensor(x), torch.tensor(w), torch.tensor(g), (kH // 2, kW // 2)
    capi.check(L.rp_hip_conv2d_same_forward(y.ptr, dx_.ptr, dw_.ptr, db_.ptr, N, Ci, H, W, Co, kH, kW, F32), "same forward")
    assert np.array_equal(y.numpy(), torch.nn.functional.conv2d(xt, wt, torch.tensor(b), padding=pad).numpy())
    with_dx = L.rp_hip_conv2d_same_supported(Co, H, W, kH, kW, F32) == 1
    capi.check(L.rp_hip_conv2d_same_backward(gx.ptr if with_dx else None, gw.ptr, dg_.ptr, dx_.ptr, dw_.ptr, N, Ci, H, W, Co, kH, kW, F32), "same backward")
    if with_dx: assert np.array_equal(gx.numpy(), torch.nn.grad.conv2d_input((N, Ci, H, W), wt, gt, padding=pad).numpy())
    assert np.array_equal(gw.numpy(), torch.nn.grad.conv2d_weight(xt, (Co, Ci, kH, kW), gt, padding=pad).numpy())


@pytest.mark.parametrize("case,forward,input_grad,weight_grad", zip(SHARED_CASES, *zip(
    ("16x16", "16x16", "32x32"), ("16x16", None, "32x32"), ("16x32", "16x32", "32x32"), ("64x64", "64x64", "32x32"), ("64x64", None, "64x64"),
    (None, None, "32x32"), (None, None, "32x32"), ("16x32", "16x32", "32x32"), (None, "16x32", "32x32"))), ids=lambda c: "x".join(map(str, c)) if isinstance(c, tuple) else str(c))
def test_tiles_of_same_convolution_in_fp32(case, forward, input_grad, weight_grad):
    """The tiles that the cases above are for (on 256 CUs); None: those whose waves do not share k."""
    N, Ci, H, W, Co, kH, kW = case
    L = capi.lib()
    d = Dev(np.zeros((N, max(Ci, Co), H, W), np.float32), F32)
    out, w = Dev.empty((N, max(Ci, Co), H, W), F32), Dev(np.zeros((Co, Ci, kH, kW), np.float32), F32)
    name = lambda tile: f"mfma32_wavek_{tile}" if tile else "conv_planes"          # noqa: E731
    capi.check(L.rp_hip_conv2d_same_forward(out.ptr, d.ptr, w.ptr, None, N, Ci, H, W, Co, kH, kW, F32), "same forward")
    assert capi.last_gemm_launch() == name(forward) and capi.last_gemm_kernel() == "conv_planes"
    if L.rp_hip_conv2d_same_supported(Co, H, W, kH, kW, F32) == 1:
        capi.check(L.rp_hip_conv2d_same_backward(out.ptr, None, d.ptr, None, w.ptr, N, Ci, H, W, Co, kH, kW, F32), "dX")
        assert capi.last_gemm_launch() == name(input_grad) and capi.last_gemm_kernel() == "conv_planes"
    capi.check(L.rp_hip_conv2d_same_backward(None, w.ptr, d.ptr, out.ptr, None, N, Ci, H, W, Co, kH, kW, F32), "dW")
    assert capi.last_gemm_launch() == name(weight_grad) and capi.last_gemm_kernel() == "conv_planes"
    capi.synchronize()


@pytest.mark.parametrize("dt", [F16, BF16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("case", [(23, 64, 56, 52, 64, 3), (29, 64, 48, 48, 64, 5), (2, 128, 12, 40, 64, 3), (1, 64, 53, 53, 128, 5)], ids=lambda c: "x".join(map(str, c)))
def test_weight_gradient_does_not_depend_on_the_input_gradient(dt, case):
    """dW alone and beside dX: the same kernel and the same bits, also where the in-place kernels take dW and refuse dX (the
    first two shapes) and where they take dX and refuse dW (the last).  Beside a dX that is stored over dY, dW is that of the planes, to tolerance."""
    N, Ci, H, W, Co, k = case
    L = capi.lib()
    rng = np.random.default_rng(88)
    x, g, w = rand_storage(rng, (N, Ci, H, W), dt), rand_storage(rng, (N, Co, H, W), dt), oracle.to_storage(rng.standard_normal((Co, Ci, k, k)) * 0.2, dt)
    dx_, dg_, dw_ = Dev(x, dt), Dev(g, dt), Dev(w, dt)
    alone_x, alone_w, gx, gw = Dev.empty((N, Ci, H, W), dt), Dev.empty((Co, Ci, k, k), dt), Dev.empty((N, Ci, H, W), dt), Dev.empty((Co, Ci, k, k), dt)
    capi.check(L.rp_hip_conv2d_same_backward(alone_x.ptr, None, dg_.ptr, None, dw_.ptr, N, Ci, H, W, Co, k, k, dt), "dX alone")
    capi.check(L.rp_hip_conv2d_same_backward(None, alone_w.ptr, dg_.ptr, dx_.ptr, None, N, Ci, H, W, Co, k, k, dt), "dW alone")
    kernel = capi.last_gemm_kernel()
    capi.check(L.rp_hip_conv2d_same_backward(gx.ptr, gw.ptr, dg_.ptr, dx_.ptr, dw_.ptr, N, Ci, H, W, Co, k, k, dt), "both")
    assert capi.last_gemm_kernel() == kernel
    assert np.array_equal(gx.numpy(), alone_x.numpy()) and np.array_equal(gw.numpy(), alone_w.numpy())
    capi.check(L.rp_hip_conv2d_same_backward(gx.ptr, dw_.ptr, dg_.ptr, dx_.ptr, dw_.ptr, N, Ci, H, W, Co, k, k, dt), "both, dW over W")
    assert np.array_equal(gx.numpy(), alone_x.numpy()) and np.array_equal(dw_.numpy(), alone_w.numpy())
    if Ci == Co:
        dw2 = Dev(w, dt)
        capi.check(L.rp_hip_conv2d_same_backward(dg_.ptr, gw.ptr, dg_.ptr, dx_.ptr, dw2.ptr, N, Ci, H, W, Co, k, k, dt), "both, dX over dY")
        # the planes round every sample's share once more: half a unit of 16 bits of each, sqrt(N) of them against sqrt(N) of the sum
        assert oracle.rel_err(oracle.to_f64(gw.numpy(), dt), oracle.to_f64(alone_w.numpy(), dt)) <= {BF16: 2.0 ** -7, F16: 2.0 ** -10}[dt]
        assert oracle.rel_err(oracle.to_f64(dg_.numpy(), dt), oracle.to_f64(alone_x.numpy(), dt)) <= {BF16: 2.0 ** -8, F16: 2.0 ** -11}[dt]


@pytest.mark.parametrize("dt", [F16, BF16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("case", [(2, 5, 9, 12, 64, 3, 3), (3, 40, 14, 14, 128, 3, 3), (1, 64, 8, 24, 64, 5, 5), (40, 64, 28, 28, 192, 3, 3), (3, 7, 3, 6, 64, 1, 3)],
                         ids=lambda c: "x".join(map(str, c)))
def test_both_gradients_in_one_call_are_those_of_two_calls(dt, case):
    """Bit for bit, apart and with dW over W, dW over x or dX over W (the last of them read before the gradient is stored)."""
    N, Ci, H, W, Co, kH, kW = case
    L = capi.lib()
    rng = np.random.default_rng(N + Ci)
    x, w, g = rand_storage(rng, (N, Ci, H, W), dt), oracle.to_storage(rng.standard_normal((Co, Ci, kH, kW)) * 0.2, dt), rand_storage(rng, (N, Co, H, W), dt)
    dx_, dw_, dg_ = Dev(x, dt), Dev(w, dt), Dev(g, dt)
    gx, gw = Dev.empty((N, Ci, H, W), dt), Dev.empty((Co, Ci, kH, kW), dt)
    capi.check(L.rp_hip_conv2d_same_backward(gx.ptr, None, dg_.ptr, None, dw_.ptr, N, Ci, H, W, Co, kH, kW, dt), "input gradient")
    capi.check(L.rp_hip_conv2d_same_backward(None, gw.ptr, dg_.ptr, dx_.ptr, None, N, Ci, H, W, Co, kH, kW, dt), "weight gradient")
    want = gx.numpy(), gw.numpy()
    size = max(x.size, w.size)
    for over_x, over_w in ((None, None), (None, "w"), (None, "x"), ("w", None)):
        bx, bw = Dev.empty((size,), dt), Dev.empty((size,), dt)
        pad = lambda a: Dev(np.concatenate([a.ravel(), np.zeros(size - a.size, a.dtype)]), dt)          # noqa: E731
        bufs = {"x": pad(x), "w": pad(w)}
        ox, ow = bufs.get(over_x, bx), bufs.get(over_w, bw)
        capi.check(L.rp_hip_conv2d_same_backward(ox.ptr, ow.ptr, dg_.ptr, bufs["x"].ptr, bufs["w"].ptr, N, Ci, H, W, Co, kH, kW, dt), "both")
        assert np.array_equal(ox.numpy()[:x.size], want[0].ravel()) and np.array_equal(ow.numpy()[:w.size], want[1].ravel()), (over_x, over_w)


@pytest.mark.parametrize("dt", [F16, BF16], ids=lambda d: NAMES[d])
def test_same_convolution_over_its_own_input(dt):
    """An output that overlaps the image it is computed from: the image is copied first, as for any other convolution."""
    N, C, H, W = 2, 64, 9, 12
    L = capi.lib()
    rng = np.random.default_rng(86)
    x, w = rand_storage(rng, (N, C, H, W), dt), oracle.to_storage(rng.standard_normal((C, C, 3, 3)) * 0.2, dt)
    dw_ = Dev(w, dt)
    for call in (lambda out, img: L.rp_hip_conv2d_same_forward(out, img, dw_.ptr, None, N, C, H, W, C, 3, 3, dt),
                 lambda out, img: L.rp_hip_conv2d_same_backward_input(out, img, dw_.ptr, N, C, H, W, C, 3, 3, dt)):
        src, out = Dev(x, dt), Dev.empty((N, C, H, W), dt)
        capi.check(call(out.ptr, src.ptr), "apart")
        capi.check(call(src.ptr, src.ptr), "in place")
        assert oracle.rel_err(oracle.to_f64(src.numpy(), dt), oracle.to_f64(out.numpy(), dt)) <= {BF16: 2.0 ** -8, F16: 2.0 ** -11}[dt]


@pytest.mark.parametrize("dt", [F16, BF16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("case", [(2, 128, 12, 16, 64), (3, 192, 14, 14, 128), (1, 64, 30, 30, 64)], ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("at", ["front", "back"])
def test_same_convolution_over_its_own_weights(dt, case, at):
    """An output that overlaps the weights it is computed from, at either end: the bits of one that does not (the weights are read before
    anything is stored)."""
    N, Ci, H, W, Co = case
    L = capi.lib()
    rng = np.random.default_rng(87)
    x, w = rand_storage(rng, (N, Ci, H, W), dt), oracle.to_storage(rng.standard_normal((Co, Ci, 3, 3)) * 0.2, dt)
    dx_, dw_, want = Dev(x, dt), Dev(w, dt), Dev.empty((N, Co, H, W), dt)
    capi.check(L.rp_hip_conv2d_same_forward(want.ptr, dx_.ptr, dw_.ptr, None, N, Ci, H, W, Co, 3, 3, dt), "apart")
    ny, nw = N * Co * H * W, w.size
    shared = 1024                                   # elements that both hold: whole 16-byte vectors, fewer than either
    both = np.zeros(ny + nw - shared, w.dtype)
    w_at, y_at = (0, nw - shared) if at == "front" else (ny - shared, 0)
    both[w_at:w_at + nw] = w.reshape(-1)
    buf = capi.DeviceBuffer.from_numpy(both)
    capi.check(L.rp_hip_conv2d_same_forward(buf.ptr + 2 * y_at, dx_.ptr, buf.ptr + 2 * w_at, None, N, Ci, H, W, Co, 3, 3, dt), "over the weights")
    got = buf.to_numpy(both.dtype, both.shape)
    assert np.array_equal(got[y_at:y_at + ny], want.numpy().reshape(-1))
    keep = got[:y_at] if at == "front" else got[ny:]
    assert np.array_equal(keep, w.reshape(-1)[:nw - shared] if at == "front" else w.reshape(-1)[shared:])


def test_same_convolution_in_chunks_of_the_batch(monkeypatch):
    """With room for two samples at a time a batch of five goes in three chunks: same bits as in one piece (the weight
    gradient adds its chunks in fp32 and rounds after each, so it is compared to tolerance)."""
    dt, (N, Ci, H, W, Co, kH, kW) = BF16, (5, 64, 6, 8, 64, 3, 3)
    L = capi.lib()
    rng = np.random.default_rng(84)
    x, w, g = rand_storage(rng, (N, Ci, H, W), dt), oracle.to_storage(rng.standard_normal((Co, Ci, kH, kW)) * 0.2, dt), rand_storage(rng, (N, Co, H, W), dt)
    dx_, dw_, dg_ = Dev(x, dt), Dev(w, dt), Dev(g, dt)

    def run():
        y, gx, gw = Dev.empty((N, Co, H, W), dt), Dev.empty((N, Ci, H, W), dt), Dev.empty((Co, Ci, kH, kW), dt)
        capi.check(L.rp_hip_conv2d_same_forward(y.ptr, dx_.ptr, dw_.ptr, None, N, Ci, H, W, Co, kH, kW, dt), "same forward")
        capi.check(L.rp_hip_conv2d_same_backward(gx.ptr, gw.ptr, dg_.ptr, dx_.ptr, dw_.ptr, N, Ci, H, W, Co, kH, kW, dt), "same backward")
        return y.numpy(), gx.numpy(), gw.numpy()

    whole = run()
    per_sample = (2 * 64 * (8 * 16 + 16) + 64 * 64 * 9) * 2          # padded dy and x planes plus the larger product, bytes
    monkeypatch.setenv("RP_CONV_WORKSPACE_BYTES", str(2 * per_sample + 64))
    parts = run()
    assert np.array_equal(whole[0], parts[0]) and np.array_equal(whole[1], parts[1])
    assert oracle.rel_err(oracle.to_f64(parts[2], dt), oracle.to_f64(whole[2], dt)) <= 2.0 ** -7
    forward_per_sample = (64 * (8 * 16 + 16) + 64 * 6 * 16) * 2      # the forward holds less per sample: give it room for two as well
    monkeypatch.setenv("RP_CONV_WORKSPACE_BYTES", str(2 * forward_per_sample + 64))
    assert np.array_equal(whole[0], run()[0])


@pytest.mark.parametrize("N,Ci,H,W,Co", [(24, 64, 28, 28, 64), (11, 192, 28, 28, 192), (5, 64, 9, 11, 96)])
def test_fp32_same_convolution_in_chunks_of_the_batch(monkeypatch, N, Ci, H, W, Co):
    """fp32 images of random values: y and dX have the same bits whether the batch goes in one piece or in several, and dX whether
    dW is asked for or not (the workspace of dW makes its chunks smaller).  The whole batches of the first two shapes have too many tiles for
    the kernel that their parts would go to."""
    L = capi.lib()
    rng = np.random.default_rng(85)
    x, w, g = rand_storage(rng, (N, Ci, H, W), F32), oracle.to_storage(rng.standard_normal((Co, Ci, 3, 3)) * 0.05, F32), rand_storage(rng, (N, Co, H, W), F32)
    dx_, dw_, dg_ = Dev(x, F32), Dev(w, F32), Dev(g, F32)

    def run(with_dw):
        y, gx, gw = Dev.empty((N, Co, H, W), F32), Dev.empty((N, Ci, H, W), F32), Dev.empty((Co, Ci, 3, 3), F32)
        capi.check(L.rp_hip_conv2d_same_forward(y.ptr, dx_.ptr, dw_.ptr, None, N, Ci, H, W, Co, 3, 3, F32), "same forward")
        capi.check(L.rp_hip_conv2d_same_backward(gx.ptr, gw.ptr if with_dw else None, dg_.ptr, dx_.ptr, dw_.ptr, N, Ci, H, W, Co, 3, 3, F32), "same backward")
        return y.numpy(), gx.numpy(), gw.numpy()

    whole = run(True)
    assert np.array_equal(whole[1], run(False)[1])
    plane = (H + 2) * ((W + 2 + 3) // 4 * 4) + 16                     # a zero-bordered plane and its slack, elements
    for samples in (2, N // 2):
        # (what a sample takes with dW: planes of dY and X and the larger product; without, and in the forward, more of them fit)
        monkeypatch.setenv("RP_CONV_WORKSPACE_BYTES", str(samples * 4 * ((Ci + Co) * plane + max(Ci * plane, Co * Ci * 9)) + 64))
        parts, without = run(True), run(False)
        assert np.array_equal(whole[0], parts[0]) and np.array_equal(whole[1], parts[1]) and np.array_equal(whole[1], without[1])
        assert oracle.rel_err(parts[2].astype(np.float64), whole[2].astype(np.float64)) <= 1e-5
    monkeypatch.delenv("RP_CONV_WORKSPACE_BYTES")


def test_same_convolution_rejects_other_shapes():
    L = capi.lib()
    assert L.rp_hip_conv2d_same_supported(48, 8, 8, 3, 3, BF16) == 0           # channels in whole k slabs: 64 for 16-bit types,
    assert L.rp_hip_conv2d_same_supported(48, 8, 8, 3, 3, F32) == 0            # 32 for float32,
    assert L.rp_hip_conv2d_same_supported(32, 8, 8, 3, 3, F32) == 1
    assert L.rp_hip_conv2d_same_supported(24, 8, 8, 3, 3, F64) == 0            # 16 for float64
    assert L.rp_hip_conv2d_same_supported(48, 8, 8, 3, 3, F64) == 1
    assert L.rp_hip_conv2d_same_supported(64, 8, 8, 3, 3, 99) == 0             # no such dtype
    assert L.rp_hip_conv2d_same_supported(64, 8, 8, 2, 2, BF16) == 0           # odd kernels only
    assert L.rp_hip_conv2d_same_supported(64, 8, 8, 1, 1, BF16) == 0           # 1 x 1 needs no lowering in the first place
    d = Dev.empty((64 * 64,), BF16)
    assert L.rp_hip_conv2d_same_forward(d.ptr, d.ptr, d.ptr, None, 1, 48, 8, 8, 64, 3, 3, BF16) == -1
    assert b"rp_hip_conv2d_same_supported" in L.rp_hip_last_error()


# ---- through the drop-in module -------------------------------------------------------------------------------
def _dev(arr, dt, grad=False):
    """storage array -> device tensor (16-bit values travel as float32, exactly)."""
    vals = oracle.to_f64(arr, dt)
    t = rp.from_numpy(np.ascontiguousarray(vals, dtype=np.float64 if dt == F64 else np.float32)).to(device="cuda", dtype=DT_NAME[dt])
    return t.requires_grad_(True) if grad else t


def _host(t):
    return t.to(device="cpu", dtype="float64").to_numpy()


def _run_conv(x, w, b, dy, s, p, d, dt):
    tx, tw = _dev(x, dt, True), _dev(w, dt, True)
    tb = _dev(b, dt, True) if b is not None else None
    y = tx.op_conv2d(tw, bias=tb, stride_h=s[0], stride_w=s[1], pad_h=p[0], pad_w=p[1], dilation_h=d[0], dilation_w=d[1])
    # upstream gradient dy: loss = y_flat . dy_flat
    n = int(np.prod(y.shape))
    y.reshape([1, n]).op_matmul(_dev(dy, dt).reshape([n, 1])).op_sum_all().backward()
    return _host(y), _host(tx.grad), _host(tw.grad), (_host(tb.grad) if tb is not None else None)


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + "_k" + "x".join(map(str, c[1][2:])))
def test_conv2d_forward_and_backward(dt, case, monkeypatch):
    import torch
    xs, ws, s, p, d, has_bias = case
    rng = np.random.default_rng(82)
    x, w = rand_storage(rng, xs, dt), oracle.to_storage(rng.standard_normal(ws) * 0.3, dt)
    b = rand_storage(rng, (ws[0],), dt) if has_bias else None
    y_ref = oracle.conv2d_forward(x, w, b, s, p, d, dt)
    dy = rand_storage(rng, y_ref.shape, dt)
    got = _run_conv(x, w, b, dy, s, p, d, dt)
    dx_ref, dw_ref, db_ref = oracle.conv2d_backward(x, w, dy, s, p, d, dt, with_bias=has_bias)
    k_fwd, k_dx, k_dw = xs[1] * ws[2] * ws[3], ws[0], y_ref.shape[2] * y_ref.shape[3] * xs[0]
    names = ("y", "dx", "dw", "db")
    refs = (y_ref, dx_ref, dw_ref, db_ref)
    ks = (k_fwd, k_dx, k_dw, k_dw)
    for name, g, r, k in zip(names, got, refs, ks):
        if r is None:
            continue
        assert g.shape == r.shape, name
        assert oracle.rel_err(g, oracle.to_f64(r, dt)) <= tol(dt, k), name
    # the same against an independent float64 implementation
    xt = torch.tensor(oracle.to_f64(x, dt), requires_grad=True); wt = torch.tensor(oracle.to_f64(w, dt), requires_grad=True)
    bt = torch.tensor(oracle.to_f64(b, dt), requires_grad=True) if has_bias else None
    yt = torch.nn.functional.conv2d(xt, wt, bt, stride=s, padding=p, dilation=d)
    yt.backward(torch.tensor(oracle.to_f64(dy, dt)))
    exact = (yt.detach().numpy(), xt.grad.numpy(), wt.grad.numpy(), bt.grad.numpy() if has_bias else None)
    for name, g, r, k in zip(names, got, exact, ks):
        if r is not None:
            assert oracle.rel_err(g, r) <= tol(dt, k), name
    # with the lowered matrix limited to one sample at a time the batch goes in chunks of one: the GEMMs then run
    # unbatched (a different kernel and split of k may be chosen), so the comparison is to tolerance, not to the bit
    monkeypatch.setenv("RP_CONV_COL_BYTES", "1")
    monkeypatch.setenv("RP_CONV_NO_DIRECT", "1")           # and always through the lowered matrix
    again = _run_conv(x, w, b, dy, s, p, d, dt)
    for name, g, r, k in zip(names, again, refs, ks):
        if r is not None:
            assert oracle.rel_err(g, oracle.to_f64(r, dt)) <= tol(dt, k), name + " (chunked)"


@pytest.mark.parametrize("dtype", ["float32", "float64", "float16", "bfloat16"])
def test_conv2d_reference_known_answers(dtype):
    """reference tests/autograd/test_conv2d.py:46-152, 188-216 with device='cuda'."""
    for case in GOLD["conv2d_known_answers"]["cases"]:
        x = rp.ones(case["x_shape"], dtype=dtype, device="cuda").requires_grad_(True)
        w = rp.ones(case["w_shape"], dtype=dtype, device="cuda").requires_grad_(True)
        b = rp.values(case["bias"], dtype=dtype, device="cuda").requires_grad_(True) if "bias" in case else None
        s, p = case.get("stride", (1, 1)), case.get("pad", (0, 0))
        y = x.op_conv2d(w, bias=b, stride_h=s[0], stride_w=s[1], pad_h=p[0], pad_w=p[1])
        assert list(y.shape) == case["out_shape"] and y.dtype == dtype
        if "out_sum" in case:
            assert _host(y).sum() == case["out_sum"]
        y.op_sum_all().backward()
        assert x.has_grad and x.grad.shape == tuple(case["x_shape"])
        assert w.has_grad and w.grad.shape == tuple(case["w_shape"])
        if "bias_grad_of_sum" in case:
            assert b.grad.shape == (1,) and list(_host(b.grad)) == case["bias_grad_of_sum"]


def test_conv2d_weight_gradient_vs_central_differences():
    """reference tests/autograd/test_conv2d.py:154-186."""
    g = GOLD["conv2d_known_answers"]["weight_gradcheck"]
    x = np.array(g["x"], dtype=np.float64).reshape(g["x_shape"]); w = np.array(g["w"], dtype=np.float64).reshape(g["w_shape"])
    tw = _dev(w, F64, True)
    _dev(x, F64).op_conv2d(tw).op_sum_all().backward()
    eps = 1e-3
    for i in range(9):
        wp, wm = w.copy().reshape(-1), w.copy().reshape(-1)
        wp[i] += eps; wm[i] -= eps
        num = (_host(_dev(x, F64).op_conv2d(_dev(wp.reshape(w.shape), F64))).sum() - _host(_dev(x, F64).op_conv2d(_dev(wm.reshape(w.shape), F64))).sum()) / (2 * eps)
        assert abs(_host(tw.grad).reshape(-1)[i] - num) <= 1e-2 * max(1.0, abs(num))


def test_conv2d_module_and_argument_errors():
    """reference recpulse/module.py:117-155 (layout of the parameters, int or pair arguments) and ops/ops.c:4726-4742 (rejections)."""
    rp.manual_seed(3)
    layer = Conv2d(3, 8, 3, stride=(2, 1), padding=1).to(device="cuda")
    assert layer.weight.shape == (8, 3, 3, 3) and layer.bias.shape == (8,) and set(layer.tracked) == {"weight", "bias"}
    assert layer.kernel_size == (3, 3) and layer.stride == (2, 1) and layer.padding == (1, 1) and layer.dilation == (1, 1)
    w = _host(layer.weight)
    assert abs(w.std() - 1.0 / np.sqrt(27)) < 0.05 and np.all(_host(layer.bias) == 0)
    x = rp.randn([2, 3, 9, 8], device="cuda")
    y = layer(x)
    assert y.shape == (2, 8, 5, 8)
    y.op_sum_all().backward()
    assert layer.weight.has_grad and layer.bias.has_grad and np.all(_host(layer.bias.grad) == 2 * 5 * 8)
    assert Conv2d(3, 4, (1, 2), bias=False).bias is None
    with pytest.raises(RuntimeError):
        x.op_conv2d(rp.ones([4, 2, 3, 3], device="cuda"))            # channel mismatch
    with pytest.raises(RuntimeError):
        x.op_conv2d(rp.ones([4, 3, 11, 3], device="cuda"))           # kernel taller than the input
    with pytest.raises(RuntimeError):
        x.op_conv2d(rp.ones([4, 3, 3, 3], device="cuda"), stride_h=0)
    with pytest.raises(RuntimeError):
        x.reshape([6, 9, 8]).op_conv2d(rp.ones([4, 3, 3, 3], device="cuda"))
