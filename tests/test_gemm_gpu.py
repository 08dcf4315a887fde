"""GPU parity of the GEMM entry points against the CPU oracle and a float64 oracle.

Every case goes through the C ABI (rp_hip_gemm_strided_batched or
matmul_kernel_device).  Small cases are compared with the oracle's full
result; integer-valued cases must match bit for bit.
"""
import json
import os

import numpy as np
import pytest

import oracle
from recpulse_amd import capi
from devhelp import Dev, ALL, BF16, F16, F32, F64, NAMES, device_gemm, elem_strides, f64_gemm, oracle_gemm, rand_storage, tol

pytestmark = pytest.mark.gpu
GOLD = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "reference_known_answers.json")))


def _check(got, a, b, dtype, k, **kw):
    want = oracle_gemm(a, b, dtype, **kw)
    want64 = f64_gemm(a, b, dtype, **kw)
    e_orc = oracle.rel_err(oracle.to_f64(got, dtype), oracle.to_f64(want, dtype))
    e_64 = oracle.rel_err(oracle.to_f64(got, dtype), want64)
    assert e_orc <= tol(dtype, k), f"vs oracle {e_orc:.3e} > {tol(dtype, k):.3e}"
    assert e_64 <= tol(dtype, k), f"vs f64 {e_64:.3e} > {tol(dtype, k):.3e}"
    return e_orc, e_64


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_reference_known_answers_bit_exact(dt):
    for key in ("matmul_2x3_3x2", "matmul_identity"):
        g = GOLD[key]
        a = oracle.to_storage(np.array(g["a"], dtype=np.float64), dt)
        b = oracle.to_storage(np.array(g["b"], dtype=np.float64), dt)
        got = device_gemm(a, b, dt)
        assert np.array_equal(oracle.to_f64(got, dt), np.array(g["c"], dtype=np.float64)), key
    for key in ("backward_a", "backward_both_2x2", "backward_nonsquare_2x4_4x3"):
        g = GOLD[key]
        a = oracle.to_storage(np.array(g["a"], dtype=np.float64), dt)
        b = oracle.to_storage(np.array(g["b"], dtype=np.float64), dt)
        dc = oracle.to_storage(np.ones((a.shape[0], b.shape[1])), dt)
        da = device_gemm(dc, b.T, dt)            # dA = dC · Bᵀ, Bᵀ passed as a stride view
        db = device_gemm(a.T, dc, dt)            # dB = Aᵀ · dC
        assert np.array_equal(oracle.to_f64(da, dt), np.array(g["da"], dtype=np.float64)), key
        assert np.array_equal(oracle.to_f64(db, dt), np.array(g["db"], dtype=np.float64)), key


def test_matmul_kernel_device_seam_f64_parity_shapes():
    rng = np.random.default_rng(30)
    g = GOLD["parity_shapes"]
    for m, k, n in g["mkn"]:
        a = rng.uniform(-1, 1, (m, k)); b = rng.uniform(-1, 1, (k, n))
        da, db = capi.DeviceBuffer.from_numpy(a), capi.DeviceBuffer.from_numpy(b)
        dc = capi.DeviceBuffer(m * n * 8)
        capi.check(capi.lib().matmul_kernel_device(dc.ptr, da.ptr, db.ptr, m, k, n, F64), "matmul_kernel_device")
        capi.synchronize()
        np.testing.assert_allclose(dc.to_numpy(np.float64, (m, n)), a @ b, rtol=g["rtol"], atol=g["atol"])


LAYOUTS = ["nn", "nt", "tn", "tt"]
HALF = [F16, BF16]


def _operands(rng, m, k, n, dt, layout, dist="normal"):
    a = rand_storage(rng, (m, k), dt, dist) if layout[0] == "n" else rand_storage(rng, (k, m), dt, dist).T
    b = rand_storage(rng, (k, n), dt, dist) if layout[1] == "n" else rand_storage(rng, (n, k), dt, dist).T
    return a, b


SHAPES = [
    (3, 4, 5), (1, 7, 1), (16, 32, 8), (33, 65, 17),          # generic (odd extents)
    (64, 64, 64), (64, 128, 64), (48, 80, 56),                # 64x64 tiles, full and edge
    (128, 192, 128), (256, 64, 384), (200, 136, 264),         # 128x128 tiles, full and edge
    (128, 784, 256),                                          # config 1 shape
]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_small_shapes_all_layouts(dt, layout):
    rng = np.random.default_rng(31)
    for m, k, n in SHAPES:
        a, b = _operands(rng, m, k, n, dt, layout)
        got = device_gemm(a, b, dt)
        _check(got, a, b, dt, k)


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_integer_valued_inputs_are_exact(dt):
    """Small integers: every partial sum is exact in every dtype's accumulator, so any order must agree bit for bit."""
    rng = np.random.default_rng(32)
    for (m, k, n), layout in [((64, 64, 64), "nn"), ((128, 128, 128), "tn"), ((40, 24, 72), "nt"), ((130, 96, 66), "tt")]:
        a = oracle.to_storage(rng.integers(-3, 4, (m, k) if layout[0] == "n" else (k, m)).astype(np.float64), dt)
        b = oracle.to_storage(rng.integers(-3, 4, (k, n) if layout[1] == "n" else (n, k)).astype(np.float64), dt)
        a = a if layout[0] == "n" else a.T
        b = b if layout[1] == "n" else b.T
        got = device_gemm(a, b, dt)
        want = oracle_gemm(a, b, dt)
        assert np.array_equal(got, want), (m, k, n, layout)


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_bias_and_accumulate_epilogue(dt):
    rng = np.random.default_rng(33)
    for m, k, n in [(5, 9, 7), (64, 64, 64), (128, 784, 256), (72, 40, 136)]:
        a, b = _operands(rng, m, k, n, dt, "nn")
        bias = rand_storage(rng, (n,), dt)
        c0 = rand_storage(rng, (m, n), dt)
        for kw in ({"bias": bias}, {"c_init": c0, "accumulate": True}, {"bias": bias, "c_init": c0, "accumulate": True}):
            got = device_gemm(a, b, dt, **kw)
            _check(got, a, b, dt, k, **kw)
    # exact epilogue: integer data makes the whole chain exact, so the three roundings of the 16-bit chain must agree
    a = oracle.to_storage(rng.integers(-2, 3, (64, 64)).astype(np.float64), dt)
    b = oracle.to_storage(rng.integers(-2, 3, (64, 64)).astype(np.float64), dt)
    bias = oracle.to_storage(rng.integers(-4, 5, (64,)).astype(np.float64), dt)
    c0 = oracle.to_storage(rng.integers(-4, 5, (64, 64)).astype(np.float64), dt)
    got = device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True)
    assert np.array_equal(got, oracle_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True))


@pytest.mark.parametrize("dt", [F16, BF16], ids=lambda d: NAMES[d])
def test_16bit_rounding_is_the_references_half_away_from_zero(dt):
    """Products chosen so the fp32 sum sits exactly on a 16-bit tie: round-to-nearest-even would differ."""
    if dt == BF16:
        vals = [257.0, 259.0, -257.0]                        # 257 = 0x1.01p8: tie between 256 and 258 in bf16
    else:
        vals = [2049.0, 2051.0, -2049.0]                     # 2049: tie between 2048 and 2050 in fp16
    m = len(vals)
    a64 = np.zeros((m, 8)); b64 = np.zeros((8, 8))
    for i, v in enumerate(vals):
        a64[i, 0] = 1.0 if v > 0 else -1.0
        a64[i, 1] = 1.0 if v > 0 else -1.0
    b64[0, :] = 1.0
    got_all = []
    for i, v in enumerate(vals):
        b = b64.copy(); b[1, :] = abs(v) - 1.0              # |v|-1 is representable in both 16-bit formats for these values
        a_s = oracle.to_storage(a64[i:i + 1], dt); b_s = oracle.to_storage(b, dt)
        assert oracle.to_f64(b_s, dt)[1, 0] == abs(v) - 1.0
        got = device_gemm(a_s, b_s, dt)
        want = oracle_gemm(a_s, b_s, dt)
        assert np.array_equal(got, want), v
        got_all.append(oracle.to_f64(got, dt)[0, 0])
    assert got_all[0] == (258.0 if dt == BF16 else 2050.0)
    assert got_all[2] == (-258.0 if dt == BF16 else -2050.0)


@pytest.mark.parametrize("m,n,k", [(256, 128, 64), (512, 512, 256)])
def test_fp16_epilogue_rounding_at_the_tile_level(m, n, k):
    """The fp16 epilogue narrows a tile with two instructions per value when every value of it rounds to a normal fp16
    number and with the general rule otherwise.  C[i, j] = hi_i + lo_i * s_j is exact in fp32 and sits on, just above
    or just below a rounding tie of the reference's add-the-first-dropped-bit rule (core/half_precision.h:50-83);
    rows in the upper half of the output also hold zeros, results below the normal range, sums that overflow, and
    infinities, so their tiles take the general path.  Either way: the oracle's bits."""
    rng = np.random.default_rng(37)
    e = rng.integers(-3, 15, m)
    hi = (1.0 + rng.integers(0, 1024, m) / 1024.0) * np.exp2(e) * rng.choice([-1.0, 1.0], m)
    ulp = np.exp2(e - 10.0)
    frac = rng.choice([0.5, 0.5 * (1 + 2.0 ** -10), 0.5 * (1 - 2.0 ** -10), 0.25, 0.0, 0.75], m)
    lo = frac * ulp * np.sign(hi) * rng.choice([-1.0, 1.0], m)
    special = np.arange(m) >= m // 2
    pick = rng.integers(0, 6, m)
    hi = np.where(special & (pick == 0), 0.0, hi); lo = np.where(special & (pick == 0), 0.0, lo)                    # exact zero
    hi = np.where(special & (pick == 1), 2.0 ** -15 * 1.5, hi); lo = np.where(special & (pick == 1), 2.0 ** -24, lo)     # subnormal result
    hi = np.where(special & (pick == 2), 65504.0, hi); lo = np.where(special & (pick == 2), 16.0, lo)               # 65520: the reference's infinity
    hi = np.where(special & (pick == 3), np.inf, hi); lo = np.where(special & (pick == 3), 0.0, lo)
    hi = np.where(special & (pick == 4), 2.0 ** -14, hi); lo = np.where(special & (pick == 4), -(2.0 ** -24), lo)   # just below the smallest normal
    a64 = np.zeros((m, k)); a64[:, 0] = hi; a64[:, 1] = lo
    b64 = np.zeros((k, n)); b64[0, :] = 1.0; b64[1, :] = rng.choice([1.0, -1.0, 0.5, 0.0], n)
    a, b = oracle.to_storage(a64, F16), oracle.to_storage(b64, F16)
    assert np.array_equal(oracle.to_f64(a, F16)[:, :2], a64[:, :2])                  # the construction is representable
    with np.errstate(invalid="ignore", over="ignore"):
        want = oracle_gemm(a, b, F16)
    got = device_gemm(a, b, F16)
    assert capi.last_gemm_kernel().startswith("mfma16_")
    assert np.array_equal(got, want)


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_batched_strided_views(dt):
    rng = np.random.default_rng(34)
    B, H, S, D = 2, 3, 64, 32
    q = rand_storage(rng, (B * H, S, D), dt); kmat = rand_storage(rng, (B * H, S, D), dt)
    kt = kmat.transpose(0, 2, 1)                       # permuted view, no copy
    s = device_gemm(q, kt, dt)
    _check(s, q, kt, dt, D)
    p = rand_storage(rng, (B * H, S, S), dt); v = rand_storage(rng, (B * H, S, D), dt)
    o = device_gemm(p, v, dt)
    _check(o, p, v, dt, S)
    # dV = Pᵀ · dO with Pᵀ a view, odd sizes (generic path with batch)
    p2 = rand_storage(rng, (4, 9, 13), dt); do = rand_storage(rng, (4, 9, 5), dt)
    dv = device_gemm(p2.transpose(0, 2, 1), do, dt)
    _check(dv, p2.transpose(0, 2, 1), do, dt, 9)


@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("batch,m,k,n", [(3, 256, 128, 384), (13, 200, 96, 136), (37, 128, 192, 128), (192, 512, 128, 128)])
def test_batched_tiled_16bit_every_matrix_and_tile_once(dt, batch, m, k, n):
    """Batched products on the 16-bit tiled kernel, whose workgroups are re-dealt so that an XCD takes a contiguous
    share of the (matrix, tile) pairs: batch sizes that are no multiple of 8, ragged tiles, integer data so that a
    tile computed twice, skipped or taken from another matrix shows as a wrong value (every matrix has its own sum)."""
    rng = np.random.default_rng(36)
    assert capi.gemm_kernel_name(batch, m, k, n, (k, 1), (n, 1), (n, 1), dt).startswith("mfma16_")
    a64 = rng.integers(-2, 3, (batch, m, k)).astype(np.float64)
    b64 = rng.integers(-2, 3, (batch, k, n)).astype(np.float64)
    b64[:, 0, :] = 1.0
    a64[:, :, 0] = (np.arange(batch) % 5 - 2)[:, None]                   # a per-matrix constant added to every output
    a = oracle.to_storage(a64, dt); b = oracle.to_storage(b64, dt)
    got = device_gemm(a, b, dt)
    want = oracle.to_storage(np.einsum("zik,zkj->zij", a64, b64), dt)
    assert np.array_equal(got, want)


def test_sliced_operand_with_offset_and_padding():
    rng = np.random.default_rng(35)
    big_a = rand_storage(rng, (96, 200), F32); big_b = rand_storage(rng, (200, 160), F32)
    a = big_a[16:80, 8:136]          # 64 x 128 window, row stride 200, base offset
    b = big_b[8:136, 32:96]
    got = device_gemm(a, b, F32)
    _check(got, a, b, F32, 128)
    a2 = big_a[::2, ::2]             # no unit stride at all -> generic
    b2 = big_b[:100:1, ::2]
    got = device_gemm(a2, b2, F32)
    _check(got, a2, b2, F32, 100)


@pytest.mark.parametrize("dt", [BF16, F16, F32], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m", [1, 2, 4, 8])
def test_skinny_rows_streaming_kernel(dt, m):
    rng = np.random.default_rng(36)
    k, n = 2048, 1024
    if m <= 4 or dt == F32:
        assert capi.gemm_kernel_name(1, m, k, n, (k, 1), (n, 1), (n, 1), dt) == "skinny"
    a, b = _operands(rng, m, k, n, dt, "nn")
    bias = rand_storage(rng, (n,), dt)
    got = device_gemm(a, b, dt, bias=bias)
    _check(got, a, b, dt, k, bias=bias)
    got2 = device_gemm(a, b, dt, bias=bias)
    assert np.array_equal(got, got2)                   # split-k partials are combined in a fixed order


@pytest.mark.parametrize("dt", [BF16, F16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_skinny_rows_mfma_split_k(dt, layout):
    rng = np.random.default_rng(38)
    for m, k, n in [(8, 4096, 1024), (5, 4160, 1032), (32, 8192, 512), (16, 4096, 1024)]:
        if layout[0] == "t" and m % 8:
            continue                                   # a transposed A needs whole 16-byte vectors along m
        a, b = _operands(rng, m, k, n, dt, layout)
        a_st = (a.strides[0] // 2, a.strides[1] // 2); b_st = (b.strides[0] // 2, b.strides[1] // 2)
        want_kernel = _stream_kernel(m, k, n) if layout == "nn" else "mfma16_skinny_32x128"
        assert capi.gemm_kernel_name(1, m, k, n, a_st, b_st, (n, 1), dt) == want_kernel
        bias = rand_storage(rng, (n,), dt); c0 = rand_storage(rng, (m, n), dt)
        got = device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True)
        _check(got, a, b, dt, k, bias=bias, c_init=c0, accumulate=True)
        assert np.array_equal(got, device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True))
    # integer data: exact in fp32 whatever the split, so the split-k path must agree with the oracle bit for bit
    a = oracle.to_storage(rng.integers(-2, 3, (8, 4096)).astype(np.float64), dt)
    b = oracle.to_storage(rng.integers(-2, 3, (4096, 1024)).astype(np.float64), dt)
    assert np.array_equal(device_gemm(a, b, dt), oracle_gemm(a, b, dt))


def _stream_kernel(m, k, n):
    """Row-major A and B with at most 32 rows take the streaming kernel unless the split of k it would need makes its
    finish too long (the dispatcher's rule, restated for a device of 256 CUs): then the tiled kernel."""
    groups = -(-n // 128)
    nsplit = min(-(-256 // groups), max(1, k // 256))            # at least two passes of 128 rows per block
    takes = m <= 32 and n % 8 == 0 and k % 8 == 0 and nsplit * m <= 256 and (nsplit <= 8 or k * n >= 1 << 24)
    return "mfma16_stream_32x128" if takes else "mfma16_skinny_32x128"


@pytest.mark.parametrize("m", [1, 3, 5, 8, 11, 16, 17, 27, 32])
def test_streaming_rows_single_launch_finish(m):
    """Row-major A times row-major B with few rows: one launch, the last block of a column group to arrive adds the
    k splits.  Repeated launches must reproduce the first result bit for bit (fixed summation order, counters left
    clean), with ragged k (a partial last round, waves with unequal numbers of rounds) and n (a partial last strip, a
    number of strips that is not a multiple of 8), a bias and an accumulating epilogue."""
    rng = np.random.default_rng(39)
    for dt, k, n in [(BF16, 8192, 4096), (F16, 4104, 4104), (BF16, 1024, 4096), (F16, 1064, 8200), (BF16, 8192, 2048)]:
        a, b = _operands(rng, m, k, n, dt, "nn")
        assert capi.gemm_kernel_name(1, m, k, n, (k, 1), (n, 1), (n, 1), dt) == _stream_kernel(m, k, n)
        if (k, n) != (8192, 2048):
            assert _stream_kernel(m, k, n) == "mfma16_stream_32x128"          # (the shapes meant for the streaming kernel do take it)
        bias = rand_storage(rng, (n,), dt); c0 = rand_storage(rng, (m, n), dt)
        first = device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True)
        _check(first, a, b, dt, k, bias=bias, c_init=c0, accumulate=True)
        for _ in range(20):
            assert np.array_equal(first, device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True))
    # integer data is exact in fp32 whatever the split: bit-equal to the oracle, NaN and Inf carried through
    a = oracle.to_storage(rng.integers(-2, 3, (m, 4096)).astype(np.float64), BF16)
    b = oracle.to_storage(rng.integers(-2, 3, (4096, 1024)).astype(np.float64), BF16)
    assert np.array_equal(device_gemm(a, b, BF16), oracle_gemm(a, b, BF16))


@pytest.mark.parametrize("dt", [BF16, F16], ids=lambda d: NAMES[d])
def test_streaming_rows_output_layouts(dt):
    """The streaming kernel writes its output in three ways (one 8-byte vector per four columns without and with
    bias / accumulation, value by value when C's layout has no such vectors), from two places (the k-split finish,
    and the block itself when k is too short to split).  Every layout of C must hold the bits of the dense result,
    and the elements of C's buffer that are not part of C must keep theirs."""
    rng = np.random.default_rng(41)
    for m, k, n in [(8, 2048, 4096), (5, 1024, 32776), (27, 4096, 4104)]:           # 8 splits; no split (257 strips); ragged, 8 splits
        assert capi.gemm_kernel_name(1, m, k, n, (k, 1), (n, 1), (n, 1), dt) == "mfma16_stream_32x128"
        a, b = _operands(rng, m, k, n, dt, "nn")
        bias = rand_storage(rng, (n,), dt); c0 = rand_storage(rng, (m, n), dt)
        for with_epilogue in (False, True):
            kw = dict(bias=bias, c_init=c0, accumulate=True) if with_epilogue else {}
            dense = device_gemm(a, b, dt, **kw)
            _check(dense, a, b, dt, k, **kw)
            da, db, dbias = capi.DeviceBuffer.from_numpy(a), capi.DeviceBuffer.from_numpy(b), capi.DeviceBuffer.from_numpy(bias)
            for what, shape, view_of in [("padded rows, vectors", (m, n + 24), lambda buf: buf[:, :n]),
                                         ("odd row pitch", (m, n + 3), lambda buf: buf[:, :n]),
                                         ("column-major", (n, m + 2), lambda buf: buf[:, :m].T)]:
                host = np.full(shape, 0x7e31, dtype=capi.NP_STORAGE[dt])           # a pattern no result has everywhere
                guard = host.copy()
                if with_epilogue:
                    view_of(host)[...] = c0
                c_view = view_of(host)
                dc = capi.DeviceBuffer.from_numpy(host)
                capi.gemm(dc.ptr, da.ptr, db.ptr, dbias.ptr if with_epilogue else None, 1, m, k, n, (0, k, 1), (0, n, 1),
                          (0,) + tuple(elem_strides(c_view)), with_epilogue, dt)
                capi.synchronize()
                out = dc.to_numpy(capi.NP_STORAGE[dt], shape)
                dc.free()
                assert np.array_equal(view_of(out), dense), (what, m, k, n, with_epilogue)
                view_of(out)[...] = 0x7e31
                assert np.array_equal(out, guard), ("wrote outside C", what, m, k, n)
            for d in (da, db, dbias):
                d.free()


@pytest.mark.parametrize("m", [1, 8, 16, 32])
def test_streaming_rows_finish_repeats_bit_for_bit_over_hundreds_of_launches(m):
    """The finish exchanges partial sums between the workgroups of a column group while other groups still stream:
    launched back to back a few hundred times on resident operands (no synchronisation in between), every launch
    must leave the bits of the first one, and the fp64 product stays inside the tolerance."""
    rng = np.random.default_rng(41)
    k = n = 8192
    dt = BF16
    a = rand_storage(rng, (m, k), dt); b = rand_storage(rng, (k, n), dt)
    assert capi.gemm_kernel_name(1, m, k, n, (k, 1), (n, 1), (n, 1), dt) == "mfma16_stream_32x128"
    da, db = capi.DeviceBuffer.from_numpy(a), capi.DeviceBuffer.from_numpy(b)
    launches = 300
    outs = [capi.DeviceBuffer(m * n * 2) for _ in range(launches)]
    for dc in outs:
        capi.gemm(dc.ptr, da.ptr, db.ptr, None, 1, m, k, n, (0, k, 1), (0, n, 1), (0, n, 1), False, dt)
    capi.synchronize()
    first = outs[0].to_numpy(np.uint16, (m, n))
    for i, dc in enumerate(outs[1:], 1):
        assert np.array_equal(first, dc.to_numpy(np.uint16, (m, n))), f"launch {i} differs from launch 0"
    want = oracle.to_f64(a, dt) @ oracle.to_f64(b, dt)
    assert oracle.rel_err(oracle.to_f64(first, dt), want) <= tol(dt, k)


@pytest.mark.parametrize("dt,m,k,n", [(BF16, 17, 1032, 16648), (F16, 32, 2056, 16904), (F16, 104, 4168, 2312), (BF16, 40, 4104, 4168), (BF16, 96, 2056, 5480)])
def test_tiled_rows_split_k_with_both_operands_k_contiguous(dt, m, k, n):
    """More 32 x 32 tiles than the kernel whose waves split k takes: the k split in two launches, k and n ragged against slabs and strips, one
    to four row tiles, with bias and accumulation, repeated; small integers bit for bit."""
    rng = np.random.default_rng(45)
    a, b = _operands(rng, m, k, n, dt, "nt")
    bias, c0 = rand_storage(rng, (n,), dt), rand_storage(rng, (m, n), dt)
    first = device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True)
    assert capi.last_gemm_kernel() == "mfma16_skinny_32x128"
    want = oracle.to_f64(a, dt) @ oracle.to_f64(b, dt) + oracle.to_f64(bias, dt) + oracle.to_f64(c0, dt)
    assert oracle.rel_err(oracle.to_f64(first, dt), want) <= tol(dt, k)
    for _ in range(3):
        assert np.array_equal(first, device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True))
    ai, bi = rng.integers(-2, 3, a.shape).astype(np.float32), rng.integers(-2, 3, b.shape).astype(np.float32)
    a[...], b[...] = oracle.to_storage(ai.astype(np.float64), dt), oracle.to_storage(bi.astype(np.float64), dt)
    assert np.array_equal(device_gemm(a, b, dt), oracle.to_storage((ai @ bi).astype(np.float64), dt))
    assert capi.last_gemm_kernel() == "mfma16_skinny_32x128"


@pytest.mark.parametrize("layout", LAYOUTS)
def test_tiled_rows_split_k_ragged(layout):
    """More rows or another operand layout: the tiled kernel splits k across the grid and a second kernel adds the
    partial tiles in split order.  Ragged k (a partial last slab, splits of unequal length) and n (a partial last
    strip, a number of strips that is not a multiple of 8), several row tiles, bias and accumulation; repeated
    launches reproduce the first bit for bit."""
    rng = np.random.default_rng(43)
    for dt, m, k, n in [(BF16, 32, 8192, 2048), (F16, 24, 4104, 1288), (BF16, 17, 1032, 4096), (F16, 104, 4160, 1160), (BF16, 8, 2048, 2048)]:
        if (layout == "nn" and _stream_kernel(m, k, n) != "mfma16_skinny_32x128") or (layout[0] == "t" and m % 8):
            continue                                   # the streaming kernel's case; a transposed A needs whole 16-byte vectors along m
        a, b = _operands(rng, m, k, n, dt, layout)
        a_st = (a.strides[0] // 2, a.strides[1] // 2); b_st = (b.strides[0] // 2, b.strides[1] // 2)
        assert capi.gemm_kernel_name(1, m, k, n, a_st, b_st, (n, 1), dt) == "mfma16_skinny_32x128"
        bias = rand_storage(rng, (n,), dt); c0 = rand_storage(rng, (m, n), dt)
        first = device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True)
        _check(first, a, b, dt, k, bias=bias, c_init=c0, accumulate=True)
        for _ in range(10):
            assert np.array_equal(first, device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True))
    # integer data is exact in fp32 whatever the split: bit-equal to the oracle
    a, b = _operands(rng, 40, 4096, 1024, BF16, layout)
    a[...] = oracle.to_storage(rng.integers(-2, 3, a.shape).astype(np.float64), BF16)
    b[...] = oracle.to_storage(rng.integers(-2, 3, b.shape).astype(np.float64), BF16)
    assert np.array_equal(device_gemm(a, b, BF16), oracle_gemm(a, b, BF16))


def test_tiled_rows_repeat_bit_for_bit_over_hundreds_of_launches():
    """The tiled k-split kernel and its combine kernel share one workspace from the pool across back-to-back launches:
    300 launches without synchronisation in between leave the bits of the first."""
    rng = np.random.default_rng(44)
    m, k, n, dt = 40, 8192, 8192, BF16
    a = rand_storage(rng, (m, k), dt); b = rand_storage(rng, (k, n), dt)
    assert capi.gemm_kernel_name(1, m, k, n, (k, 1), (n, 1), (n, 1), dt) == "mfma16_skinny_32x128"
    da, db = capi.DeviceBuffer.from_numpy(a), capi.DeviceBuffer.from_numpy(b)
    outs = [capi.DeviceBuffer(m * n * 2) for _ in range(300)]
    for dc in outs:
        capi.gemm(dc.ptr, da.ptr, db.ptr, None, 1, m, k, n, (0, k, 1), (0, n, 1), (0, n, 1), False, dt)
    capi.synchronize()
    first = outs[0].to_numpy(np.uint16, (m, n))
    for i, dc in enumerate(outs[1:], 1):
        assert np.array_equal(first, dc.to_numpy(np.uint16, (m, n))), f"launch {i} differs from launch 0"
    want = oracle.to_f64(a, dt) @ oracle.to_f64(b, dt)
    assert oracle.rel_err(oracle.to_f64(first, dt), want) <= tol(dt, k)


def test_streaming_rows_both_exchanges_give_the_same_bits(tmp_path):
    """The k-split finish goes through the XCD's own L2 when workgroup placement was verified, and through memory at
    device scope otherwise (RP_HIP_DISABLE=l2_exchange forces that, read once per process): a child process computes
    the same products the other way, and the bits must agree (same partial sums, same order)."""
    import subprocess
    import sys
    code = (
        "import sys, numpy as np\n"
        "sys.path.insert(0, %r); sys.path.insert(0, %r)\n"
        "from devhelp import device_gemm, rand_storage, BF16, F16\n"
        "rng = np.random.default_rng(42)\n"
        "out = {}\n"
        "for i, (dt, m, k, n) in enumerate([(BF16, 1, 8192, 8192), (BF16, 8, 8192, 8192), (F16, 16, 4104, 1288), (BF16, 11, 2048, 2048), (BF16, 32, 8192, 8192), (F16, 27, 4104, 1288)]):\n"
        "    a = rand_storage(rng, (m, k), dt); b = rand_storage(rng, (k, n), dt)\n"
        "    out[str(i)] = device_gemm(a, b, dt)\n"
        "np.savez(sys.argv[1], **out)\n"
    ) % (os.path.dirname(os.path.abspath(__file__)), os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    results = []
    for flag in ("", "l2_exchange"):
        path = str(tmp_path / f"exchange_{flag or 'on'}.npz")
        env = dict(os.environ, RP_HIP_DISABLE=flag)
        subprocess.run([sys.executable, "-c", code, path], check=True, env=env, timeout=300)
        results.append(np.load(path))
    for key in results[0].files:
        assert np.array_equal(results[0][key], results[1][key]), f"case {key}: the two exchanges disagree"


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_pair_of_separately_allocated_matrices_in_one_launch(dt):
    """Batch strides of either sign: a batch of two whose second matrices are separate allocations, addressed by their
    distances from the first (how a recurrent cell's backward issues its input-side and recurrent-side products
    together).  Every matrix must equal the oracle's product of its own operands, whichever of the two allocations
    lies higher in memory; the deep-k shape takes the k-split kernel with a batch, the short-k one the resident kernel."""
    rng = np.random.default_rng(45)
    es = np.dtype(capi.NP_STORAGE[dt]).itemsize
    cases = [(64, 4096, 1024, "nt"), (1024, 64, 4096, "tn"), (33, 70, 65, "nn"), (64, 2048, 512, "nn")]
    if dt == F64:
        cases = cases[2:]
    for m, k, n, layout in cases:
        mats = []
        for _ in range(2):
            a, b = _operands(rng, m, k, n, dt, layout)
            c0 = rand_storage(rng, (m, n), dt)
            mats.append((a, b, c0))
        for accumulate in (False, True):
            for order in ((0, 1), (1, 0)):
                # allocations in the given order, so that both signs of every distance occur
                bufs = {}
                for i in order:
                    a, b, c0 = mats[i]
                    # (an operand view starts at its buffer's first element: uploading a dense copy of the view's
                    # transpose-free form and passing the view's strides addresses the same elements)
                    bufs[i] = (capi.DeviceBuffer.from_numpy(np.ascontiguousarray(a if layout[0] == "n" else a.T)),
                               capi.DeviceBuffer.from_numpy(np.ascontiguousarray(b if layout[1] == "n" else b.T)),
                               capi.DeviceBuffer.from_numpy(c0))
                a0, b0, _ = mats[0]
                dist = [(bufs[1][j].ptr - bufs[0][j].ptr) for j in range(3)]
                assert all(d % es == 0 for d in dist)
                a_st = (dist[0] // es,) + tuple(elem_strides(a0)); b_st = (dist[1] // es,) + tuple(elem_strides(b0))
                capi.gemm(bufs[0][2].ptr, bufs[0][0].ptr, bufs[0][1].ptr, None, 2, m, k, n, a_st, b_st, (dist[2] // es, n, 1), accumulate, dt)
                capi.synchronize()
                if dt in (BF16, F16) and k >= 2048 and k * n >= 1 << 22:
                    assert capi.last_gemm_kernel() == "mfma16_skinny_32x128"
                for i in (0, 1):
                    a, b, c0 = mats[i]
                    got = bufs[i][2].to_numpy(capi.NP_STORAGE[dt], (m, n))
                    _check(got, a, b, dt, k, c_init=c0 if accumulate else None, accumulate=accumulate)
                for i in (0, 1):
                    for d in bufs[i]:
                        d.free()


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_ragged_small_outputs_deep_k(dt):
    """Outputs that no vector kernel takes (n = 10, odd strides) with a deep k.  16-bit: the generic kernel splits k
    across blocks and a scalar kernel adds the partials in split order.  fp32: the one-launch 16 x 16-tile kernel, whose
    four waves add their partial tiles in wave order.  Either way results repeat bit for bit.  fp64 does not split."""
    rng = np.random.default_rng(40)
    for m, k, n, layout in [(128, 256, 10, "tn"), (256, 128, 10, "nn"), (17, 1000, 3, "nn"), (70, 333, 65, "nt"), (10, 96, 130, "tt")]:
        a, b = _operands(rng, m, k, n, dt, layout)
        es = a.itemsize
        if dt != F64:              # 2-element vectors fit some of these shapes, which then take the fp64 MFMA kernel
            name = capi.gemm_kernel_name(1, m, k, n, (a.strides[0] // es, a.strides[1] // es), (b.strides[0] // es, b.strides[1] // es), (n, 1), dt)
            assert name == ("tiny32_16x16" if dt == F32 else "generic")
        bias = rand_storage(rng, (n,), dt); c0 = rand_storage(rng, (m, n), dt)
        got = device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True)
        _check(got, a, b, dt, k, bias=bias, c_init=c0, accumulate=True)
        assert np.array_equal(got, device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True))


def test_large_tile_kernel_multi_slab():
    """4096 x 4096 outputs select the 256x256 tile; checked against float64 everywhere and the oracle on a row slab."""
    rng = np.random.default_rng(37)
    m = n = 4096; k = 320
    for dt, layout in [(BF16, "nn"), (F16, "tn"), (BF16, "nt"), (F16, "tt")]:
        assert capi.gemm_kernel_name(1, m, k, n, (k, 1), (n, 1), (n, 1), dt) == "mfma16_256x256"
        a, b = _operands(rng, m, k, n, dt, layout)
        got = device_gemm(a, b, dt)
        e64 = oracle.rel_err(oracle.to_f64(got, dt), f64_gemm(a, b, dt))
        assert e64 <= tol(dt, k), e64
        rows = np.array([0, 1, 255, 256, 1023, 2048, 4095])
        want = oracle.matmul(np.ascontiguousarray(a[rows]), np.ascontiguousarray(b), dt)
        assert oracle.rel_err(oracle.to_f64(got[rows], dt), oracle.to_f64(want, dt)) <= tol(dt, k)


def test_large_tile_kernel_with_ragged_edges():
    """The 256 x 256 tile (16 x 16 x 32 MFMAs) on extents that are whole vectors but not whole tiles or slabs: rows and
    columns past the edge, a last slab of 8, every layout, bias and accumulation.  Float64 everywhere, the oracle on
    sampled rows (first and last of tiles, the ragged last tile)."""
    rng = np.random.default_rng(43)
    m, k, n = 2856, 264, 3080
    for dt, layout, epilogue in [(BF16, "nn", True), (F16, "nt", False), (BF16, "tn", False), (F16, "tt", True)]:
        a, b = _operands(rng, m, k, n, dt, layout)
        es = a.itemsize
        assert capi.gemm_kernel_name(1, m, k, n, (a.strides[0] // es, a.strides[1] // es), (b.strides[0] // es, b.strides[1] // es), (n, 1), dt) == "mfma16_256x256"
        bias = rand_storage(rng, (n,), dt) if epilogue else None
        c0 = rand_storage(rng, (m, n), dt) if epilogue else None
        got = device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=epilogue)
        assert oracle.rel_err(oracle.to_f64(got, dt), f64_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=epilogue)) <= tol(dt, k)
        rows = np.array([0, 15, 16, 255, 256, 2559, 2560, 2815, 2816, 2855])
        _check(got[rows], np.ascontiguousarray(a[rows]), b, dt, k, bias=bias, c_init=None if c0 is None else np.ascontiguousarray(c0[rows]), accumulate=epilogue)


def test_wide_tiles_for_outputs_of_at_most_64_rows():
    """Up to 64 rows and many columns: 64 x 128 tiles while k is short, 64 x 256 beyond (one row of waves, no MFMA
    spent on rows past m).  Full tiles and ragged ones, every layout, bias and accumulation; checked against float64
    everywhere and against the oracle on a slab of columns."""
    rng = np.random.default_rng(41)
    cases = [(64, 192, 32768, BF16, "nn", "mfma16_64x128", False), (33, 64, 32776, F16, "nt", "mfma16_64x128", True),
             (64, 1088, 32768, BF16, "tn", "mfma16_64x256", True), (40, 1096, 32776, F16, "nn", "mfma16_64x256", False)]
    for m, k, n, dt, layout, kernel, epilogue in cases:
        a, b = _operands(rng, m, k, n, dt, layout)
        es = a.itemsize
        assert capi.gemm_kernel_name(1, m, k, n, (a.strides[0] // es, a.strides[1] // es), (b.strides[0] // es, b.strides[1] // es), (n, 1), dt) == kernel
        bias = rand_storage(rng, (n,), dt) if epilogue else None
        c0 = rand_storage(rng, (m, n), dt) if epilogue else None
        got = device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=epilogue)
        assert oracle.rel_err(oracle.to_f64(got, dt), f64_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=epilogue)) <= tol(dt, k)
        cols = np.r_[0:8, 250:262, n - 9:n]
        _check(got[:, cols], a, np.ascontiguousarray(b[:, cols]), dt, k, bias=None if bias is None else bias[cols],
               c_init=None if c0 is None else np.ascontiguousarray(c0[:, cols]), accumulate=epilogue)


RAGGED_SHAPES = [  # (batch, m, k, n, kernel): every 16-bit tile, k of one slab and its tails, free axes that end 1 .. 7 past a vector
    (1, 1000, 9, 9, "mfma16_64x64"), (1, 131, 8, 65, "mfma16_64x64"), (1, 203, 63, 129, "mfma16_64x64"), (3, 121, 65, 71, "mfma16_64x64"),
    (1, 199, 391, 137, "mfma16_64x64"), (1, 1450, 127, 1403, "mfma16_128x128"), (130, 33, 77, 261, "mfma16_64x128"), (66, 35, 1025, 305, "mfma16_64x256"),
    (1, 3000, 259, 2821, "mfma16_256x256"), (1, 65, 2561, 127, "generic"), (1, 65, 2557, 127, "mfma16_64x64"), (1, 5, 4099, 1027, "mfma16_skinny_32x128"), (1, 33, 4102, 1035, "mfma16_skinny_32x128")]


RAGGED_WIDE_SHAPES = [  # the same for fp32 (with and without a k split) and fp64
    (F32, 1, 600, 33, 517, "mfma32_64x64"), (F32, 1, 530, 261, 527, "mfma32_64x64"), (F32, 70, 65, 7, 71, "mfma32_64x64"), (F32, 1, 1450, 67, 1403, "mfma32_128x128"),
    (F64, 1, 131, 5, 67, "mfma64_64x64"), (F64, 3, 121, 65, 71, "mfma64_64x64"), (F64, 1, 1450, 33, 1403, "mfma64_64x64"), (F32, 1, 1450, 31, 1403, "mfma32_64x64")]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("dt,batch,m,k,n,kernel", [(dt,) + shape for dt in HALF for shape in RAGGED_SHAPES] + RAGGED_WIDE_SHAPES)
def test_ragged_rows(dt, batch, m, k, n, kernel, layout):
    """Rows at any element and of any length on the MFMA kernels.  The operands are slices of NaN-filled arrays that end
    with the operand's last element, so a value taken from outside the slice shows; integers, so the bits are known."""
    rng = np.random.default_rng(46)
    fill = oracle.to_storage(np.full(1, np.nan), dt)[0]
    es = capi.DTYPE_SIZE[dt]

    def operand(rows, cols):                       # [batch, rows, cols], pitch cols + 3, everything around it NaN, nothing after it
        flat = np.full(1 + batch * rows * (cols + 3) - 3, fill)
        view = np.lib.stride_tricks.as_strided(flat[1:], (batch, rows, cols), (rows * (cols + 3) * es, (cols + 3) * es, es))
        vals = rng.integers(-2, 3, (batch, rows, cols)).astype(np.float64)
        view[...] = oracle.to_storage(vals, dt)
        return capi.DeviceBuffer.from_numpy(flat), vals, (rows * (cols + 3), cols + 3, 1)

    da, a64, a_st = operand(m, k) if layout[0] == "n" else operand(k, m)
    db, b64, b_st = operand(k, n) if layout[1] == "n" else operand(n, k)
    if layout[0] == "t":
        a64, a_st = a64.transpose(0, 2, 1), (a_st[0], a_st[2], a_st[1])
    if layout[1] == "t":
        b64, b_st = b64.transpose(0, 2, 1), (b_st[0], b_st[2], b_st[1])
    exact = np.matmul(a64, b64)
    bias = oracle.to_storage(rng.integers(-2, 3, n).astype(np.float64), dt)
    dbias = capi.DeviceBuffer.from_numpy(bias)
    pitch = n + 5
    c0 = oracle.to_storage(rng.integers(-2, 3, (batch, m, pitch)).astype(np.float64), dt)
    for with_bias, accumulate in ((False, False), (True, True)):
        dc = capi.DeviceBuffer.from_numpy(c0)
        capi.gemm(dc.at(es), da.at(es), db.at(es), dbias.ptr if with_bias else None, batch, m, k, n, a_st, b_st, (m * pitch, pitch, 1), accumulate, dt)
        assert capi.last_gemm_kernel() == ("generic" if layout[0] == "t" and m < 8 else kernel)      # fewer than a vector of rows to load along
        want = oracle.to_storage(exact, dt)
        if with_bias:
            want = oracle.to_storage(oracle.to_f64(want, dt) + oracle.to_f64(bias, dt), dt)
        expect = c0.reshape(-1).copy()
        inner = np.lib.stride_tricks.as_strided(expect[1:], (batch, m, n), (m * pitch * es, pitch * es, es))
        inner[...] = oracle.to_storage(oracle.to_f64(inner.copy(), dt) + oracle.to_f64(want, dt), dt) if accumulate else want
        assert np.array_equal(dc.to_numpy(c0.dtype, (expect.size,)), expect)      # C, and nothing around it
        dc.free()


# (dtype, batch, m, k, n, name, launched, layouts): ragged rows on waves that share k in the place of the kernel named, and those that are left to it
RAGGED_LAUNCHES = [(BF16, 1, 5, 4099, 1027, "mfma16_skinny_32x128", "mfma16_wavek_ragged", ["nt"]), (F16, 1, 65, 2561, 127, "generic", "mfma16_wavek_ragged", ["nn", "nt"]),
                   (F32, 1, 530, 261, 527, "mfma32_64x64", "mfma32_wavek_32x32", LAYOUTS), (F64, 1, 131, 5, 67, "mfma64_64x64", "mfma64_wavek_16x16", LAYOUTS),
                   (F32, 1, 16, 5745, 49, "mfma32_64x64", "mfma32_64x64", LAYOUTS), (F32, 1, 60, 2049, 131, "mfma32_64x64", "mfma32_64x64", LAYOUTS),
                   (F32, 1, 1450, 31, 1403, "mfma32_64x64", "mfma32_64x64", LAYOUTS), (F64, 1, 1450, 33, 1403, "mfma64_64x64", "mfma64_64x64", LAYOUTS),
                   (F64, 2, 1100, 41, 563, "mfma64_64x64", "mfma64_64x64", LAYOUTS), (BF16, 1, 105, 4165, 2311, "mfma16_skinny_32x128", "mfma16_skinny_32x128", ["nt"]),
                   (F16, 1, 105, 4165, 2311, "mfma16_skinny_32x128", "mfma16_skinny_32x128", ["nt"]), (BF16, 1, 11, 3261, 63, "generic", "generic", ["nn"])]


@pytest.mark.parametrize("dt,batch,m,k,n,kernel,launched,layout", [c[:-1] + (layout,) for c in RAGGED_LAUNCHES for layout in c[-1]])
def test_ragged_rows_by_the_kernel_launched(dt, batch, m, k, n, kernel, launched, layout):
    test_ragged_rows(dt, batch, m, k, n, kernel, layout)
    assert capi.last_gemm_launch() == launched


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m,k,n", [(64, 704, 128), (64, 768, 128), (128, 832, 64), (64, 896, 192), (72, 712, 136), (136, 776, 200), (200, 840, 72), (8, 904, 72), (64, 961, 129), (130, 1535, 66)])
def test_deep_prefetch_small_tiles(m, k, n, dt, layout):
    """64 x 64 tiles around the number of k slabs from which three of them travel at a time, for every remainder of the slabs by
    three, whole and hanging over; sums of small integers, so every slab must be added exactly once."""
    rng = np.random.default_rng(m * 7 + k + n)
    a = oracle.to_storage(rng.integers(-2, 3, (m, k) if layout[0] == "n" else (k, m)).astype(np.float64), dt)
    b = oracle.to_storage(rng.integers(-2, 3, (k, n) if layout[1] == "n" else (n, k)).astype(np.float64), dt)
    av, bv = (a if layout[0] == "n" else a.T), (b if layout[1] == "n" else b.T)
    bias = oracle.to_storage(rng.integers(-3, 4, n).astype(np.float64), dt)
    got = device_gemm(av, bv, dt, bias=bias)
    # sums of at most 1535 products of at most 4 in magnitude whose spread is about 80: rounded to 16 bits once, then the bias once
    assert np.array_equal(got, oracle_gemm(av, bv, dt, bias=bias))


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m,k,n", [(576, 704, 512), (576, 768, 512), (576, 832, 512), (576, 896, 512), (520, 712, 504), (520, 776, 504), (520, 840, 504), (520, 904, 504)])
def test_deep_prefetch_small_tiles_of_every_layout(m, k, n, dt, layout):
    """The same for outputs of more tiles than the kernel whose waves split k takes, whichever way round A lies: eleven slabs (one at a time)
    to fifteen (three at a time, every remainder), whole and hanging over."""
    rng = np.random.default_rng(m + k)
    a, b = rng.integers(-2, 3, (m, k)).astype(np.float32), rng.integers(-2, 3, (k, n)).astype(np.float32)
    bias = rng.integers(-3, 4, n).astype(np.float64)
    sa, sb = (oracle.to_storage(np.ascontiguousarray(v if lay == "n" else v.T).astype(np.float64), dt) for v, lay in zip((a, b), layout))
    got = device_gemm(sa if layout[0] == "n" else sa.T, sb if layout[1] == "n" else sb.T, dt, bias=oracle.to_storage(bias, dt))
    assert capi.last_gemm_kernel() == "mfma16_64x64"
    # sums of at most 904 products of at most 4 in magnitude, exact in fp32; one rounding each for the product and the bias
    product = oracle.to_f64(oracle.to_storage((a @ b).astype(np.float64), dt), dt)
    assert np.array_equal(got, oracle.to_storage(product + bias, dt))


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m,n", [(256, 784), (251, 785), (4096, 9), (9, 4096), (128, 96)])
def test_outer_products(dt, m, n):
    """k = 1, where the strides of k may hold anything: those of a contiguous [m, 1] and of an expanded row are 1 and 0.  An
    infinity and a NaN spoil their own row and column and nothing beside them."""
    rng = np.random.default_rng(52)
    a64, b64 = rng.integers(-2, 3, (m, 1)).astype(np.float64), rng.integers(-2, 3, (1, n)).astype(np.float64)
    a64[m // 2], b64[0, n - 1] = np.inf, np.nan
    a, b = oracle.to_storage(a64, dt), oracle.to_storage(b64, dt)
    da, db, dc = Dev(a, dt), Dev(b, dt), Dev.empty((m, n), dt)
    with np.errstate(invalid="ignore"):
        want = oracle.to_f64(oracle.to_storage(a64 * b64, dt), dt)
    for a_k in (0, 1, m, m + 3):
        for b_k in (0, 1, n, n + 5):
            capi.gemm(dc.ptr, da.ptr, db.ptr, None, 1, m, 1, n, (0, 1, a_k), (0, b_k, 1), (0, n, 1), False, dt)
            assert np.array_equal(oracle.to_f64(dc.numpy(), dt), want, equal_nan=True), (a_k, b_k, capi.last_gemm_kernel())
    # the gradients of a layer with one output: dx = dy . w^T is such a product, dw = x^T . dy has one column
    x = rand_storage(rng, (m, n), dt)
    dy = oracle.to_storage(rng.integers(-2, 3, (m, 1)).astype(np.float64), dt)
    w = oracle.to_storage(rng.integers(-2, 3, (n, 1)).astype(np.float64), dt)
    d_x, d_w, d_dy, d_dx, d_dw, d_db = Dev(x, dt), Dev(w, dt), Dev(dy, dt), Dev.empty((m, n), dt), Dev.empty((n, 1), dt), Dev.empty((1,), dt)
    capi.check(capi.lib().rp_hip_linear_backward(d_dx.ptr, d_dw.ptr, d_db.ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, n, 1, n, 1, 1, 1, n, 1, 1, 1, 0, 0, 0, dt), "linear_backward")
    assert np.array_equal(oracle.to_f64(d_dx.numpy(), dt), oracle.to_f64(dy, dt) @ oracle.to_f64(w, dt).T)
    want_dw = oracle.to_f64(x, dt).T @ oracle.to_f64(dy, dt)
    assert oracle.rel_err(oracle.to_f64(d_dw.numpy(), dt), want_dw) <= tol(dt, m)
    assert d_db.numpy()[0] == oracle.to_storage(oracle.to_f64(dy, dt).sum(0), dt)[0]


@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("k", [8, 72, 128, 1032])
def test_operands_expanded_along_k(dt, k):
    """Both operands with k stride 0 or rows of k that overlap: what lies behind the last k row is inside the buffer."""
    rng = np.random.default_rng(53)
    m, n = 128, 256
    for a_k, b_k in ((0, 0), (8, 8), (0, n), (m, 8)):
        a, b = rng.integers(-2, 3, m + max(a_k, 8) * k).astype(np.float64), rng.integers(-2, 3, n + max(b_k, 8) * k).astype(np.float64)
        b[n + b_k * (k - 1):] = np.nan
        es = a.itemsize
        av = np.lib.stride_tricks.as_strided(a, (m, k), (es, a_k * es))
        bv = np.lib.stride_tricks.as_strided(b, (k, n), (b_k * es, es))
        da, db, dc = Dev(oracle.to_storage(a, dt), dt), Dev(oracle.to_storage(b, dt), dt), Dev.empty((m, n), dt)
        capi.gemm(dc.ptr, da.ptr, db.ptr, None, 1, m, k, n, (0, 1, a_k), (0, b_k, 1), (0, n, 1), False, dt)
        assert np.array_equal(dc.numpy(), oracle.to_storage(np.matmul(av, bv), dt)), (a_k, b_k, capi.last_gemm_kernel())


@pytest.mark.parametrize("dt", ALL, ids=lambda d: NAMES[d])
def test_linear_backward_in_one_call(dt):
    """rp_hip_linear_backward against two GEMM calls with swapped strides and rp_hip_reduce_rows: the same bits,
    whether the three run as one launch (small float32 layers) or one after the other; outputs that are absent,
    accumulated into, and a transposed x view."""
    rng = np.random.default_rng(42)
    L = capi.lib()
    for m, k, n in ((256, 784, 256), (256, 128, 10), (37, 50, 21), (512, 1024, 512)):
        x, w, dy = rand_storage(rng, (m, k), dt), rand_storage(rng, (k, n), dt), rand_storage(rng, (m, n), dt)
        dx0, dw0, db0 = rand_storage(rng, (m, k), dt), rand_storage(rng, (k, n), dt), rand_storage(rng, (n,), dt)
        d_x, d_w, d_dy = Dev(x, dt), Dev(w, dt), Dev(dy, dt)
        for acc in (0, 1):
            want_dx, want_dw, want_db = Dev(dx0, dt), Dev(dw0, dt), Dev(db0, dt)
            capi.gemm(want_dx.ptr, d_dy.ptr, d_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n), (0, k, 1), bool(acc), dt)
            capi.gemm(want_dw.ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n, 1), bool(acc), dt)
            capi.check(L.rp_hip_reduce_rows(want_db.ptr, d_dy.ptr, m, n, acc, dt), "reduce_rows")
            got_dx, got_dw, got_db = Dev(dx0, dt), Dev(dw0, dt), Dev(db0, dt)
            capi.check(L.rp_hip_linear_backward(got_dx.ptr, got_dw.ptr, got_db.ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n,
                                                k, 1, n, 1, k, 1, n, 1, acc, acc, acc, dt), "linear_backward")
            assert np.array_equal(got_dx.numpy(), want_dx.numpy()) and np.array_equal(got_dw.numpy(), want_dw.numpy())
            assert np.array_equal(got_db.numpy(), want_db.numpy())
        # only some of the outputs, and x given as the transpose of a [k, m] array
        xt = Dev(np.ascontiguousarray(x.T), dt)
        only_w, only_b = Dev(dw0, dt), Dev(db0, dt)
        capi.check(L.rp_hip_linear_backward(None, only_w.ptr, None, d_dy.ptr, xt.ptr, None, m, k, n, 1, m, n, 1, k, 1, n, 1, 0, 0, 0, dt), "dw only")
        capi.check(L.rp_hip_linear_backward(None, None, only_b.ptr, d_dy.ptr, None, None, m, k, n, k, 1, n, 1, k, 1, n, 1, 0, 0, 0, dt), "db only")
        ref_w = Dev(dw0, dt)
        capi.gemm(ref_w.ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n, 1), False, dt)
        assert oracle.rel_err(oracle.to_f64(only_w.numpy(), dt), oracle.to_f64(ref_w.numpy(), dt)) <= tol(dt, m)     # another layout may take another kernel
        ref_b = Dev(db0, dt)
        capi.check(L.rp_hip_reduce_rows(ref_b.ptr, d_dy.ptr, m, n, 0, dt), "reduce_rows")
        assert np.array_equal(only_b.numpy(), ref_b.numpy())
        _, dwant = oracle.matmul_backward(x, w, dy, dt)
        assert oracle.rel_err(oracle.to_f64(only_w.numpy(), dt), oracle.to_f64(dwant, dt)) <= tol(dt, m)
    assert L.rp_hip_linear_backward(None, None, None, None, None, None, 4, 4, 4, 4, 1, 4, 1, 4, 1, 4, 1, 0, 0, 0, dt) == -1


@pytest.mark.parametrize("dt", [BF16, F16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("shape", [(64, 64, 64), (72, 136, 264), (8, 512, 520), (200, 1032, 72), (448, 704, 1024), (1024, 1024, 1024)], ids=lambda s: "x".join(map(str, s)))
def test_linear_backward_pair_16bit(dt, shape):
    """dX and dW of a 16-bit layer in one launch: the bits of the two products, also accumulated and in padded rows; dW written
    over W (which dX reads) is the two products one after the other."""
    m, k, n = shape
    rng = np.random.default_rng(43)
    L = capi.lib()
    x, w, dy = rand_storage(rng, (m, k), dt), rand_storage(rng, (k, n), dt), rand_storage(rng, (m, n), dt)
    pad = 3                                             # rows of the gradients that start anywhere
    dx0, dw0 = rand_storage(rng, (m, k + pad), dt), rand_storage(rng, (k, n + pad), dt)
    d_x, d_w, d_dy = Dev(x, dt), Dev(w, dt), Dev(dy, dt)
    for acc in (0, 1):
        want_dx, want_dw, got_dx, got_dw = Dev(dx0, dt), Dev(dw0, dt), Dev(dx0, dt), Dev(dw0, dt)
        capi.gemm(want_dx.ptr, d_dy.ptr, d_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n), (0, k + pad, 1), bool(acc), dt)
        capi.gemm(want_dw.ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n + pad, 1), bool(acc), dt)
        capi.check(L.rp_hip_linear_backward(got_dx.ptr, got_dw.ptr, None, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n,
                                            k, 1, n, 1, k + pad, 1, n + pad, 1, acc, acc, 0, dt), "linear_backward")
        assert capi.last_gemm_kernel() == "linear_backward16_64x64"
        assert np.array_equal(got_dx.numpy(), want_dx.numpy()) and np.array_equal(got_dw.numpy(), want_dw.numpy())
    want_dx, want_dw, got_dx = Dev.empty((m, k), dt), Dev.empty((k, n), dt), Dev.empty((m, k), dt)
    capi.gemm(want_dx.ptr, d_dy.ptr, d_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n), (0, k, 1), False, dt)
    capi.gemm(want_dw.ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n, 1), False, dt)
    capi.check(L.rp_hip_linear_backward(got_dx.ptr, d_w.ptr, None, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n,
                                        k, 1, n, 1, k, 1, n, 1, 0, 0, 0, dt), "dW over W")
    assert capi.last_gemm_kernel() != "linear_backward16_64x64"
    assert np.array_equal(got_dx.numpy(), want_dx.numpy()) and np.array_equal(d_w.numpy(), want_dw.numpy())


@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("shape", [(8, 8, 640), (72, 136, 648), (40, 24, 4104), (33, 72, 1032), (64, 256, 4096), (300, 304, 640), (264, 312, 1600),
                                   (248, 1000, 1544), (512, 512, 640), (1024, 256, 704), (64, 1024, 1024)], ids=lambda s: "x".join(map(str, s)))
def test_linear_backward_pair_whose_dx_splits_k(dt, shape):
    """Layers whose dX has few tiles and a deep reduction: in one launch with dW and db, alone in its own call and as a separate product
    the same bits (every tile size of the kernel whose waves split k, whole and ragged), accumulated and in padded rows too."""
    m, k, n = shape
    rng = np.random.default_rng(m + k + n)
    L, pad = capi.lib(), 3
    x, w, dy = rand_storage(rng, (m, k), dt), rand_storage(rng, (k, n), dt), rand_storage(rng, (m, n), dt)
    dx0, dw0, db0 = rand_storage(rng, (m, k + pad), dt), rand_storage(rng, (k, n + pad), dt), rand_storage(rng, (n,), dt)
    d_x, d_w, d_dy = Dev(x, dt), Dev(w, dt), Dev(dy, dt)
    for acc in (0, 1):
        want = Dev(dx0, dt), Dev(dw0, dt), Dev(db0, dt)
        capi.gemm(want[0].ptr, d_dy.ptr, d_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n), (0, k + pad, 1), bool(acc), dt)
        assert capi.last_gemm_kernel() == "mfma16_wavek"
        capi.gemm(want[1].ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n + pad, 1), bool(acc), dt)
        capi.check(L.rp_hip_reduce_rows(want[2].ptr, d_dy.ptr, m, n, acc, dt), "reduce_rows")
        got, alone = (Dev(dx0, dt), Dev(dw0, dt), Dev(db0, dt)), Dev(dx0, dt)
        capi.check(L.rp_hip_linear_backward(got[0].ptr, got[1].ptr, got[2].ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n,
                                            k, 1, n, 1, k + pad, 1, n + pad, 1, acc, acc, acc, dt), "linear_backward")
        assert capi.last_gemm_kernel() == "linear_backward16_64x64"
        capi.check(L.rp_hip_linear_backward(alone.ptr, None, None, d_dy.ptr, None, d_w.ptr, m, k, n,
                                            0, 0, n, 1, k + pad, 1, 0, 0, acc, 0, 0, dt), "linear_backward (dX alone)")
        for name, a, b in zip(("dX", "dW", "db"), got, want):
            assert np.array_equal(a.numpy(), b.numpy()), name
        assert np.array_equal(alone.numpy(), want[0].numpy())


@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m,n", [(8, 8), (64, 72), (248, 40), (256, 264), (264, 32), (520, 1032), (768, 40), (776, 40), (1024, 128), (1024, 136), (1032, 64), (2048, 136), (2056, 64)])
def test_bias_gradient_beside_the_paired_gradients(dt, m, n):
    """db in the launch of dX and dW (up to 1024 rows, 768 where a strip of columns hangs over), around its chunks of rows and strips of columns: the bits of
    rp_hip_reduce_rows, written and added; over W, which the launch still reads, it comes in a launch of its own."""
    rng = np.random.default_rng(m + n)
    L, k = capi.lib(), 64
    x, w, dy, db0 = rand_storage(rng, (m, k), dt), rand_storage(rng, (k, n), dt), rand_storage(rng, (m, n), dt), rand_storage(rng, (n,), dt)
    d_x, d_w, d_dy, d_dx, d_dw = Dev(x, dt), Dev(w, dt), Dev(dy, dt), Dev.empty((m, k), dt), Dev.empty((k, n), dt)
    for acc in (0, 1):
        want, got = Dev(db0, dt), Dev(db0, dt)
        capi.check(L.rp_hip_reduce_rows(want.ptr, d_dy.ptr, m, n, acc, dt), "reduce_rows")
        capi.check(L.rp_hip_linear_backward(d_dx.ptr, d_dw.ptr, got.ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n, k, 1, n, 1, k, 1, n, 1, 0, 0, acc, dt), "backward")
        assert L.rp_hip_last_gemm_kernel() == b"linear_backward16_64x64"
        assert np.array_equal(got.numpy(), want.numpy())
    want_dx = d_dx.numpy()
    capi.check(L.rp_hip_linear_backward(d_dx.ptr, d_dw.ptr, d_w.ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n, k, 1, n, 1, k, 1, n, 1, 0, 0, 0, dt), "db over W")
    capi.check(L.rp_hip_reduce_rows(want.ptr, d_dy.ptr, m, n, 0, dt), "reduce_rows")
    assert np.array_equal(d_dx.numpy(), want_dx) and np.array_equal(d_w.numpy().reshape(-1)[:n], want.numpy())


@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("m,k,n", [(119, 57, 245), (57, 50, 859), (754, 43, 201), (33, 1033, 71), (9, 1001, 9), (300, 305, 641), (64, 72, 1001), (72, 65, 1024), (1030, 129, 77), (130, 1025, 9)])
def test_gradients_of_ragged_layers_in_one_launch(m, k, n, dt):
    """Layers whose rows are no whole vectors: dX, dW and db together have the bits of the three on their own, also accumulated."""
    rng = np.random.default_rng(m + k + n)
    L = capi.lib()
    x, w, dy = rand_storage(rng, (m, k), dt), rand_storage(rng, (k, n), dt), rand_storage(rng, (m, n), dt)
    d_x, d_w, d_dy = Dev(x, dt), Dev(w, dt), Dev(dy, dt)
    init = [rand_storage(rng, s, dt) for s in ((m, k), (k, n), (n,))]
    for acc in (0, 1):
        want, got = [Dev(i, dt) for i in init], [Dev(i, dt) for i in init]
        capi.gemm(want[0].ptr, d_dy.ptr, d_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n), (0, k, 1), bool(acc), dt)
        capi.gemm(want[1].ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n, 1), bool(acc), dt)
        capi.check(L.rp_hip_reduce_rows(want[2].ptr, d_dy.ptr, m, n, acc, dt), "reduce_rows")
        capi.check(L.rp_hip_linear_backward(got[0].ptr, got[1].ptr, got[2].ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n, k, 1, n, 1, k, 1, n, 1, acc, acc, acc, dt), "linear_backward")
        assert capi.last_gemm_kernel() == "linear_backward16_64x64"
        for g, t in zip(got, want):
            assert np.array_equal(g.numpy(), t.numpy())


@pytest.mark.parametrize("dt,m,k,n", [(F32,) + s for s in ((935, 213, 862), (20, 100, 700), (700, 30, 40), (600, 200, 600), (600, 900, 50), (513, 64, 2000), (33, 1200, 600), (600, 130, 500),
                                                          (520, 420, 500), (64, 1024, 1024), (1100, 40, 600))]
                         + [(F64,) + s for s in ((89, 2787, 286), (64, 60, 70), (500, 40, 600), (200, 1000, 33), (33, 100, 2000), (1030, 64, 96))])
def test_gradients_whose_waves_share_k_in_one_launch(dt, m, k, n):
    """fp32 and fp64 layers, every pair of tiles that the two products can be on: dX, dW and db together have the bits of the three on their own, also
    accumulated; dW written over W (which dX reads) is the three one after the other."""
    rng = np.random.default_rng(m + k + n)
    L = capi.lib()
    x, w, dy = rand_storage(rng, (m, k), dt), rand_storage(rng, (k, n), dt), rand_storage(rng, (m, n), dt)
    d_x, d_w, d_dy = Dev(x, dt), Dev(w, dt), Dev(dy, dt)
    init = [rand_storage(rng, s, dt) for s in ((m, k), (k, n), (n,))]
    for acc in (0, 1):
        want, got = [Dev(i, dt) for i in init], [Dev(i, dt) for i in init]
        capi.gemm(want[0].ptr, d_dy.ptr, d_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n), (0, k, 1), bool(acc), dt)
        capi.gemm(want[1].ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n, 1), bool(acc), dt)
        capi.check(L.rp_hip_reduce_rows(want[2].ptr, d_dy.ptr, m, n, acc, dt), "reduce_rows")
        capi.check(L.rp_hip_linear_backward(got[0].ptr, got[1].ptr, got[2].ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n, k, 1, n, 1, k, 1, n, 1, acc, acc, acc, dt), "linear_backward")
        assert capi.last_gemm_kernel() == "linear_backward_wavek"
        for g, t in zip(got, want):
            assert np.array_equal(g.numpy(), t.numpy())
    want, got = [Dev(i, dt) for i in init[:2]], Dev(init[0], dt)
    capi.gemm(want[0].ptr, d_dy.ptr, d_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n), (0, k, 1), False, dt)
    capi.gemm(want[1].ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n, 1), False, dt)
    capi.check(L.rp_hip_linear_backward(got.ptr, d_w.ptr, None, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n, k, 1, n, 1, k, 1, n, 1, 0, 0, 0, dt), "dW over W")
    assert capi.last_gemm_kernel() != "linear_backward_wavek"
    assert np.array_equal(got.numpy(), want[0].numpy()) and np.array_equal(d_w.numpy(), want[1].numpy())


@pytest.mark.parametrize("dt,m,k,n", [(F32, 1040, 160, 272), (F32, 1536, 32, 512), (F32, 1537, 32, 512), (F32, 1280, 33, 130), (F32, 1281, 33, 130), (F32, 832, 160, 800), (F32, 272, 544, 624), (F32, 720, 256, 2100),
                                      (F64, 1536, 64, 72), (F64, 1280, 64, 75), (F64, 1281, 64, 75), (F64, 1540, 64, 72)])
def test_gradients_in_one_launch_of_more_rows_and_tiles(dt, m, k, n):
    """The bias gradient beside the others around the rows up to which it rides, and two to three rounds of 16 x 16 tiles beside another product: the bits of the three on their own."""
    rng = np.random.default_rng(m + k + n)
    L = capi.lib()
    x, w, dy = rand_storage(rng, (m, k), dt), rand_storage(rng, (k, n), dt), rand_storage(rng, (m, n), dt)
    d_x, d_w, d_dy = Dev(x, dt), Dev(w, dt), Dev(dy, dt)
    want, got = ([Dev.empty(s, dt) for s in ((m, k), (k, n), (n,))] for _ in range(2))
    capi.gemm(want[0].ptr, d_dy.ptr, d_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n), (0, k, 1), False, dt)
    capi.gemm(want[1].ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n, 1), False, dt)
    capi.check(L.rp_hip_reduce_rows(want[2].ptr, d_dy.ptr, m, n, 0, dt), "reduce_rows")
    capi.check(L.rp_hip_linear_backward(got[0].ptr, got[1].ptr, got[2].ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n, k, 1, n, 1, k, 1, n, 1, 0, 0, 0, dt), "linear_backward")
    assert capi.last_gemm_kernel() == "linear_backward_wavek"
    for g, t in zip(got, want):
        assert np.array_equal(g.numpy(), t.numpy())


@pytest.mark.parametrize("m,k,n", [(37, 50, 21), (256, 128, 10), (200, 240, 160)])
def test_gradients_of_small_layers_over_operands(m, k, n):
    """Small fp32 layers, whose gradients go out in one launch: a gradient over what another product reads gives what the calls
    one after the other give.  Small integers, so the bits do not depend on the kernels."""
    rng = np.random.default_rng(m + k + n)
    L = capi.lib()
    x, w, dy = (rng.integers(-2, 3, s).astype(np.float32) for s in ((m, k), (k, n), (m, n)))
    dx_, dw_, db_ = dy @ w.T, x.T @ dy, dy.sum(0)

    def call(over):
        d_x, d_w, d_dy = Dev(x, F32), Dev(w, F32), Dev(dy, F32)
        out = {"dx": Dev.empty((m, k), F32), "dw": Dev.empty((k, n), F32), "db": Dev.empty((n,), F32)}
        place = dict(out)
        for name, operand in over.items():
            place[name] = {"x": d_x, "w": d_w}[operand]
        capi.check(L.rp_hip_linear_backward(place["dx"].ptr, place["dw"].ptr, place["db"].ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n,
                                            k, 1, n, 1, k, 1, n, 1, 0, 0, 0, F32), str(over))
        return {name: d.numpy() for name, d in place.items()}

    got = call({"dw": "w"})
    assert np.array_equal(got["dx"], dx_) and np.array_equal(got["dw"], dw_) and np.array_equal(got["db"], db_)
    got = call({"dx": "x"})                             # (dX is stored before dW is computed from what then stands there)
    assert np.array_equal(got["dx"], dx_) and np.array_equal(got["dw"], (dx_.T.astype(np.float64) @ dy).astype(np.float32)) and np.array_equal(got["db"], db_)
    got = call({"db": "w"})
    assert np.array_equal(got["dx"], dx_) and np.array_equal(got["dw"], dw_) and np.array_equal(got["db"].reshape(-1)[:n], db_)


def test_batch_longer_than_a_grid_axis():
    """70 000 tiny matrices in one call (the batch index rides on a grid axis of at most 65 535 blocks), A shared by
    all of them through a zero batch stride."""
    rng = np.random.default_rng(41)
    Z, m, k, n = 70000, 4, 8, 4
    a = rand_storage(rng, (m, k), F32); b = rand_storage(rng, (Z, k, n), F32)
    da, db, dc = capi.DeviceBuffer.from_numpy(a), capi.DeviceBuffer.from_numpy(b), capi.DeviceBuffer(Z * m * n * 4)
    capi.gemm(dc.ptr, da.ptr, db.ptr, None, Z, m, k, n, (0, k, 1), (k * n, n, 1), (m * n, n, 1), False, F32)
    got = dc.to_numpy(np.float32, (Z, m, n))
    want = np.einsum("ik,zkj->zij", a.astype(np.float64), b.astype(np.float64))
    assert oracle.rel_err(got.astype(np.float64), want) <= 1e-6
    assert oracle.rel_err(got[69999].astype(np.float64), oracle.matmul(a, np.ascontiguousarray(b[69999]), F32).astype(np.float64)) <= tol(F32, k)


def test_more_tiles_than_workgroups_fit_a_launch():
    """2^23 tiles of 16 x 16, whose workgroups of 512 threads are more than a launch holds: fp64 with a row-major B of 24 columns (A's rows are one
    row, expanded; 1.3e10 bytes of C, of which a few rows are looked at)."""
    rng = np.random.default_rng(47)
    m, k, n = 1 << 26, 50, 24
    a, b = rng.integers(-3, 4, k).astype(np.float64), rng.integers(-3, 4, (k, n)).astype(np.float64)
    da, db, dc = capi.DeviceBuffer.from_numpy(a), capi.DeviceBuffer.from_numpy(b), capi.DeviceBuffer(m * n * 8)
    capi.gemm(dc.ptr, da.ptr, db.ptr, None, 1, m, k, n, (0, 0, 1), (0, n, 1), (0, n, 1), False, F64)
    got = np.empty((2, n))
    for row in (0, 12345678, m // 2 - 1, m - 2):
        capi.check(capi.lib().rp_hip_memcpy_d2h(got.ctypes.data, dc.at(row * n * 8), got.nbytes), "memcpy_d2h")
        assert np.array_equal(got, np.stack([a @ b] * 2))
    dc.free()


def test_rejects_bad_arguments():
    lib = capi.lib()
    d = capi.DeviceBuffer(64)
    assert lib.rp_hip_gemm_strided_batched(d.ptr, d.ptr, None, None, 1, 2, 2, 2, 0, 2, 1, 0, 2, 1, 0, 2, 1, 0, F32) == -1
    assert lib.rp_hip_gemm_strided_batched(d.ptr, d.ptr, d.ptr, None, 1, 0, 2, 2, 0, 2, 1, 0, 2, 1, 0, 2, 1, 0, F32) == -1
    assert lib.rp_hip_gemm_strided_batched(d.ptr, d.ptr, d.ptr, None, 1, 2, 2, 2, 0, 2, 1, 0, 2, 1, 0, 2, 1, 0, 7) == -1
    assert lib.matmul_kernel_device(d.ptr, d.ptr, d.ptr, 2, -1, 2, F32) == -1
    assert b"extent" in lib.rp_hip_last_error()


def test_small_fp32_outputs_take_one_launch():
    """fp32 outputs of fewer than 64 tiles of 64 x 64 with k <= 2048 (the layers of the configuration-2 MLP): every layout,
    ragged extents, batches, bias and accumulation, against the oracle and float64; repeatable bit for bit."""
    rng = np.random.default_rng(43)
    cases = [(256, 784, 256, "nn"), (256, 256, 784, "nt"), (784, 256, 256, "tn"), (256, 128, 10, "nn"), (1, 5, 1, "nn"), (33, 2048, 47, "tt"),
             (100, 17, 300, "nt"), (16, 16, 16, "nn"), (250, 1, 250, "tn")]
    for m, k, n, layout in cases:
        a, b = _operands(rng, m, k, n, F32, layout)
        assert capi.gemm_kernel_name(1, m, k, n, (a.strides[0] // 4, a.strides[1] // 4), (b.strides[0] // 4, b.strides[1] // 4), (n, 1), F32) == "tiny32_16x16"
        bias = rand_storage(rng, (n,), F32); c0 = rand_storage(rng, (m, n), F32)
        for kw in ({}, {"bias": bias}, {"bias": bias, "c_init": c0, "accumulate": True}):
            got = device_gemm(a, b, F32, **kw)
            _check(got, a, b, F32, k, **kw)
            assert np.array_equal(got, device_gemm(a, b, F32, **kw))
    # beyond the limits the tiled kernels take over
    assert capi.gemm_kernel_name(1, 256, 4096, 256, (4096, 1), (256, 1), (256, 1), F32) != "tiny32_16x16"
    assert capi.gemm_kernel_name(1, 512, 512, 512, (512, 1), (512, 1), (512, 1), F32) != "tiny32_16x16"
    # a small batch of small matrices on stride views
    a3 = rand_storage(rng, (5, 40, 24), F32); b3 = rand_storage(rng, (5, 24, 56), F32)
    assert capi.gemm_kernel_name(5, 40, 24, 56, (24, 1), (56, 1), (56, 1), F32) == "tiny32_16x16"
    got = device_gemm(a3, b3, F32)
    assert oracle.rel_err(got, oracle_gemm(a3, b3, F32)) <= tol(F32, 24)
    got_t = device_gemm(a3, np.ascontiguousarray(b3.transpose(0, 2, 1)).transpose(0, 2, 1), F32)
    assert oracle.rel_err(got_t, oracle_gemm(a3, b3, F32)) <= tol(F32, 24)



@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("m,k,n", [(17, 33, 19), (100, 131, 77), (35, 509, 18), (3, 257, 301)])
def test_small_fp32_outputs_of_rows_at_any_element(m, k, n, layout):
    """Rows of odd length that start at an odd element: whole vectors along k are loaded there.  Small integers, so the sums are exact."""
    rng = np.random.default_rng(44)

    def operand(rows, cols, transposed):
        shape = (cols, rows + 1) if transposed else (rows, cols + 1)
        x = rng.integers(-3, 4, shape).astype(np.float32)[:, 1:]
        return x.T if transposed else x

    a, b = operand(m, k, layout[0] == "t"), operand(k, n, layout[1] == "t")
    got = device_gemm(a, b, F32)
    assert capi.last_gemm_kernel() == "tiny32_16x16"
    assert np.array_equal(got, (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))


# fp32 and fp64 products whose waves share k: every tile, k of no whole piece (32 values in fp32, 16 in fp64), of fewer pieces than waves and of many
# rounds of them, last tiles that start early, batches
WAVEKW_SHAPES = [(F32, 1, 16, 513, 16, "mfma32_wavek"), (F32, 1, 5, 700, 333, "mfma32_wavek"), (F32, 1, 35, 2047, 18, "mfma32_wavek"), (F32, 1, 70, 545, 300, "mfma32_wavek"),
                 (F32, 1, 497, 577, 401, "mfma32_wavek"), (F32, 1, 63, 1024, 2113, "mfma32_wavek"), (F32, 1, 3, 1001, 1100, "mfma32_wavek"), (F32, 1, 900, 519, 901, "mfma32_64x64"),
                 (F32, 3, 67, 1027, 35, "mfma32_wavek"), (F32, 9, 131, 61, 260, "mfma32_64x64"), (F32, 1, 33, 3000, 1100, "mfma32_64x64"), (F64, 1, 16, 1, 16, "mfma64_wavek"),
                 (F64, 1, 17, 16, 19, "mfma64_wavek"), (F64, 1, 60, 131, 50, "mfma64_wavek"), (F64, 1, 20, 2001, 17, "mfma64_wavek"), (F64, 1, 390, 257, 401, "mfma64_64x64"), (F64, 5, 33, 130, 31, "mfma64_wavek"),
                 (F32, 253, 64, 512, 64, "mfma32_64x64"), (F32, 301, 20, 600, 24, "mfma32_64x64"), (F64, 130, 64, 70, 130, "mfma64_64x64")]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("dt,batch,m,k,n,kernel", WAVEKW_SHAPES)
def test_waves_that_share_k_in_fp32_and_fp64(dt, batch, m, k, n, kernel, layout):
    """The operands are slices, at an odd element, of NaN-filled arrays that end with their last element; small integers, so the bits are known."""
    rng = np.random.default_rng(m + k + n)
    es = capi.DTYPE_SIZE[dt]
    np_t = capi.NP_STORAGE[dt]

    def operand(rows, cols):
        flat = np.full(1 + batch * rows * (cols + 3) - 3, np.nan, np_t)
        vals = rng.integers(-2, 3, (batch, rows, cols)).astype(np_t)
        np.lib.stride_tricks.as_strided(flat[1:], (batch, rows, cols), (rows * (cols + 3) * es, (cols + 3) * es, es))[...] = vals
        return capi.DeviceBuffer.from_numpy(flat), vals, (rows * (cols + 3), cols + 3, 1)

    da, a, a_st = operand(m, k) if layout[0] == "n" else operand(k, m)
    db, b, b_st = operand(k, n) if layout[1] == "n" else operand(n, k)
    if layout[0] == "t":
        a, a_st = a.transpose(0, 2, 1), (a_st[0], a_st[2], a_st[1])
    if layout[1] == "t":
        b, b_st = b.transpose(0, 2, 1), (b_st[0], b_st[2], b_st[1])
    want = np.matmul(a.astype(np.float64), b.astype(np.float64))
    bias = rng.integers(-2, 3, n).astype(np_t)
    dbias = capi.DeviceBuffer.from_numpy(bias)
    pitch = n + 5
    c0 = rng.integers(-2, 3, (batch, m, pitch)).astype(np_t)
    for with_bias, accumulate in ((False, False), (True, True)):
        dc = capi.DeviceBuffer.from_numpy(c0)
        capi.gemm(dc.at(es), da.at(es), db.at(es), dbias.ptr if with_bias else None, batch, m, k, n, a_st, b_st, (m * pitch, pitch, 1), accumulate, dt)
        if not ((layout[0] == "t" and m < 16) or (layout[1] == "n" and n < 16)):       # a row of k shorter than a tile's edge: the kernels of before
            assert capi.last_gemm_kernel() == kernel
        expect = c0.reshape(-1).copy()
        inner = np.lib.stride_tricks.as_strided(expect[1:], (batch, m, n), (m * pitch * es, pitch * es, es))
        inner[...] = (inner if accumulate else 0) + want + (bias if with_bias else 0)
        assert np.array_equal(dc.to_numpy(np_t, (expect.size,)), expect)      # C, and nothing around it
        dc.free()


@pytest.mark.parametrize("dt,batch,m,k,n,tile", [(F32, 1, 16, 513, 16, "16x16"), (F32, 1, 70, 545, 300, "16x16"), (F32, 1, 497, 577, 401, "16x64"), (F32, 1, 900, 519, 901, "64x64"), (F32, 9, 131, 77, 260, "32x32"),
                                                 (F32, 253, 64, 512, 64, "64x64"), (F32, 1, 63, 1024, 2113, "16x64"), (F32, 1, 3, 1001, 1100, "few_rows"), (F32, 1, 33, 3000, 1500, "16x32"),
                                                 (F64, 1, 60, 131, 50, "16x16"), (F64, 1, 390, 257, 401, "32x32"), (F64, 130, 64, 70, 130, "32x32")])
def test_tiles_of_waves_that_share_k(dt, batch, m, k, n, tile):
    """Which of the tiles shapes like those above are on (A and B row-major, on 256 CUs)."""
    es = capi.DTYPE_SIZE[dt]
    da, db, dc = (capi.DeviceBuffer(batch * size * es) for size in (m * k, k * n, m * n))
    capi.gemm(dc.ptr, da.ptr, db.ptr, None, batch, m, k, n, (m * k, k, 1), (k * n, n, 1), (m * n, n, 1), False, dt)
    assert capi.last_gemm_launch() == f"mfma{8 * es}_wavek_{tile}"
    capi.synchronize()


@pytest.mark.parametrize("dt,m,k,n", [(F32, 935, 213, 862), (F32, 64, 1024, 1024), (F32, 600, 900, 50), (F64, 89, 287, 286), (F64, 500, 40, 600), (BF16, 119, 57, 245), (F16, 300, 305, 641), (F32, 37, 50, 21)])
def test_gradients_in_one_launch_with_pitches_and_over_operands(dt, m, k, n):
    """x, w, dx and dw with pitches of their own, dx and dw also transposed: the bits of the three on their own and nothing around them written; and gradients
    over what the launch still reads, which come one after the other."""
    rng = np.random.default_rng(m + k + n)
    L = capi.lib()
    dy = rand_storage(rng, (m, n), dt)
    x, w = rand_storage(rng, (m, k + 3), dt), rand_storage(rng, (k, n + 5), dt)
    d_dy, d_x, d_w = Dev(dy, dt), Dev(x, dt), Dev(w, dt)
    want_b, got_b = Dev.empty((n,), dt), Dev.empty((n,), dt)
    capi.check(L.rp_hip_reduce_rows(want_b.ptr, d_dy.ptr, m, n, 0, dt), "reduce_rows")
    for transposed in (False, True):
        shape_x, st_x = ((k, m + 2), (1, m + 2)) if transposed else ((m, k + 7), (k + 7, 1))
        shape_w, st_w = ((n, k + 1), (1, k + 1)) if transposed else ((k, n + 9), (n + 9, 1))
        init_x, init_w = rand_storage(rng, shape_x, dt), rand_storage(rng, shape_w, dt)
        want, got = [Dev(v, dt) for v in (init_x, init_w)], [Dev(v, dt) for v in (init_x, init_w)]
        capi.gemm(want[0].ptr, d_dy.ptr, d_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n + 5), (0,) + st_x, False, dt)
        capi.gemm(want[1].ptr, d_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k + 3), (0, n, 1), (0,) + st_w, False, dt)
        capi.check(L.rp_hip_linear_backward(got[0].ptr, got[1].ptr, got_b.ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n, k + 3, 1, n + 5, 1, *st_x, *st_w, 0, 0, 0, dt), "linear_backward")
        for g, t in zip(got + [got_b], want + [want_b]):
            assert np.array_equal(g.numpy(), t.numpy())
    # db over W: written after dX has read W; dX over X: dW is computed from what then stands there; dW over W, as deep as the pitches
    want = [Dev.empty((m, k), dt), Dev(rand_storage(rng, (k, n + 5), dt), dt)]
    xs, ws = np.ascontiguousarray(x[:, :k]), np.ascontiguousarray(w)
    for over in ("db", "dx", "dw"):
        d_x, d_w = Dev(xs, dt), Dev(ws, dt)
        place = {"dx": Dev.empty((m, k), dt), "dw": Dev(w, dt), "db": Dev.empty((n,), dt)}
        place[over] = d_x if over == "dx" else d_w
        capi.check(L.rp_hip_linear_backward(place["dx"].ptr, place["dw"].ptr, place["db"].ptr, d_dy.ptr, d_x.ptr, d_w.ptr, m, k, n, k, 1, n + 5, 1, k, 1, n + 5, 1, 0, 0, 0, dt), over)
        e_x, e_w = Dev(xs, dt), Dev(ws, dt)
        capi.gemm(want[0].ptr, d_dy.ptr, e_w.ptr, None, 1, m, n, k, (0, n, 1), (0, 1, n + 5), (0, k, 1), False, dt)
        capi.gemm(want[1].ptr, want[0].ptr if over == "dx" else e_x.ptr, d_dy.ptr, None, 1, k, m, n, (0, 1, k), (0, n, 1), (0, n + 5, 1), False, dt)
        assert np.array_equal(place["dx"].numpy(), want[0].numpy()), over
        assert np.array_equal(place["dw"].numpy()[:, :n], want[1].numpy()[:, :n]), over
        assert np.array_equal(place["db"].numpy().reshape(-1)[:n], want_b.numpy()), over


@pytest.mark.parametrize("batch,m,k,n,launched", [(3000, 64, 5, 64, "generic"), (3000, 33, 5, 65, "generic"), (1, 3001, 3, 2001, "generic"), (3000, 20, 5, 20, "generic"), (3000, 64, 17, 64, "generic"),
                                                  (3000, 64, 48, 64, "generic"), (100, 64, 5, 64, "mfma64_wavek_32x32"), (3000, 20, 17, 20, "mfma64_wavek_16x16"), (400, 64, 48, 64, "mfma64_wavek_32x32"),
                                                  (3000, 33, 33, 65, "mfma64_wavek_32x32"), (400, 64, 130, 64, "mfma64_wavek_32x32"), (1, 300, 17, 301, "mfma64_wavek_16x16")])
def test_overlapping_rows_in_fp64(batch, m, k, n, launched):
    """A's rows are windows that move on by one value (on 256 CUs: few slabs of k and many tiles on the generic kernel); small integers, so the bits are known."""
    rng = np.random.default_rng(m + k)
    a, b = rng.integers(-2, 3, (batch, k + m)).astype(np.float64), rng.integers(-2, 3, (batch, k, n)).astype(np.float64)
    da, db, dc = Dev(a, F64), Dev(b, F64), Dev.empty((batch, m, n), F64)
    capi.gemm(dc.ptr, da.ptr, db.ptr, None, batch, m, k, n, (k + m, 1, 1), (k * n, n, 1), (m * n, n, 1), False, F64)
    assert capi.last_gemm_launch() == launched
    windows = np.lib.stride_tricks.as_strided(a, (batch, m, k), (a.strides[0], 8, 8))
    assert np.array_equal(dc.numpy(), np.matmul(np.ascontiguousarray(windows), b))


def _sums_of_short_chains(a, b):
    """a @ b in float32 as the row-streaming kernel sums it: chains of 32 products with fused multiply-adds (a float64 step holds a product and
    its sum, rounded once), eight chains to a block of 256, blocks one after the other."""
    (m, k), n = a.shape, b.shape[1]
    chains = -(-k // 32)
    ap, bp = np.zeros((m, 32 * chains)), np.zeros((32 * chains, n))
    ap[:, :k], bp[:k] = a, b
    parts = np.zeros((chains, m, n), np.float32)
    for i in range(32):
        parts = (parts + ap[:, i::32].T[:, :, None] * bp[i::32][:, None, :]).astype(np.float32)
    total = np.zeros((m, n), np.float32)
    for c in range(0, chains, 8):
        block = parts[c].copy()
        for j in range(c + 1, min(c + 8, chains)):
            block += parts[j]
        total += block
    return total


@pytest.mark.parametrize("m,k,n", [(1, 168, 16384), (2, 1000, 1088), (3, 1024, 8192), (2, 797, 13688), (3, 896, 11964), (4, 641, 9584), (2, 424, 16640), (2, 1024, 24576), (8, 100, 12288), (1, 200, 49152)])
def test_few_rows_in_fp32_keep_short_chains(m, k, n):
    """Up to eight rows against a row-major B: whichever kernel takes them, the error against 64 bits is no larger than that of sums in chains of 32
    (1.05: two such measures over these many values differ by less than 2 %, and by 3 % more for the order within the MFMAs)."""
    rng = np.random.default_rng(m * k + n)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    got = device_gemm(a, b, F32).astype(np.float64)
    short = _sums_of_short_chains(a, b).astype(np.float64)
    assert np.linalg.norm(got - exact) <= 1.05 * np.linalg.norm(short - exact), (np.linalg.norm(got - exact) / np.linalg.norm(exact), np.linalg.norm(short - exact) / np.linalg.norm(exact))


# ---- fp32 products with a short reduction (k <= 64) and many tiles: the resident cross-tile kernel (every layout, ragged
# extents, k below a whole slab, bias, accumulation) and, for operands with unit stride along their free index, the
# kernel that multiplies straight out of registers
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("batch,m,k,n", [(8, 512, 64, 512), (9, 500, 64, 456), (33, 250, 44, 300), (16, 384, 36, 512), (40, 256, 20, 256)])
def test_fp32_short_reduction_batched(layout, batch, m, k, n):
    rng = np.random.default_rng(61)
    a = rand_storage(rng, (batch, m, k), F32) if layout[0] == "n" else rand_storage(rng, (batch, k, m), F32).transpose(0, 2, 1)
    b = rand_storage(rng, (batch, k, n), F32) if layout[1] == "n" else rand_storage(rng, (batch, n, k), F32).transpose(0, 2, 1)
    a_rc, b_rc = [s // 4 for s in a.strides[1:]], [s // 4 for s in b.strides[1:]]
    kernel = capi.gemm_kernel_name(batch, m, k, n, a_rc, b_rc, (n, 1), F32)
    if layout == "tn" and k > 32 and m % 4 == 0 and n % 4 == 0:
        assert kernel == "direct32_128x128"
    elif m % 4 == 0 and n % 4 == 0 and k % 4 == 0:
        assert kernel == "mfma32_128x128"
    got = device_gemm(a, b, F32)
    _check(got, a, b, F32, k)
    bias = rand_storage(rng, (n,), F32)
    c0 = rand_storage(rng, (batch, m, n), F32)
    got = device_gemm(a, b, F32, bias=bias, c_init=c0, accumulate=True)
    _check(got, a, b, F32, k, bias=bias, c_init=c0, accumulate=True)


# ---- fp32, k <= 64, both operands contiguous along k, at least one 128 x 128 tile per CU: the resident kernel whose
# fetching waves fill LDS directly and whose multiplying waves store the previous tile between the MFMAs
PIPE32_SHAPES = [(16, 512, 64, 512), (20, 500, 64, 456), (48, 250, 44, 300), (32, 384, 36, 512), (70, 256, 20, 256), (300, 130, 8, 129), (260, 128, 32, 128),
                   (1, 2048, 64, 2048), (3, 1100, 60, 1300)]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("batch,m,k,n", PIPE32_SHAPES)
def test_fp32_pipelined_kernel(batch, m, k, n, layout):
    rng = np.random.default_rng(63)
    # free-index-major operands need 16-byte aligned k rows: pad the storage, view the first m (n) entries
    mp, npad = (m + 3) // 4 * 4, (n + 3) // 4 * 4
    a = rand_storage(rng, (batch, m, k), F32) if layout[0] == "n" else rand_storage(rng, (batch, k, mp), F32)[:, :, :m].transpose(0, 2, 1)
    b = rand_storage(rng, (batch, k, npad), F32)[:, :, :n] if layout[1] == "n" else rand_storage(rng, (batch, n, k), F32).transpose(0, 2, 1)
    a_rc, b_rc = [x // 4 for x in a.strides[1:]], [x // 4 for x in b.strides[1:]]
    assert capi.gemm_kernel_name(batch, m, k, n, a_rc, b_rc, (n, 1), F32) == "pipe32_128x128"
    got = device_gemm(a, b, F32)
    _check(got, a, b, F32, k)
    assert capi.last_gemm_kernel() == "pipe32_128x128"
    # the bias per column is this kernel's too
    bias = rand_storage(rng, (n,), F32)
    got = device_gemm(a, b, F32, bias=bias)
    assert capi.last_gemm_kernel() == "pipe32_128x128"
    _check(got, a, b, F32, k, bias=bias)
    # an accumulated C is not (reading C back leaves the product bound by memory either way): the same call must still be
    # right through the kernel that takes over
    c0 = rand_storage(rng, (batch, m, n), F32)
    got = device_gemm(a, b, F32, bias=bias, c_init=c0, accumulate=True)
    assert capi.last_gemm_kernel() != "pipe32_128x128"
    _check(got, a, b, F32, k, bias=bias, c_init=c0, accumulate=True)


def test_fp32_pipelined_kernel_views_and_strided_output():
    """Rows that are slices of wider arrays (row pitch above k), a batch stride that skips entries, and C written through
    row / column strides of a transposed, padded output: nothing outside the addressed elements may change."""
    rng = np.random.default_rng(64)
    batch, m, k, n = 24, 384, 48, 512
    wide_a = rand_storage(rng, (2 * batch, m, 80), F32)
    wide_b = rand_storage(rng, (batch, n, 96), F32)
    a = wide_a[::2, :, 16:16 + k]                              # every other batch entry, columns 16..63 of 80
    b = wide_b[:, :, 32:32 + k].transpose(0, 2, 1)
    assert capi.gemm_kernel_name(batch, m, k, n, (80, 1), (1, 96), (n, 1), F32) == "pipe32_128x128"
    got = device_gemm(a, b, F32)
    _check(got, a, b, F32, k)
    # C[z] stored transposed inside a padded [n + 3, m + 5] plane
    pitch = m + 5
    plane = (n + 3) * pitch
    c0 = rand_storage(rng, (batch, n + 3, pitch), F32)
    da, db, dc = capi.DeviceBuffer.from_numpy(wide_a), capi.DeviceBuffer.from_numpy(wide_b), capi.DeviceBuffer.from_numpy(c0)
    capi.gemm(dc.ptr, da.at(16 * 4), db.at(32 * 4), None, batch, m, k, n, (2 * m * 80, 80, 1), (n * 96, 1, 96), (plane, 1, pitch), False, F32)
    capi.synchronize()
    out = dc.to_numpy(np.float32, (batch, n + 3, pitch))
    for d in (da, db, dc):
        d.free()
    assert np.array_equal(out[:, :n, :m], got.transpose(0, 2, 1))
    assert np.array_equal(out[:, n:, :], c0[:, n:, :]) and np.array_equal(out[:, :, m:], c0[:, :, m:])


# ---- the same for bf16 / fp16 (C row-major, n in whole eights): narrowing and stores between the MFMAs of the next tile
PIPE16_SHAPES = [(16, 512, 64, 512), (20, 500, 64, 456), (48, 250, 40, 296), (32, 384, 32, 512), (70, 256, 16, 256), (300, 130, 8, 136), (3, 1100, 56, 1304)]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("batch,m,k,n", PIPE16_SHAPES)
def test_16bit_pipelined_kernel(batch, m, k, n, dt, layout):
    rng = np.random.default_rng(65)
    mp = (m + 7) // 8 * 8                                   # m-major A needs 16-byte aligned k rows: pad the storage
    a = rand_storage(rng, (batch, m, k), dt) if layout[0] == "n" else rand_storage(rng, (batch, k, mp), dt)[:, :, :m].transpose(0, 2, 1)
    b = rand_storage(rng, (batch, k, n), dt) if layout[1] == "n" else rand_storage(rng, (batch, n, k), dt).transpose(0, 2, 1)
    es = a.itemsize
    a_rc, b_rc = [x // es for x in a.strides[1:]], [x // es for x in b.strides[1:]]
    if layout[0] == "n" or m % 8 == 0:
        assert capi.gemm_kernel_name(batch, m, k, n, a_rc, b_rc, (n, 1), dt) == "pipe16_128x128"
    got = device_gemm(a, b, dt)
    _check(got, a, b, dt, k)
    resident = layout[0] == "n" or m % 8 == 0
    bias = rand_storage(rng, (n,), dt)
    got = device_gemm(a, b, dt, bias=bias)                                     # the bias per column is this kernel's too
    if resident:
        assert capi.last_gemm_kernel() == "pipe16_128x128"
    _check(got, a, b, dt, k, bias=bias)
    c0 = rand_storage(rng, (batch, m, n), dt)
    got = device_gemm(a, b, dt, bias=bias, c_init=c0, accumulate=True)          # accumulation is not: through the one that takes over
    assert capi.last_gemm_kernel() != "pipe16_128x128"
    _check(got, a, b, dt, k, bias=bias, c_init=c0, accumulate=True)


def test_16bit_pipelined_kernel_free_index_major_bit_exact():
    """The lowered convolution's dcol = W^T.dy shape (both operands with unit stride along their free index), small
    integers: every sum is exact, so the product must equal the oracle's bits."""
    rng = np.random.default_rng(73)
    batch, m, k, n = 8, 576, 64, 3136
    for dt in HALF:
        w64 = rng.integers(-2, 3, (k, m)).astype(np.float64)            # shared by the batch (batch stride 0)
        dy64 = rng.integers(-2, 3, (batch, k, n)).astype(np.float64)
        w_st, dy_st = oracle.to_storage(w64, dt), oracle.to_storage(dy64, dt)
        dw, ddy, dc = capi.DeviceBuffer.from_numpy(w_st), capi.DeviceBuffer.from_numpy(dy_st), capi.DeviceBuffer(batch * m * n * 2)
        assert capi.gemm_kernel_name(batch, m, k, n, (1, m), (n, 1), (n, 1), dt) == "pipe16_128x128"
        capi.gemm(dc.ptr, dw.ptr, ddy.ptr, None, batch, m, k, n, (0, 1, m), (k * n, n, 1), (m * n, n, 1), False, dt)
        capi.synchronize()
        out = dc.to_numpy(capi.NP_STORAGE[dt], (batch, m, n))
        for d in (dw, ddy, dc):
            d.free()
        assert np.array_equal(out, oracle.to_storage(np.matmul(w64.T[None], dy64), dt)), dt


@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
def test_16bit_pipelined_kernel_bit_exact_and_padded_rows(dt):
    """Small integers (every sum exact, so any order gives the oracle's bits), operands that are slices of wider arrays,
    and C with a row pitch above n: nothing outside the addressed elements may change."""
    rng = np.random.default_rng(66)
    batch, m, k, n = 24, 384, 48, 504
    wide_a = oracle.to_storage(rng.integers(-3, 4, (2 * batch, m, 80)).astype(np.float64), dt)
    wide_b = oracle.to_storage(rng.integers(-3, 4, (batch, n, 96)).astype(np.float64), dt)
    a = wide_a[::2, :, 16:16 + k]
    b = wide_b[:, :, 32:32 + k].transpose(0, 2, 1)
    want = np.matmul(oracle.to_f64(np.ascontiguousarray(a), dt), oracle.to_f64(np.ascontiguousarray(b), dt))
    pitch = n + 16
    c0 = rand_storage(rng, (batch, m + 2, pitch), dt)
    da, db, dc = capi.DeviceBuffer.from_numpy(wide_a), capi.DeviceBuffer.from_numpy(wide_b), capi.DeviceBuffer.from_numpy(c0)
    assert capi.gemm_kernel_name(batch, m, k, n, (80, 1), (1, 96), (pitch, 1), dt) == "pipe16_128x128"
    capi.gemm(dc.ptr, da.at(16 * 2), db.at(32 * 2), None, batch, m, k, n, (2 * m * 80, 80, 1), (n * 96, 1, 96), ((m + 2) * pitch, pitch, 1), False, dt)
    capi.synchronize()
    out = dc.to_numpy(capi.NP_STORAGE[dt], (batch, m + 2, pitch))
    for d in (da, db, dc):
        d.free()
    assert np.array_equal(oracle.to_f64(out[:, :m, :n], dt), want)
    assert np.array_equal(out[:, m:, :], c0[:, m:, :]) and np.array_equal(out[:, :, n:], c0[:, :, n:])


# ---- bf16 / fp16 outputs of at most 64 columns with at least one 128-row tile per CU: the resident kernel that streams k
# slabs of A and B into LDS, every operand layout, ragged m, n below 64, k that ends inside a slab
PIPE16K_SHAPES = [(64, 512, 512, 64), (70, 504, 200, 40), (300, 136, 72, 64), (1, 32768, 96, 56), (130, 256, 64, 64), (33, 1000, 328, 8)]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("dt", HALF, ids=lambda d: NAMES[d])
@pytest.mark.parametrize("batch,m,k,n", PIPE16K_SHAPES)
def test_16bit_narrow_output_kernel(batch, m, k, n, dt, layout):
    rng = np.random.default_rng(67)
    a = rand_storage(rng, (batch, m, k), dt) if layout[0] == "n" else rand_storage(rng, (batch, k, m), dt).transpose(0, 2, 1)
    b = rand_storage(rng, (batch, k, n), dt) if layout[1] == "n" else rand_storage(rng, (batch, n, k), dt).transpose(0, 2, 1)
    es = a.itemsize
    a_rc, b_rc = [x // es for x in a.strides[1:]], [x // es for x in b.strides[1:]]
    assert capi.gemm_kernel_name(batch, m, k, n, a_rc, b_rc, (n, 1), dt) == "pipe16k_128x64"
    got = device_gemm(a, b, dt)
    _check(got, a, b, dt, k)
    # the bias per column and the accumulation into C (the gradient rule of ops/ops.c:6781-6788) are this kernel's too
    bias = rand_storage(rng, (n,), dt)
    c0 = rand_storage(rng, (batch, m, n), dt)
    for kw in ({"bias": bias}, {"c_init": c0, "accumulate": True}, {"bias": bias, "c_init": c0, "accumulate": True}):
        got = device_gemm(a, b, dt, **kw)
        assert capi.last_gemm_kernel() == "pipe16k_128x64", kw.keys()
        _check(got, a, b, dt, k, **kw)


@pytest.mark.parametrize("layout", LAYOUTS)
def test_16bit_narrow_output_kernel_bit_exact(layout):
    """Small integers: every partial sum is exact in fp32, so the product must equal the oracle's bits in any summation
    order; C rows with a pitch above n must keep what lies between them."""
    rng = np.random.default_rng(68)
    batch, m, k, n, dt = 40, 1024, 448, 48, BF16
    a64 = rng.integers(-2, 3, (batch, m, k) if layout[0] == "n" else (batch, k, m)).astype(np.float64)
    b64 = rng.integers(-2, 3, (batch, k, n) if layout[1] == "n" else (batch, n, k)).astype(np.float64)
    a_st, b_st = oracle.to_storage(a64, dt), oracle.to_storage(b64, dt)
    a = a_st if layout[0] == "n" else a_st.transpose(0, 2, 1)
    b = b_st if layout[1] == "n" else b_st.transpose(0, 2, 1)
    want = np.matmul(a64 if layout[0] == "n" else a64.transpose(0, 2, 1), b64 if layout[1] == "n" else b64.transpose(0, 2, 1))
    pitch = 64
    c0 = rand_storage(rng, (batch, m, pitch), dt)
    da, db, dc = capi.DeviceBuffer.from_numpy(a_st), capi.DeviceBuffer.from_numpy(b_st), capi.DeviceBuffer.from_numpy(c0)
    es = 2
    a_str = (m * k,) + tuple(x // es for x in a.strides[1:])
    b_str = (k * n,) + tuple(x // es for x in b.strides[1:])
    assert capi.gemm_kernel_name(batch, m, k, n, a_str[1:], b_str[1:], (pitch, 1), dt) == "pipe16k_128x64"
    capi.gemm(dc.ptr, da.ptr, db.ptr, None, batch, m, k, n, a_str, b_str, (m * pitch, pitch, 1), False, dt)
    capi.synchronize()
    out = dc.to_numpy(capi.NP_STORAGE[dt], (batch, m, pitch))
    for d in (da, db, dc):
        d.free()
    assert np.array_equal(oracle.to_f64(out[:, :, :n], dt), want)
    assert np.array_equal(out[:, :, n:], c0[:, :, n:])
    # with a bias and an accumulated C every rounding of the reference's three ops is visible (sums up to 1800 need more
    # than bf16's 8 bits): the oracle's bits, from this kernel and from the tiled one that a misaligned bias falls back to
    bias = oracle.to_storage(rng.integers(-40, 41, (n + 8,)).astype(np.float64), dt)
    cacc = oracle.to_storage(rng.integers(-300, 301, (batch, m, n)).astype(np.float64), dt)
    want_bits = oracle_gemm(a, b, dt, bias=bias[:n], c_init=cacc, accumulate=True)
    got = device_gemm(a, b, dt, bias=bias[:n], c_init=cacc, accumulate=True)
    assert capi.last_gemm_kernel() == "pipe16k_128x64"
    assert np.array_equal(got, want_bits)
    dbias_all = capi.DeviceBuffer.from_numpy(bias)
    da, db, dc = capi.DeviceBuffer.from_numpy(a_st), capi.DeviceBuffer.from_numpy(b_st), capi.DeviceBuffer.from_numpy(cacc)
    capi.gemm(dc.ptr, da.ptr, db.ptr, dbias_all.at(2), batch, m, k, n, a_str, b_str, (m * n, n, 1), True, dt)      # bias at a 2-byte offset
    capi.synchronize()
    assert capi.last_gemm_kernel() != "pipe16k_128x64"
    tiled = dc.to_numpy(capi.NP_STORAGE[dt], (batch, m, n))
    assert np.array_equal(tiled, oracle_gemm(a, b, dt, bias=bias[1:n + 1], c_init=cacc, accumulate=True))
    for d in (da, db, dc, dbias_all):
        d.free()


# ---- and its fp32 twin (any n up to 64, any C strides)
PIPE32K_SHAPES = [(64, 512, 512, 64), (70, 500, 200, 40), (300, 130, 72, 64), (1, 32768, 96, 50), (130, 256, 32, 64), (33, 1000, 324, 7)]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("batch,m,k,n", PIPE32K_SHAPES)
def test_fp32_narrow_output_kernel(batch, m, k, n, layout):
    rng = np.random.default_rng(69)
    # free-index-major operands need 16-byte aligned k rows: pad the storage, view the first m (n) entries
    mp, npad = (m + 3) // 4 * 4, (n + 3) // 4 * 4
    a = rand_storage(rng, (batch, m, k), F32) if layout[0] == "n" else rand_storage(rng, (batch, k, mp), F32)[:, :, :m].transpose(0, 2, 1)
    b = rand_storage(rng, (batch, k, npad), F32)[:, :, :n] if layout[1] == "n" else rand_storage(rng, (batch, n, k), F32).transpose(0, 2, 1)
    a_rc, b_rc = [x // 4 for x in a.strides[1:]], [x // 4 for x in b.strides[1:]]
    assert capi.gemm_kernel_name(batch, m, k, n, a_rc, b_rc, (n, 1), F32) == "pipe32k_128x64"
    got = device_gemm(a, b, F32)
    _check(got, a, b, F32, k)
    # the bias per column and the accumulation into C are this kernel's too
    bias = rand_storage(rng, (n,), F32)
    c0 = rand_storage(rng, (batch, m, n), F32)
    for kw in ({"bias": bias}, {"c_init": c0, "accumulate": True}, {"bias": bias, "c_init": c0, "accumulate": True}):
        got = device_gemm(a, b, F32, **kw)
        assert capi.last_gemm_kernel() == "pipe32k_128x64", kw.keys()
        _check(got, a, b, F32, k, **kw)


@pytest.mark.parametrize("layout", LAYOUTS)
def test_fp32_narrow_output_kernel_bit_exact_strided_c(layout):
    """Small integers (every partial sum exact: the oracle's bits in any order) into a transposed, padded C."""
    rng = np.random.default_rng(70)
    batch, m, k, n = 40, 1024, 448, 48
    a64 = rng.integers(-3, 4, (batch, m, k) if layout[0] == "n" else (batch, k, m)).astype(np.float32)
    b64 = rng.integers(-3, 4, (batch, k, n) if layout[1] == "n" else (batch, n, k)).astype(np.float32)
    a = a64 if layout[0] == "n" else a64.transpose(0, 2, 1)
    b = b64 if layout[1] == "n" else b64.transpose(0, 2, 1)
    want = np.matmul(a.astype(np.float64), b.astype(np.float64)).astype(np.float32)
    pitch = m + 3
    c0 = rand_storage(rng, (batch, n + 1, pitch), F32)
    da, db, dc = capi.DeviceBuffer.from_numpy(a64), capi.DeviceBuffer.from_numpy(b64), capi.DeviceBuffer.from_numpy(c0)
    a_str = (m * k,) + tuple(x // 4 for x in a.strides[1:])
    b_str = (k * n,) + tuple(x // 4 for x in b.strides[1:])
    assert capi.gemm_kernel_name(batch, m, k, n, a_str[1:], b_str[1:], (1, pitch), F32) == "pipe32k_128x64"
    capi.gemm(dc.ptr, da.ptr, db.ptr, None, batch, m, k, n, a_str, b_str, ((n + 1) * pitch, 1, pitch), False, F32)
    capi.synchronize()
    out = dc.to_numpy(np.float32, (batch, n + 1, pitch))
    for d in (da, db, dc):
        d.free()
    assert np.array_equal(out[:, :n, :m], want.transpose(0, 2, 1))
    assert np.array_equal(out[:, n:, :], c0[:, n:, :]) and np.array_equal(out[:, :, m:], c0[:, :, m:])
    # integers with a bias and an accumulated C: exact in fp32, so the oracle's bits
    bias = rng.integers(-40, 41, (n,)).astype(np.float32)
    cacc = rng.integers(-300, 301, (batch, m, n)).astype(np.float32)
    got = device_gemm(a, b, F32, bias=bias, c_init=cacc, accumulate=True)
    assert capi.last_gemm_kernel() == "pipe32k_128x64"
    assert np.array_equal(got, oracle_gemm(a, b, F32, bias=bias, c_init=cacc, accumulate=True))


def test_fp32_short_reduction_integers_bit_exact():
    """Small integers: every partial sum is exact, so the product must equal the oracle's bit for bit in any summation order."""
    rng = np.random.default_rng(62)
    batch, m, k, n = 16, 512, 64, 512
    for layout in LAYOUTS:
        a = rng.integers(-3, 4, (batch, m, k) if layout[0] == "n" else (batch, k, m)).astype(np.float32)
        b = rng.integers(-3, 4, (batch, k, n) if layout[1] == "n" else (batch, n, k)).astype(np.float32)
        a = a if layout[0] == "n" else a.transpose(0, 2, 1)
        b = b if layout[1] == "n" else b.transpose(0, 2, 1)
        got = device_gemm(a, b, F32)
        assert np.array_equal(got, np.matmul(a.astype(np.float64), b.astype(np.float64)).astype(np.float32)), layout


# fp32 tiles of 128 x 128 run on the bf16 matrix cores with every value split in three.  Shapes: whole tiles and slabs of 32;
# k one past and one short of a slab, free axes one past and one short of a tile, a batch.
SPLIT32_SHAPES = [(1, 1408, 96, 1536), (1, 1409, 97, 1535), (1, 1407, 95, 1537), (1, 1500, 69, 1500), (1, 1411, 1029, 1404), (2, 1024, 68, 1160)]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("batch,m,k,n", SPLIT32_SHAPES)
def test_split32_is_as_close_as_fp32_sums(batch, m, k, n, layout):
    """Against float64.  Every step of 16 k rounds the running sum once (2^-24 of it at most, of random sign), two more
    roundings join the small products and the bias; a plane of either operand left out would cost 2^-18 and more."""
    rng = np.random.default_rng(47)

    def operand(rows, cols, transposed):
        x = rng.normal(0, 1, (batch, rows, cols)).astype(np.float32)
        return (x, capi.DeviceBuffer.from_numpy(np.ascontiguousarray(x.transpose(0, 2, 1))), (rows * cols, 1, rows)) if transposed else (x, capi.DeviceBuffer.from_numpy(x), (rows * cols, cols, 1))

    a, da, a_st = operand(m, k, layout[0] == "t")
    b, db, b_st = operand(k, n, layout[1] == "t")
    bias, c0 = rng.normal(0, 1, n).astype(np.float32), rng.normal(0, 1, (batch, m, n)).astype(np.float32)
    exact = np.matmul(a.astype(np.float64), b.astype(np.float64))
    dbias = capi.DeviceBuffer.from_numpy(bias)
    for with_bias, accumulate in ((False, False), (True, True)):
        dc = capi.DeviceBuffer.from_numpy(c0)
        capi.gemm(dc.ptr, da.ptr, db.ptr, dbias.ptr if with_bias else None, batch, m, k, n, a_st, b_st, (m * n, n, 1), accumulate, F32)
        assert capi.last_gemm_kernel() == "mfma32_128x128"
        want = exact + (bias if with_bias else 0.0) + (c0 if accumulate else 0.0)
        got = dc.to_numpy(np.float32, (batch, m, n)).astype(np.float64)
        assert np.linalg.norm(got - want) <= 2.0 ** -24 * (np.sqrt(k / 16) + 4) * np.linalg.norm(want)
        dc.free()


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, np.finfo(np.float32).max, -np.finfo(np.float32).max, 2.0 ** -105, 2.0 ** -111, 2.0 ** -120])
@pytest.mark.parametrize("m,k,n", [(1408, 96, 1536), (1411, 99, 1405)])
def test_split32_values_that_do_not_split(m, k, n, value):
    """Infinities, NaN, magnitudes that round to bf16 infinity and magnitudes whose last bits bf16 cannot hold: a tile that meets
    one is computed with fp32 MFMAs.  One row of A is `value` times N(0, 1) where that is tiny (fp32 sums of k products then
    bound the row's error by itself), otherwise `value` stands in two places."""
    rng = np.random.default_rng(48)
    a, b = rng.normal(0, 1, (m, k)).astype(np.float32), rng.normal(0, 1, (k, n)).astype(np.float32)
    tiny = abs(value) < 1
    if tiny:
        a[5] = (rng.normal(0, 1, k) * value).astype(np.float32)
        b *= np.float32(2.0 ** 60)
    else:
        a[5, 7] = value
        b[k - 1, n - 2] = value
    dc, da, db = capi.DeviceBuffer(m * n * 4), capi.DeviceBuffer.from_numpy(a), capi.DeviceBuffer.from_numpy(b)
    capi.gemm(dc.ptr, da.ptr, db.ptr, None, 1, m, k, n, (0, k, 1), (0, n, 1), (0, n, 1), False, F32)
    assert capi.last_gemm_kernel() == "mfma32_128x128"
    got = dc.to_numpy(np.float32, (m, n))
    with np.errstate(all="ignore"):
        want = np.matmul(a.astype(np.float64), b.astype(np.float64))
        as32 = want.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(as32)) and np.array_equal(np.isinf(got), np.isinf(as32))
    there = np.isinf(as32)
    assert np.array_equal(got[there], as32[there])
    for rows in (slice(5, 6), slice(0, 5), slice(6, m)):
        w, g = want[rows], got[rows].astype(np.float64)
        keep = np.isfinite(as32[rows])
        keep[:, n - 2] &= tiny                             # (one huge value sets the scale of that column's errors)
        if not tiny and rows.start == 5:
            continue
        assert np.linalg.norm((g - w)[keep]) <= 2.0 ** -24 * (np.sqrt(k) + 4) * np.linalg.norm(w[keep])


def _split32_error(a, b, rows):
    """2-norm error of these rows of A.B against float64, in units of 2^-24 of the result, and the largest relative one of a value."""
    m, k = a.shape
    n = b.shape[1]
    dc, da, db = capi.DeviceBuffer(m * n * 4), capi.DeviceBuffer.from_numpy(a), capi.DeviceBuffer.from_numpy(b)
    capi.gemm(dc.ptr, da.ptr, db.ptr, None, 1, m, k, n, (0, k, 1), (0, n, 1), (0, n, 1), False, F32)
    assert capi.last_gemm_kernel() == "mfma32_128x128"
    got = dc.to_numpy(np.float32, (m, n))[rows].astype(np.float64)
    want = a[rows].astype(np.float64) @ b.astype(np.float64)
    return np.linalg.norm(got - want) / np.linalg.norm(want) * 2 ** 24, np.max(np.abs(got - want)[want != 0] / np.abs(want[want != 0])) * 2 ** 24


@pytest.mark.parametrize("exponent", [-115, -127, -130, -136, -140])
def test_split32_subnormal_operands(exponent):
    """A row of A around 2^exponent (subnormal below 2^-126, a bf16 zero below 2^-134) against values around 2^100."""
    rng = np.random.default_rng(49)
    m, k, n = 1408, 96, 1536
    a, b = rng.normal(0, 1, (m, k)).astype(np.float32), (rng.normal(0, 1, (k, n)) * 2.0 ** 100).astype(np.float32)
    a[5] = (rng.normal(0, 1, k) * 2.0 ** exponent).astype(np.float32)
    for rows in (slice(5, 6), slice(0, 5), slice(128, m)):
        assert _split32_error(a, b, rows)[0] <= np.sqrt(k) + 4


@pytest.mark.parametrize("k", [96, 2048])
def test_split32_at_the_ends_of_its_range(k):
    """Operands just above the limit of what splits (their last planes are bf16 subnormals) stay on the split path.  Results near
    the smallest normal number, whose small products would be subnormal, are fp32 sums; a single product is then rounded once."""
    rng = np.random.default_rng(50)
    m, n = 1408, 1536
    sign = rng.choice([-1.0, 1.0], (m, k))
    a, b = (sign * 2.0 ** rng.uniform(-110, -104, (m, k))).astype(np.float32), (rng.normal(0, 1, (k, n)) * 2.0 ** 60).astype(np.float32)
    assert np.min(np.abs(a)) >= 2.0 ** -110
    assert _split32_error(a, b, slice(0, m))[0] <= np.sqrt(k / 16) + 4
    for e in (-58, -60, -61):
        a, b = (rng.normal(0, 1, (m, k)) * 2.0 ** e).astype(np.float32), (rng.normal(0, 1, (k, n)) * 2.0 ** e).astype(np.float32)
        assert _split32_error(a, b, slice(0, m))[0] <= np.sqrt(k) + 4
    a = np.zeros((m, k), np.float32)
    a[np.arange(m), np.arange(m) % k] = rng.uniform(1, 2, m) * 2.0 ** -62.5
    b = (rng.uniform(1, 2, (k, n)) * 2.0 ** -62.5).astype(np.float32)
    assert _split32_error(a, b, slice(0, m))[1] <= 1 + 1e-6


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("m,k,n", [(1408, 288, 1536), (1411, 170, 1405), (1501, 69, 1499)])
def test_split32_tiles_that_change_over(m, k, n, layout):
    """From the first slab of k on that holds a value whose last bits bf16 cannot hold, a tile is multiplied with fp32 MFMAs: at the
    first, an inner and the last k, from either operand.  Integers otherwise, so every sum that is not zero has known bits; then an infinity as well."""
    rng = np.random.default_rng(54)
    a0, b0 = rng.integers(-4, 5, (m, k)).astype(np.float32), rng.integers(-4, 5, (k, n)).astype(np.float32)
    whole = a0.astype(np.float64) @ b0.astype(np.float64)
    dc = capi.DeviceBuffer(m * n * 4)

    def product(a, b):
        a_st, b_st = ((0, k, 1) if layout[0] == "n" else (0, 1, m)), ((0, n, 1) if layout[1] == "n" else (0, 1, k))
        da, db = capi.DeviceBuffer.from_numpy(np.ascontiguousarray(a if layout[0] == "n" else a.T)), capi.DeviceBuffer.from_numpy(np.ascontiguousarray(b if layout[1] == "n" else b.T))
        capi.gemm(dc.ptr, da.ptr, db.ptr, None, 1, m, k, n, a_st, b_st, (0, n, 1), False, F32)
        assert capi.last_gemm_kernel() == "mfma32_128x128"
        out = dc.to_numpy(np.float32, (m, n))
        da.free(); db.free()
        return out

    for at in sorted({0, min(33, k - 1), k // 2, k - 1}):
        a, b = a0.copy(), b0.copy()
        a[7, at], a[m - 1, at], b[at, 9], b[at, n - 1] = 1.2345 * 2.0 ** -115, 2.0 ** -140, -1.2345 * 2.0 ** -120, 1.2345 * 2.0 ** -130
        want = a.astype(np.float64) @ b.astype(np.float64)
        sure = np.abs(want) >= 1                               # (a tiny term beside an integer sum is rounded away)
        got = product(a, b)
        assert np.array_equal(got[sure], np.rint(want)[sure].astype(np.float32)) and np.all(np.abs(got[~sure]) < 1e-30)
        a[200, k - 1 - at // 2] = np.inf
        got = product(a, b)
        with np.errstate(invalid="ignore"):
            row = (a[200].astype(np.float64)[:, None] * b.astype(np.float64)).sum(0)
        assert np.array_equal(got[200], row.astype(np.float32), equal_nan=True)
        sure[200] = False
        assert np.array_equal(got[sure], np.rint(want)[sure].astype(np.float32))
    assert np.array_equal(product(a0, b0), whole.astype(np.float32))


def test_split32_single_products_and_repeated_values():
    """The three smallest of the nine partial products are left out: at most 2^-24 of a product (8 significant bits leave
    |m| <= 2^-8 |h|, |l| <= 2^-17 |h|), beside the sum's own rounding of 2^-24.  That shows where a row of A has one significant term,
    and, always to the same side, where the values repeat (1.0038986 is close to the worst one)."""
    rng = np.random.default_rng(51)
    m, k, n = 1408, 512, 1536
    a = np.zeros((m, k), np.float32)
    a[np.arange(m), np.arange(m) % k] = rng.normal(0, 1, m)
    b = rng.normal(0, 1, (k, n)).astype(np.float32)
    assert _split32_error(a, b, slice(0, m))[1] <= 2 + 1e-3
    a[a != 0], b[:] = 1.0038986, 1.0038986
    assert _split32_error(a, b, slice(0, m))[1] <= 2 + 1e-3
    a[:] = 1.0038986
    assert _split32_error(a, b, slice(0, m))[1] <= 2 + k / 16      # a rounding per 16 k, which may all go one way too


@pytest.mark.parametrize("dt", [BF16, F16], ids=lambda d: NAMES[d])
@pytest.mark.parametrize("layout,m,k,n",
                         [("nt", *s) for s in [(1, 640, 1), (16, 648, 16), (17, 1024, 33), (65, 1032, 129), (31, 4096, 5), (40, 4104, 47), (300, 1536, 300),
                                               (1024, 640, 250), (96, 2048, 2055), (100, 4096, 4088)]] +
                         [("nn", *s) for s in [(1, 640, 8), (17, 1024, 40), (65, 1032, 136), (300, 1536, 304), (33, 5000, 72), (64, 2048, 2048), (10, 1016, 64)]])
def test_waves_that_split_k(dt, layout, m, k, n):
    """Few tiles, deep k, B either way round: every tile size, ragged ends of m, n and k, one and several rounds of loads.
    Operands are small integers (sums below 2^24: exact in any order) between NaNs that must not be read into a sum."""
    rng = np.random.default_rng(m + k + n)
    a64, b64 = rng.integers(-2, 3, (m, k)).astype(np.float64), rng.integers(-2, 3, (k, n)).astype(np.float64)
    pad = 8
    bt = b64.T if layout == "nt" else b64
    arow, brow = np.full((m + 1, k + pad), np.nan), np.full((bt.shape[0] + 1, bt.shape[1] + pad), np.nan)
    arow[:m, :k] = a64
    brow[:bt.shape[0], :bt.shape[1]] = bt
    b_st = (0, 1, k + pad) if layout == "nt" else (0, n + pad, 1)
    bias, old = oracle.to_storage(rng.integers(-4, 5, (n,)).astype(np.float64), dt), oracle.to_storage(rng.integers(-4, 5, (m, n)).astype(np.float64), dt)
    da, db, dbias = (capi.DeviceBuffer.from_numpy(v) for v in (oracle.to_storage(arow, dt), oracle.to_storage(brow, dt), bias))
    for with_bias, accumulate, transposed in ((False, False, False), (True, True, False), (True, False, True)):
        c0 = np.ascontiguousarray(old.T) if transposed else old
        dc = capi.DeviceBuffer.from_numpy(c0)
        capi.gemm(dc.ptr, da.ptr, db.ptr, dbias.ptr if with_bias else None, 1, m, k, n, (0, k + pad, 1), b_st, (0, 1, m) if transposed else (0, n, 1), accumulate, dt)
        assert capi.last_gemm_kernel() == "mfma16_wavek"
        capi.synchronize()
        got = dc.to_numpy(capi.NP_STORAGE[dt], c0.shape)
        # one rounding per operation: product, then bias, then accumulation
        want = oracle.to_storage(a64 @ b64, dt)
        if with_bias:
            want = oracle.to_storage(oracle.to_f64(want, dt) + oracle.to_f64(bias, dt), dt)
        if accumulate:
            want = oracle.to_storage(oracle.to_f64(old, dt) + oracle.to_f64(want, dt), dt)
        assert np.array_equal(got.T if transposed else got, want), (with_bias, accumulate, transposed)
