"""The work that users of this library have it do, as cases for timing and for comparing results.

A case is a dict of plain values with a "kind" (which path) and its sizes.  `listed()` holds the fixed ones, `draw(rng)`
makes others of the same ranges.  Everything but the drop-in case calls the C ABI through `recpulse_amd.capi` on torch
tensors (torch's current stream is the null stream, which is the library's default too, so work is stream-ordered).

Kinds and the ranges they stand for:

  linear            y = x.W (+ b), and with backward dx, dW, db in one call: every dense product of a training step.
                    16-bit, fp32 and fp64; widths that are multiples of 64 up to 8192, and sizes that come from data
                    (row counts, class counts, feature counts), which are arbitrary integers.
  decode            y = x.W for 1 to 32 rows against a large weight: one step of token-by-token inference.
  attention_ops     softmax(scale Q.K^T).V as separate operations on stride views, forward and backward, the scores and
                    probabilities in memory: what the operation-by-operation API of the reference runs.
  attention_fused   the same value and gradients without the score matrix in memory; any sequence lengths, forward
                    alone for inference (a single query row is decoding against a cache of keys).
  conv2d            stride-1 convolution with "same" padding, forward and all gradients.
  lstm              one step of an LSTM cell, forward and all gradients.
  mlp_train         forward, mean cross-entropy and backward of a ReLU network over its flat layers.
  mlp_infer         logits of a ReLU network through the drop-in `recpulse` modules, read back to the host.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

import recpulse_amd
from recpulse_amd import capi

DTYPES = {"bf16": (capi.BF16, torch.bfloat16), "f16": (capi.F16, torch.float16),
          "f32": (capi.F32, torch.float32), "f64": (capi.F64, torch.float64)}
# the MLP of the configurations: 784 -> 256 -> 128 -> 10, batch 256
MLP = {"batch": 256, "d0": 784, "d1": 256, "d2": 128, "classes": 10}


def listed():
    return [
        # a classifier answering requests: host latency, five launches and one small copy back
        {"name": "mlp_infer_784", "kind": "mlp_infer", **MLP},
        # a training step of the same network: a dozen launches of a few microseconds each
        {"name": "mlp_train_784", "kind": "mlp_train", **MLP},
        # a layer of a small model, forward and backward
        {"name": "linear_bf16_1024", "kind": "linear", "dtype": "bf16", "m": 1024, "k": 1024, "n": 1024, "bias": True, "backward": True},
        # a large dense layer, forward and backward: the headline product size
        {"name": "linear_bf16_8192", "kind": "linear", "dtype": "bf16", "m": 8192, "k": 8192, "n": 8192, "bias": True, "backward": True},
        # sizes that come from data: a ragged batch, an odd feature count, an odd class count
        {"name": "linear_f16_ragged", "kind": "linear", "dtype": "f16", "m": 1500, "k": 2049, "n": 3003, "bias": True, "backward": True},
        # single precision training and double precision (scientific) use, square as in the configurations
        {"name": "linear_f32_4096", "kind": "linear", "dtype": "f32", "m": 4096, "k": 4096, "n": 4096, "bias": True, "backward": True},
        {"name": "linear_f64_2048", "kind": "linear", "dtype": "f64", "m": 2048, "k": 2048, "n": 2048, "bias": False, "backward": True},
        # token-by-token inference of eight sequences against one large weight
        {"name": "decode_bf16_m8", "kind": "decode", "dtype": "bf16", "m": 8, "k": 8192, "n": 8192},
        # batch 16, 12 heads, 512 positions, head width 64: op by op, and fused
        {"name": "attention_ops_bf16", "kind": "attention_ops", "dtype": "bf16", "z": 192, "s": 512, "d": 64},
        {"name": "attention_fused_bf16", "kind": "attention_fused", "dtype": "bf16", "z": 192, "sq": 512, "sk": 512, "d": 64, "backward": True},
        # a residual network's 3 x 3 layer
        {"name": "conv2d_bf16_56", "kind": "conv2d", "dtype": "bf16", "batch": 64, "c_in": 64, "h": 56, "w": 56, "c_out": 64, "ksize": 3},
        # one step of a recurrent layer
        {"name": "lstm_bf16_1024", "kind": "lstm", "dtype": "bf16", "batch": 64, "input": 1024, "hidden": 1024},
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _log_multiple(rng, lo, hi, step):
    return max(1, _log_int(rng, lo, hi) // step) * step


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "decode", "attention_ops", "attention_fused", "attention_fused",
                       "conv2d", "lstm", "mlp_train", "mlp_infer"])
    if kind == "linear":
        dtype = rng.choice(["bf16", "bf16", "f16", "f16", "f32", "f64"])
        # multiply-adds of one product: bounded so that no drawn case costs more than the listed ones of its type
        if rng.random() < 0.5:       # model widths
            most = {"f32": 2 ** 35, "f64": 2 ** 32}.get(dtype, 2 ** 37)
            pick = lambda: _log_multiple(rng, 64, 8192, 64)  # noqa: E731
        else:                        # sizes that come from data
            most = {"f32": 2 ** 32, "f64": 2 ** 31}.get(dtype, 2 ** 33)
            pick = lambda: _log_int(rng, 33, 5000)  # noqa: E731
        m, k, n = pick(), pick(), pick()
        while m * k * n > most:
            m, k, n = pick(), pick(), pick()
        return {"kind": kind, "dtype": dtype, "m": m, "k": k, "n": n, "bias": rng.random() < 0.7, "backward": rng.random() < 0.7}
    if kind == "decode":
        size = (lambda: _log_multiple(rng, 1024, 8192, 64)) if rng.random() < 0.7 else (lambda: _log_int(rng, 1024, 8192))
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "m": _log_int(rng, 1, 32), "k": size(), "n": size()}
    if kind == "attention_ops":
        dtype = rng.choice(["bf16", "f16", "f32"])
        s = rng.choice([64, 128, 256, 512]) if rng.random() < 0.5 else _log_int(rng, 16, 512)
        return {"kind": kind, "dtype": dtype, "z": _log_int(rng, 1, 192 if dtype != "f32" else 96), "s": s, "d": rng.choice([32, 64, 128])}
    if kind == "attention_fused":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        backward = rng.random() < 0.6
        d = rng.choice([32, 64, 128])
        sk = _log_int(rng, 32, 4096)
        sq = sk if rng.random() < 0.6 else (_log_int(rng, 1, 4096))
        z = _log_int(rng, 1, 192)
        most = 2 ** 25 if dtype == "f32" else 2 ** 27        # scores over all heads
        while z * sq * sk > most:
            z = max(1, z // 2)
        return {"kind": kind, "dtype": dtype, "z": z, "sq": sq, "sk": sk, "d": d, "backward": backward}
    if kind == "conv2d":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        hw = rng.choice([7, 14, 28, 56]) if rng.random() < 0.6 else rng.randint(7, 56)
        c_in, c_out = 64 * rng.choice([1, 1, 2, 3, 4]), 64 * rng.choice([1, 1, 2, 3, 4])
        ksize = rng.choice([3, 3, 3, 5])
        batch = _log_int(rng, 1, 64)
        most = 2 ** 32 if dtype == "f32" else 2 ** 34
        while batch > 1 and batch * c_in * c_out * hw * hw * ksize * ksize > most:
            batch = max(1, batch // 2)
        return {"kind": kind, "dtype": dtype, "batch": batch, "c_in": c_in, "h": hw, "w": hw if rng.random() < 0.7 else rng.randint(7, 56), "c_out": c_out, "ksize": ksize}
    if kind == "lstm":
        hidden = _log_multiple(rng, 64, 1536, 8) if rng.random() < 0.7 else _log_int(rng, 64, 1536)
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "batch": _log_int(rng, 1, 256),
                "input": hidden if rng.random() < 0.6 else _log_int(rng, 64, 1536), "hidden": hidden}
    return {"kind": kind, "batch": _log_int(rng, 1, 1024), "d0": _log_int(rng, 64, 1024), "d1": _log_int(rng, 32, 1024),
            "d2": _log_int(rng, 16, 512), "classes": _log_int(rng, 2, 1000)}


# ---- inputs ------------------------------------------------------------------------------------------------------
class _Source:
    """Tensors on the GPU from one seed."""

    def __init__(self, seed, dtype):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.code, self.dtype = DTYPES[dtype]

    def normal(self, *shape, std=1.0):
        wide = torch.float64 if self.dtype == torch.float64 else torch.float32
        return torch.randn(shape, generator=self.gen, device="cuda", dtype=wide).mul_(std).to(self.dtype)

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda", dtype=torch.float32).to(self.dtype)

    def empty(self, *shape):
        return torch.empty(shape, device="cuda", dtype=self.dtype)


def prepare(case, seed):
    return {"linear": _prepare_linear, "decode": _prepare_linear, "attention_ops": _prepare_attention_ops,
            "attention_fused": _prepare_attention_fused, "conv2d": _prepare_conv2d, "lstm": _prepare_lstm,
            "mlp_train": _prepare_mlp_train, "mlp_infer": _prepare_mlp_infer}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


# ---- linear, decode ----------------------------------------------------------------------------------------------
def _prepare_linear(case, seed):
    src = _Source(seed, case["dtype"])
    m, k, n = case["m"], case["k"], case["n"]
    backward = case.get("backward", False)
    st = {"run": _run_linear, "m": m, "k": k, "n": n, "code": src.code, "x": src.normal(m, k), "w": src.normal(k, n, std=1 / math.sqrt(k)),
          "b": src.normal(n, std=0.1) if case.get("bias") else None, "y": src.empty(m, n), "backward": backward}
    if backward:
        st.update(dy=src.normal(m, n), dx=src.empty(m, k), dw=src.empty(k, n), db=src.empty(n) if case.get("bias") else None)
    return st


def _run_linear(st):
    m, k, n, b = st["m"], st["k"], st["n"], st["b"]
    capi.gemm(st["y"].data_ptr(), st["x"].data_ptr(), st["w"].data_ptr(), b.data_ptr() if b is not None else None,
              1, m, k, n, (0, k, 1), (0, n, 1), (0, n, 1), False, st["code"])
    if not st["backward"]:
        return st["y"]
    db = st["db"]
    capi.check(capi.lib().rp_hip_linear_backward(st["dx"].data_ptr(), st["dw"].data_ptr(), db.data_ptr() if db is not None else None,
                                                 st["dy"].data_ptr(), st["x"].data_ptr(), st["w"].data_ptr(), m, k, n,
                                                 k, 1, n, 1, k, 1, n, 1, 0, 0, 0, st["code"]), "rp_hip_linear_backward")
    return [st["y"], st["dx"], st["dw"]] + ([db] if db is not None else [])


# ---- attention ---------------------------------------------------------------------------------------------------
def _prepare_attention_ops(case, seed):
    src = _Source(seed, case["dtype"])
    z, s, d = case["z"], case["s"], case["d"]
    st = {"run": _run_attention_ops, "z": z, "s": s, "d": d, "code": src.code, "scale": (ctypes.c_float * 1)(1 / math.sqrt(d))}
    for name in ("q", "k", "v", "do"):
        st[name] = src.normal(z, s, d)
    for name in ("o", "dq", "dk", "dv"):
        st[name] = src.empty(z, s, d)
    for name in ("scores", "p", "dp", "ds"):
        st[name] = src.empty(z, s, s)
    return st


def _run_attention_ops(st):
    z, s, d, code, scale = st["z"], st["s"], st["d"], st["code"], st["scale"]
    L = capi.lib()
    p = {name: st[name].data_ptr() for name in ("q", "k", "v", "do", "o", "dq", "dk", "dv", "scores", "p", "dp", "ds")}
    sd, ss = s * d, s * s
    narrow, wide = (sd, d, 1), (ss, s, 1)            # [s, d] and [s, s] matrices of a head
    narrow_t, wide_t = (sd, 1, d), (ss, 1, s)        # their transposes as stride views
    capi.gemm(p["scores"], p["q"], p["k"], None, z, s, d, s, narrow, narrow_t, wide, False, code)
    capi.check(L.rp_hip_scaled_softmax(p["p"], p["scores"], scale, z * s, s, 1, code), "rp_hip_scaled_softmax")
    capi.gemm(p["o"], p["p"], p["v"], None, z, s, s, d, wide, narrow, narrow, False, code)
    capi.gemm(p["dp"], p["do"], p["v"], None, z, s, d, s, narrow, narrow_t, wide, False, code)
    capi.gemm(p["dv"], p["p"], p["do"], None, z, s, s, d, wide_t, narrow, narrow, False, code)
    capi.check(L.rp_hip_backwards_scaled_softmax(p["dp"], p["p"], p["ds"], scale, z * s, s, 1, code), "rp_hip_backwards_scaled_softmax")
    capi.gemm(p["dq"], p["ds"], p["k"], None, z, s, s, d, wide, narrow, narrow, False, code)
    capi.gemm(p["dk"], p["ds"], p["q"], None, z, s, s, d, wide_t, narrow, narrow, False, code)
    return [st["o"], st["dq"], st["dk"], st["dv"]]


def _prepare_attention_fused(case, seed):
    src = _Source(seed, case["dtype"])
    z, sq, sk, d = case["z"], case["sq"], case["sk"], case["d"]
    st = {"run": _run_attention_fused, "z": z, "sq": sq, "sk": sk, "d": d, "code": src.code, "backward": case["backward"],
          "q": src.normal(z, sq, d), "k": src.normal(z, sk, d), "v": src.normal(z, sk, d), "o": src.empty(z, sq, d), "lse": None}
    if case["backward"]:
        st.update(do=src.normal(z, sq, d), dq=src.empty(z, sq, d), dk=src.empty(z, sk, d), dv=src.empty(z, sk, d),
                  lse=torch.empty((z, sq), device="cuda", dtype=torch.float32))
    return st


def _run_attention_fused(st):
    z, sq, sk, d, code, L = st["z"], st["sq"], st["sk"], st["d"], st["code"], capi.lib()
    q, k, v, o, lse = (st[name].data_ptr() if st[name] is not None else None for name in ("q", "k", "v", "o", "lse"))
    scale = 1 / math.sqrt(d)
    capi.check(L.rp_hip_attention_forward(o, q, k, v, lse, z, sq, sk, d, sq * d, d, sk * d, d, sk * d, d, sq * d, d, scale, code),
               "rp_hip_attention_forward")
    if not st["backward"]:
        return st["o"]
    capi.check(L.rp_hip_attention_backward(st["dq"].data_ptr(), st["dk"].data_ptr(), st["dv"].data_ptr(), q, k, v, o, st["do"].data_ptr(), lse,
                                           z, sq, sk, d, sq * d, d, sk * d, d, sk * d, d, sq * d, d, sq * d, d, scale, code),
               "rp_hip_attention_backward")
    return [st["o"], st["dq"], st["dk"], st["dv"]]


# ---- conv2d ------------------------------------------------------------------------------------------------------
def _prepare_conv2d(case, seed):
    src = _Source(seed, case["dtype"])
    n, ci, h, w, co, ks = (case[name] for name in ("batch", "c_in", "h", "w", "c_out", "ksize"))
    return {"run": _run_conv2d, "n": n, "ci": ci, "h": h, "wd": w, "co": co, "ks": ks, "code": src.code,
            "x": src.normal(n, ci, h, w), "w": src.normal(co, ci, ks, ks, std=1 / math.sqrt(ci * ks * ks)), "b": src.normal(co, std=0.1),
            "dy": src.normal(n, co, h, w), "y": src.empty(n, co, h, w), "dx": src.empty(n, ci, h, w), "dw": src.empty(co, ci, ks, ks), "db": src.empty(co)}


def _run_conv2d(st):
    n, ci, h, w, co, ks, code, L = st["n"], st["ci"], st["h"], st["wd"], st["co"], st["ks"], st["code"], capi.lib()
    p = {name: st[name].data_ptr() for name in ("x", "w", "b", "dy", "y", "dx", "dw", "db")}
    capi.check(L.rp_hip_conv2d_same_forward(p["y"], p["x"], p["w"], p["b"], n, ci, h, w, co, ks, ks, code), "rp_hip_conv2d_same_forward")
    capi.check(L.rp_hip_conv2d_same_backward(p["dx"], p["dw"], p["dy"], p["x"], p["w"], n, ci, h, w, co, ks, ks, code), "rp_hip_conv2d_same_backward")
    capi.check(L.rp_hip_channel_sums(p["db"], p["dy"], n, co, h * w, 0, code), "rp_hip_channel_sums")
    return [st["y"], st["dx"], st["dw"], st["db"]]


# ---- lstm --------------------------------------------------------------------------------------------------------
def _prepare_lstm(case, seed):
    src = _Source(seed, case["dtype"])
    b, i, h = case["batch"], case["input"], case["hidden"]
    g = 4 * h
    return {"run": _run_lstm, "b": b, "i": i, "h": h, "code": src.code,
            "x": src.normal(b, i), "hp": src.normal(b, h, std=0.5), "cp": src.normal(b, h, std=0.5),
            "wi": src.normal(i, g, std=1 / math.sqrt(h)), "wh": src.normal(h, g, std=1 / math.sqrt(h)),
            "bi": src.normal(g, std=0.1), "bh": src.normal(g, std=0.1), "dhc": src.normal(b, 2 * h),
            "gates": src.empty(b, g), "act": src.empty(b, g), "hc": src.empty(b, 2 * h), "dg": src.empty(b, g), "dc": src.empty(b, h),
            "dx": src.empty(b, i), "dh": src.empty(b, h), "dwi": src.empty(i, g), "dwh": src.empty(h, g), "db": src.empty(g)}


def _run_lstm(st):
    b, i, h, code, L = st["b"], st["i"], st["h"], st["code"], capi.lib()
    g = 4 * h
    p = {name: st[name].data_ptr() for name in ("x", "hp", "cp", "wi", "wh", "bi", "bh", "dhc", "gates", "act", "hc", "dg", "dc", "dx", "dh", "dwi", "dwh", "db")}
    capi.gemm(p["gates"], p["x"], p["wi"], None, 1, b, i, g, (0, i, 1), (0, g, 1), (0, g, 1), False, code)
    capi.gemm(p["gates"], p["hp"], p["wh"], None, 1, b, h, g, (0, h, 1), (0, g, 1), (0, g, 1), True, code)
    capi.check(L.rp_hip_lstm_cell_forward(p["hc"], p["act"], p["gates"], p["bi"], p["bh"], p["cp"], h, b, h, code), "rp_hip_lstm_cell_forward")
    capi.check(L.rp_hip_lstm_cell_backward(p["dg"], p["dc"], p["dhc"], p["act"], p["hc"], p["cp"], h, b, h, code), "rp_hip_lstm_cell_backward")
    capi.gemm(p["dx"], p["dg"], p["wi"], None, 1, b, g, i, (0, g, 1), (0, 1, g), (0, i, 1), False, code)
    capi.gemm(p["dh"], p["dg"], p["wh"], None, 1, b, g, h, (0, g, 1), (0, 1, g), (0, h, 1), False, code)
    capi.gemm(p["dwi"], p["x"], p["dg"], None, 1, i, b, g, (0, 1, i), (0, g, 1), (0, g, 1), False, code)
    capi.gemm(p["dwh"], p["hp"], p["dg"], None, 1, h, b, g, (0, 1, h), (0, g, 1), (0, g, 1), False, code)
    capi.check(L.rp_hip_reduce_rows(p["db"], p["dg"], b, g, 0, code), "rp_hip_reduce_rows")      # both biases have this gradient
    return [st[name] for name in ("hc", "dx", "dh", "dc", "dwi", "dwh", "db")]


# ---- MLP ---------------------------------------------------------------------------------------------------------
def _prepare_mlp_train(case, seed):
    src = _Source(seed, "f32")
    dims, batch = [case["d0"], case["d1"], case["d2"], case["classes"]], case["batch"]
    st = {"run": _run_mlp_train, "dims": dims, "batch": batch, "x": src.uniform(batch, dims[0]), "loss": src.empty(1),
          "labels": torch.randint(0, dims[3], (batch,), generator=src.gen, device="cuda", dtype=torch.int32)}
    for i in range(3):
        st.update({"w%d" % i: src.normal(dims[i], dims[i + 1], std=math.sqrt(2 / dims[i])), "b%d" % i: src.normal(dims[i + 1], std=0.05),
                   "z%d" % i: src.empty(batch, dims[i + 1]), "h%d" % i: src.empty(batch, dims[i + 1]),
                   "gz%d" % i: src.empty(batch, dims[i + 1]), "gh%d" % i: src.empty(batch, dims[i]),
                   "dw%d" % i: src.empty(dims[i], dims[i + 1]), "db%d" % i: src.empty(dims[i + 1])})
    return st


def _run_mlp_train(st):
    dims, batch, L, code = st["dims"], st["batch"], capi.lib(), capi.F32
    ptr = lambda name: st[name].data_ptr()  # noqa: E731
    for i in range(3):
        k, n = dims[i], dims[i + 1]
        capi.gemm(ptr("z%d" % i), ptr("h%d" % (i - 1) if i else "x"), ptr("w%d" % i), ptr("b%d" % i), 1, batch, k, n, (0, k, 1), (0, n, 1), (0, n, 1), False, code)
        if i < 2:
            capi.check(L.relu_kernel_device(ptr("h%d" % i), ptr("z%d" % i), batch * n, code), "relu_kernel_device")
    capi.check(L.rp_hip_cross_entropy_mean(ptr("loss"), ptr("gz2"), ptr("z2"), ptr("labels"), batch, dims[3], 1.0, code), "rp_hip_cross_entropy_mean")
    for i in (2, 1, 0):
        k, n = dims[i], dims[i + 1]
        capi.check(L.rp_hip_linear_backward(ptr("gh%d" % i), ptr("dw%d" % i), ptr("db%d" % i), ptr("gz%d" % i), ptr("h%d" % (i - 1) if i else "x"), ptr("w%d" % i),
                                            batch, k, n, k, 1, n, 1, k, 1, n, 1, 0, 0, 0, code), "rp_hip_linear_backward")
        if i:
            capi.check(L.backwards_relu_device(ptr("gh%d" % i), ptr("z%d" % (i - 1)), ptr("gz%d" % (i - 1)), batch * k, code), "backwards_relu_device")
    return [st[name] for name in ("loss", "z2", "gh0", "dw0", "db0", "dw1", "db1", "dw2", "db2")]


def _dropin():
    """The drop-in modules (`recpulse`, `recpulse_cuda`), which live in the package's dropin folder."""
    path = os.path.join(os.path.dirname(os.path.abspath(recpulse_amd.__file__)), "dropin")
    if path not in sys.path:
        sys.path.insert(0, path)
    import recpulse.module
    import recpulse_cuda
    return recpulse_cuda, recpulse.module


def _prepare_mlp_infer(case, seed):
    rp, modules = _dropin()

    class Net(modules.Module):
        def __init__(self):
            super().__init__()
            self.fc1 = modules.Linear(case["d0"], case["d1"])
            self.fc2 = modules.Linear(case["d1"], case["d2"])
            self.fc3 = modules.Linear(case["d2"], case["classes"])

        def forward(self, x):
            return self.fc3(self.fc2(self.fc1(x).op_relu()).op_relu())

    rng = np.random.default_rng(seed)
    rp.manual_seed(seed)
    net = Net().to(device="cuda")
    x = rp.from_numpy(rng.uniform(0, 1, (case["batch"], case["d0"])).astype(np.float32)).to(device="cuda")
    return {"run": _run_mlp_infer, "net": net, "x": x}


def _run_mlp_infer(st):
    return st["net"](st["x"]).to_numpy()


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    e = {"bf16": 2, "f16": 2, "f32": 4, "f64": 8}[case.get("dtype", "f32")]
    if kind in ("linear", "decode"):
        m, k, n = case["m"], case["k"], case["n"]
        bias = n if case.get("bias") else 0
        once = m * k + k * n + m * n + bias
        if not case.get("backward"):
            return {"bytes": e * once, "flops": 2 * m * k * n}
        return {"bytes": e * (2 * once), "flops": 6 * m * k * n}         # x, w, b, dy in; y, dx, dw, db out
    if kind == "attention_ops":
        z, s, d = case["z"], case["s"], case["d"]
        # the operations are separate calls on tensors in memory: six products of two narrow (one narrow, one wide in)
        # matrices, the softmax (one in, one out) and its gradient (two in, one out)
        return {"bytes": e * z * (6 * (2 * s * d + s * s) + 5 * s * s), "flops": 12 * z * s * s * d}
    if kind == "attention_fused":
        z, sq, sk, d = case["z"], case["sq"], case["sk"], case["d"]
        forward = e * z * (2 * sq * d + 2 * sk * d)
        if not case["backward"]:
            return {"bytes": forward, "flops": 4 * z * sq * sk * d}
        return {"bytes": e * z * (4 * sq * d + 4 * sk * d), "flops": 14 * z * sq * sk * d}      # scores are computed again in the backward
    if kind == "conv2d":
        n, ci, h, w, co, ks = (case[name] for name in ("batch", "c_in", "h", "w", "c_out", "ksize"))
        return {"bytes": e * (2 * n * h * w * (ci + co) + 2 * co * ci * ks * ks + 2 * co), "flops": 6 * n * h * w * ci * co * ks * ks}
    if kind == "lstm":
        b, i, h = case["batch"], case["input"], case["hidden"]
        weights = 4 * h * (i + h)
        return {"bytes": e * (2 * weights + 12 * h + 2 * b * i + 8 * b * h), "flops": 6 * b * weights}
    b, d0, d1, d2, c = (case[name] for name in ("batch", "d0", "d1", "d2", "classes"))
    weights = d0 * d1 + d1 * d2 + d2 * c + d1 + d2 + c
    if kind == "mlp_infer":
        return {"bytes": 4 * (b * d0 + weights + b * c), "flops": 2 * b * weights}
    return {"bytes": 4 * (2 * b * d0 + 2 * weights + b * c), "flops": 6 * b * weights}


# Largest relative errors (2-norm) of the listed and sixty drawn cases against the same path in float64, times about four.
# One rounding of the output is 1.7e-3 in bf16 and 2.1e-4 in f16, two (product, then bias) 2.4e-3 and 3.0e-4; the chains
# that round every intermediate reach 5.3e-3 and 5.5e-4; fp32 sums 1.4e-6 (3.2e-6 through exp), fp64 sums 1.9e-15.
def tolerance(case):
    kind, dtype = case["kind"], case.get("dtype", "f32")
    if kind in ("attention_ops", "lstm"):
        return {"rel": {"bf16": 2e-2, "f16": 2.2e-3, "f32": 1.2e-5}[dtype]}
    if kind == "attention_fused":
        return {"rel": {"bf16": 1e-2, "f16": 1.2e-3, "f32": 1.2e-5}[dtype]}
    return {"rel": {"bf16": 1e-2, "f16": 1.2e-3, "f32": 6e-6, "f64": 8e-15}[dtype]}
