"""The work this framework is used for, as timed cases: FP32 SGEMMs on device
memory through the extension table's sgemm_device, and whole session calls
through the v1 table (host write, execute, host read; out of core).

A device case is one xvram_amd_sgemm_v1 descriptor a program keeps and enqueues
on its current stream; its matrices are column-major with leading dimensions of
whole float4s, as the entry point asks, and the four N/T forms are those of
xvram_amd_ext.h. A linear layer's forward is T/N (m = outputs, n = batch, k =
inputs; the weight row-major outputs x inputs), its input gradient N/N (m =
inputs, k = outputs) and its weight gradient N/T (k = batch).
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch  # before the library is loaded: both then share one HIP runtime

import xvram_amd as xv
from xvram_amd import abi

MiB = 1 << 20


def _device(name, form, m, n, k, *, alpha=1.0, beta=0.0, bias="none", relu=False, pad=0,
            workspace_mib=0, data="uniform", calls=1, gram=False):
    return {"name": name, "kind": "device", "form": form, "m": m, "n": n, "k": k, "alpha": alpha,
            "beta": beta, "bias": bias, "relu": relu, "pad": pad, "workspace_mib": workspace_mib,
            "data": data, "calls": calls, "gram": gram}


def listed():
    return [
        # The smallest calls: an odd-sized product of a few hundred rows, where
        # the launches and the host's share decide.
        _device("tiny_nn", "NN", 100, 84, 260),
        # Config 1, the ordinary small square.
        _device("square_1024_nn", "NN", 1024, 1024, 1024),
        # Config 2: ragged in every dimension, a residual update (alpha 1.5,
        # beta 0.5) of a C that the program sets first.
        _device("ragged_3001x2047x4099_tn", "TN", 3001, 2047, 4099, alpha=1.5, beta=0.5),
        # Decode: one 16384-wide linear + bias + ReLU layer (config 5's) for a
        # batch of 4. Reads 1 GiB of weights for 2 GFLOP.
        _device("linear_batch4_tn", "TN", 16384, 4, 16384, bias="row", relu=True, data="linear"),
        # The config-5 chain's launch: batch 256, a program that keeps its workspace.
        _device("linear_batch256_tn", "TN", 4096, 256, 4096, bias="row", relu=True,
                workspace_mib=128, data="linear"),
        # Backward of a linear layer, with respect to its input, an odd batch.
        _device("input_gradient_nn", "NN", 4096, 300, 16384, data="linear"),
        # ... and to its weight, over two micro-batches of 256: the first call
        # writes the gradient, the second adds to it (beta 1).
        _device("weight_gradient_nt", "NT", 4096, 4096, 256, data="gradient", calls=2),
        # X^T X of 60000 samples with 500 features: both operands one buffer, a
        # small result and a very deep K.
        _device("gram_500x60000_tn", "TN", 500, 500, 60000, gram=True),
        # A large square that fits no tile and no whole round of the chip.
        _device("square_5000_tt", "TT", 5000, 5000, 5000),
        # Config 3: the large resident square.
        _device("square_8192_nt", "NT", 8192, 8192, 8192),
        # A small layer through a session, as a host program serves it: write
        # the activations, execute the plan (weights resident), read the result.
        {"name": "session_linear", "kind": "session", "m": 1000, "n": 33, "k": 784},
        # Out of core: operands of 1 GiB in pinned host memory under a third of
        # that in VRAM, executed and read back.
        {"name": "out_of_core_nt", "kind": "out_of_core", "m": 4096, "n": 4096, "k": 32768,
         "frame_mib": 32, "frames": 12},
    ]


def _log(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _size(rng, low, high):
    """Log-uniform; half of the sizes as they come (mostly odd), half rounded to whole tiles of 32."""
    v = _log(rng, low, high)
    return v if rng.random() < 0.5 else max(32, v // 32 * 32)


def draw(rng):
    what = rng.choice(["square", "square", "square", "box", "box", "linear", "linear", "decode",
                       "decode", "input_gradient", "weight_gradient", "gram", "session",
                       "out_of_core"])
    if what == "square":
        s = _size(rng, 64, 8192)
        c = _device("", rng.choice(["NN", "NT", "TN", "TT"]), s, s, s)
    elif what == "box":
        m, n, k = (_size(rng, 64, 8192) for _ in range(3))
        c = _device("", rng.choice(["NN", "NT", "TN", "TT"]), m, n, k,
                    alpha=rng.choice([1.0, 1.5, -0.75]), beta=rng.choice([0.0, 0.0, 0.5]),
                    bias=rng.choice(["none", "row", "col"]), relu=rng.random() < 0.3,
                    pad=rng.choice([0, 0, 4, 64]), workspace_mib=rng.choice([0, 128]))
    elif what in ("linear", "decode"):
        batch = _log(rng, 1, 32) if what == "decode" else _log(rng, 33, 1024)
        c = _device("", "TN", _size(rng, 1024, 16384), batch, _size(rng, 1024, 16384), bias="row",
                    relu=rng.random() < 0.5, data="linear", workspace_mib=rng.choice([0, 128]))
    elif what == "input_gradient":
        c = _device("", "NN", _size(rng, 1024, 16384), _log(rng, 16, 1024), _size(rng, 1024, 16384),
                    data="linear")
    elif what == "weight_gradient":
        c = _device("", "NT", _size(rng, 1024, 8192), _size(rng, 1024, 8192), _log(rng, 16, 1024),
                    data="gradient", calls=2)
    elif what == "gram":
        s = _size(rng, 64, 1024)
        c = _device("", "TN", s, s, _log(rng, 8192, 65536), gram=True)
    elif what == "session":
        c = {"kind": "session", "m": _log(rng, 64, 4096), "n": _log(rng, 1, 256),
             "k": _log(rng, 64, 4096)}
    else:
        c = {"kind": "out_of_core", "m": 4 * _log(rng, 256, 1024), "n": 4 * _log(rng, 256, 1024),
             "k": 4 * _log(rng, 2048, 8192), "frame_mib": 32, "frames": 12}
    c.pop("name", None)
    return c


# ---- inputs -----------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _fill(gen, rows, cols, ld, data, scale=1.0):
    """A column-major rows x cols matrix as a (cols, ld) tensor; padding rows zero."""
    t = torch.zeros((cols, ld), dtype=torch.float32, device="cuda")
    if data == "uniform":
        t[:, :rows].uniform_(-1.0, 1.0, generator=gen)
    else:
        t[:, :rows].normal_(0.0, scale, generator=gen)
    return t


def _up4(v):
    return (v + 3) // 4 * 4


def _operands(case, seed):
    """(a's, b's, c0, bias) of a device case; one a and b for each of its calls."""
    gen = _generator(seed)
    m, n, k, form = case["m"], case["n"], case["k"], case["form"]
    data = "uniform" if case["data"] == "uniform" else "normal"
    # A layer's weight is N(0, 1 / inputs); a gradient's operands are activations and deltas.
    wscale = 1.0 / math.sqrt(k) if case["data"] == "linear" else 1.0
    a_rows, a_cols = (m, k) if form[0] == "N" else (k, m)
    b_rows, b_cols = (k, n) if form[1] == "N" else (n, k)
    a, b = [], []
    for _ in range(case["calls"]):
        a.append(_fill(gen, a_rows, a_cols, _up4(a_rows) + case["pad"], data, wscale))
        b.append(a[-1] if case["gram"] else
                 _fill(gen, b_rows, b_cols, _up4(b_rows) + case["pad"], data))
    c0 = None
    if case["beta"] != 0.0:
        c0 = _fill(gen, m, n, _up4(m) + case["pad"], data)
    bias = None
    if case["bias"] != "none":
        bias = _fill(gen, m if case["bias"] == "row" else n, 1, _up4(max(m, n)), "normal", 0.1)
    return a, b, c0, bias


class _HostGemm:
    """A session with its allocations and plan; closed when the program drops it."""

    def __init__(self, case, seed):
        m, n, k = case["m"], case["n"], case["k"]
        a, b, bias = _host_operands(case, seed)
        resident = case["kind"] == "session"
        frame = (16 if resident else case["frame_mib"]) * MiB
        frames = 16 if resident else case["frames"]
        self.session = xv.Session(xv.load(), chunk_size_bytes=frame, cache_target_bytes=frames * frame,
                                  workspace_cap_bytes=0, device_headroom_bytes=0,
                                  max_transaction_ms=600000)
        s = self.session
        self.a, self.b, self.c = (s.allocation(v) for v in (a.nbytes, b.nbytes, 4 * m * n))
        self.a.write(a)
        if resident:
            self.activations = b
            self.bias = s.allocation(bias.nbytes)
            self.bias.write(bias)
            # Y^T = ReLU(W X^T + b): W row-major m x k, X row-major n x k.
            self.plan = xv.GemmPlan(s, xv.matrix(self.a, k, m, k), xv.matrix(self.b, k, n, k),
                                    xv.matrix(self.c, m, n, m), abi.OP_T, abi.OP_N,
                                    epilogue=xv.epilogue(self.bias, abi.BIAS_PER_ROW, relu=True))
        else:
            self.activations = None
            self.b.write(b)
            self.plan = xv.GemmPlan(s, xv.matrix(self.a, m, k, m), xv.matrix(self.b, n, k, n),
                                    xv.matrix(self.c, m, n, m), abi.OP_N, abi.OP_T)
        self.out = np.zeros((n, m), dtype=np.float32)

    def run(self):
        if self.activations is not None:
            self.b.write(self.activations)
        self.plan.execute()
        return self.c.read_into(self.out)

    def __del__(self):
        if getattr(self, "plan", None) is not None:
            self.plan.release()
        if getattr(self, "session", None) is not None:
            self.session.close()
            self.session.release()


def _host_operands(case, seed):
    gen = _generator(seed)
    m, n, k = case["m"], case["n"], case["k"]
    if case["kind"] == "session":
        a = _fill(gen, k, m, k, "normal", 1.0 / math.sqrt(k))
        b = _fill(gen, k, n, k, "normal")
        bias = _fill(gen, m, 1, m, "normal", 0.1)
        return a.cpu().numpy(), b.cpu().numpy(), bias.cpu().numpy()
    return (_fill(gen, m, k, m, "uniform").cpu().numpy(),
            _fill(gen, n, k, n, "uniform").cpu().numpy(), None)


def prepare(case, seed):
    if case["kind"] != "device":
        return _HostGemm(case, seed)
    a, b, c0, bias = _operands(case, seed)
    m, n = case["m"], case["n"]
    c = torch.zeros((n, _up4(m) + case["pad"]), dtype=torch.float32, device="cuda")
    workspace = None
    if case["workspace_mib"]:
        workspace = torch.empty(case["workspace_mib"] * MiB, dtype=torch.uint8, device="cuda")
    descs = []
    for i in range(case["calls"]):
        d = abi.sgemm_device_init()
        d.a, d.b, d.c = a[i].data_ptr(), b[i].data_ptr(), c.data_ptr()
        d.m, d.n, d.k = m, n, case["k"]
        d.lda, d.ldb, d.ldc = a[i].shape[1], b[i].shape[1], c.shape[1]
        d.operation_a = abi.OP_T if case["form"][0] == "T" else abi.OP_N
        d.operation_b = abi.OP_T if case["form"][1] == "T" else abi.OP_N
        d.alpha = case["alpha"]
        d.beta = case["beta"] if i == 0 else 1.0
        if bias is not None:
            d.bias = bias.data_ptr()
            d.bias_axis = abi.BIAS_PER_ROW if case["bias"] == "row" else abi.BIAS_PER_COLUMN
        d.activation = abi.ACTIVATION_RELU if case["relu"] else abi.ACTIVATION_NONE
        if workspace is not None:
            d.workspace, d.workspace_bytes = workspace.data_ptr(), workspace.numel()
        descs.append(d)
    return {"m": m, "c": c, "c0": c0, "descs": descs, "keep": (a, b, bias, workspace),
            "call": xv.load().ext.sgemm_device}


def run(state):
    if isinstance(state, _HostGemm):
        return state.run()
    if state["c0"] is not None:
        state["c"].copy_(state["c0"])
    stream = torch.cuda.current_stream().cuda_stream
    for d in state["descs"]:
        status = state["call"](ctypes.byref(d), stream)
        if status != abi.SUCCESS:
            raise xv.XvramError(status, "sgemm_device")
    return state["c"][:, :state["m"]]


def work(case):
    m, n, k = case["m"], case["n"], case["k"]
    if case["kind"] != "device":
        # Through host memory: what is written, multiplied and read back (the
        # session's weights stay on the device from one call to the next).
        return {"bytes": 4 * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    calls = case["calls"]
    operands = m * k if case["gram"] else m * k + n * k
    c_passes = 1 + (2 if case["beta"] != 0.0 else 0) + 2 * (calls - 1)
    bias = {"none": 0, "row": m, "col": n}[case["bias"]]
    return {"bytes": 4 * (calls * operands + c_passes * m * n + bias), "flops": 2 * calls * m * n * k}


def tolerance(case):
    """FP32 sums over K: rounding grows with the length of one accumulator's
    chain, about 2^-24 * sqrt(K) / 2 of the result for zero-mean products."""
    return {"rel": 1e-5 if case["k"] > 2048 else 2e-6, "max": 1e-4}


def exact(case, seed):
    if case["kind"] == "session":
        w, x, bias = (torch.from_numpy(v).cuda().double() for v in _host_operands(case, seed))
        return torch.relu(x @ w.t() + bias)
    if case["kind"] == "out_of_core":
        a, b, _ = _host_operands(case, seed)
        return torch.from_numpy(b).cuda().double().t() @ torch.from_numpy(a).cuda().double()
    a, b, c0, bias = _operands(case, seed)
    m, n, k = case["m"], case["n"], case["k"]
    out = torch.zeros((n, m), dtype=torch.float64, device="cuda")
    for x, y in zip(a, b):
        xt = x[:, :m] if case["form"][0] == "N" else x[:, :k].t()  # (k, m)
        yt = y[:, :k] if case["form"][1] == "N" else y[:, :n].t()  # (n, k)
        out += yt.double() @ xt.double()
    out *= float(np.float32(case["alpha"]))
    if c0 is not None:
        out += float(np.float32(case["beta"])) * c0[:, :m].double()
    if bias is not None:
        v = bias.double().reshape(-1)
        out += v[:m].unsqueeze(0) if case["bias"] == "row" else v[:n].unsqueeze(1)
    return torch.relu(out) if case["relu"] else out
