"""Performance cases of the library: the calls a user's program makes, through the public entry points.

A case is a dict of plain values; `kind` names the entry point:

  dropin   BatchedPcForward.infer_get_top_batch, host arrays in and out
  settle   PcDeviceModel.relax_device (pcd_pc_relax) on device pointers
  ragged   PcDeviceModel.relax_ragged_device: packed requests, early exit
  classify PcDeviceModel.classify_device: every label clamped in turn
  adaptive PcDeviceModel.classify_adaptive_device under an effort preset
  learn    an epoch of PcDeviceModel.learn_device, then get_weights
  gemm     pcd_gemm_{f32,bf16,f16}, the provider's matrix product
  batched  pcd_gemm_{f32,bf16,f16}_batched

Networks are given as "784-256-256-10" (layer 0, the clamped input, first).
Weights are random at the scale of the initialisers the library is used with
(Xavier-normal for tanh and sigmoid, 1/fan_in for GELU), biases small and not
zero, as in a network that has been trained; 16-bit models get weights that
their operand type holds exactly.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from predicitivecoding_amd import BatchedPcForward, EffortLevel, EffortPresets, GenerativeSnapshot, PcDeviceModel
from predicitivecoding_amd._native import call

ACT = {"linear": 0, "tanh": 1, "relu": 2, "sigmoid": 3, "gelu": 4}
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
NBYTES = {"f32": 4, "bf16": 2, "f16": 2}


def _sizes(case):
    return [int(s) for s in case["net"].split("-")]


def _net(*sizes):
    return "-".join(str(s) for s in sizes)


# ------------------------------------------------------------------- the cases


def listed():
    return [
        # The published workload of the reference: one inference request from host arrays through the drop-in.
        {"name": "dropin_3072_f32", "kind": "dropin", "net": "3072-512-128-10", "act": "tanh", "dtype": "f32",
         "batch": 64, "steps": 20, "eta": 0.05, "input": "normal"},
        # The smallest benchmark network, inputs resident: 40 phases of a 64-row batch, bound by latency.
        {"name": "settle_784_f32", "kind": "settle", "net": "784-256-256-10", "act": "tanh", "dtype": "f32",
         "batch": 64, "steps": 20, "eta": 0.1, "input": "uniform", "energy": True, "states": True},
        # A middle-sized fp32 settling with its energy trace.
        {"name": "settle_1024_f32", "kind": "settle", "net": "1024-1024-1024-1024-256", "act": "tanh", "dtype": "f32",
         "batch": 1024, "steps": 50, "eta": 0.05, "input": "normal", "energy": True, "states": False},
        # The wide bf16 network: batch inference that reads the top latents alone.
        {"name": "settle_4096_bf16", "kind": "settle", "net": _net(*[4096] * 6), "act": "gelu", "dtype": "bf16",
         "batch": 4096, "steps": 32, "eta": 0.05, "input": "normal", "energy": False, "states": False},
        # The largest network one GPU runs in the benchmark, with its energy trace.
        {"name": "settle_8192_bf16", "kind": "settle", "net": _net(*[8192] * 12), "act": "gelu", "dtype": "bf16",
         "batch": 8192, "steps": 16, "eta": 0.02, "input": "normal", "energy": True, "states": False},
        # Continuous batching: 64 requests of 1 to 512 rows and 8 to 64 steps in one packed call.
        {"name": "ragged_2048_f32", "kind": "ragged", "net": _net(*[2048] * 4), "act": "tanh", "dtype": "f32",
         "requests": 64, "max_rows": 512, "min_steps": 8, "max_steps": 64, "rule": "absolute", "threshold": 1e-3,
         "eta": 0.1, "input": "normal", "mix": 4},
        # Classification of a test batch with the cheapest effort preset: B x C one-row requests that leave early.
        {"name": "adaptive_784_f32", "kind": "adaptive", "net": "784-256-256-10", "act": "tanh", "dtype": "f32",
         "batch": 200, "effort": "Low", "eta": 0.1, "input": "uniform"},
        # The trainer's loop on the small network: 16 minibatches of 64, then the weights exported.
        {"name": "learn_784_f32", "kind": "learn", "net": "784-256-256-10", "act": "tanh", "dtype": "f32",
         "batch": 64, "batches": 16, "steps": 20, "eta": 0.1, "eta_w": 2e-4, "decay": 1e-4, "input": "uniform"},
        # The same loop with large minibatches on the middle network.
        {"name": "learn_1024_f32", "kind": "learn", "net": "1024-1024-1024-1024-256", "act": "tanh", "dtype": "f32",
         "batch": 2048, "batches": 4, "steps": 20, "eta": 0.05, "eta_w": 1e-5, "decay": 1e-4, "input": "normal"},
        # Gemm.MatMul's own layout (both row-major) in fp32, with a row count that fills no whole tile.
        {"name": "gemm_1000_f32", "kind": "gemm", "dtype": "f32", "m": 1000, "k": 1024, "n": 4096,
         "trans_a": False, "trans_b": False, "beta": 0.0},
        # The same with 16-bit operands and a larger weight.
        {"name": "gemm_1000_bf16", "kind": "gemm", "dtype": "bf16", "m": 1000, "k": 4096, "n": 4096,
         "trans_a": False, "trans_b": False, "beta": 0.0},
        # Strided batches of small products (MatMulBatchedDevice), edges of no tile.
        {"name": "batched_96_f32", "kind": "batched", "dtype": "f32", "batch": 96, "m": 200, "k": 64, "n": 200},
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layout_size(rng, lo, hi):
    """A size over [lo, hi]: as drawn, or (half of the time) a multiple of 64 where the range reaches one."""
    v = _log(rng, lo, hi)
    return max(lo, v // 64 * 64) if v >= 64 and rng.random() < 0.5 else v


def draw(rng):
    kind = rng.choice(["dropin", "settle", "settle", "settle", "ragged", "classify", "adaptive", "learn", "gemm",
                       "gemm", "batched"])
    while True:
        case = _draw_kind(rng, kind)
        w = work(case)
        rate = 4e13 if case["dtype"] == "f32" else 4e14
        # far below the largest listed case's time, and quick to prepare and to compute in 64 bits
        if w["flops"] / rate < 0.15 and w["flops"] < 3e13 and w["bytes"] < 3e9:
            return case


def _draw_net(rng, lo, hi, depth):
    wide = _layout_size(rng, lo, hi)
    if rng.random() < 0.5:
        return _net(*[wide] * depth)
    return _net(*[_layout_size(rng, lo, max(lo, wide)) for _ in range(depth)])


def _draw_kind(rng, kind):
    dtype = rng.choice(["f32", "f32", "bf16", "f16"])
    act = rng.choice(["tanh", "tanh", "gelu", "sigmoid"])
    if kind == "dropin":
        net = _net(_layout_size(rng, 100, 3072), _layout_size(rng, 64, 512), _layout_size(rng, 32, 512),
                   rng.randint(2, 40))
        return {"kind": kind, "net": net, "act": "tanh", "dtype": rng.choice(["f32", "f16"]),
                "batch": _log(rng, 1, 300), "steps": rng.randint(5, 40), "eta": 0.05, "input": "normal"}
    if kind == "settle":
        return {"kind": kind, "net": _draw_net(rng, 48, 4096, rng.randint(3, 10)), "act": act, "dtype": dtype,
                "batch": _log(rng, 1, 4096), "steps": rng.randint(4, 40), "eta": 0.05, "input": "normal",
                "energy": rng.random() < 0.6, "states": rng.random() < 0.3}
    if kind == "ragged":
        lo = rng.randint(1, 12)
        return {"kind": kind, "net": _draw_net(rng, 64, 2048, rng.randint(3, 6)), "act": "tanh", "dtype": dtype,
                "requests": _log(rng, 2, 100), "max_rows": _log(rng, 1, 512), "min_steps": lo,
                "max_steps": rng.randint(lo + 1, 64), "rule": rng.choice(["none", "absolute"]), "threshold": 1e-3,
                "eta": 0.1, "input": "normal", "mix": rng.randrange(1 << 20)}
    if kind in ("classify", "adaptive"):
        net = _net(_layout_size(rng, 64, 1024), _layout_size(rng, 32, 512), _layout_size(rng, 32, 512),
                   rng.randint(2, 20))
        case = {"kind": kind, "net": net, "act": "tanh", "dtype": "f32" if kind == "adaptive" else dtype,
                "batch": _log(rng, 1, 500), "eta": 0.1, "input": "uniform"}
        case.update({"effort": "Low"} if kind == "adaptive" else {"steps": rng.randint(5, 30)})
        return case
    if kind == "learn":
        net = _net(_layout_size(rng, 64, 1024), _layout_size(rng, 32, 1024), _layout_size(rng, 32, 1024),
                   rng.randint(2, 256))
        batch = _log(rng, 1, 4096)
        return {"kind": kind, "net": net, "act": "tanh", "dtype": dtype, "batch": batch,
                "batches": rng.randint(2, 8), "steps": rng.randint(5, 30), "eta": 0.05, "eta_w": 0.02 / batch,
                "decay": 1e-4, "input": "normal"}
    if kind == "gemm":
        return {"kind": kind, "dtype": dtype, "m": _layout_size(rng, 1, 8192), "k": _layout_size(rng, 8, 8192),
                "n": _layout_size(rng, 8, 8192), "trans_a": rng.random() < 0.3, "trans_b": rng.random() < 0.5,
                "beta": 0.0}
    return {"kind": kind, "dtype": dtype, "batch": _log(rng, 2, 200), "m": _layout_size(rng, 8, 512),
            "k": _layout_size(rng, 8, 512), "n": _layout_size(rng, 8, 512)}


# --------------------------------------------------------------------- inputs


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) % (1 << 62))


def _weights(case, seed):
    """(W, b) of the case's network as fp32 tensors on the GPU: W_l [s_{l-1} x s_l], b_l [s_{l-1}]."""
    s, g = _sizes(case), _gen(seed, 1)
    W, b = [], []
    for l in range(1, len(s)):
        std = math.sqrt(1.0 / s[l]) if case["act"] == "gelu" else math.sqrt(2.0 / (s[l] + s[l - 1]))
        w = torch.randn((s[l - 1], s[l]), generator=g, device="cuda") * std
        W.append(w.to(TORCH[case["dtype"]]).float())
        b.append(0.05 * torch.randn((s[l - 1],), generator=g, device="cuda"))
    return W, b


def _inputs(case, seed, rows):
    shape, g = (rows, _sizes(case)[0]), _gen(seed, 2)
    if case["input"] == "uniform":
        return torch.rand(shape, generator=g, device="cuda")
    return torch.randn(shape, generator=g, device="cuda")


def _labels(case, seed, rows):
    c = _sizes(case)[-1]
    return torch.nn.functional.one_hot(torch.randint(c, (rows,), generator=_gen(seed, 3), device="cuda"), c).float()


def _requests(case):
    """(row offsets, step budgets) of a ragged case: rows log-uniform in [1, max_rows], budgets uniform."""
    rng = np.random.default_rng(case["mix"])
    rows = np.exp(rng.uniform(0.0, math.log(case["max_rows"]), case["requests"])) if case["max_rows"] > 1 else \
        np.ones(case["requests"])
    rows = np.clip(np.floor(rows), 1, case["max_rows"]).astype(np.int32)
    steps = rng.integers(case["min_steps"], case["max_steps"] + 1, case["requests"]).astype(np.int32)
    return np.concatenate([[0], np.cumsum(rows)]).astype(np.int32), steps


def _snapshot(case, seed):
    W, b = _weights(case, seed)
    return GenerativeSnapshot(_sizes(case), ACT[case["act"]], case["eta"], 0.0, False, [w.cpu().numpy() for w in W],
                              [v.cpu().numpy() for v in b])


def _operands(case, seed):
    g, n = _gen(seed, 4), case.get("batch")
    lead = () if n is None else (n,)
    a = (case["k"], case["m"]) if case.get("trans_a") else (case["m"], case["k"])
    b = (case["n"], case["k"]) if case.get("trans_b") else (case["k"], case["n"])
    A = torch.randn(lead + a, generator=g, device="cuda").to(TORCH[case["dtype"]])
    B = (torch.randn(lead + b, generator=g, device="cuda") / math.sqrt(case["k"])).to(TORCH[case["dtype"]])
    return A, B


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind in ("gemm", "batched"):
        st["A"], st["B"] = _operands(case, seed)
        lead = (case["batch"],) if kind == "batched" else ()
        st["C"] = torch.zeros(lead + (case["m"], case["n"]), device="cuda")
        return st
    snap, s = _snapshot(case, seed), _sizes(case)
    if kind == "dropin":
        st["snapshot"] = snap
        st["inputs"] = list(_inputs(case, seed, case["batch"]).cpu().numpy())
        return st
    st["model"] = PcDeviceModel(snap, case["dtype"])
    if kind == "ragged":
        st["offsets"], st["steps"] = _requests(case)
        rows = int(st["offsets"][-1])
    else:
        rows = case["batch"] * case.get("batches", 1)
    st["x"] = _inputs(case, seed, rows)
    if kind in ("settle", "ragged"):
        st["top"] = torch.zeros((rows, s[-1]), device="cuda")
    if kind == "settle":
        if case["states"]:
            st["states"] = torch.zeros(rows * sum(s), device="cuda")
        if case["energy"]:
            st["energy"] = torch.zeros((case["steps"], rows), device="cuda")
    if kind in ("classify", "adaptive"):
        st["class_energies"] = torch.zeros((rows, s[-1]), device="cuda")
        st["class"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
        st["energy"] = torch.zeros(rows, device="cuda")
        if kind == "adaptive":
            st["class_steps"] = torch.zeros((rows, s[-1]), dtype=torch.int32, device="cuda")
            st["steps_used"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
    if kind == "learn":
        st["labels"] = _labels(case, seed, rows)
        st["energy"] = torch.zeros(rows, device="cuda")
    return st


# ------------------------------------------------------------------- one pass


def _ptr(t):
    return None if t is None else t.data_ptr()


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "gemm":
        call("pcd_gemm_" + case["dtype"], _ptr(st["A"]), _ptr(st["B"]), _ptr(st["C"]), case["m"], case["k"],
             case["n"], int(case["trans_a"]), int(case["trans_b"]), case["beta"], None)
        return st["C"]
    if kind == "batched":
        call("pcd_gemm_" + case["dtype"] + "_batched", _ptr(st["A"]), _ptr(st["B"]), _ptr(st["C"]), case["batch"],
             case["m"], case["k"], case["n"], None)
        return st["C"]
    if kind == "dropin":
        return np.stack(BatchedPcForward.infer_get_top_batch(st["snapshot"], st["inputs"], case["steps"],
                                                             mixed=case["dtype"] == "f16"))
    model = st["model"]
    if kind == "settle":
        model.relax_device(_ptr(st["x"]), case["batch"], case["steps"], _ptr(st["top"]), _ptr(st.get("states")),
                           _ptr(st.get("energy")))
        return {k: st[k] for k in ("top", "states", "energy") if k in st}
    if kind == "ragged":
        used, energy = model.relax_ragged_device(_ptr(st["x"]), st["offsets"], st["steps"], _ptr(st["top"]),
                                                 case["rule"], case["threshold"])
        return {"top": st["top"], "used": used, "energy": energy}
    if kind == "classify":
        model.classify_device(_ptr(st["x"]), case["batch"], case["steps"], _ptr(st["class_energies"]),
                              _ptr(st["class"]), _ptr(st["energy"]))
        return {k: st[k] for k in ("class_energies", "class", "energy")}
    if kind == "adaptive":
        steps, epsilon = EffortPresets.for_level(EffortLevel[case["effort"]])
        model.classify_adaptive_device(_ptr(st["x"]), case["batch"], steps, epsilon, _ptr(st["class_energies"]),
                                       _ptr(st["class_steps"]), _ptr(st["class"]), _ptr(st["energy"]),
                                       _ptr(st["steps_used"]))
        return {k: st[k] for k in ("class_energies", "class_steps", "class", "energy", "steps_used")}
    n, s = case["batch"], _sizes(case)
    for i in range(case["batches"]):
        model.learn_device(st["x"].data_ptr() + 4 * i * n * s[0], st["labels"].data_ptr() + 4 * i * n * s[-1], n,
                           case["steps"], case["eta_w"], case["decay"], st["energy"].data_ptr() + 4 * i * n)
    W, b = model.get_weights()
    return {"W": W, "b": b, "energy": st["energy"]}


# ------------------------------------------------------------------------ work


def _macs(s, steps, clamped):
    """Multiply-adds per sample of a settling.  Free states start at zero, so at step t the states of the layers
    the input (or a clamped top) has not reached yet are the same for every sample, and so are their products:
    those are one row's work for the whole batch, and not counted here."""
    L = len(s)
    total = 0.0
    for t in range(steps):
        for l in range(1, L):
            mul = float(s[l]) * s[l - 1]
            above = clamped and L - 1 - l <= t        # M_l depends on the clamped top
            if l <= t or above:                       # pre_l = W_l M_l
                total += mul
            if clamped and l == L - 1:
                continue                              # a clamped top is not updated
            if l <= t + 1 or above:                   # G_l = W_l^T Delta_l
                total += mul
    return total


def work(case):
    kind, ob = case["kind"], NBYTES[case["dtype"]]
    if kind in ("gemm", "batched"):
        n = case.get("batch", 1)
        m, k, c = case["m"], case["k"], case["n"]
        return {"bytes": n * (m * k + k * c) * ob + n * m * c * 4, "flops": 2.0 * n * m * k * c}
    s = _sizes(case)
    weights = sum(s[l] * s[l - 1] for l in range(1, len(s)))
    biases = sum(s[:-1])
    if kind == "ragged":
        offs, steps = _requests(case)
        rows = int(offs[-1])
        flops = sum(2.0 * int(n) * _macs(s, int(t), False) for n, t in zip(np.diff(offs), steps))
        return {"bytes": weights * ob + biases * 4 + rows * (s[0] + s[-1]) * 4, "flops": flops}
    batch = case["batch"]
    if kind in ("classify", "adaptive"):
        # the adaptive form's exits depend on the data: the first step never exits, so two steps are certain
        steps = case["steps"] if kind == "classify" else 2
        return {"bytes": weights * ob + biases * 4 + batch * (s[0] + s[-1] + 2) * 4,
                "flops": 2.0 * batch * s[-1] * _macs(s, steps, True)}
    if kind == "learn":
        n = case["batches"]
        flops = 2.0 * batch * n * (_macs(s, case["steps"], True) + weights)
        # weights and biases are read and written by every minibatch's update, the inputs read once
        return {"bytes": n * (2 * weights * 4 + 2 * biases * 4 + batch * (s[0] + s[-1] + 1) * 4), "flops": flops}
    out = s[-1]
    out += case["steps"] if case.get("energy") else 0
    out += sum(s) if case.get("states") else 0
    return {"bytes": weights * ob + biases * 4 + batch * (s[0] + out) * 4,
            "flops": 2.0 * batch * _macs(s, case["steps"], False)}


# ------------------------------------------------------------------- tolerance


def tolerance(case):
    """About four times the distance from 64-bit results that was measured over these ranges (relative, then largest):
    fp32 settlings up to 4e-7 and 1.4e-6, bf16 operands 6e-4 and 3e-3, f16 operands 1e-4 and 4e-4.  A product's fp32
    sums of exact operands are up to 6e-7 away at K = 1024 and grow with K."""
    kind, dtype = case["kind"], case["dtype"]
    if kind in ("gemm", "batched"):
        return {"rel": 4e-6, "max": 2e-5}
    if kind == "adaptive":
        # A candidate whose energy falls by almost exactly epsilon may leave a step earlier or later; its energy then
        # differs by about epsilon (one such candidate seen in 60 drawn cases).
        return {"rel": 1e-4, "max": 5e-3, "differ": 5e-3}
    if dtype == "f32":
        return {"rel": 2e-6, "max": 1e-5, "differ": 2e-3}
    return {"rel": 2e-3, "max": 1e-2, "differ": 5e-3} if dtype == "bf16" else \
        {"rel": 5e-4, "max": 2e-3, "differ": 5e-3}


# -------------------------------------------------------------- 64-bit results


def _act64(name, x):
    if name == "tanh":
        y = torch.tanh(x)
        return y, 1 - y * y
    if name == "relu":
        return torch.clamp(x, min=0), (x > 0).double()
    if name == "sigmoid":
        y = torch.sigmoid(x)
        return y, y * (1 - y)
    if name == "gelu":   # the tanh form
        c, a = math.sqrt(2 / math.pi), 0.044715
        t = torch.tanh(c * (x + a * x ** 3))
        return 0.5 * x * (1 + t), 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * c * (1 + 3 * a * x * x)
    return x, torch.ones_like(x)


class _Settling64:
    """The relaxation in 64 bits, a step at a time; `runs` (a mask of rows) freezes the others."""

    def __init__(self, case, W, b, x, top=None):
        s = _sizes(case)
        self.act, self.eta, self.L = case["act"], case["eta"], len(s)
        self.W, self.b, self.clamped = W, b, top is not None
        self.M = [x.double()] + [torch.zeros((x.shape[0], n), dtype=torch.float64, device="cuda") for n in s[1:]]
        if top is not None:
            self.M[-1] = top.double()

    def step(self, runs=None):
        """One step of the rows that run; returns every row's energy before it moved."""
        E, self.D, energy = [], [], 0.0
        for l in range(1, self.L):
            y, dy = _act64(self.act, self.M[l] @ self.W[l - 1].T + self.b[l - 1])
            e = self.M[l - 1] - y
            energy = energy + 0.5 * (e * e).sum(1)
            E.append(e)
            self.D.append(dy.mul_(e))
        for l in range(1, self.L):
            if l == self.L - 1 and self.clamped:
                break
            g = self.D[l - 1] @ self.W[l - 1]
            if l < self.L - 1:
                g = g.sub_(E[l])
            g = g.mul_(self.eta)
            self.M[l] = self.M[l] + (g if runs is None else g * runs[:, None])
        return energy


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gemm", "batched"):
        A, B = _operands(case, seed)
        A = A.transpose(-1, -2).contiguous() if case.get("trans_a") else A
        B = B.transpose(-1, -2).contiguous() if case.get("trans_b") else B
        return A.double() @ B.double()
    s = _sizes(case)
    W, b = _weights(case, seed)
    W, b = [w.double() for w in W], [v.double() for v in b]
    if kind == "ragged":
        offs, budget = _requests(case)
        rows = int(offs[-1])
        req = torch.repeat_interleave(torch.arange(len(budget), device="cuda"),
                                      torch.from_numpy(np.diff(offs)).to("cuda", torch.int64))
        count = torch.bincount(req, minlength=len(budget)).double()
        done = torch.from_numpy(budget.astype(np.int64)).cuda()
        last = torch.zeros(len(budget), dtype=torch.float64, device="cuda")
        z = _Settling64(case, W, b, _inputs(case, seed, rows))
        for t in range(int(budget.max())):
            live = done > t
            # a request's rows move in the step after which it leaves too
            e = z.step(live[req].double())
            total = torch.zeros_like(last).index_add_(0, req, e)
            last = torch.where(live, total, last)
            if case["rule"] == "absolute":
                done = torch.where(live & (total / count < case["threshold"]), torch.full_like(done, t + 1), done)
        return {"top": z.M[-1], "used": None, "energy": last}
    if kind in ("classify", "adaptive"):
        n, c = case["batch"], s[-1]
        x = _inputs(case, seed, n).repeat_interleave(c, 0)
        z = _Settling64(case, W, b, x, torch.eye(c, device="cuda").repeat(n, 1))
        steps, eps = (case["steps"], 0.0) if kind == "classify" else EffortPresets.for_level(EffortLevel[case["effort"]])
        live = torch.ones(n * c, dtype=torch.bool, device="cuda")
        last = torch.zeros(n * c, dtype=torch.float64, device="cuda")
        for t in range(steps):
            e = z.step(live.double())
            leaves = live & (last - e < eps * torch.clamp(last, min=1e-12)) if t > 0 and eps > 0 else \
                torch.zeros_like(live)
            last = torch.where(live, e, last)
            live = live & ~leaves
        table = last.reshape(n, c)
        out = {"class_energies": table, "class": None, "energy": table.min(1).values}
        if kind == "adaptive":
            out.update({"class_steps": None, "steps_used": None})
        return out
    if kind == "learn":
        n = case["batch"]
        x, labels = _inputs(case, seed, n * case["batches"]), _labels(case, seed, n * case["batches"])
        energies, keep = [], 1.0 - case["eta_w"] * case["decay"]
        for i in range(case["batches"]):
            z = _Settling64(case, W, b, x[i * n:(i + 1) * n], labels[i * n:(i + 1) * n])
            for _ in range(case["steps"]):
                e = z.step()
            energies.append(e)
            for l in range(len(W)):
                W[l] = keep * (W[l] + case["eta_w"] * (z.D[l].T @ z.M[l + 1]))
                b[l] = b[l] + case["eta_w"] * z.D[l].sum(0)
        return {"W": W, "b": b, "energy": torch.cat(energies)}
    z = _Settling64(case, W, b, _inputs(case, seed, case["batch"]))
    trace = [z.step() for _ in range(case["steps"])]
    if kind == "dropin":
        return z.M[-1]
    out = {"top": z.M[-1]}
    if case["states"]:
        out["states"] = torch.cat([m.reshape(-1) for m in z.M])
    if case["energy"]:
        out["energy"] = torch.stack(trace)
    return out
