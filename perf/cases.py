"""What this framework's speed is measured on: whole programs, taken through the C ABI as a compiled caller takes them.

A program is written with the caller-side API (`autodiff`, `nn`), serialised once, and handed to the library in one of
the two ways that `include/adhip.h` offers:

* call: one `adhip_execute`, the counterpart of the reference's `Device::execute`: every payload goes up, the program
  runs, every kept tensor comes back.  This is how a training program (a loop inside the IR) is run.
* resident: the program was created and its payloads uploaded beforehand; a pass queues its runs and reads the kept
  tensors back.  This is how a model that serves, or a step that is repeated from the host, is run.

Kept tensors are returned as the library hands them over: views of host memory that the context owns.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

# the package's folder, in the tree that is the working folder
sys.path.insert(0, os.path.join(os.getcwd(), "autodiff-ir-rust_amd"))

from adhip import autodiff, ir as IR, nn, workloads  # noqa: E402
from adhip.core import concat, constant  # noqa: E402
from adhip.device import Device, load_library  # noqa: E402


def listed():
    return [
        # the smallest call there is: the README's two-layer perceptron, one training step per call (latency alone)
        {"name": "readme step", "kind": "readme"},
        # a small perceptron trained for a hundred steps in the IR's loop: every kernel is short, launches count
        {"name": "mlp small", "kind": "mlp", "batch": 64, "d0": 32, "d1": 64, "d2": 48, "d3": 8, "iters": 100},
        # the same at the sizes of a digit classifier, none of them a multiple of a tile
        {"name": "mlp ragged", "kind": "mlp", "batch": 1000, "d0": 784, "d1": 500, "d2": 300, "d3": 10, "iters": 40},
        # the benchmark's training configuration: batch 4096, 4096-4096-4096-1024, ten steps
        {"name": "mlp large", "kind": "mlp", "batch": 4096, "d0": 4096, "d1": 4096, "d2": 4096, "d3": 1024, "iters": 10},
        # an encoder layer trained at the size the tests use: a hundred short kernels per step
        {"name": "encoder training small", "kind": "encoder_train", "seq": 64, "d_model": 32, "heads": 4, "ff": 64, "iters": 20},
        # an encoder layer trained on a sequence and widths between the tiles
        {"name": "encoder training ragged", "kind": "encoder_train", "seq": 500, "d_model": 320, "heads": 5, "ff": 1000, "iters": 10},
        # the benchmark's encoder layer, forward and backward, all gradients returned
        {"name": "encoder gradients", "kind": "encoder_grad", "seq": 2048, "d_model": 1024, "heads": 8, "ff": 4096},
        # inference: the benchmark's multi-head attention, forward only
        {"name": "attention", "kind": "attention", "seq": 2048, "d_model": 1024, "heads": 8},
        # inference on a sequence that fits no tile, narrower heads
        {"name": "attention ragged", "kind": "attention", "seq": 1001, "d_model": 512, "heads": 8},
        # the benchmark's reductions: row sums of squares, column sums and their total over 16384 x 4096
        {"name": "reductions", "kind": "reductions", "rows": 16384, "cols": 4096},
        # the benchmark's element-wise function with broadcast, forward and backward, as descent steps on its operands
        {"name": "descent", "kind": "descent", "rows": 4096, "cols": 4096, "steps": 50},
        # permute, concat, slice, scale, then a data-dependent loop over row sums: the benchmark's manipulation program
        {"name": "gather and loop", "kind": "gather", "nb": 64, "n1": 512, "n2": 1024, "n3": 256, "lo": 128, "hi": 896},
    ]


def draw(rng):
    def size(lo, hi):
        """Between lo and hi, evenly over the logarithm; one in three rounded to a multiple of 16, the rest as they fall."""
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return max(16, n // 16 * 16) if n >= 16 and rng.random() < 0.34 else n

    kind = rng.choice(["mlp", "mlp", "encoder_train", "encoder_grad", "attention", "reductions", "descent", "gather"])
    if kind == "mlp":
        batch, dims = size(16, 4096), [size(8, 4096) for _ in range(3)] + [size(2, 1024)]
        per_step = 6.0 * batch * sum(a * b for a, b in zip(dims, dims[1:]))
        return {"kind": kind, "batch": batch, "d0": dims[0], "d1": dims[1], "d2": dims[2], "d3": dims[3],
                "iters": max(5, min(100, int(2e12 / per_step)))}
    if kind in ("encoder_train", "encoder_grad", "attention"):
        heads = rng.choice([1, 2, 4, 5, 8])
        c = {"kind": kind, "seq": size(32, 2048), "d_model": heads * 4 * max(2, size(32, 1024) // (4 * heads)), "heads": heads}
        if kind != "attention":
            c["ff"] = size(64, 4096)
        if kind == "encoder_train":
            c["iters"] = rng.randint(5, 20)
        return c
    if kind == "reductions":
        return {"kind": kind, "rows": size(64, 16384), "cols": size(64, 4096)}
    if kind == "descent":
        return {"kind": kind, "rows": size(64, 4096), "cols": size(64, 4096), "steps": rng.randint(20, 50)}
    n2 = size(32, 1024)
    lo = rng.randint(0, n2 // 4)
    return {"kind": kind, "nb": size(1, 64), "n1": size(32, 512), "n2": n2, "n3": size(16, 256), "lo": lo,
            "hi": rng.randint(n2 // 2, n2)}


# ---- the C ABI, as a compiled caller uses it ------------------------------------------------------------


class Context:
    """One context of the library (`adhip_create`), which a program keeps for its whole life."""

    def __init__(self):
        self.lib = load_library()
        self.h = ctypes.c_void_p()
        if self.lib.adhip_create(0, ctypes.byref(self.h)) != 0:
            raise RuntimeError("adhip_create failed")

    def check(self, rc):
        if rc != 0:
            raise RuntimeError(self.lib.adhip_last_error(self.h).decode())

    def tensor(self, name):
        """A kept tensor of the last read-back: the context's own host memory."""
        data, dims, ndim = ctypes.POINTER(ctypes.c_float)(), ctypes.POINTER(ctypes.c_uint64)(), ctypes.c_size_t()
        self.check(self.lib.adhip_get_tensor(self.h, name, ctypes.byref(data), ctypes.byref(dims), ctypes.byref(ndim)))
        return np.ctypeslib.as_array(data, tuple(dims[i] for i in range(ndim.value)))


_context = None


def context():
    global _context
    if _context is None:
        _context = Context()
    return _context


class Caller:
    """A serialised program with its keep list, and, if it is resident, its handle."""

    def __init__(self, workload, keep, runs=None):
        self.ctx = context()
        proc, _ = workload.finish()
        self.outputs = [(k, workload.outputs[k].id.encode()) for k in keep]
        self.blob, self.payloads = IR.serialize(proc)
        ids = sorted({i for _, i in self.outputs})
        self.ids, self.n_ids = (ctypes.c_char_p * len(ids))(*ids), len(ids)
        self.runs = runs
        self.program = ctypes.c_void_p()
        if runs is not None:
            lib = self.ctx.lib
            self.ctx.check(lib.adhip_program_create(self.ctx.h, self.blob, len(self.blob), self.ids, self.n_ids,
                                                    ctypes.byref(self.program)))
            self.ctx.check(lib.adhip_program_upload(self.program))

    def run(self):
        ctx, lib = self.ctx, self.ctx.lib
        if self.runs is None:
            ctx.check(lib.adhip_execute(ctx.h, self.blob, len(self.blob), self.ids, self.n_ids))
        else:
            for _ in range(self.runs):
                ctx.check(lib.adhip_program_enqueue(self.program))
            ctx.check(lib.adhip_program_readback(self.program))
        return {k: ctx.tensor(i) for k, i in self.outputs}

    def __del__(self):
        if self.program:
            self.ctx.lib.adhip_program_destroy(self.program)


# ---- programs that adhip.workloads does not hold in this form ------------------------------------------


def descent(rows, cols, seed, lr=0.01):
    """One descent step on the squares of y = sigmoid(a*b + c + bias) - 0.5*exp(a) + sin(b)*cos(c), taken on all four
    operands: forward, backward with the broadcast operand's column sums, four updates in place."""
    autodiff.set_device(Device())
    autodiff.eager_dep_opt()
    rng = np.random.default_rng(seed)

    def uniform(*dim):
        return autodiff.tensor(rng.random(dim, dtype=np.float32) * np.float32(2.0) - np.float32(1.0), list(dim))

    a, b, c, bias = uniform(rows, cols), uniform(rows, cols), uniform(rows, cols), uniform(cols)
    y = (a * b + c + bias).sigmoid() - 0.5 * a.exp() + b.sin() * c.cos()
    loss = (y * y).sum(0).sum(0)
    loss.forward()
    loss.backward()
    nn.SGD([a, b, c], lr).step()
    nn.SGD([bias], lr / rows).step()
    outs = {"loss": loss.val(), "a": a.val(), "b": b.val(), "c": c.val(), "bias": bias.val()}
    return workloads.Workload("descent", outs, {})


def gather(nb, n1, n2, n3, lo, hi, seed):
    """r = concat(p.permute(0,2,1), q, dim=2)[:, lo:hi, :] * w as rows; then r -= step * r.sum(1) until every row sum is
    below 1.  The step takes three tenths off a row's sum, so a dozen iterations are needed; the counter bounds them."""
    autodiff.set_device(Device())
    autodiff.eager_dep_opt()
    rng = np.random.default_rng(seed)

    def uniform(*dim):
        return autodiff.tensor(rng.random(dim, dtype=np.float32) * np.float32(2.0) - np.float32(1.0), list(dim))

    p, q, w = uniform(nb, n1, n2), uniform(nb, n2, n3), uniform(n1 + n3)
    rows, width = nb * (hi - lo), n1 + n3
    r = concat([p.permute([0, 2, 1]), q], 2).r(range(lo, hi), 1).view([rows, width]) * w
    i = constant(0.0, [1]).contigious()   # set by the program, so that a resident one can be run again
    not_done = 1.0 - r.sum(1).less_than(constant(1.0, [rows])).all()
    pred = not_done * i.less_than(constant(50.0, [1]))
    r.forward()
    state = {"r": r, "i": i}

    def body():
        rv = state["r"].val().to_node()
        state["r"] -= (0.3 / width) * rv.sum(1).unsqueeze(-1)
        state["i"] += 1.0

    autodiff.ir_while(pred, body)
    return workloads.Workload("gather", {"r": r.val(), "i": i.val()}, {})


# ---- the interface ---------------------------------------------------------------------------------------


def prepare(case, seed):
    k = case["kind"]
    dev = Device()   # builders only record the program; the library is driven below
    if k == "readme":
        wl = workloads.readme_mlp(dev, seed=seed)
        return Caller(wl, list(wl.outputs))
    if k == "mlp":
        wl = workloads.mlp_train(dev, case["batch"], (case["d0"], case["d1"], case["d2"], case["d3"]), case["iters"], seed=seed)
        return Caller(wl, list(wl.outputs))
    if k == "encoder_train":
        wl = workloads.encoder_train(dev, case["seq"], case["d_model"], case["heads"], case["ff"], case["iters"], seed=seed)
        return Caller(wl, list(wl.outputs))
    if k == "encoder_grad":
        wl = workloads.encoder_layer(dev, case["seq"], case["d_model"], case["heads"], case["ff"], seed=seed)
        return Caller(wl, list(wl.outputs), runs=1)
    if k == "attention":
        wl = workloads.attention_forward(dev, case["seq"], case["d_model"], case["heads"], seed=seed)
        return Caller(wl, ["y"], runs=1)
    if k == "reductions":
        wl = workloads.reductions(dev, case["rows"], case["cols"], seed=seed, backward=False)
        return Caller(wl, list(wl.outputs), runs=1)
    if k == "descent":
        wl = descent(case["rows"], case["cols"], seed)
        return Caller(wl, list(wl.outputs), runs=case["steps"])
    wl = gather(case["nb"], case["n1"], case["n2"], case["n3"], case["lo"], case["hi"], seed)
    return Caller(wl, list(wl.outputs), runs=1)


def run(state):
    return state.run()


def work(case):
    k, f = case["kind"], 4.0   # bytes of a float
    if k == "readme":
        return {"bytes": f * (2 * (15 + 6 + 2) + 10 + 4 + 33), "flops": 3 * 2.0 * 2 * (15 + 6)}
    if k == "mlp":
        d, b = [case["d0"], case["d1"], case["d2"], case["d3"]], case["batch"]
        w = sum(p * q for p, q in zip(d, d[1:]))
        return {"bytes": f * (2 * (w + sum(d[1:])) + 2 * b * d[0] + b * d[3]), "flops": 6.0 * b * w * case["iters"]}
    if k in ("encoder_train", "encoder_grad", "attention"):
        s, d, h = case["seq"], case["d_model"], case["heads"]
        w, products = 4 * d * d, 2.0 * s * d * 4 * d + 4.0 * s * s * d
        if k == "attention":
            return {"bytes": f * (w + 2 * s * d), "flops": products}
        w, products = w + 2 * d * case["ff"] + case["ff"] + 3 * d, products + 4.0 * s * d * case["ff"]
        if k == "encoder_train":
            return {"bytes": f * (2 * w + 2 * s * d), "flops": 3 * products * case["iters"]}
        return {"bytes": f * (2 * w + 4 * s * d), "flops": 3 * products}
    if k == "reductions":
        r, c = case["rows"], case["cols"]
        return {"bytes": f * (r * c + r + c), "flops": 3.0 * r * c}
    if k == "descent":
        n, c = case["rows"] * case["cols"], case["cols"]
        return {"bytes": case["steps"] * f * (6 * n + 2 * c), "flops": case["steps"] * 60.0 * n}
    n = case["nb"] * (case["hi"] - case["lo"]) * (case["n1"] + case["n3"])
    return {"bytes": f * 2 * n, "flops": 3.0 * n}


def tolerance(case):
    """About four times the distance from the same program in 64 bits, over the listed cases and a dozen drawn ones
    (largest relative error; largest single difference): perceptrons 1.3e-5, 3.6e-5 (the gradient of x, behind a hundred
    updates of narrow layers); encoder layers 1.1e-6, 7.8e-6, and more for the total of a gradient program, a sum of
    values of both signs; attention 9.6e-7, 5.6e-6; reductions 1.3e-7, 4.8e-7; descent 1.8e-7, 1.5e-6; gather 8.3e-8, 5.2e-7."""
    return {"readme": {"rel": 1e-6, "max": 1e-6},
            "mlp": {"rel": 5e-5, "max": 1.5e-4},
            "encoder_train": {"rel": 5e-6, "max": 3e-5},
            "encoder_grad": {"rel": 2e-5, "max": 3e-5},
            "attention": {"rel": 4e-6, "max": 2.5e-5},
            "reductions": {"rel": 1e-6, "max": 2e-6},
            "descent": {"rel": 1e-6, "max": 6e-6},
            "gather": {"rel": 4e-7, "max": 2e-6}}[case["kind"]]


# ---- what the outputs are in 64 bits ----------------------------------------------------------------------


def built(case, seed):
    """The program of a case that `adhip.workloads` builds; its `inputs` are the values that go in."""
    k, dev = case["kind"], Device()
    if k == "readme":
        return workloads.readme_mlp(dev, seed=seed)
    if k == "mlp":
        return workloads.mlp_train(dev, case["batch"], (case["d0"], case["d1"], case["d2"], case["d3"]), case["iters"], seed=seed)
    if k == "encoder_train":
        return workloads.encoder_train(dev, case["seq"], case["d_model"], case["heads"], case["ff"], case["iters"], seed=seed)
    if k == "encoder_grad":
        return workloads.encoder_layer(dev, case["seq"], case["d_model"], case["heads"], case["ff"], seed=seed)
    if k == "attention":
        return workloads.attention_forward(dev, case["seq"], case["d_model"], case["heads"], seed=seed)
    return workloads.reductions(dev, case["rows"], case["cols"], seed=seed, backward=False)


def attention_exact(t, x, heads, d_model):
    out = []
    for h in range(heads):
        q, k, v = x @ t["wq%d" % h], x @ t["wk%d" % h], x @ t["wv%d" % h]
        out.append(torch.softmax(q @ k.T / math.sqrt(float(d_model)), -1) @ v)
    return torch.cat(out, -1) @ t["wo"]


def encoder_exact(t, heads, d_model):
    def norm(v, scale):
        c = v - v.mean(-1, keepdim=True)
        return c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-9) * scale

    y = norm(t["x"] + attention_exact(t, t["x"], heads, d_model), t["ln1_scale"])
    return norm(y + (y @ t["w1"] + t["b1"]) @ t["w2"] + t["b2"], t["ln2_scale"])


def exact(case, seed):
    k = case["kind"]
    on = "cuda" if torch.cuda.is_available() else "cpu"
    f32 = lambda v: float(np.float32(v))   # a constant as the program holds it

    def wide(a, grad=False):
        return torch.tensor(a, dtype=torch.float64, device=on, requires_grad=grad)

    def host(outs):
        return {n: v.detach().cpu().numpy() for n, v in outs.items()}

    if k in ("descent", "gather"):
        rng = np.random.default_rng(seed)

        def uniform(*dim):
            return wide(rng.random(dim, dtype=np.float32) * np.float32(2.0) - np.float32(1.0))

        if k == "gather":
            nb, n1, n2, n3, lo, hi = (case[n] for n in ("nb", "n1", "n2", "n3", "lo", "hi"))
            p, q, w = uniform(nb, n1, n2), uniform(nb, n2, n3), uniform(n1 + n3)
            r = torch.cat([p.permute(0, 2, 1), q], 2)[:, lo:hi].reshape(nb * (hi - lo), n1 + n3) * w
            del p, q
            i, step = 0, f32(0.3 / (n1 + n3))
            while i < 50:
                s = r.sum(1, keepdim=True)
                if bool((s < 1.0).all()):
                    break
                r -= step * s
                i += 1
            return host({"r": r, "i": torch.tensor([float(i)])})
        a, b, c, bias = uniform(case["rows"], case["cols"]), uniform(case["rows"], case["cols"]), uniform(case["rows"], case["cols"]), uniform(case["cols"])
        lr, lr_bias = f32(0.01), f32(0.01 / case["rows"])
        for _ in range(case["steps"]):
            g = torch.sigmoid(a * b + c + bias)
            y = g - 0.5 * a.exp() + b.sin() * c.cos()
            loss, dy = (y * y).sum().reshape(1), 2.0 * y
            g = g * (1.0 - g) * dy
            da, db, dc = g * b - 0.5 * a.exp() * dy, g * a + b.cos() * c.cos() * dy, g - b.sin() * c.sin() * dy
            a -= lr * da
            b -= lr * db
            c -= lr * dc
            bias -= lr_bias * g.sum(0)
        return host({"loss": loss, "a": a, "b": b, "c": c, "bias": bias})
    given = built(case, seed).inputs
    if k == "reductions":
        x = wide(given["x"])
        return host({"s0": (x * x).sum(1), "s1": x.sum(0), "s2": (x * x).sum().reshape(1)})
    if k == "readme":
        t = {n: wide(v, True) for n, v in given.items()}
        y = torch.sigmoid(t["x"].reshape(2, 5) @ t["W1"]) @ t["W2"] + t["b2"]
        y.sum().backward()
        outs = {"y": y, "dW1": t["W1"].grad, "dW2": t["W2"].grad, "db2": t["b2"].grad, "dx": t["x"].grad.reshape(2, 5)}
        outs.update({n: t[n] - f32(0.1) * t[n].grad for n in ("W1", "W2", "b2")})
        return host(outs)
    if k == "attention":
        t = {n: wide(v) for n, v in given.items()}
        return host({"y": attention_exact(t, t["x"], case["heads"], case["d_model"])})
    ones = np.ones(case.get("d_model", 1), dtype=np.float32)
    if k == "encoder_grad":
        t = {n: wide(v, n != "r") for n, v in dict(given, ln1_scale=ones, ln2_scale=ones).items()}
        y = encoder_exact(t, case["heads"], case["d_model"])
        loss = (y * t["r"]).sum().reshape(1)
        loss.backward()
        return host(dict({"y": y, "L": loss}, **{"d" + n: v.grad for n, v in t.items() if n != "r"}))
    if k == "encoder_train":
        t = {n: wide(v, n not in ("x", "t")) for n, v in dict(given, ln1_scale=ones, ln2_scale=ones).items()}
        scale, lr = f32(1.0 / (case["seq"] * case["d_model"])), f32(0.05)
        forward = lambda: encoder_exact(t, case["heads"], case["d_model"])
    else:
        t = {n: wide(v, n != "t") for n, v in given.items()}
        scale, lr = f32(1.0 / (case["batch"] * case["d3"])), f32(0.01)

        def forward():
            h = torch.sigmoid(t["x"] @ t["W0"] + t["b0"])
            h = torch.sigmoid(h @ t["W1"] + t["b1"])
            return h @ t["W2"] + t["b2"]
    weights = [n for n in t if n not in ("x", "t")]
    for _ in range(case["iters"]):
        for v in t.values():
            v.grad = None
        loss = ((forward() - t["t"]) ** 2).sum() * scale
        loss.backward()
        with torch.no_grad():
            for n in weights:
                t[n] -= lr * t[n].grad
    outs = {"loss": loss.reshape(1)}
    if k == "mlp":
        outs["dx"] = t["x"].grad
    return host(dict(outs, **{n: t[n] for n in weights}))
