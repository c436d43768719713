"""What the framework is timed on: the calls its users make, through the
public entry points (the C ABI of tensor.h, autograd.h, tt_data.h and
tt_hip.h), over the sizes they are made with.

Kinds of case:

  gemm    one tt_k_gemm on device buffers, any transposition.
  matmul  an ag_matmul layer: forward, then both gradients.
  mlp     784 -> 512 -> 256 -> 10 and its like: a training step (softmax-CE,
          backward, optimizer) or the forward pass of a trained one.
  cnn     conv -> relu -> pool twice, flatten, classifier: a training step or
          the evaluation of a batch.
  conv    one ag_conv2d layer with bias: forward, then dX, dW and db.

Everything is fp32, the one type the framework computes in.
"""
import ctypes
import math

import numpy as np
import torch

import tinytorch_amd

#: CIFAR-10's usual normalisation, what its batches are read with
MEAN = np.array([0.4914, 0.4822, 0.4465], np.float32)
STD = np.array([0.2023, 0.1994, 0.2010], np.float32)
DATASET = 2000  # samples resident on the device in the cases that draw batches from them


# ---------------------------------------------------------------- the cases

def _gemm(name, M, N, K, ta=False, tb=False):
    return dict(name=name, kind="gemm", M=M, N=N, K=K, ta=ta, tb=tb)


def _mlp(name, B, d0, d1, d2, classes, train, opt):
    return dict(name=name, kind="mlp", B=B, d0=d0, d1=d1, d2=d2, classes=classes, train=train,
                opt=opt)


def _cnn(name, B, C, H, W, F1, F2, k, classes, train, opt, dataset):
    return dict(name=name, kind="cnn", B=B, C=C, H=H, W=W, F1=F1, F2=F2, k=k, classes=classes,
                train=train, opt=opt, dataset=dataset)


def _conv(name, N, C, H, W, F, kh, kw, stride, ph, pw):
    return dict(name=name, kind="conv", N=N, C=C, H=H, W=W, F=F, kh=kh, kw=kw, stride=stride,
                ph=ph, pw=pw)


def listed():
    return [
        # one sample through a trained MLP: the smallest call a serving
        # program makes, all latency and launches
        _mlp("mlp_eval_1", 1, 784, 512, 256, 10, False, "none"),
        # the benchmark's MLP training step
        _mlp("mlp_train_256", 256, 784, 512, 256, 10, True, "sgd"),
        # a wider MLP at a round decimal batch, with momentum as the MNIST
        # harness trains
        _mlp("mlp_train_1000_wide", 1000, 784, 2048, 1024, 10, True, "momentum"),
        # the benchmark's CNN training step on resident inputs
        _cnn("cnn_train_128", 128, 3, 32, 32, 32, 64, 3, 10, True, "sgd", False),
        # the last batch of an epoch (50,000 images in batches of 128 leave
        # 80), gathered from a resident dataset and stepped with Adam as the
        # CIFAR harness does
        _cnn("cnn_train_80_adam", 80, 3, 32, 32, 32, 64, 3, 10, True, "adam", True),
        # a test set read through the trained CNN, a thousand images a call
        _cnn("cnn_eval_1000", 1000, 3, 32, 32, 32, 64, 3, 10, False, "none", False),
        # a convolution layer of a larger network, forward and backward
        _conv("conv_56", 32, 64, 56, 56, 128, 3, 3, 1, 1, 1),
        # a strided layer with a larger kernel over odd sizes
        _conv("conv_odd_stride2", 50, 24, 45, 37, 40, 5, 5, 2, 2, 2),
        # the benchmark's secondary GEMMs
        _gemm("gemm_1024", 1024, 1024, 1024),
        _gemm("gemm_ragged", 1000, 1003, 997),
        _gemm("gemm_tall", 65536, 64, 4096),
        # a matmul and both its gradients at the headline size
        dict(name="matmul_4096", kind="matmul", M=4096, N=4096, K=4096),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm; odd ones too."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


MOST_FLOPS, MOST_BYTES = 4.0e11, 1.2e9  # no drawn case costs more than the largest listed ones


def draw(rng):
    while True:
        kind = rng.choice(["gemm", "matmul", "mlp", "mlp", "cnn", "cnn", "conv", "conv"])
        if kind == "gemm":
            c = _gemm("", _log(rng, 32, 65536), _log(rng, 10, 8192), _log(rng, 32, 8192),
                      rng.random() < 0.3, rng.random() < 0.3)
        elif kind == "matmul":
            c = dict(name="", kind="matmul", M=_log(rng, 32, 4096), N=_log(rng, 10, 4096),
                     K=_log(rng, 32, 4096))
        elif kind == "mlp":
            train = rng.random() < 0.7
            c = _mlp("", _log(rng, 1, 2048), rng.choice([784, 3072, _log(rng, 64, 3072)]),
                     _log(rng, 32, 2048), _log(rng, 16, 1024), rng.choice([10, 10, rng.randint(2, 100)]),
                     train, rng.choice(["sgd", "momentum"]) if train else "none")
        elif kind == "cnn":
            train, dataset = rng.random() < 0.7, rng.random() < 0.3
            C = rng.choice([1, 3])
            H = 32 if dataset else rng.choice([28, 32, rng.randint(16, 48)])
            c = _cnn("", _log(rng, 1, 512 if train else 1000), 3 if dataset else C, H, H,
                     rng.choice([16, 32, _log(rng, 8, 64)]), rng.choice([32, 64, _log(rng, 16, 128)]),
                     rng.choice([3, 3, 5]), 10, train,
                     rng.choice(["sgd", "adam"]) if train else "none", dataset)
        else:
            k = rng.choice([1, 3, 3, 5])
            c = _conv("", _log(rng, 1, 64), _log(rng, 1, 128), rng.randint(7, 64), rng.randint(7, 64),
                      _log(rng, 4, 256), k, k, rng.choice([1, 1, 2]), rng.randint(0, k // 2),
                      rng.randint(0, k // 2))
        w = work(c)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            del c["name"]
            return c


# ---------------------------------------------------------------- inputs

def _rng(seed, k):
    return np.random.default_rng([int(seed), k])


def _uniform(seed, k, shape, lo=-1.0, hi=1.0):
    u = _rng(seed, k).random(shape, dtype=np.float32)
    return u * np.float32(hi - lo) + np.float32(lo)


def _normal(seed, k, shape, scale=1.0):
    return _rng(seed, k).standard_normal(shape, dtype=np.float32) * np.float32(scale)


def _he(seed, k, shape, fan_in):
    return _normal(seed, k, shape, math.sqrt(2.0 / fan_in))


def _dense(seed, k, fan_in, fan_out):
    """He-normal weights with a small bias row."""
    w = np.empty((fan_in + 1, fan_out), np.float32)
    w[:fan_in] = _he(seed, k, (fan_in, fan_out), fan_in)
    w[fan_in] = _normal(seed, k + 50, (fan_out,), 0.05)
    return w


def _flat(case):
    return case["F2"] * (case["H"] // 4) * (case["W"] // 4)


def _arrays(case, seed):
    """The case's inputs on the host, by name; "params" in the order of the model."""
    kind = case["kind"]
    if kind == "matmul":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(a=_uniform(seed, 1, (M, K)), b=_uniform(seed, 2, (K, N)),
                    seed=_normal(seed, 3, (M, N)))
    if kind == "conv":
        N, C, H, W, F = (case[k] for k in "NCHWF")
        kh, kw = case["kh"], case["kw"]
        Ho, Wo = _conv_out(case)
        return dict(x=_normal(seed, 1, (N, C, H, W)), w=_he(seed, 2, (F, C, kh, kw), C * kh * kw),
                    b=_normal(seed, 3, (F,), 0.05), seed=_normal(seed, 4, (N, F, Ho, Wo)))
    B = case["B"]
    d = dict(labels=_rng(seed, 2).integers(0, case["classes"], B).astype(np.int32))
    if kind == "mlp":
        dims = [case["d0"], case["d1"], case["d2"], case["classes"]]
        d["x"] = _uniform(seed, 1, (B, dims[0]), 0.0, 1.0)
        d["params"] = [_dense(seed, 10 + i, dims[i], dims[i + 1]) for i in range(3)]
    else:
        C, H, W, F1, F2, k = (case[n] for n in ("C", "H", "W", "F1", "F2", "k"))
        d["params"] = [_he(seed, 10, (F1, C, k, k), C * k * k), _normal(seed, 11, (F1,), 0.05),
                       _he(seed, 12, (F2, F1, k, k), F1 * k * k), _normal(seed, 13, (F2,), 0.05),
                       _dense(seed, 14, _flat(case), case["classes"])]
        if case["dataset"]:
            d["samples"] = _rng(seed, 1).integers(0, 256, (DATASET, C, H, W), dtype=np.uint8)
            d["all_labels"] = _rng(seed, 3).integers(0, case["classes"], DATASET).astype(np.int32)
            d["idx"] = _rng(seed, 4).permutation(DATASET)[:_spare(case)].astype(np.int64)
        else:
            d["x"] = _uniform(seed, 1, (_spare(case), C, H, W), 0.0, 1.0)
    if case["train"]:
        _clear(case, d)
    return d


def _spare(case):
    """The images drawn for a batch: a few more than it has for a training
    step, which leaves some out (_clear)."""
    return case["B"] + case["B"] // 2 + 8 if case["train"] else case["B"]


def _clear(case, d):
    """Moves the hidden units' drawn biases a little, each to where its
    pre-activations keep clear of the relu's edge, and leaves out the images
    with a pool window whose two largest values are within rounding of each
    other: a value that a rounding carries across moves a whole term of the
    gradients, and then says nothing of the sums' precision."""
    ws = [_f64(p) for p in d["params"]]
    x = _inputs64(case, d)
    steps = torch.arange(-8, 9, device="cuda", dtype=torch.float64) * 1e-3

    def moved(z, b):  # z: units x samples, without the bias
        best, at = torch.full_like(b, -1.0), b
        for s in steps:
            t = (b + s).float().double()
            gap = (z + t[:, None]).abs().amin(1)
            at, best = torch.where(gap > best, t, at), torch.maximum(gap, best)
        return at

    if case["kind"] == "mlp":
        for i in range(2):
            z = x.mm(ws[i][:-1])
            ws[i][-1] = moved(z.t(), ws[i][-1])
            d["params"][i][-1] = ws[i][-1].cpu().numpy()
            x = (z + ws[i][-1]).relu()
        return
    for i in (0, 2):
        z = _conv64(x, ws[i], None, 1, case["k"] // 2, case["k"] // 2)
        ws[i + 1] = moved(z.permute(1, 0, 2, 3).reshape(z.shape[1], -1), ws[i + 1])
        d["params"][i + 1][:] = ws[i + 1].cpu().numpy()
        r = (z + ws[i + 1][None, :, None, None]).relu()
        x = torch.nn.functional.max_pool2d(r, 2)
        h, w = r.shape[2] // 2 * 2, r.shape[3] // 2 * 2
        top = torch.stack([r[:, :, a:h:2, b:w:2] for a in (0, 1) for b in (0, 1)], -1).topk(2).values
        close = (top[..., 0] > 0) & (top[..., 0] - top[..., 1] < 4e-6)
        bad = close.flatten(1).any(1) if i == 0 else bad | close.flatten(1).any(1)
    keep = torch.argsort(bad, stable=True)[:case["B"]].cpu().numpy()
    for k in ("idx", "x"):
        if k in d:
            d[k] = np.ascontiguousarray(d[k][keep])


def _f64(a, grad=False):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda().double().requires_grad_(grad)


def _inputs64(case, d):
    """The model's input batch in 64 bits."""
    if case["kind"] == "cnn" and case["dataset"]:
        u = d["samples"][d["idx"]].astype(np.float32) / np.float32(255)
        return _f64((u - MEAN[None, :, None, None]) / STD[None, :, None, None])
    return _f64(d["x"])


def _conv_out(case):
    s = case["stride"]
    return ((case["H"] + 2 * case["ph"] - case["kh"]) // s + 1,
            (case["W"] + 2 * case["pw"] - case["kw"]) // s + 1)


# ---------------------------------------------------------------- the program's side

LR = {"sgd": 0.01, "momentum": 0.01, "adam": 0.003, "none": 0.0}


class _Owner:
    """The library objects of one state: its tensors, optimizer and dataset,
    and the graph of its latest pass, given back with it."""

    def __init__(self):
        self.L = tinytorch_amd.lib()
        self.tensors, self.nodes, self.opt, self.data = [], [], None, None

    def tensor(self, a):
        shape = (ctypes.c_long * a.ndim)(*a.shape)
        t = self.L.tt_fromdata(np.ascontiguousarray(a).ctypes.data_as(tinytorch_amd.F32P), shape, a.ndim)
        if not t:
            raise MemoryError("tt_fromdata failed")
        self.tensors.append(t)
        return t

    def keep(self, node):
        if not node:
            raise RuntimeError("an operation returned NULL")
        self.nodes.append(node)
        return node

    def drop_graph(self):
        release = self.L.ag_release
        for n in self.nodes:
            release(n)
        self.nodes = []

    def __del__(self):
        self.drop_graph()
        for t in self.tensors:
            self.L.tt_release(t)
        if self.opt:
            self.L.ag_optim_release(self.opt)
        if self.data:
            self.L.tt_dataset_release(self.data)


class _Device:
    """A tensor of the library's, as torch reads it: its memory, kept by `owner`."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False), version=2)


class _State:
    def __init__(self, case):
        self.case, self.own, self.views = case, _Owner(), {}
        self.L = self.own.L

    def view(self, tensor, shape):
        """What a Tensor holds on the device, without a copy."""
        ptr = self.L.tt_dev(tensor)
        v = self.views.get((ptr, shape))
        if v is None:
            if not ptr:
                raise RuntimeError("tt_dev returned NULL")
            v = self.views[ptr, shape] = torch.as_tensor(_Device(ptr, shape, self.own), device="cuda")
        return v


def prepare(case, seed):
    tinytorch_amd.require_gpu()
    s = _State(case)
    if case["kind"] == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        g = torch.Generator(device="cuda")
        g.manual_seed(int(seed))
        s.a = torch.rand((K, M) if case["ta"] else (M, K), generator=g, device="cuda") * 2 - 1
        s.b = torch.rand((N, K) if case["tb"] else (K, N), generator=g, device="cuda") * 2 - 1
        s.c = torch.empty((M, N), device="cuda")
        s.args = (M, N, K, s.a.data_ptr(), M if case["ta"] else K, int(case["ta"]),
                  s.b.data_ptr(), K if case["tb"] else N, int(case["tb"]), s.c.data_ptr(), N)
        return s
    d = _arrays(case, seed)
    if case["kind"] in ("matmul", "conv"):
        s.t = {k: s.own.tensor(v) for k, v in d.items()}
        s.shapes = {k: v.shape for k, v in d.items()}
        return s
    s.labels = d["labels"]
    s.params = [s.own.tensor(p) for p in d["params"]]
    s.shapes = [p.shape for p in d["params"]]
    s.weights = [s.view(t, shape) for t, shape in zip(s.params, s.shapes)]
    if case["kind"] == "cnn" and case["dataset"]:
        s.idx = d["idx"]
        s.own.data = s.L.tt_dataset_from_u8(d["samples"].ctypes.data, d["all_labels"].ctypes.data,
                                            *d["samples"].shape)
        s.x = None
    else:
        s.x = s.own.tensor(d["x"])
    if case["opt"] == "momentum":
        s.own.opt = s.L.ag_optim_sgd_momentum(LR["momentum"], 0.9)
    elif case["opt"] == "adam":
        s.own.opt = s.L.ag_optim_adam(LR["adam"], 0.9, 0.999, 1e-8)
    if case["kind"] == "cnn":
        s.flat = (ctypes.c_long * 2)(case["B"], _flat(case))
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    return _RUN[s.case["kind"]](s)


def _run_gemm(s):
    if s.L.tt_k_gemm(*s.args) != 0:
        raise RuntimeError("tt_k_gemm failed")
    return s.c


def _run_matmul(s):
    L, own, t = s.L, s.own, s.t
    own.drop_graph()
    k = own.keep
    a, b = k(L.ag_leaf(t["a"], 1)), k(L.ag_leaf(t["b"], 1))
    y = k(L.ag_matmul(a, b))
    L.ag_backward_from_tensor(y, t["seed"])
    return [s.view(L.ag_value(y), s.shapes["seed"]), s.view(L.ag_grad(a), s.shapes["a"]),
            s.view(L.ag_grad(b), s.shapes["b"])]


def _run_conv(s):
    L, own, t, c = s.L, s.own, s.t, s.case
    own.drop_graph()
    k = own.keep
    x, w, b = (k(L.ag_leaf(t[n], 1)) for n in ("x", "w", "b"))
    y = k(L.ag_conv2d(x, w, b, c["stride"], c["stride"], c["ph"], c["pw"]))
    L.ag_backward_from_tensor(y, t["seed"])
    return [s.view(L.ag_value(y), s.shapes["seed"])] + [
        s.view(L.ag_grad(n), s.shapes[name]) for n, name in ((x, "x"), (w, "w"), (b, "b"))]


def _run_mlp(s):
    L, own, c = s.L, s.own, s.case
    own.drop_graph()
    k = own.keep
    train = 1 if c["train"] else 0
    ws = [k(L.ag_leaf(t, train)) for t in s.params]
    h = k(L.ag_padones(k(L.ag_leaf(s.x, 0))))
    h = k(L.ag_padones(k(L.ag_relu(k(L.ag_matmul(h, ws[0]))))))
    h = k(L.ag_padones(k(L.ag_relu(k(L.ag_matmul(h, ws[1]))))))
    return _finish(s, k(L.ag_matmul(h, ws[2])), ws)


def _run_cnn(s):
    L, own, c = s.L, s.own, s.case
    own.drop_graph()
    k = own.keep
    train, pad = (1 if c["train"] else 0), c["k"] // 2
    ws = [k(L.ag_leaf(t, train)) for t in s.params]
    if s.x is None:
        x = L.tt_dataset_batch(own.data, s.idx.ctypes.data, s.idx.size,
                               MEAN.ctypes.data_as(tinytorch_amd.F32P),
                               STD.ctypes.data_as(tinytorch_amd.F32P), 0, s.labels.ctypes.data)
        h = k(L.ag_leaf(x, 0))
        L.tt_release(x)
    else:
        h = k(L.ag_leaf(s.x, 0))
    h = k(L.ag_relu(k(L.ag_conv2d(h, ws[0], ws[1], 1, 1, pad, pad))))
    h = k(L.ag_maxpool2d(h, 2, 2, 2, 2))
    h = k(L.ag_relu(k(L.ag_conv2d(h, ws[2], ws[3], 1, 1, pad, pad))))
    h = k(L.ag_maxpool2d(h, 2, 2, 2, 2))
    h = k(L.ag_padones(k(L.ag_reshape(h, s.flat, 2))))
    return _finish(s, k(L.ag_matmul(h, ws[4])), ws)


def _finish(s, logits, ws):
    """The end of a model's pass: the probabilities, or the loss, the backward
    pass and the optimizer's step."""
    L, c = s.L, s.case
    shape = (c["B"], c["classes"])
    if not c["train"]:
        probs = s.own.keep(L.ag_softmax(logits))
        return dict(logits=s.view(L.ag_value(logits), shape), probs=s.view(L.ag_value(probs), shape))
    loss = s.own.keep(L.ag_softmax_ce(logits, s.labels.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
                                      c["B"]))
    L.ag_backward(loss)
    nodes = (ctypes.c_void_p * len(ws))(*ws)
    if s.own.opt:
        rc = L.ag_optim_step(s.own.opt, nodes, len(ws))
    else:
        rc = L.ag_sgd_step_many(nodes, len(ws), LR["sgd"])
    if rc != 0:
        raise RuntimeError("the optimizer's step failed")
    return dict(logits=s.view(L.ag_value(logits), shape), weights=s.weights,
                grads=[s.view(L.ag_grad(n), sh) for n, sh in zip(ws, s.shapes)])


_RUN = dict(gemm=_run_gemm, matmul=_run_matmul, conv=_run_conv, mlp=_run_mlp, cnn=_run_cnn)


# ---------------------------------------------------------------- what a pass needs

def work(case):
    """Inputs and weights read once, outputs written once; the multiply-adds
    of the products (a first layer has no input gradient)."""
    kind = case["kind"]
    if kind in ("gemm", "matmul"):
        M, N, K = case["M"], case["N"], case["K"]
        if kind == "gemm":
            return dict(bytes=4.0 * (M * K + K * N + M * N), flops=2.0 * M * N * K)
        return dict(bytes=4.0 * (2 * M * K + 2 * K * N + 2 * M * N), flops=6.0 * M * N * K)
    if kind == "conv":
        Ho, Wo = _conv_out(case)
        x = case["N"] * case["C"] * case["H"] * case["W"]
        y = case["N"] * case["F"] * Ho * Wo
        taps = case["C"] * case["kh"] * case["kw"]
        w = case["F"] * (taps + 1)
        return dict(bytes=4.0 * (2 * x + 2 * y + 2 * w), flops=6.0 * y * taps)
    B = case["B"]
    if kind == "mlp":
        d = [case["d0"], case["d1"], case["d2"], case["classes"]]
        layers = [2.0 * B * (d[i] + 1) * d[i + 1] for i in range(3)]
        weights = sum((d[i] + 1) * d[i + 1] for i in range(3))
        x = B * d[0]
    else:
        C, H, W, F1, F2, k = (case[n] for n in ("C", "H", "W", "F1", "F2", "k"))
        layers = [2.0 * B * F1 * H * W * C * k * k, 2.0 * B * F2 * (H // 2) * (W // 2) * F1 * k * k,
                  2.0 * B * (_flat(case) + 1) * case["classes"]]
        weights = F1 * (C * k * k + 1) + F2 * (F1 * k * k + 1) + (_flat(case) + 1) * case["classes"]
        x = B * C * H * W
    logits = B * case["classes"]
    if not case["train"]:
        return dict(bytes=4.0 * (x + weights + 2 * logits), flops=sum(layers))
    state = {"sgd": 3, "momentum": 5, "adam": 7}[case["opt"]]  # weight, gradient and optimizer state
    return dict(bytes=4.0 * (x + state * weights + logits), flops=3.0 * sum(layers) - layers[0])


def tolerance(case):
    """fp32 sums in another order: four times what was measured between the
    framework's own paths and between them and 64 bits (1.6e-6 at most in one
    layer).  In a network's second and later passes a rounding can move a
    value across a relu's or a pool's edge, and with it single terms of the
    gradients (2.5e-3 measured)."""
    if case["kind"] in ("gemm", "matmul"):
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "conv":
        return {"rel": 1e-5, "max": 1e-4}
    if not case["train"]:
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 1e-2, "max": 0.4}


# ---------------------------------------------------------------- the same in 64 bits

def _conv64(x, w, b, stride, ph, pw):
    F, kh, kw = w.shape[0], w.shape[2], w.shape[3]
    N, _, H, W = x.shape
    Ho, Wo = (H + 2 * ph - kh) // stride + 1, (W + 2 * pw - kw) // stride + 1
    col = torch.nn.functional.unfold(x, (kh, kw), padding=(ph, pw), stride=stride)
    col = col.permute(1, 0, 2).reshape(col.shape[1], -1)
    y = w.reshape(F, -1).mm(col).reshape(F, N, Ho * Wo)
    y = y.permute(1, 0, 2).reshape(N, F, Ho, Wo)
    return y if b is None else y + b[None, :, None, None]


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        s = prepare(case, seed)
        a, b = s.a.double(), s.b.double()
        return (a.t() if case["ta"] else a).mm(b.t() if case["tb"] else b)
    d = _arrays(case, seed)

    if kind == "matmul":
        a, b, g = _f64(d["a"]), _f64(d["b"]), _f64(d["seed"])
        return [a.mm(b), g.mm(b.t()), a.t().mm(g)]
    if kind == "conv":
        x, w, b = _f64(d["x"], True), _f64(d["w"], True), _f64(d["b"], True)
        y = _conv64(x, w, b, case["stride"], case["ph"], case["pw"])
        y.backward(_f64(d["seed"]))
        return [y.detach(), x.grad, w.grad, b.grad]
    ws = [_f64(p, case["train"]) for p in d["params"]]
    labels = d["all_labels"][d["idx"]] if kind == "cnn" and case["dataset"] else d["labels"]
    x = _inputs64(case, d)
    if kind == "mlp":
        h = (x.mm(ws[0][:-1]) + ws[0][-1]).relu()
        h = (h.mm(ws[1][:-1]) + ws[1][-1]).relu()
        logits = h.mm(ws[2][:-1]) + ws[2][-1]
    else:
        pad = case["k"] // 2
        pool = torch.nn.functional.max_pool2d
        h = pool(_conv64(x, ws[0], ws[1], 1, pad, pad).relu(), 2)
        h = pool(_conv64(h, ws[2], ws[3], 1, pad, pad).relu(), 2).reshape(case["B"], -1)
        logits = h.mm(ws[4][:-1]) + ws[4][-1]
    if not case["train"]:
        return dict(logits=logits, probs=torch.softmax(logits, 1))
    logp = torch.log_softmax(logits, 1)
    y = torch.from_numpy(labels.astype(np.int64)).cuda()
    (-logp.gather(1, y[:, None]).mean()).backward()
    lr = LR[case["opt"]]
    new = []
    for w in ws:
        g, w = w.grad, w.detach()
        # Adam's first step divides a gradient by itself: of one near its
        # epsilon it keeps the rounding, so only the gradients are compared
        new.append(None if case["opt"] == "adam" else w - lr * g)
    return dict(logits=logits.detach(), weights=new, grads=[w.grad for w in ws])
