"""Measured cases of the training and inference path, as a user's program
calls it through the package's public entry points.

Kinds of case:
  step        a captured MLP training step (forward, softmax + cross-entropy,
              backward, optimiser) replayed through GpuContext.launch_step
  infer       the eager forward of an MLP plan up to its logits
  linear      one Linear layer through the direct calls: forward with bias and
              activation (Z stored), then the gradients of input, weight, bias
  softmax_ce  fused row softmax + cross-entropy, loss and logit gradient
  softmax     plain row softmax and its backward
  optim       one multi-tensor Adam or SGD update
  eltwise     an elementwise graph: forward, MSE loss, backward (eager)

Whole models appear in `step` and `infer` only; 16-bit types are measured
layer by layer (and in `infer`), since a rounding difference in one layer of a
16-bit model travels through all that follow.
"""
import math

import torch

import ferrograd_amd as fa
from ferrograd_amd import graph as G

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
CODE = {"f32": fa.DTYPE_F32, "f16": fa.DTYPE_F16, "bf16": fa.DTYPE_BF16}
ACT = {"none": fa.ACT_NONE, "relu": fa.ACT_RELU, "gelu": fa.ACT_GELU}
WORKSPACE = 256 << 20  # reserved once per program, so that direct calls never allocate

# lr, beta1, beta2, eps as the fp32 values that the update uses.
ADAM = tuple(torch.tensor(v, dtype=torch.float32).item() for v in (1e-3, 0.9, 0.999, 1e-8))


# ------------------------------------------------------------------- cases
def listed():
    return [
        # The smallest whole step: a 2-layer classifier at batch 64, where
        # launches and latency count.
        dict(name="step_small", kind="step", batch=64, dims="784,256,10", act="relu",
             optim="sgd"),
        # The headline workload: an 8-layer 4096-wide MLP step at batch 2048.
        dict(name="step_large", kind="step", batch=2048,
             dims="1024,4096,4096,4096,4096,4096,4096,4096,1000", act="gelu", optim="adam"),
        # Serving the same model in 16 bits at a small batch: every weight is
        # read for a few rows.
        dict(name="infer_bf16_b16", kind="infer", dtype="bf16", batch=16,
             dims="1024,4096,4096,4096,4096,4096,4096,4096,1000", act="gelu"),
        # A small layer of a small model, every size odd.
        dict(name="linear_f32_small", kind="linear", dtype="f32", m=50, k=215, n=101,
             act="relu", bwd="linear"),
        # A layer of ordinary size in training.
        dict(name="linear_f32_1024", kind="linear", dtype="f32", m=1024, k=1024, n=1024,
             act="gelu", bwd="matmul"),
        # A layer whose sizes are no multiple of anything (a vocabulary or
        # feature count that nobody rounded).
        dict(name="linear_f32_odd", kind="linear", dtype="f32", m=1000, k=1501, n=2003,
             act="gelu", bwd="linear"),
        # The hidden layer of the 8-layer model with 16-bit tensors.
        dict(name="linear_bf16_4096", kind="linear", dtype="bf16", m=2048, k=4096, n=4096,
             act="gelu", bwd="matmul"),
        # A 16-bit layer with ragged sizes.
        dict(name="linear_f16_odd", kind="linear", dtype="f16", m=777, k=2049, n=1333,
             act="gelu", bwd="matmul"),
        # The loss over a large vocabulary in fp32, rows that fit a workgroup's
        # registers.
        dict(name="softmax_ce_f32", kind="softmax_ce", dtype="f32", rows=8192, cols=32000),
        # The loss over an odd vocabulary in 16 bits, rows longer than that.
        dict(name="softmax_ce_bf16_odd", kind="softmax_ce", dtype="bf16", rows=2048, cols=50257),
        # An optimiser step over a model's list: wide matrices, narrow ones and
        # biases, half of the tensors in 16 bits.
        dict(name="adam_mixed", kind="optim", optim="adam", tensors=96, largest=4194304,
             dtypes="mixed"),
        # A custom elementwise block with its loss and gradients.
        dict(name="eltwise_mid", kind="eltwise", dtype="f32", rows=1000, cols=777,
             chain="tanh_mul_add"),
    ]


def _size(rng, lo, hi):
    """Log-uniform in [lo, hi]; half of them rounded to a multiple of 64 (8 below 64)."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        q = 64 if n >= 64 else 8
        n = max(q, n // q * q)
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choices(
        ["linear", "step", "infer", "softmax_ce", "softmax", "optim", "eltwise"],
        [40, 10, 12, 14, 8, 8, 8])[0]
    if kind == "linear":
        dtype = rng.choice(["f32", "f32", "bf16", "f16"])
        while True:
            m, k, n = (_size(rng, 16, 4096) for _ in range(3))
            if m * k * n <= 2048 * 4096 * 4096:
                break
        return dict(kind=kind, dtype=dtype, m=m, k=k, n=n,
                    act=rng.choice(["none", "relu", "gelu", "gelu"]),
                    bwd=rng.choice(["linear", "matmul"]) if dtype == "f32" else "matmul")
    if kind == "step":
        layers = rng.randint(2, 4)
        dims = [_size(rng, 32, 2048) for _ in range(layers)] + [_size(rng, 10, 1000)]
        return dict(kind=kind, batch=_size(rng, 16, 2048), dims=",".join(map(str, dims)),
                    act=rng.choice(["relu", "gelu"]), optim=rng.choice(["sgd", "adam"]))
    if kind == "infer":
        layers = rng.randint(2, 4)
        dims = [_size(rng, 64, 4096) for _ in range(layers)] + [_size(rng, 10, 1000)]
        return dict(kind=kind, dtype=rng.choice(["f32", "bf16", "f16"]),
                    batch=_size(rng, 1, 256), dims=",".join(map(str, dims)),
                    act=rng.choice(["relu", "gelu"]))
    if kind in ("softmax_ce", "softmax"):
        while True:
            rows, cols = _size(rng, 16, 16384), _size(rng, 10, 131072)
            if 1 << 12 <= rows * cols <= 8192 * 32000:
                break
        return dict(kind=kind, dtype=rng.choice(["f32", "f32", "bf16", "f16"]), rows=rows,
                    cols=cols)
    if kind == "optim":
        return dict(kind=kind, optim=rng.choice(["adam", "adam", "sgd"]),
                    tensors=rng.randint(4, 160), largest=_size(rng, 4096, 4194304),
                    dtypes=rng.choice(["f32", "mixed", "bf16"]))
    return dict(kind="eltwise", dtype=rng.choice(["f32", "f32", "bf16"]),
                rows=_size(rng, 16, 4096), cols=_size(rng, 16, 8192),
                chain=rng.choice(["tanh_mul_add", "gelu_gate", "elu_sub_div"]))


# ----------------------------------------------------------------- inputs
_CTX = []


def _context():
    """The program's one context (its stream is torch's current one)."""
    if not _CTX:
        c = G.GpuContext.new(0)
        c.ctx.reserve_workspace(WORKSPACE)
        _CTX.append(c)
    return _CTX[0]


class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, shape, std=1.0, dtype="f32"):
        return torch.empty(shape, device="cuda").normal_(0.0, std, generator=self.g).to(DT[dtype])

    def uniform(self, shape, bound, dtype="f32"):
        return torch.empty(shape, device="cuda").uniform_(-bound, bound,
                                                          generator=self.g).to(DT[dtype])

    def labels(self, rows, classes):
        return torch.randint(0, classes, (rows,), device="cuda", generator=self.g,
                             dtype=torch.int32)


def _dims(case):
    return [int(d) for d in case["dims"].split(",")]


def _hidden(act, z):
    return torch.relu(z) if act == "relu" else torch.nn.functional.gelu(z, approximate="tanh")


def _mlp_inputs(case, seed):
    """x ~ N(0,1), Kaiming-uniform weights, zero biases, uniform labels."""
    r, dims, dtype = _Rand(seed), _dims(case), case.get("dtype", "f32")
    x = r.normal((case["batch"], dims[0]), 1.0, dtype)
    params = []
    for a, b in zip(dims, dims[1:]):
        params.append(r.uniform((a, b), math.sqrt(6.0 / a), dtype))
        params.append(torch.zeros(b, device="cuda", dtype=DT[dtype]))
    return x, params, r.labels(case["batch"], dims[-1])


def _linear_inputs(case, seed):
    r, d = _Rand(seed), case["dtype"]
    m, k, n = case["m"], case["k"], case["n"]
    t = dict(x=r.normal((m, k), 1.0, d), w=r.uniform((k, n), math.sqrt(6.0 / k), d),
             b=r.normal((n,), 0.1, d), dy=r.normal((m, n), 1.0, d))
    if case["bwd"] == "matmul":
        t["zprev"] = r.normal((m, k), 1.0, d)
    return t


def _optim_sizes(case):
    """A model's list: matrices of `largest` elements and fewer, each followed
    by a bias-sized vector."""
    sizes = []
    for i in range(case["tensors"]):
        sizes.append(max(1, case["largest"] >> (i // 2 % 4)) if i % 2 == 0
                     else max(1, math.isqrt(case["largest"]) + i % 3))
    return sizes


def _optim_dtypes(case):
    return [("bf16" if i // 2 % 2 else "f32") if case["dtypes"] == "mixed" else case["dtypes"]
            for i in range(case["tensors"])]


def _optim_inputs(case, seed):
    """Tensors of one type are views of one allocation, each on a 256-byte line."""
    r = _Rand(seed)
    sizes, dts = _optim_sizes(case), _optim_dtypes(case)
    flat, views = {}, [None] * len(sizes)
    for d in sorted(set(dts)):
        at, offs = 0, {}
        for i, n in enumerate(sizes):
            if dts[i] == d:
                offs[i] = at
                at += -(-n // 128) * 128
        p, g = r.normal((at,), 0.02, d), r.normal((at,), 1e-3, d)
        m, v = torch.zeros(at, device="cuda"), torch.zeros(at, device="cuda")
        for i, o in offs.items():
            views[i] = [t[o:o + sizes[i]] for t in (p, g, m, v)]
        keep = torch.zeros(at, device="cuda", dtype=torch.bool)
        for i, o in offs.items():
            keep[o:o + sizes[i]] = True
        flat[d] = dict(p=p, g=g, m=m, v=v, keep=keep)
    return sizes, dts, flat, views


def _eltwise_inputs(case, seed):
    r, d, s = _Rand(seed), case["dtype"], (case["rows"], case["cols"])
    return [r.normal(s, 1.0, d) for _ in range(3)], r.normal(s, 1.0, d)


class _View:
    """A plan-owned device tensor as torch sees it."""

    def __init__(self, ptr, n, code):
        self.__cuda_array_interface__ = dict(
            shape=(n,), typestr={0: "<f4", 1: "<f2", 2: "<i2"}[code], data=(ptr, False),
            version=3, strides=None)


def _view(at, t, dtype, shape):
    v = torch.as_tensor(_View(t.ptr, t.len(), CODE[dtype]), device="cuda")
    v = (v.view(torch.bfloat16) if dtype == "bf16" else v).view(shape)
    v.plan = at.plan  # the plan's memory lives as long as the tensor
    return v


def _mlp_plan(c, case, softmax):
    dims, dtype = _dims(case), case.get("dtype", "f32")
    opt = G.Optim.adam() if case.get("optim") == "adam" else G.Optim.sgd()
    graph, meta = G.Graph(G.CROSS_ENTROPY if softmax else G.MEAN_SQUARED_ERROR, opt.lower), \
        G.Metadata.new()
    fb, fd = meta.new_field(), [meta.new_field() for _ in dims]
    with graph.define_ops() as ops:
        h = ops.input([fb, fd[0]], dtype, trainable=False, requires_grad=softmax)
        for l in range(len(dims) - 1):
            w = ops.input([fd[l], fd[l + 1]], dtype)
            b = ops.input([fd[l + 1]], dtype)
            z = ops.bias_add(ops.matmul(h, w), b)
            h = getattr(ops, case["act"])(z) if l < len(dims) - 2 else z
        if softmax:
            ops.softmax(h)
    binding = [G.f32_bits(1e-4 if case.get("optim") == "sgd" else ADAM[0]), case["batch"]] + dims
    return graph, meta, binding, c.alloc_tensors(graph, graph.compute_saved_nodes(), binding)


def prepare(case, seed):
    c = _context()
    kind = case["kind"]
    st = dict(kind=kind, case=case, c=c, ctx=c.ctx)
    if kind in ("step", "infer"):
        x, params, labels = _mlp_inputs(case, seed)
        graph, meta, binding, at = _mlp_plan(c, case, kind == "step")
        sched = c.schedule(graph.lower(meta), binding, [x] + params, at)
        st.update(x=x, params=params, labels=labels, at=at, sched=sched)
        if kind == "step":
            c.capture_step(sched, labels)
            of = {t.node: t for t in at.grad_tensors}
            ins = [i for i, nd in enumerate(graph.nodes) if nd.op == G.OP_INPUT]
            st["grads"] = [_view(at, of[i], "f32", t.shape) for i, t in zip(ins, [x] + params)]
            st["loss"] = _view(at, at.mean_loss, "f32", (1,))
        else:
            st["out"] = _view(at, at.forward_out, case["dtype"], (case["batch"], _dims(case)[-1]))
    elif kind == "linear":
        st.update(_linear_inputs(case, seed))
        m, k, n, dt = case["m"], case["k"], case["n"], DT[case["dtype"]]
        for name, shape in dict(h=(m, n), z=(m, n), dx=(m, k), dw=(k, n), db=(n,),
                                dz=(m, n)).items():
            st[name] = torch.empty(shape, device="cuda", dtype=dt)
    elif kind in ("softmax_ce", "softmax"):
        r, s = _Rand(seed), (case["rows"], case["cols"])
        st["x"] = r.normal(s, 2.0, case["dtype"])
        if kind == "softmax_ce":
            st["labels"] = r.labels(*s)
            st["row_loss"] = torch.empty(s[0], device="cuda")
            st["mean"] = torch.empty(1, device="cuda")
            st["argmax"] = torch.empty(s[0], device="cuda", dtype=torch.int32)
        else:
            st["dy"] = r.normal(s, 1.0, case["dtype"])
            st["y"] = torch.empty_like(st["x"])
        st["dx"] = torch.empty_like(st["x"])
    elif kind == "optim":
        sizes, dts, flat, views = _optim_inputs(case, seed)
        adam = case["optim"] == "adam"
        st.update(flat=flat, t=0, mt=fa.MultiTensor(
            c.ctx, [v[0] for v in views], [v[1] for v in views],
            [v[2] for v in views] if adam else None, [v[3] for v in views] if adam else None,
            dtypes=[CODE[d] for d in dts]))
    else:
        ins, target = _eltwise_inputs(case, seed)
        graph, meta = G.Graph(G.MEAN_SQUARED_ERROR, G.Optim.sgd().lower), G.Metadata.new()
        shape = [meta.new_field(), meta.new_field()]
        d = case["dtype"]
        with graph.define_ops() as ops:
            a, b, e = (ops.input(shape, d) for _ in range(3))
            if case["chain"] == "tanh_mul_add":
                ops.tanh(ops.add(ops.mul(a, b), e))
            elif case["chain"] == "gelu_gate":
                ops.add(ops.mul(ops.gelu(a), b), e)
            else:
                one = getattr(ops, "constant_" + d)(1.0)
                ops.div(ops.elu(ops.sub(a, b)), ops.add(ops.abs(e), one))
        binding = [G.f32_bits(1e-3), case["rows"], case["cols"]]
        at = c.alloc_tensors(graph, graph.compute_saved_nodes(), binding)
        s2 = (case["rows"], case["cols"])
        of = {t.node: t for t in at.grad_tensors}
        st.update(ins=ins, target=target, at=at,
                  sched=c.schedule(graph.lower(meta), binding, ins, at),
                  out=_view(at, at.forward_out, d, s2), loss=_view(at, at.loss_t, d, s2),
                  grads=[_view(at, of[i], d, s2) for i in range(3)])
    return st


# -------------------------------------------------------------------- run
def run(st):
    kind, case, ctx = st["kind"], st["case"], st["ctx"]
    if kind == "step":
        st["c"].launch_step(st["sched"])
        return dict(loss=st["loss"], grads=st["grads"], params=st["params"])
    if kind == "infer":
        st["c"].dispatch_forward(st["sched"])
        return st["out"]
    if kind == "linear":
        m, k, n, act = case["m"], case["k"], case["n"], ACT[case["act"]]
        x, w, b, h, z, dy, dx, dw, db = (st[i] for i in
                                         ("x", "w", "b", "h", "z", "dy", "dx", "dw", "db"))
        if case["dtype"] == "f32":
            ctx.gemm(fa.NN, m, n, k, x, k, w, n, h, n, bias=b, act=act, Z=z, ldz=n)
            if case["bwd"] == "linear":
                ctx.linear_bwd(act, m, n, k, x, k, w, n, z, n, dy, n, dX=dx, dW=dw, dbias=db,
                               dZ=st["dz"])
            else:
                ctx.matmul_bwd(m, n, k, x, k, w, n, dy, n, dx, k, dw, n, dbias=db, act=act,
                               Zs=st["zprev"], ldzs=k)
        else:
            code = CODE[case["dtype"]]
            ctx.gemm_x16(code, fa.NN, m, n, k, x, k, w, n, h, n, bias=b, act=act, Z=z, ldz=n)
            ctx.matmul_bwd_x16(code, m, n, k, x, k, w, n, dy, n, dx, k, dw, n, dbias=db, act=act,
                               Zs=st["zprev"], ldzs=k)
        return dict(h=h, z=z, dx=dx, dw=dw, db=db)
    if kind == "softmax_ce":
        R, C = case["rows"], case["cols"]
        ctx.softmax_ce(st["x"], C, st["labels"], R, C, row_loss=st["row_loss"],
                       mean_loss=st["mean"], dlogits=st["dx"], ldd=C, argmax=st["argmax"],
                       dtype=CODE[case["dtype"]])
        return dict(row_loss=st["row_loss"], mean=st["mean"], dx=st["dx"], argmax=st["argmax"])
    if kind == "softmax":
        R, C, code = case["rows"], case["cols"], CODE[case["dtype"]]
        ctx.softmax(st["x"], R, C, st["y"], dtype=code)
        ctx.softmax_bwd(st["y"], st["dy"], R, C, st["dx"], dtype=code)
        return dict(y=st["y"], dx=st["dx"])
    if kind == "optim":
        st["t"] += 1
        if case["optim"] == "adam":
            st["mt"].adam(*ADAM, st["t"])
            return {d: [f["p"], f["m"], f["v"]] for d, f in st["flat"].items()}
        st["mt"].sgd(1e-3, zero_grad=False)
        return {d: [f["p"]] for d, f in st["flat"].items()}
    st["c"].dispatch_forward(st["sched"])
    st["c"].dispatch_loss(st["sched"], st["target"])
    st["c"].dispatch_backward(st["sched"])
    return dict(out=st["out"], loss=st["loss"], grads=st["grads"])


# ------------------------------------------------------------ work, limits
def _bytes(dtype):
    return 4 if dtype == "f32" else 2


def work(case):
    kind = case["kind"]
    if kind in ("step", "infer"):
        dims, B = _dims(case), case["batch"]
        params = sum(a * b + b for a, b in zip(dims, dims[1:]))
        mac = sum(a * b for a, b in zip(dims, dims[1:])) * B
        if kind == "infer":
            return dict(flops=2 * mac,
                        bytes=_bytes(case["dtype"]) * (params + B * (dims[0] + dims[-1])))
        # Weights read, gradients and updated weights written (Adam: m and v
        # read and written too); the input read and its gradient written.
        per = 7 if case["optim"] == "adam" else 3
        return dict(flops=6 * mac, bytes=4 * (per * params + B * (2 * dims[0] + 1)))
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        mats = 3 * m * n + 2 * m * k + 2 * k * n + 2 * n
        mats += m * k if case["bwd"] == "matmul" else 0
        return dict(flops=6 * m * k * n, bytes=_bytes(case["dtype"]) * mats)
    if kind in ("softmax_ce", "softmax"):
        rc, b = case["rows"] * case["cols"], _bytes(case["dtype"])
        if kind == "softmax":
            return dict(flops=8 * rc, bytes=4 * rc * b)
        return dict(flops=5 * rc, bytes=2 * rc * b + 12 * case["rows"] + 4)
    if kind == "optim":
        total = 0
        for n, d in zip(_optim_sizes(case), _optim_dtypes(case)):
            total += n * (3 * _bytes(d) + (16 if case["optim"] == "adam" else 0))
        return dict(flops=0, bytes=total)
    rc = case["rows"] * case["cols"]
    return dict(flops=20 * rc, bytes=9 * rc * _bytes(case["dtype"]))


def tolerance(case):
    kind, dtype = case["kind"], case.get("dtype", "f32")
    # Two jumps that fp32 rounding can cross.  ReLU's backward: a pre-activation
    # within rounding of 0 switches one term of the gradients.  Adam's first
    # step is lr * sign(g): a gradient within rounding of 0 moves its parameter
    # the other way.
    if kind == "step" and (case["optim"] == "adam" or case["act"] == "relu"):
        return {"rel": 2e-3, "max": 0.5}
    if kind == "linear" and dtype == "f32" and case["act"] == "relu" and case["bwd"] == "linear":
        return {"rel": 2e-3, "max": 0.5}
    if kind == "optim":  # element by element: the order of no sum to choose
        return {"rel": 1e-6, "max": 1e-2} if case["dtypes"] != "f32" else {"rel": 1e-6}
    # fp32: layers were seen at 2e-7 to 1.2e-6 off the 64-bit result (sums of
    # up to 4096 products), whole models at 6e-6, rows and chains at 1e-7.
    if dtype == "f32":
        return {"rel": {"step": 2e-5, "infer": 1e-5, "linear": 5e-6}.get(kind, 2e-6), "max": 1e-3}
    # 16 bits: layers were seen at 3e-3 (bf16) and 4e-4 (f16) off, each node
    # value rounded once; eight bf16 layers at 8e-3.
    unit = 4e-3 if dtype == "bf16" else 5e-4
    return {"rel": 2.5 * unit if kind == "infer" else unit, "max": 25 * unit}


# ------------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "infer"):
        x, params, labels = _mlp_inputs(case, seed)
        ts = [t.double().requires_grad_(kind == "step") for t in [x] + params]
        h, last = ts[0], len(params) // 2 - 1
        for l in range(last + 1):
            h = h @ ts[1 + 2 * l] + ts[2 + 2 * l]
            h = _hidden(case["act"], h) if l < last else h
        if kind == "infer":
            return h
        loss = torch.nn.functional.cross_entropy(h, labels.long(), reduction="none")
        grads = torch.autograd.grad(loss.sum(), ts)
        new = []
        for p, g in zip(ts[1:], grads[1:]):
            if case["optim"] == "sgd":
                new.append((p - 1e-4 * g).detach())
            else:
                new.append((p - ADAM[0] * g / (g.abs() + ADAM[3])).detach())
        if case["optim"] == "sgd":  # the update clears the gradients it has used
            grads = list(grads[:1]) + [torch.zeros_like(g) for g in grads[1:]]
        return dict(loss=loss.mean().detach().view(1), grads=list(grads), params=new)
    if kind == "linear":
        t = {i: v.double() for i, v in _linear_inputs(case, seed).items()}
        z = t["x"] @ t["w"] + t["b"]

        def act(v):
            return v if case["act"] == "none" else _hidden(case["act"], v)

        def slope(v):
            v = v.detach().requires_grad_()
            return torch.autograd.grad(act(v).sum(), v)[0]

        dz = t["dy"] * slope(z) if case["bwd"] == "linear" else t["dy"]
        dx = dz @ t["w"].t()
        if case["bwd"] == "matmul":
            dx = dx * slope(t["zprev"])
        return dict(h=act(z), z=z, dx=dx, dw=t["x"].t() @ dz, db=dz.sum(0))
    if kind in ("softmax_ce", "softmax"):
        r, s = _Rand(seed), (case["rows"], case["cols"])
        x = r.normal(s, 2.0, case["dtype"]).double()
        if kind == "softmax":
            dy, y = r.normal(s, 1.0, case["dtype"]).double(), torch.softmax(x, 1)
            return dict(y=y, dx=y * (dy - (dy * y).sum(1, keepdim=True)))
        labels = r.labels(*s).long()
        rows = torch.nn.functional.cross_entropy(x, labels, reduction="none")
        dx = torch.softmax(x, 1)
        dx[torch.arange(s[0], device="cuda"), labels] -= 1.0
        return dict(row_loss=rows, mean=rows.mean().view(1), dx=dx, argmax=None)
    if kind == "optim":
        _, _, flat, _ = _optim_inputs(case, seed)
        out = {}
        for d, f in flat.items():
            p, g = f["p"].double(), f["g"].double() * f["keep"]
            if case["optim"] == "sgd":
                out[d] = [p - 1e-3 * g]
            else:
                out[d] = [p - ADAM[0] * g / (g.abs() + ADAM[3]), (1 - ADAM[1]) * g,
                          (1 - ADAM[2]) * g * g]
        return out
    ins, target = _eltwise_inputs(case, seed)
    a, b, e = (t.double().requires_grad_() for t in ins)
    if case["chain"] == "tanh_mul_add":
        out = torch.tanh(a * b + e)
    elif case["chain"] == "gelu_gate":
        out = _hidden("gelu", a) * b + e
    else:
        out = torch.nn.functional.elu(a - b) / (e.abs() + 1.0)
    loss = (out - target.double()) ** 2
    return dict(out=out.detach(), loss=loss.detach(),
                grads=list(torch.autograd.grad(loss.sum(), [a, b, e])))
