"""The work whose time counts: compiled programs called through the framework's public entry points (`compile` gives a
`Thunk`, the thunk is called on device arrays), from a reduction of a few thousand numbers to fields of half a gigabyte.

A case names a program and its sizes:

    loss      sum(sin.(x) .+ y) of two vectors, a scalar result                        f32, f64
    stencil   explicit time steps of 3-D advection and diffusion, a halo of 3 cells    f64, f32
    gemm      C = alpha A B + beta C, what `mul!` on device matrices compiles to        f32, f64
    mlp       dense + bias + gelu layers and a softmax: a network's inference pass      bf16, f32
    train     loss and gradients of a two-layer network (forward and reverse pass)      bf16, f32
    fp8       absmax quantization, an e4m3 linear layer, RMSNorm                        bf16 activations
    vgg       forward pass of VGG-11, the convolutional model of the vision benchmark   f32, bf16

`listed()` are fixed cases, `draw(rng)` gives others of the same ranges.  A program is compiled once per process, as a
user's program does; inputs are made on the device from the seed."""
import importlib
import importlib.util
import math
import os
import sys

import torch


def _package():
    if "reactant_jl_amd" not in sys.modules:
        d = os.path.abspath("reactant.jl_amd")
        spec = importlib.util.spec_from_file_location("reactant_jl_amd", os.path.join(d, "__init__.py"), submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["reactant_jl_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["reactant_jl_amd"]


def listed():
    return [
        # a loss over a small batch, called once per step of an optimizer: launches and the host's work per call
        {"name": "loss_small", "kind": "loss", "n": 4099, "dt": "f32"},
        # the same over vectors that fill the memory system
        {"name": "loss_large", "kind": "loss", "n": 1 << 26, "dt": "f32"},
        # a coarse grid of uneven extents: the development run of a simulation
        {"name": "stencil_small", "kind": "stencil", "nx": 61, "ny": 47, "nz": 33, "steps": 10, "dt": "f64"},
        # the production grid: fields of 562 MB, ten time steps per call
        {"name": "stencil_large", "kind": "stencil", "nx": 512, "ny": 512, "nz": 256, "steps": 10, "dt": "f64"},
        # a matrix product of sizes that come from data, no multiples of anything
        {"name": "gemm_odd", "kind": "gemm", "m": 1001, "n": 777, "k": 1531, "dt": "f32"},
        # a large dense product in Julia's single precision
        {"name": "gemm_large", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096, "dt": "f32"},
        # a served network: a small batch, bound by reading the weights
        {"name": "mlp_serve", "kind": "mlp", "batch": 16, "w0": 1024, "w1": 4096, "w2": 4096, "w3": 1024, "dt": "bf16"},
        # the same network over a large batch
        {"name": "mlp_large", "kind": "mlp", "batch": 8192, "w0": 1024, "w1": 4096, "w2": 4096, "w3": 1024, "dt": "bf16"},
        # one training step's loss and gradients at an ordinary batch
        {"name": "train_step", "kind": "train", "batch": 1024, "w0": 784, "w1": 2048, "w2": 1000, "dt": "bf16"},
        # a quantized layer on a ragged number of tokens
        {"name": "fp8_ragged", "kind": "fp8", "batch": 200, "k": 4096, "n": 6144},
        # the same layer, large and square
        {"name": "fp8_large", "kind": "fp8", "batch": 8192, "k": 8192, "n": 8192},
        # the vision benchmark's model and input
        {"name": "vgg_4", "kind": "vgg", "batch": 4, "hw": 224, "dt": "f32"},
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["loss", "stencil", "gemm", "mlp", "train", "fp8", "vgg"])
    if kind == "loss":
        return {"kind": kind, "n": _log(rng, 1 << 10, 1 << 26), "dt": rng.choice(["f32", "f32", "f64"])}
    if kind == "stencil":
        return {"kind": kind, "nx": _log(rng, 24, 512), "ny": _log(rng, 24, 512), "nz": _log(rng, 16, 256), "steps": rng.randint(4, 10),
                "dt": rng.choice(["f64", "f64", "f32"])}
    if kind == "gemm":
        m, n, k = (_log(rng, 64, 4096) for _ in range(3))
        if rng.random() < 0.5:   # half of them are whole vectors in every dimension, as chosen sizes are
            m, n, k = (max(64, v - v % 64) for v in (m, n, k))
        return {"kind": kind, "m": m, "n": n, "k": k, "dt": rng.choice(["f32", "f32", "f64"])}
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 1, 8192), "w0": rng.choice([512, 784, 1024]), "w1": rng.choice([1024, 2048, 3000, 4096]),
                "w2": rng.choice([1024, 2048, 4096]), "w3": rng.choice([10, 1000, 1024]), "dt": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "train":
        return {"kind": kind, "batch": _log(rng, 64, 4096), "w0": rng.choice([512, 784, 1024]), "w1": rng.choice([1024, 2048, 4096]),
                "w2": rng.choice([10, 1000, 1024]), "dt": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "fp8":
        return {"kind": kind, "batch": _log(rng, 1, 8192), "k": rng.choice([1024, 2048, 4096, 5120, 8192]),
                "n": rng.choice([1024, 2048, 4096, 6144, 8192])}
    if rng.random() < 0.6:
        return {"kind": kind, "batch": rng.randint(1, 8), "hw": 32 * rng.randint(2, 7), "dt": "f32"}
    return {"kind": kind, "batch": rng.randint(4, 32), "hw": 32 * rng.randint(2, 7), "dt": "bf16"}


# ----------------------------------------------------------------------------
# programs
# ----------------------------------------------------------------------------
def _train_text(batch, w0, w1, w2, dt):
    """Mean squared error of `relu(x W1 + b1) W2 + b2` against targets and its gradients with respect to the four
    parameters, with the products in the form the reverse pass leaves them: dW = h' dy contracts the batch of both
    operands, dh = dy W' the minor dimension of both.  Results: loss (f32), dW1, db1, dW2, db2."""
    P = importlib.import_module("reactant_jl_amd.programs")
    tt, b = P._tt, P._B()
    X, T, W1, B1, W2, B2 = ([batch, w0], [batch, w2], [w0, w1], [w1], [w1, w2], [w2])
    args = []
    for k, s in enumerate((X, T, W1, B1, W2, B2)):
        b.types["%%arg%d" % k] = tt(s, dt)
        args.append("%%arg%d: %s" % (k, tt(s, dt)))
    H, Y, S = [batch, w1], [batch, w2], "tensor<f32>"

    def op(text, shape, ty=None):
        r = b.new(tt(shape, ty or dt))
        b.lines.append("    %s = %s -> %s" % (r, text, tt(shape, ty or dt)))
        return r

    def dot(x, y, dims, shape):
        return op("stablehlo.dot_general %s, %s, contracting_dims = %s, precision = [DEFAULT, DEFAULT] : (%s, %s)"
                  % (x, y, dims, b.types[x], b.types[y]), shape)

    def rows(v, shape):
        return op("stablehlo.broadcast_in_dim %s, dims = [1] : (%s)" % (v, b.types[v]), shape)

    def column_sum(x, shape):
        zero = b.const(0.0, [], dt)
        return op("stablehlo.reduce(%s init: %s) applies stablehlo.add across dimensions = [0] : (%s, %s)"
                  % (x, zero, b.types[x], b.types[zero]), shape)

    z = b.bin("add", dot("%arg0", "%arg2", "[1] x [0]", H), rows("%arg3", H))
    h = b.bin("maximum", z, b.const(0.0, H, dt))
    y = b.bin("add", dot(h, "%arg4", "[1] x [0]", Y), rows("%arg5", Y))
    d = b.bin("subtract", y, "%arg1")
    df = op("stablehlo.convert %s : (%s)" % (d, b.types[d]), Y, "f32") if dt != "f32" else d
    zf = b.const(0.0, [], "f32")
    total = op("stablehlo.reduce(%s init: %s) applies stablehlo.add across dimensions = [0, 1] : (%s, %s)"
               % (b.bin("multiply", df, df), zf, b.types[df], S), [], "f32")
    loss = b.bin("multiply", total, b.const(1.0 / (batch * w2), [], "f32"))
    dy = b.bin("multiply", d, b.const(2.0 / w2, Y, dt))
    dw2, db2 = dot(h, dy, "[0] x [0]", W2), column_sum(dy, B2)
    dh = dot(dy, "%arg4", "[1] x [1]", H)
    pred = b.new(tt(H, "i1"))
    zh = b.const(0.0, H, dt)
    b.lines.append("    %s = stablehlo.compare  GT, %s, %s,  FLOAT : (%s, %s) -> %s" % (pred, z, zh, b.types[z], b.types[zh], tt(H, "i1")))
    dz = b.new(tt(H, dt))
    b.lines.append("    %s = stablehlo.select %s, %s, %s : %s, %s" % (dz, pred, dh, zh, tt(H, "i1"), tt(H, dt)))
    dw1, db1 = dot("%arg0", dz, "[0] x [0]", W1), column_sum(dz, B1)
    res = [loss, dw1, db1, dw2, db2]
    rt = ", ".join(b.types[r] for r in res)
    return ("module @reactant_train {\n  func.func @main(" + ", ".join(args) + ") -> (" + rt + ") {\n" + b.text()
            + "    return %s : %s\n  }\n}\n" % (", ".join(res), rt))


def _program(case):
    """(module text, [(shape, element type, distribution)] of the arguments); shapes are those of the module's tensors."""
    _package()
    P = importlib.import_module("reactant_jl_amd.programs")
    kind, dt = case["kind"], case.get("dt", "bf16")
    if kind == "loss":
        n = case["n"]
        return P.sinsum_add(n, dt), [([n], dt, ("uniform", -math.pi, math.pi)), ([n], dt, ("uniform", 0.0, 1.0))]
    if kind == "stencil":
        full = [case["nz"] + 6, case["ny"] + 6, case["nx"] + 6]
        return (P.stencil(case["nx"], case["ny"], case["nz"], steps=case["steps"], elt=dt),
                [(full, dt, ("interior", 0.0, 1.0))] + [(full, dt, ("uniform", -1.0, 1.0))] * 3)
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return P.gemm(m, n, k, dt=dt), [([k, m], dt, ("normal", 1.0)), ([n, k], dt, ("normal", 1.0)), ([n, m], dt, ("normal", 1.0))]
    if kind == "mlp":
        w = [case["w0"], case["w1"], case["w2"], case["w3"]]
        args = [([case["batch"], w[0]], dt, ("normal", 1.0))]
        for a, b in zip(w, w[1:]):
            args += [([a, b], dt, ("uniform", -math.sqrt(6.0 / (a + b)), math.sqrt(6.0 / (a + b)))), ([b], dt, ("uniform", -0.1, 0.1))]
        return P.mlp(case["batch"], tuple(w), dt=dt), args
    if kind == "train":
        bt, w0, w1, w2 = case["batch"], case["w0"], case["w1"], case["w2"]
        g = lambda a, b: ("uniform", -math.sqrt(6.0 / (a + b)), math.sqrt(6.0 / (a + b)))   # noqa: E731
        return _train_text(bt, w0, w1, w2, dt), [([bt, w0], dt, ("normal", 1.0)), ([bt, w2], dt, ("normal", 1.0)), ([w0, w1], dt, g(w0, w1)),
                                                 ([w1], dt, ("uniform", -0.1, 0.1)), ([w1, w2], dt, g(w1, w2)), ([w2], dt, ("uniform", -0.1, 0.1))]
    if kind == "fp8":
        bt, k, n = case["batch"], case["k"], case["n"]
        return P.fp8_linear(bt, k, n), [([bt, k], "bf16", ("normal", 1.0)), ([n, k], "f8E4M3FN", ("normal", 80.0)), ([], "f32", ("uniform", 1e-4, 3e-4))]
    if kind == "vgg":
        N = importlib.import_module("reactant_jl_amd.nn_programs")
        text, shapes, _ = N.vgg11(batch=case["batch"], hw=case["hw"], dt=dt)
        nconv = sum(1 for l in N.VGG11_LAYERS if l != "M")
        args = []
        for k, s in enumerate(shapes):
            if len(s) == 4 and k > 0:
                how = ("normal", math.sqrt(2.0 / (s[1] * s[2] * s[3])))
            elif len(s) == 2:
                how = ("normal", math.sqrt(2.0 / s[0]))
            elif 0 < k <= 5 * nconv and (k - 1) % 5 in (1, 4):
                how = ("uniform", 0.5, 2.0)       # a batch norm's scale and running variance
            elif len(s) == 1:
                how = ("normal", 0.1)
            else:
                how = ("normal", 1.0)
            args.append((s, dt, how))
        return text, args
    raise KeyError(kind)


# ----------------------------------------------------------------------------
# device arrays and torch's view of them
# ----------------------------------------------------------------------------
_TORCH = {"f32": ("<f4", torch.float32), "f64": ("<f8", torch.float64), "bf16": ("<i2", torch.bfloat16), "f8E4M3FN": ("|u1", torch.float8_e4m3fn)}


class _Bytes:
    """A device array's memory as torch takes it; torch keeps this object, and with it the array, while its view lives."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {"shape": array.shape[::-1], "typestr": _TORCH[array.dtype][0], "version": 2,
                                         "data": (array.data.buffer.unsafe_pointer(), False)}


def _view(array):
    t = torch.as_tensor(_Bytes(array), device="cuda")
    want = _TORCH[array.dtype][1]
    return t if t.dtype == want else t.view(want)


def _fill(gen, shape, dt, how):
    if how[0] == "normal":
        t = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * how[1]
    else:
        t = torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64 if dt == "f64" else torch.float32) * (how[2] - how[1]) + how[1]
        if how[0] == "interior":                  # zeros in the halo
            inner = t[3:-3, 3:-3, 3:-3].clone()
            t.zero_()
            t[3:-3, 3:-3, 3:-3] = inner
    return t.clamp_(-448.0, 448.0) if dt == "f8E4M3FN" else t


_compiled = {}


def prepare(case, seed):
    text, args = _program(case)
    rx = _package()
    client = rx.set_default_backend("gpu")
    if text not in _compiled:
        _compiled[text] = rx.compile(text)
    client.default_device().synchronize()         # a recycled block may still be in use on the framework's stream
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    arrays = []
    for shape, dt, how in args:
        array = rx.ConcreteRArray(rx.AsyncBuffer(rx.Buffer.uninitialized(client, shape, dt)), tuple(shape)[::-1], dt)
        _view(array).copy_(_fill(gen, shape, dt, how))
        arrays.append(array)
    torch.cuda.synchronize()                      # nor does that stream wait for torch's
    return {"thunk": _compiled[text], "args": arrays}


def run(state):
    out = state["thunk"](*state["args"])
    return [_view(o) for o in out] if isinstance(out, tuple) else _view(out)


# ----------------------------------------------------------------------------
# what a pass cannot do without, and how far another correct implementation may be
# ----------------------------------------------------------------------------
_SIZE = {"f32": 4, "f64": 8, "bf16": 2, "f8E4M3FN": 1}


def work(case):
    kind, e = case["kind"], _SIZE[case.get("dt", "bf16")]
    if kind == "loss":
        return {"bytes": 2.0 * e * case["n"], "flops": 3.0 * case["n"]}
    if kind == "stencil":
        cells = float(case["nx"]) * case["ny"] * case["nz"]
        full = (case["nx"] + 6.0) * (case["ny"] + 6) * (case["nz"] + 6)
        return {"bytes": e * (4 * cells + full), "flops": 30.0 * cells * case["steps"]}
    if kind == "gemm":
        m, n, k = float(case["m"]), case["n"], case["k"]
        return {"bytes": e * (m * k + k * n + 2 * m * n), "flops": 2 * m * n * k + 3 * m * n}
    if kind == "mlp":
        w = [case["w0"], case["w1"], case["w2"], case["w3"]]
        mats = sum(float(a) * b for a, b in zip(w, w[1:]))
        return {"bytes": e * (mats + sum(w[1:]) + case["batch"] * (w[0] + w[3])), "flops": 2.0 * case["batch"] * mats}
    if kind == "train":
        bt, w0, w1, w2 = float(case["batch"]), case["w0"], case["w1"], case["w2"]
        params = w0 * w1 + w1 + w1 * w2 + w2
        return {"bytes": e * (2 * params + bt * (w0 + w2)), "flops": 2 * bt * (2 * w0 * w1 + 3 * w1 * w2)}
    if kind == "fp8":
        bt, k, n = float(case["batch"]), case["k"], case["n"]
        return {"bytes": 2 * bt * k + k * n + 2 * bt * n, "flops": 2 * bt * k * n}
    N = importlib.import_module("reactant_jl_amd.nn_programs") if _package() else None
    _, shapes, flops = N.vgg11(batch=case["batch"], hw=case["hw"], dt=case["dt"])
    return {"bytes": e * (sum(float(math.prod(s)) for s in shapes) + case["batch"] * 1000), "flops": flops}


def tolerance(case):
    """About four times the distance from the same program in 64 bits (2-norm, as measured on the listed cases and
    others of their kinds): loss 1e-8 (f32) and 1e-16 (f64), stencil 4e-8 and 1e-16, vgg 1e-6 and 6e-3 (bf16), gemm 1e-6 and 1e-15, mlp and train 3e-7 to 7e-7 (f32) and
    2e-3 to 3e-3 (bf16), fp8 2e-3; sums of many terms in another order add their own rounding."""
    kind, dt = case["kind"], case.get("dt", "bf16")
    if dt == "bf16":
        return {"rel": 3e-2 if kind == "vgg" else 1e-2}
    if dt == "f64":
        return {"rel": 1e-14}
    return {"rel": {"loss": 1e-6, "stencil": 1e-6, "vgg": 1e-5}.get(kind, 5e-6)}
