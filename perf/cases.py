"""The work this library is used for, as cases a timing program can run.

A case is one problem C = epilogue(prologue(C) + A x B) and the way a program calls it:

  bound     accera_amd.GemmCall: a program that keeps its operands in place binds the call once and launches it again and again
  eager     accera_amd.gemm_relu: operands that change from call to call
  package   a HAT package's function on NumPy arrays, as a consumer of an Accera package calls it

listed() holds problems of the benchmark (bench.py), of the shape lists (accera_amd/shapes, the reference's sweep rows) and
a few generic ones; draw() gives more of the same ranges: general problems of 16 to 8192 rows and columns in every type,
layout and class of ops, decode and short-prefill problems against a large B, batches, and package functions.
"""
import functools
import math
import os
import tempfile

import numpy as np
import torch

import accera_amd as acc

_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8, "i32": torch.int32, "i16": torch.int16}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "i8": 1, "i32": 4, "i16": 2}
_SCALAR = {"f32": "float32", "f16": "float16", "bf16": "bfloat16", "i8": "int8", "i32": "int32", "i16": "int16"}
# classes of ops: (prologue, its operand, epilogue, its operand)
_OPS = {
    "set": (acc.PROLOGUE_SET0, 0.0, acc.EPILOGUE_NONE, 0.0),           # C = A x B
    "relu": (acc.PROLOGUE_SET0, 0.0, acc.EPILOGUE_RELU, 0.0),          # C = relu(A x B): the fused nest
    "accumulate": (acc.PROLOGUE_NONE, 0.0, acc.EPILOGUE_NONE, 0.0),    # C += A x B
    "blend": (acc.PROLOGUE_SCALE, 0.5, acc.EPILOGUE_RELU, 0.0),        # C = relu(beta C + A x B)
    "scale": (acc.PROLOGUE_SET0, 0.0, acc.EPILOGUE_SCALE, 0.125),      # C = alpha A x B
}
_READS_C = ("accumulate", "blend")


def _case(call, tin, tout, M, N, K, a="row", b="row", ops="relu", batch=1, name=None):
    c = {"call": call, "in": tin, "out": tout, "M": M, "N": N, "K": K, "a": a, "b": b, "ops": ops, "batch": batch}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the README's quick start: the smallest thing anybody runs, all launch latency
        _case("bound", "f32", "f32", 512, 512, 512, name="quickstart f32 512"),
        # a small layer of the reference's sweep lists, called with new operands each time: host work per call and latency
        _case("eager", "f16", "f16", 289, 896, 128, name="eager f16 289x896x128"),
        # the headline problem
        _case("bound", "f16", "f32", 4096, 4096, 4096, name="f16 4096"),
        # the largest: the int8 benchmark problem
        _case("bound", "i8", "i32", 8192, 8192, 8192, name="i8 8192"),
        # an FFN's forward product, weights as a framework keeps them (K contiguous)
        _case("bound", "bf16", "bf16", 4096, 3072, 768, b="col", name="ffn bf16 4096x3072x768"),
        # the same layer's weight gradient: A column-major, summed into the fp32 gradient of earlier micro-batches
        _case("bound", "bf16", "f32", 768, 3072, 4096, a="col", ops="accumulate", name="wgrad bf16 768x3072x4096"),
        # one decode step of eight sequences: a stream of B out of HBM
        _case("bound", "f16", "f16", 8, 11008, 4096, name="decode f16 8x11008x4096"),
        # prefill of a short prompt against a layer whose weights are far larger than the caches
        _case("bound", "f16", "f16", 128, 8192, 28672, b="col", ops="set", name="prefill f16 128x8192x28672"),
        # sizes that are multiples of nothing
        _case("bound", "f16", "f16", 1234, 5678, 4321, ops="set", name="ragged f16 1234x5678x4321"),
        # attention scores of 32 heads: Q x K^T, scaled
        _case("bound", "f16", "f16", 2048, 2048, 128, b="col", ops="scale", batch=32, name="scores f16 32x2048x2048x128"),
        # fp32 in earnest
        _case("bound", "f32", "f32", 2048, 2048, 2048, ops="set", name="f32 2048"),
        # the package boundary: NumPy arrays in, NumPy array out
        _case("package", "f16", "f32", 4096, 4096, 4096, name="package f16 4096"),
    ]


# ---- drawn cases --------------------------------------------------------------------------------------------------

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size between lo and hi: half of them a multiple of 64 (of 16 below 128), a quarter of 8, a quarter any number."""
    n, r = _log(rng, lo, hi), rng.random()
    step = (64 if n >= 128 else 16) if r < 0.5 else 8 if r < 0.75 else 1
    return max(lo, min(hi, n // step * step)) if n >= step else n


def _types(rng, package=False):
    tin = rng.choice(["f16", "f16", "bf16", "bf16", "i8", "f32"])
    out = {"f16": ["f16", "f32"], "bf16": ["bf16", "f32"], "i8": ["i32"], "f32": ["f32"]}[tin]
    return tin, rng.choice(out)


# operations a drawn problem of a type may have: none costs more than the largest listed problem
_MOST_FLOPS = {"f16": 4e11, "bf16": 4e11, "i8": 1e12, "f32": 5e10}


def draw(rng):
    family = rng.choice(["general", "general", "general", "decode", "prefill", "batch", "package"])
    tin, tout = _types(rng)
    a = "col" if rng.random() < 0.2 else "row"
    b = "col" if rng.random() < 0.5 else "row"
    ops = rng.choice(["set", "relu", "relu", "accumulate", "blend", "scale"])
    if family == "general":
        M, N, K = _size(rng, 16, 8192), _size(rng, 16, 8192), _size(rng, 32, 8192)
        while 2.0 * M * N * K > _MOST_FLOPS[tin]:
            K = max(32, K // 2 if K % 16 == 0 else K // 2 + 1)
            M = max(16, M // 2 if M % 16 == 0 else M // 2 + 1)
        return _case(rng.choice(["bound", "bound", "eager"]), tin, tout, M, N, K, a, b, ops)
    if family in ("decode", "prefill"):
        tin = rng.choice(["f16", "bf16", "i8"])
        tout = tin if tin != "i8" else "i32"
        M = rng.randint(1, 32) if family == "decode" else _log(rng, 33, 256)
        N, K = _log(rng, 2048, 65536) // 64 * 64, _log(rng, 1024, 32768) // 64 * 64
        if b == "col" and rng.random() < 0.3:
            N += rng.randint(1, 63)  # an odd vocabulary
        while N * K * _BYTES[tin] > 600e6:
            K = K // 128 * 64
        return _case("bound", tin, tout, M, N, K, "row", b, rng.choice(["set", "relu"]))
    if family == "batch":
        M, N, K = _size(rng, 16, 2048), _size(rng, 16, 2048), _size(rng, 32, 1024)
        batch = _log(rng, 4, 256)
        while batch > 4 and (batch * (M * K + K * N + M * N) * 4 > 400e6 or 2.0 * batch * M * N * K > _MOST_FLOPS[tin] / 4):
            batch = batch // 2
        return _case(rng.choice(["bound", "eager"]), tin, tout, M, N, K, "row", b, ops, max(batch, 4))
    # (a package's array is written by every call: C = A x B, with or without the ReLU)
    M, N, K = _size(rng, 64, 4096), _size(rng, 64, 4096), _size(rng, 64, 4096)
    return _case("package", tin, tout, M, N, K, "row", b, "relu" if ops == "relu" else "set")


# ---- running one ----------------------------------------------------------------------------------------------------

def _values(shape, t, std, g):
    if t == "i8":
        return torch.randint(-128, 128, shape, device="cuda", dtype=torch.int8, generator=g)
    if t in ("i32", "i16"):
        return torch.randint(-1000, 1001, shape, device="cuda", dtype=torch.int32, generator=g).to(_TORCH[t])
    x = torch.empty(shape, device="cuda", dtype=_TORCH[t])
    return x.normal_(0.0, std, generator=g)


def _matrix(rows, cols, batch, layout, t, std, g):
    lead = (batch,) if batch > 1 else ()
    if layout == "col":
        return _values(lead + (cols, rows), t, std, g).transpose(-1, -2)
    return _values(lead + (rows, cols), t, std, g)


@functools.lru_cache(maxsize=None)
def _package_function(tin, tout, M, N, K, b, ops):
    """The one function of a package built for this problem (what a program builds once and loads)."""
    L, T = acc.Array.Layout, acc.ScalarType
    A = acc.Array(role=acc.Role.INPUT, element_type=getattr(T, _SCALAR[tin]), shape=(M, K))
    B = acc.Array(role=acc.Role.INPUT, element_type=getattr(T, _SCALAR[tin]), shape=(K, N), layout=L.LAST_MAJOR if b == "col" else L.FIRST_MAJOR)
    C = acc.Array(role=acc.Role.INPUT_OUTPUT, element_type=getattr(T, _SCALAR[tout]), shape=(M, N))
    nest = acc.Nest(shape=(M, N, K))
    i, j, k = nest.get_indices()

    @nest.iteration_logic
    def _():
        C[i, j] += A[i, k] * B[k, j]

    plan = nest.create_schedule().create_plan(acc.Target(acc.Target.Model.AMD_MI355X))
    shape = acc.MMAShape.M16xN16xK64_B1 if tin == "i8" else acc.MMAShape.M32xN32xK2_B1 if tin == "f32" else acc.MMAShape.M16xN16xK32_B1
    plan.tensorize(indices=(i, j, k), mma_shape=shape, prologue_op=acc.MMAFragmentOp.SET, prologue_arg=0,
                   epilogue_op=acc.MMAFragmentOp.ReLU if ops == "relu" else acc.MMAFragmentOp.NONE)
    package = acc.Package()
    package.add(plan, args=(A, B, C), base_name="gemm")
    with tempfile.TemporaryDirectory() as where:
        package.build("gemm_package", format=acc.Package.Format.HAT_DYNAMIC, output_dir=where)
        _, functions = acc.hat.load(os.path.join(where, "gemm_package.hat"))
    return functions["gemm"]


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    tin, tout, M, N, K, batch = case["in"], case["out"], case["M"], case["N"], case["K"], case["batch"]
    # activations N(0, 1), weights scaled so that the sums are of order one; C holds earlier sums where it is read
    A = _matrix(M, K, batch, case["a"], tin, 1.0, g)
    B = _matrix(K, N, batch, case["b"], tin, K ** -0.5, g)
    C = _matrix(M, N, batch, "row", tout, 1.0, g)
    if case["call"] == "package":
        def host(t):
            x = t.view(torch.int16) if t.dtype == torch.bfloat16 else t  # (bfloat16 travels as 16-bit words)
            x = x.cpu().numpy()
            return x.view(np.uint16) if t.dtype == torch.bfloat16 else x
        B = host(B.t().contiguous()).T if case["b"] == "col" else host(B)
        return {"call": "package", "f": _package_function(tin, tout, M, N, K, case["b"], case["ops"]), "args": (host(A), B, host(C)), "bf16": tout == "bf16"}
    pro, pro_arg, epi, epi_arg = _OPS[case["ops"]]
    if tin == "i8":
        pro_arg, epi_arg = 2.0, 3.0  # (the operands of the ops are cast to the sums' type)
    ops = dict(prologue=pro, prologue_arg=pro_arg, epilogue=epi, epilogue_arg=epi_arg)
    if case["call"] == "bound":
        return {"call": "bound", "f": acc.GemmCall(A, B, C, **ops)}
    return {"call": "eager", "args": (A, B, C), "ops": ops}


def run(state):
    if state["call"] == "bound":
        return state["f"]()
    if state["call"] == "eager":
        return acc.gemm_relu(*state["args"], **state["ops"])
    state["f"](*state["args"])
    C = state["args"][2]
    return torch.from_numpy(C.view(np.int16)).view(torch.bfloat16) if state["bf16"] else C


def work(case):
    M, N, K, batch = case["M"], case["N"], case["K"], case["batch"]
    c = M * N * _BYTES[case["out"]] * (2 if case["ops"] in _READS_C else 1)
    return {"bytes": batch * ((M * K + K * N) * _BYTES[case["in"]] + c), "flops": 2.0 * batch * M * N * K}


def tolerance(case):
    """Integers are exact.  Against float64, the largest 2-norm error measured was 2.1e-4 for fp16 results and 1.7e-3 for bf16
    ones (their last rounding) and 8.1e-7 for fp32 ones (the order of the sums); about four times that."""
    if case["in"] == "i8":
        return "exact"
    return {"rel": {"f16": 8e-4, "bf16": 6.6e-3, "f32": 3.5e-6}[case["out"]]}
