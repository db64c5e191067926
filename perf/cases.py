"""The work whose speed counts: what a program does with this library, from one fragment to 8192^3.

A case is a dict of plain values.  `path` names the entry point (`GEMM.gemm`, `GEMM.gemm_splitk`, or the
fragment operations of `WMMA` one by one); the other keys are what a caller writes into the descriptor.
Inputs live in HBM before the call, as they do in a program that chains such products; device memory,
streams and synchronisation are torch's, the library gets raw addresses.

    listed()              the cases that stand for the ranges
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   inputs and descriptor, on the GPU
    run(state)            one pass through the public entry points; returns D
    work(case)            bytes and operations that one pass cannot do without
    tolerance(case)       how far another correct implementation may be off
    exact(case, seed)     what D would be in 64 bits, from the same inputs
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

LARGEST_FLOPS = 2.0 * 8192 ** 3
LARGEST_BYTES = 8192 * 8192 * (2 + 2 + 4 + 4)

_module = None


def _package():
    global _module
    if _module is None:
        _module = load_package()
        _module.init(0)
    return _module


def _gemm(name, m, n, k, **more):
    case = dict(name=name, path="gemm", m=m, n=n, k=k, batch=1, a="col", b="col", d="col", c="f32", out="f32", acc="f32",
                alpha=1.0, beta=1.0, values="uniform")
    case.update(more)
    return case


def listed():
    return [
        # The reference's own example (one warp, one 16x16x16 tile) written with load_a, load_b, load_c, mma
        # and store_d, as the test suite and every first program with this library have it.
        dict(name="fragment", path="fragment", a="col", b="col", d="col", c="f32", out="f32", space="global"),
        # A small product of odd extents, where the launch counts as much as the arithmetic.
        _gemm("small_720x656x784", 720, 656, 784),
        # One decoding step of a projection: 16 sequences, activations row-major, weights stored N x K,
        # Float16 result, nothing to add.  Bound by reading the weights.
        _gemm("decode_16", 16, 4096, 4096, a="row", d="row", c="none", out="f16", values="weights"),
        # The same with 128 sequences in the batch, or a short prefill.
        _gemm("decode_128", 128, 4096, 4096, a="row", d="row", c="none", out="f16", values="weights"),
        # Forward pass of a projection over 8192 tokens (the benchmark's mixed-layout configuration).
        _gemm("forward_8192x1024x4096", 8192, 1024, 4096, a="row", values="weights"),
        # Its backward pass to the input, over a packed batch whose token count no tile divides.
        _gemm("dgrad_4144x4096x4096", 4144, 4096, 4096, a="row", b="row", d="row", c="none", out="f16", values="weights"),
        # Backward pass to the weights of a narrow layer: few output tiles, a long sum over tokens, added to
        # the Float32 gradient; the program keeps the workspace.
        _gemm("wgrad_512x512x16384", 512, 512, 16384, path="splitk", a="col", b="row", d="row"),
        # The headline benchmark.
        _gemm("square_4096", 4096, 4096, 4096),
        # Everything Float16, the running sum too.
        _gemm("f16acc_2048", 2048, 2048, 2048, c="f16", out="f16", acc="f16", values="half"),
        # Many small problems in one call.
        _gemm("batched_512x128", 128, 128, 128, batch=512),
        # The trailing update of a blocked factorisation: C and D far larger than the operands, alpha = -1.
        _gemm("update_8192x8192x1024", 8192, 8192, 1024, b="row", alpha=-1.0),
        # The largest.
        _gemm("square_8192", 8192, 8192, 8192),
    ]


def _size(rng, low, high):
    """A multiple of 16, spread over the logarithm of the range; half of them multiples of 64 or more."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    step = rng.choice((16, 16, 64, 128))
    return max(low, min(high, int(round(v / step)) * step))


def _draw(rng):
    side = lambda: rng.choice(("row", "col"))  # noqa: E731
    kind = rng.choice(("fragment", "small", "small", "decode", "decode", "layer", "layer", "wgrad", "half", "batched", "update", "square"))
    if kind == "fragment":
        return dict(path="fragment", a=side(), b=side(), d=side(), c=rng.choice(("f16", "f32")), out=rng.choice(("f16", "f32")),
                    space=rng.choice(("generic", "global", "shared")))
    if kind == "small":
        return _gemm("", _size(rng, 400, 1280), _size(rng, 400, 1280), _size(rng, 400, 1280), a=side(), b=side(), d=side(),
                     c=rng.choice(("none", "f16", "f32")), out=rng.choice(("f16", "f32")))
    if kind == "decode":
        return _gemm("", 16 * rng.randint(1, 8), _size(rng, 2048, 8192), _size(rng, 2048, 8192), a="row", d="row",
                     c=rng.choice(("none", "none", "f16")), out=rng.choice(("f16", "f16", "f32")), values="weights")
    if kind == "layer":  # forward and both backward products of one layer
        form = rng.choice((dict(a="row"), dict(a="row", b="row"), dict(a="col", b="row")))
        return _gemm("", _size(rng, 512, 8192), _size(rng, 512, 8192), _size(rng, 512, 8192), d="row",
                     c=rng.choice(("none", "f16", "f32")), out=rng.choice(("f16", "f32")), values="weights", **form)
    if kind == "wgrad":
        return _gemm("", _size(rng, 128, 1024), _size(rng, 128, 1024), 128 * rng.randint(32, 256), path="splitk", a="col", b="row",
                     d="row", c=rng.choice(("none", "f32")), values="weights")
    if kind == "half":
        return _gemm("", _size(rng, 256, 4096), _size(rng, 256, 4096), _size(rng, 256, 4096), a=side(), b=side(), c="f16", out="f16",
                     acc="f16", values="half")
    if kind == "batched":
        return _gemm("", _size(rng, 64, 256), _size(rng, 64, 256), _size(rng, 64, 256), batch=rng.randint(64, 512), a=side(), b=side(),
                     c=rng.choice(("none", "f32")), out=rng.choice(("f16", "f32")))
    if kind == "update":
        return _gemm("", _size(rng, 1024, 8192), _size(rng, 1024, 8192), _size(rng, 16, 1024), b="row",
                     alpha=rng.choice((-1.0, 1.0, 0.5)), beta=rng.choice((1.0, 1.0, 0.5)))
    return _gemm("", _size(rng, 1024, 6144), _size(rng, 1024, 6144), _size(rng, 1024, 6144), a=side(), b=side(),
                 c=rng.choice(("none", "f32")))


def draw(rng):
    while True:
        case = _draw(rng)
        case.pop("name", None)
        w = work(case)
        if w["flops"] <= LARGEST_FLOPS and w["bytes"] <= LARGEST_BYTES:
            return case


_TORCH = {"f16": torch.float16, "f32": torch.float32}
_NUMPY = {"f16": np.float16, "f32": np.float32}


def _matrix(gen, case, rows, cols, order, dtype, scale):
    """`batch` matrices, each stored row- or column-major without padding, values as the case's use has them."""
    shape = (case.get("batch", 1), rows, cols) if order == "row" else (case.get("batch", 1), cols, rows)
    x = torch.empty(shape, dtype=torch.float32, device="cuda")
    if scale < 0:
        x.normal_(0.0, -scale, generator=gen)
    else:
        x.uniform_(-scale, scale, generator=gen)
    return x.to(dtype)


def prepare(case, seed):
    pkg = _package()
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    W, G = pkg.WMMA, pkg.GEMM
    order = {"row": W.RowMajor, "col": W.ColMajor}
    if case["path"] == "fragment":
        A = _matrix(gen, case, 16, 16, case["a"], torch.float16, 1.0)
        B = _matrix(gen, case, 16, 16, case["b"], torch.float16, 1.0)
        C = _matrix(gen, case, 16, 16, case["d"], _TORCH[case["c"]], 1.0)
        D = torch.empty((16, 16), dtype=_TORCH[case["out"]], device="cuda")
        space = {"generic": pkg.AS.Generic, "global": pkg.AS.Global, "shared": pkg.AS.Shared}[case["space"]]
        pointer = lambda x, t: pkg.DevicePtr(t, x.data_ptr(), space, x)  # noqa: E731
        return dict(path="fragment", W=W, D=D, a=pointer(A, np.float16), b=pointer(B, np.float16), c=pointer(C, _NUMPY[case["c"]]),
                    d=pointer(D, _NUMPY[case["out"]]), la=order[case["a"]], lb=order[case["b"]], ld=order[case["d"]],
                    config=W.Config(16, 16, 16, _NUMPY[case["out"]]))
    m, n, k = case["m"], case["n"], case["k"]
    # uniform: the benchmark's operands; half: small enough for a Float16 running sum; weights: activations
    # (or their gradients) of unit variance times weights of standard deviation 0.02
    sa, sb, sc = {"uniform": (1.0, 1.0, 1.0), "half": (0.5, 0.5, 0.1), "weights": (-1.0, -0.02, -1.0)}[case["values"]]
    A = _matrix(gen, case, m, k, case["a"], torch.float16, sa)
    B = _matrix(gen, case, k, n, case["b"], torch.float16, sb)
    C = None if case["c"] == "none" else _matrix(gen, case, m, n, case["d"], _TORCH[case["c"]], sc)
    shape = (case["batch"], m, n) if case["d"] == "row" else (case["batch"], n, m)
    D = torch.empty(shape, dtype=_TORCH[case["out"]], device="cuda")
    desc = G.make_desc(m, n, k, a_layout=order[case["a"]], b_layout=order[case["b"]], c_layout=order[case["d"]],
                       d_layout=order[case["d"]], c_type=_NUMPY["f32" if C is None else case["c"]], d_type=_NUMPY[case["out"]],
                       acc_type=_NUMPY[case["acc"]], alpha=case["alpha"], beta=case["beta"], use_c=C is not None,
                       batch=case["batch"])
    state = dict(path=case["path"], G=G, desc=desc, A=A, B=B, C=C, D=D,
                 addresses=(A.data_ptr(), B.data_ptr(), None if C is None else C.data_ptr(), D.data_ptr()))
    if case["path"] == "splitk":
        state["workspace"] = pkg.DeviceArray.undef(np.float32, max(4, G.splitk_workspace(desc)[1] // 4))
    return state


def run(state):
    if state["path"] == "fragment":
        W, config = state["W"], state["config"]
        a = W.load_a(state["a"], 16, state["la"], config)
        b = W.load_b(state["b"], 16, state["lb"], config)
        c = W.load_c(state["c"], 16, state["ld"], config)
        W.store_d(state["d"], W.mma(a, b, c, config), 16, state["ld"], config)
    elif state["path"] == "splitk":
        state["G"].gemm_splitk(*state["addresses"], state["desc"], workspace=state["workspace"])
    else:
        state["G"].gemm(*state["addresses"], state["desc"])
    return state["D"]


def exact(case, seed):
    """alpha*A*B + beta*C in 64 bits, laid out as D; every case takes well under a second on the GPU."""
    if case["path"] == "fragment":
        gen = torch.Generator(device="cuda").manual_seed(int(seed))
        A, B, C = (_matrix(gen, case, 16, 16, case[x], t, 1.0)
                   for x, t in (("a", torch.float16), ("b", torch.float16), ("d", _TORCH[case["c"]])))
        D = torch.empty((16, 16), device="cuda")
        alpha = beta = 1.0
    else:
        state = prepare(case, seed)
        A, B, C, D = (state[x] for x in "ABCD")
        alpha, beta = case["alpha"], case["beta"]
    wide = lambda x, order: (x if order == "row" else x.transpose(1, 2)).double().contiguous()  # noqa: E731
    P = alpha * torch.bmm(wide(A, case["a"]), wide(B, case["b"]))
    if C is not None:
        P += beta * wide(C, case["d"])
    return (P if case["d"] == "row" else P.transpose(1, 2).contiguous()).reshape(D.shape)


def work(case):
    size = {"none": 0, "f16": 2, "f32": 4}
    m, n, k = (case.get(x, 16) for x in "mnk")
    batch = case.get("batch", 1)
    return {"bytes": batch * (2 * (m * k + k * n) + m * n * (size[case["c"]] + size[case["out"]])), "flops": 2.0 * batch * m * n * k}


def tolerance(case):
    # Four times the largest distance to the same product in float64, over the listed and four dozen drawn
    # cases.  Float32 results: rel 7.7e-7, max 5.2e-6.  Float16 results: rel 2.2e-4, max 4.9e-4
    # (half a unit in the last place).  Float16 running sums: rel 9.8e-4, max 6.3e-3, growing with the
    # square root of the number of roundings.
    if case.get("acc") == "f16":
        return {"rel": 5e-3, "max": 3e-2}
    if case["out"] == "f16":
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 3e-6, "max": 2e-5}
