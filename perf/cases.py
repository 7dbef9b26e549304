"""The work that a program using this backend spends its time in, as cases to measure.

Every case calls a public entry point the way a user's program does: the C ABI
(trs_backend.abi, the functions of include/trs_hip.h) for single ops and fused
programs, and torch_rs for training steps.  Sizes are those of the repository's
benchmark configurations and tests, or generic ones around them, odd and ragged
ones included.

  kind          what it stands for
  bias_relu     relu(x + b), a row-broadcast bias and activation, one fused program
  chain         relu(exp(x*y + z) - 1) over flat tensors, one fused program
  permuted      (a + b) * c.mT, broadcast and transposed operands, one fused program
  bias_grad     the gradient of a row-broadcast operand: rows summed in order
  linear        x @ W or x @ W.mT with 1 to 32 rows: a decode step, a small batch
  matmul        one product, square or not, plain or transposed operands
  bmm           a batch of products
  mlp           a two-layer MLP training step: forward, dropout, backward through autograd
"""
import ctypes
import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "pytorch-rs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from trs_backend import abi  # noqa: E402
from trs_backend.abi import check, layout_of  # noqa: E402

_KEEP = 0.9  # dropout keep probability of the training steps
_SCALE = 1 / 0.9


def listed():
    return [
        # A small activation, where the call itself is the cost.
        {"name": "bias_relu_small", "kind": "bias_relu", "rows": 32, "cols": 1000},
        # Activations of a batch: the benchmark's rows x cols, and rows of odd length.
        {"name": "bias_relu", "kind": "bias_relu", "rows": 4096, "cols": 4096},
        # The benchmark's fused chain at its full 2^28 elements (4 GiB moved).
        {"name": "chain", "kind": "chain", "n": 1 << 28},
        # The benchmark's broadcast + transposed view, at sizes no tile divides.
        {"name": "permuted_ragged", "kind": "permuted", "batch": 60, "rows": 500, "cols": 1001},
        # Backward of the bias: a layer of odd width.
        {"name": "bias_grad", "kind": "bias_grad", "rows": 8192, "cols": 1000},
        # A small batch through a linear layer (inference).
        {"name": "linear_8", "kind": "linear", "rows": 8, "k": 4096, "n": 4096, "wt": False},
        # A prefill-sized batch through the same layer.
        {"name": "matmul_512", "kind": "matmul", "m": 512, "k": 4096, "n": 4096, "ta": False, "tb": False},
        # Ragged in every dim, with the weight stored as its transpose.
        {"name": "matmul_ragged", "kind": "matmul", "m": 1000, "k": 2047, "n": 1500, "ta": False, "tb": True},
        # The benchmark's square product.
        {"name": "matmul_4096", "kind": "matmul", "m": 4096, "k": 4096, "n": 4096, "ta": False, "tb": False},
        # The benchmark's batch of products.
        {"name": "bmm", "kind": "bmm", "batch": 32, "m": 512, "k": 512, "n": 512, "tb": False},
        # The benchmark's training step, and a small ragged one.
        {"name": "mlp", "kind": "mlp", "rows": 8192, "d": 4096, "h": 4096, "o": 1024},
        {"name": "mlp_small", "kind": "mlp", "rows": 300, "d": 784, "h": 500, "o": 100},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, even over its logarithm; half of them multiples of 32 where that fits."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and n >= 64:
        n = n // 32 * 32
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(("bias_relu", "chain", "permuted", "bias_grad", "linear", "matmul", "matmul", "bmm", "mlp"))
    if kind == "bias_relu":
        return {"kind": kind, "rows": _size(rng, 16, 8192), "cols": _size(rng, 32, 8192)}
    if kind == "chain":
        return {"kind": kind, "n": int(math.exp(rng.uniform(math.log(1 << 12), math.log(1 << 28))))}
    if kind == "permuted":
        return {"kind": kind, "batch": _size(rng, 1, 64), "rows": _size(rng, 64, 1024), "cols": _size(rng, 64, 1024)}
    if kind == "bias_grad":
        return {"kind": kind, "rows": _size(rng, 64, 8192), "cols": _size(rng, 64, 4096)}
    if kind == "linear":
        return {"kind": kind, "rows": rng.choice((1, 2, 3, 5, 8, 13, 16, 24, 32)), "k": _size(rng, 512, 8192),
                "n": _size(rng, 512, 8192), "wt": rng.random() < 0.5}
    if kind == "matmul":
        return {"kind": kind, "m": _size(rng, 64, 6144), "k": _size(rng, 64, 6144), "n": _size(rng, 64, 6144),
                "ta": rng.random() < 0.3, "tb": rng.random() < 0.4}
    if kind == "bmm":
        return {"kind": kind, "batch": _size(rng, 2, 64), "m": _size(rng, 48, 768), "k": _size(rng, 48, 768),
                "n": _size(rng, 48, 768), "tb": rng.random() < 0.4}
    return {"kind": kind, "rows": _size(rng, 64, 4096), "d": _size(rng, 128, 2048), "h": _size(rng, 128, 2048),
            "o": _size(rng, 32, 1024)}


# ---- inputs -----------------------------------------------------------------

def _inputs(case, seed):
    """The case's operands as torch tensors on the GPU, made from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device="cuda").mul_(std)

    def uniform(lim, *shape):
        return torch.rand(*shape, generator=g, device="cuda").mul_(2 * lim).sub_(lim)

    kind = case["kind"]
    if kind == "bias_relu":
        return normal(case["rows"], case["cols"]), normal(case["cols"])
    if kind == "chain":
        return tuple(uniform(4.0, case["n"]) for _ in range(3))
    if kind == "permuted":
        b, m, n = case["batch"], case["rows"], case["cols"]
        return normal(b, 1, n), normal(1, m, n), normal(b, n, m)
    if kind == "bias_grad":
        return (normal(case["rows"], case["cols"]),)
    if kind == "linear":
        w = (case["n"], case["k"]) if case["wt"] else (case["k"], case["n"])
        return normal(case["rows"], case["k"]), uniform(1 / math.sqrt(case["k"]), *w)
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        std = 1 / math.sqrt(k)
        return normal(*((k, m) if case["ta"] else (m, k)), std=std), normal(*((n, k) if case["tb"] else (k, n)), std=std)
    if kind == "bmm":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        std = 1 / math.sqrt(k)
        return normal(b, m, k, std=std), normal(*((b, n, k) if case["tb"] else (b, k, n)), std=std)
    r, d, h, o = case["rows"], case["d"], case["h"], case["o"]
    mask = (torch.rand(r, h, generator=g, device="cuda") < _KEEP).to(torch.uint8)
    return normal(r, d), uniform(1 / math.sqrt(d), d, h), uniform(1 / math.sqrt(h), h, o), mask


# ---- calls ------------------------------------------------------------------

def _fused(ir, devs, lays, out, lo):
    """A fused launch: the program compiled, its argument arrays laid out once."""
    kid = ctypes.c_uint64()
    check(abi.lib.trs_fusion_compile(ir.encode(), len(ir), ctypes.byref(kid)))
    n = len(devs)
    args = (kid.value, n, (ctypes.c_void_p * n)(*[t.data_ptr() for t in devs]), (abi.Layout * n)(*lays),
            ctypes.c_void_p(out.data_ptr()), ctypes.byref(lo))
    return {"fn": abi.lib.trs_fusion_launch, "args": args, "out": out, "keep": (devs, lays, lo)}


def _product(a, la, b, lb, out, lo):
    args = (ctypes.c_void_p(a.data_ptr()), ctypes.byref(la), ctypes.c_void_p(b.data_ptr()), ctypes.byref(lb),
            ctypes.c_void_p(out.data_ptr()), ctypes.byref(lo))
    return {"fn": abi.lib.trs_matmul_f32, "args": args, "out": out, "keep": (a, la, b, lb, lo)}


def _matrix(rows, cols, transposed, batch=0):
    """The layout of a rows x cols matrix (or a batch of them), stored as its transpose or not."""
    st = (1, rows) if transposed else (cols, 1)
    return layout_of((batch, rows, cols), (rows * cols,) + st) if batch else layout_of((rows, cols), st)


class _Device:
    """A torch_rs tensor as torch sees it: the same memory, no copy."""

    def __init__(self, t):
        self.keep = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": "<f4", "data": (t.data_ptr(), False),
                                         "strides": None, "version": 2}


def _as_torch(t):
    return torch.as_tensor(_Device(t), device="cuda")


def prepare(case, seed):
    check(abi.lib.trs_init())
    ins = _inputs(case, seed)
    kind = case["kind"]
    if kind == "mlp":
        return _prepare_mlp(ins)

    def empty(*shape):
        return torch.empty(*shape, device="cuda")

    if kind == "bias_relu":
        x, b = ins
        lx, lb = layout_of(x.shape), layout_of(b.shape)
        # relu(x + b) as torch_rs.fuse writes it: the broadcast operand first.
        return _fused("in f32\nin f32\nadd %1 %0\nrelu %2\nout %3\n", [b, x], [lb, lx], torch.empty_like(x), lx)
    if kind == "chain":
        lay = layout_of((case["n"],))
        ir = "in f32\nin f32\nin f32\nmul %0 %1\nadd %3 %2\nexp %4\nconst 0x3f800000\nsub %5 %6\nrelu %7\nout %8\n"
        return _fused(ir, list(ins), [lay] * 3, empty(case["n"]), lay)
    if kind == "permuted":
        a, b, c = ins
        nb, m, n = case["batch"], case["rows"], case["cols"]
        lo = layout_of((nb, m, n))
        return _fused("in f32\nin f32\nin f32\nadd %0 %1\nmul %3 %2\nout %4\n", [a, b, c],
                      [layout_of((nb, 1, n)), layout_of((1, m, n)), _matrix(m, n, True, nb)], empty(nb, m, n), lo)
    if kind == "bias_grad":
        up, = ins
        lu, ls, out = layout_of(up.shape), layout_of((case["cols"],)), empty(case["cols"])
        args = (ctypes.c_void_p(up.data_ptr()), ctypes.byref(lu), ctypes.byref(ls), ctypes.c_void_p(out.data_ptr()))
        return {"fn": abi.lib.trs_reduce_to_shape_f32, "args": args, "out": out, "keep": (up, lu, ls)}
    a, b = ins
    if kind == "linear":
        r, k, n = case["rows"], case["k"], case["n"]
        return _product(a, _matrix(r, k, False), b, _matrix(k, n, case["wt"]), empty(r, n), layout_of((r, n)))
    m, k, n = case["m"], case["k"], case["n"]
    if kind == "matmul":
        return _product(a, _matrix(m, k, case["ta"]), b, _matrix(k, n, case["tb"]), empty(m, n), layout_of((m, n)))
    nb = case["batch"]
    return _product(a, _matrix(m, k, False, nb), b, _matrix(k, n, case["tb"], nb), empty(nb, m, n), layout_of((nb, m, n)))


def _prepare_mlp(ins):
    import torch_rs

    x, w1, w2, mask = (t.cpu().numpy() for t in ins)
    X, W1, W2 = (torch_rs.tensor(t, device="cuda") for t in (x, w1, w2))
    return {"X": X, "W1": W1, "W2": W2, "mask": torch_rs.nn.functional.keep_mask(mask),
            "b1": torch_rs.zeros(w1.shape[1], device="cuda"), "b2": torch_rs.zeros(w2.shape[1], device="cuda"),
            "act": torch_rs.fuse(lambda z, b, m: ((z + b).relu() * m) * _SCALE)}


def run(state):
    fn = state.get("fn")
    if fn is not None:
        check(fn(*state["args"]))
        return state["out"]
    # A training step: fresh leaves, so that the gradients are the step's own.
    x, w1, w2 = (state[n].with_requires_grad(True) for n in ("X", "W1", "W2"))
    out = state["act"](x @ w1, state["b1"], state["mask"]) @ w2 + state["b2"]
    out.sum().backward()
    return {"out": _as_torch(out.detach()), "dX": _as_torch(x.grad), "dW1": _as_torch(w1.grad), "dW2": _as_torch(w2.grad)}


# ---- what a pass cannot do without, and how exact it is -----------------------

def work(case):
    kind = case["kind"]
    if kind == "bias_relu":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * (2 * n + case["cols"]), "flops": 2 * n}
    if kind == "chain":
        return {"bytes": 16 * case["n"], "flops": 5 * case["n"]}
    if kind == "permuted":
        b, m, n = case["batch"], case["rows"], case["cols"]
        return {"bytes": 4 * (b * n + m * n + 2 * b * m * n), "flops": 2 * b * m * n}
    if kind == "bias_grad":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * (n + case["cols"]), "flops": n}
    if kind == "mlp":
        r, d, h, o = case["rows"], case["d"], case["h"], case["o"]
        return {"bytes": 4 * (2 * r * d + 2 * d * h + 2 * h * o + r * o) + r * h, "flops": 6 * r * h * (d + o)}
    nb = case.get("batch", 1)
    m = case["rows"] if kind == "linear" else case["m"]
    k, n = case["k"], case["n"]
    return {"bytes": 4 * nb * (m * k + k * n + m * n), "flops": 2 * nb * m * k * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("bias_relu", "permuted"):
        return "exact"  # one rounding per op, in the written order
    if kind == "chain":
        return {"rel": 1e-6, "max": 1e-5}  # exp within 2 ulp
    if kind == "bias_grad":
        return {"rel": 4e-6, "max": 4e-5}  # up to 8192 additions in 32 bits
    if kind == "mlp":
        # relu's mask flips where z is within a rounding of zero: a share f of
        # the elements flipped moves the gradients by about sqrt(f).
        return {"rel": 4e-3, "max": 0.9}
    return {"rel": 4e-6, "max": 4e-5}  # 32-bit sums of up to 8192 products


def exact(case, seed):
    ins = _inputs(case, seed)
    kind = case["kind"]
    d = [t.double() for t in ins]
    if kind == "bias_relu":
        return (d[0] + d[1]).relu()
    if kind == "chain":
        return d[0].mul_(d[1]).add_(d[2]).exp_().sub_(1.0).relu_()
    if kind == "permuted":
        return (d[0] + d[1]) * d[2].transpose(1, 2)
    if kind == "bias_grad":
        return d[0].sum(0)
    if kind == "linear":
        return d[0] @ (d[1].t().contiguous() if case["wt"] else d[1])
    if kind == "matmul":
        a = d[0].t().contiguous() if case["ta"] else d[0]
        return a @ (d[1].t().contiguous() if case["tb"] else d[1])
    if kind == "bmm":
        return torch.bmm(d[0], d[1].transpose(1, 2).contiguous() if case["tb"] else d[1])
    x, w1, w2, mask = d
    scale = float(torch.tensor(_SCALE, dtype=torch.float32))
    z = x @ w1
    keep = mask * scale
    h = z.relu() * keep
    up = torch.ones(x.shape[0], w2.shape[1], dtype=torch.float64, device="cuda")
    dz = (up @ w2.t().contiguous()) * keep * (z > 0)
    return {"out": h @ w2, "dX": dz @ w1.t().contiguous(), "dW1": x.t().contiguous() @ dz, "dW2": h.t().contiguous() @ up}
