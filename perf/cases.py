"""Performance cases of the offloaded hot path, through its public entry points.

Each case is one call as a user's program makes it: functions under ``njit``,
bodies under ``@kernel`` and the array functions of ``mlir.ops``, over device
arrays, in the default mode in which a call returns when its result is there.
Sizes are this repository's benchmark configurations, the presets and odd
shapes of its tests, and generic ones.

Array results come back as torch tensors over the framework's own device memory,
so that nothing is copied for the comparison.
"""

import math

import numpy as np
import torch

from numba_mlir_amd import kernel as kapi
from numba_mlir_amd.decorators import njit
from numba_mlir_amd.mlir import device_array as hip
from numba_mlir_amd.mlir import ops

get_global_id = kapi.get_global_id

RATE = np.float32(0.1)
VOLATILITY = np.float32(0.2)

_NUMPY = {"float32": np.float32, "float64": np.float64, "int32": np.int32,
          "int64": np.int64}


# -- device arrays and their torch views -------------------------------------

class _Exported:
    """A device array under the interface torch reads; keeps it alive."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {
            "data": (array.ptr, False), "shape": array.shape, "version": 2,
            "typestr": array.dtype.str, "strides": array.strides,
        }


def _tensor(array):
    return torch.as_tensor(_Exported(array), device="cuda")


def _empty(shape, dtype):
    return hip.empty(shape, _NUMPY[dtype])


def _array(values):
    """A device array holding a torch tensor's values."""
    out = _empty(tuple(values.shape), str(values.dtype).replace("torch.", ""))
    _tensor(out).copy_(values)
    return out


class _Random:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def uniform(self, low, high, shape, dtype):
        return torch.empty(shape, dtype=getattr(torch, dtype), device="cuda").uniform_(
            low, high, generator=self.g)

    def normal(self, shape, dtype):
        return torch.empty(shape, dtype=getattr(torch, dtype), device="cuda").normal_(
            generator=self.g)

    def integers(self, low, high, shape, dtype):
        return torch.randint(low, high + 1, shape, dtype=getattr(torch, dtype), device="cuda",
                             generator=self.g)

    def values(self, shape, dtype):
        """Data of an ordinary array: centred floats, integers up to 1000."""
        if dtype.startswith("int"):
            return self.integers(-1000, 1000, shape, dtype)
        return self.normal(shape, dtype)


# -- the user's functions -----------------------------------------------------

@njit
def _add(a, b):
    return a + b


@njit
def _scaled_add(a, b):
    return a * 2.0 + b


@njit
def _sum_rows(x):
    return np.sum(x, axis=1)


@njit
def _sum_columns(x):
    return np.sum(x, axis=0)


@njit
def _norm(x):
    return np.sqrt(np.sum(x * x))


@njit
def _dot(a, b, out):
    return np.dot(a, b, out)


@njit
def _black_scholes(price, strike, t, rate, volatility, call, put):
    mr = -rate
    sig_sig_two = volatility * volatility * 2
    P = price
    S = strike
    T = t
    a = np.log(P / S)
    b = T * mr
    z = T * sig_sig_two
    c = 0.25 * z
    y = 1.0 / np.sqrt(z)
    w1 = (a - b + c) * y
    w2 = (a - b - c) * y
    d1 = 0.5 + 0.5 * math.erf(w1)
    d2 = 0.5 + 0.5 * math.erf(w2)
    Se = np.exp(b) * S
    r = P * d1 - Se * d2
    call[:] = r
    put[:] = r - P + Se


@kapi.kernel
def _small_kernel(a, b, c, d, out1, out2):
    i = get_global_id(0)
    out1[i] = a[i] + b[i]
    out2[i] = c[i] - d[i]


@kapi.kernel
def _pairwise(X1, X2, D):
    i = get_global_id(0)
    j = get_global_id(1)
    d = 0.0
    for k in range(X1.shape[1]):
        tmp = X1[i, k] - X2[j, k]
        d += tmp * tmp
    D[i, j] = np.sqrt(d)


# -- the cases ------------------------------------------------------------------

def listed():
    return [
        # a kernel over eight elements with six array arguments: what a launch
        # costs (the benchmark's dispatch entry)
        {"name": "launch_8", "kind": "launch", "n": 8},
        # bias added to a batch: the benchmark's broadcast configuration
        {"name": "add_broadcast", "kind": "add", "rows": 4096, "cols": 4096,
         "dtype": "float64", "broadcast": True, "scale": False},
        # option pricing over a whole book: the benchmark's headline
        {"name": "black_scholes", "kind": "black_scholes", "n": 1 << 24, "fused": True},
        # the same formula as the user writes it under njit, an odd number of options
        {"name": "black_scholes_njit", "kind": "black_scholes", "n": 1000003, "fused": False},
        # row sums of a large matrix: the benchmark's first reduction
        {"name": "sum_rows", "kind": "sum", "rows": 16384, "cols": 8192, "axis": 1,
         "dtype": "float32"},
        # column totals of an integer table whose rows end anywhere
        {"name": "sum_columns_odd", "kind": "sum", "rows": 5003, "cols": 3001, "axis": 0,
         "dtype": "int32"},
        # the norm of an ordinary vector (a solver's stopping test)
        {"name": "norm_1m", "kind": "norm", "n": 1000000},
        # all distances of two point sets: the benchmark's @kernel configuration
        {"name": "pairwise", "kind": "pairwise", "n1": 8192, "n2": 8192, "dims": 3},
        # the benchmark's matrix product
        {"name": "dot_4096", "kind": "dot", "m": 4096, "n": 4096, "k": 4096,
         "dtype": "float32", "ta": False, "tb": False},
        # odd extents, the left operand given as a transposed view (X.T @ Y)
        {"name": "dot_odd_transposed", "kind": "dot", "m": 2047, "n": 2049, "k": 2051,
         "dtype": "float32", "ta": True, "tb": False},
        # the gemm benchmark's small and large double precision presets
        {"name": "dot_f64_small", "kind": "dot", "m": 1000, "n": 1100, "k": 1200,
         "dtype": "float64", "ta": False, "tb": False},
        {"name": "dot_f64_large", "kind": "dot", "m": 7000, "n": 7500, "k": 8000,
         "dtype": "float64", "ta": False, "tb": False},
    ]


def _spread(rng, low, high):
    """A whole number spread over the logarithm of [low, high]."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["launch", "add", "black_scholes", "sum", "norm", "pairwise", "dot",
                       "dot", "dot"])
    if kind == "launch":
        return {"kind": kind, "n": _spread(rng, 1, 10000)}
    if kind == "add":
        return {"kind": kind, "rows": _spread(rng, 16, 4096), "cols": _spread(rng, 16, 4096),
                "dtype": rng.choice(["float32", "float64", "int32", "int64"]),
                "broadcast": rng.random() < 0.5, "scale": rng.random() < 0.3}
    if kind == "black_scholes":
        return {"kind": kind, "n": _spread(rng, 1000, 1 << 24), "fused": rng.random() < 0.5}
    if kind == "sum":
        return {"kind": kind, "rows": _spread(rng, 16, 16384), "cols": _spread(rng, 16, 8192),
                "axis": rng.choice([0, 1]),
                "dtype": rng.choice(["float32", "float64", "int32", "int64"])}
    if kind == "norm":
        return {"kind": kind, "n": _spread(rng, 1000, 1 << 27)}
    if kind == "pairwise":
        return {"kind": kind, "n1": _spread(rng, 64, 8192), "n2": _spread(rng, 64, 8192),
                "dims": rng.choice([2, 3, 4])}
    case = {"kind": "dot", "dtype": rng.choice(["float32", "float64"]),
            "ta": rng.random() < 0.5, "tb": rng.random() < 0.5}
    if rng.random() < 0.2:                  # a matrix times a vector
        return dict(case, m=_spread(rng, 64, 16384), n=1, k=_spread(rng, 64, 16384), tb=False)
    return dict(case, m=_spread(rng, 64, 6000), n=_spread(rng, 64, 6000),
                k=_spread(rng, 64, 6000))


def prepare(case, seed):
    rnd, kind = _Random(seed), case["kind"]
    state = {"kind": kind}
    if kind == "launch":
        n = case["n"]
        arrays = [_array(rnd.integers(-1000, 1000, (n,), "int32")) for _ in range(4)]
        outs = [_array(torch.zeros(n, dtype=torch.int32, device="cuda")) for _ in range(2)]
        state.update(args=arrays + outs, n=n, out=[_tensor(o) for o in outs])
    elif kind == "add":
        rows, cols, dtype = case["rows"], case["cols"], case["dtype"]
        state.update(scale=case["scale"], a=_array(rnd.values((rows, cols), dtype)),
                     b=_array(rnd.values((1 if case["broadcast"] else rows, cols), dtype)))
    elif kind == "black_scholes":
        n = case["n"]
        args = [_array(rnd.uniform(low, high, (n,), "float32"))
                for low, high in ((10.0, 50.0), (10.0, 50.0), (1.0, 2.0))]
        outs = [_empty((n,), "float32") for _ in range(2)]
        state.update(args=args + [RATE, VOLATILITY] + outs, fused=case["fused"],
                     out=[_tensor(o) for o in outs])
    elif kind == "sum":
        state.update(x=_array(rnd.values((case["rows"], case["cols"]), case["dtype"])),
                     axis=case["axis"])
    elif kind == "norm":
        state.update(x=_array(rnd.normal((case["n"],), "float32")))
    elif kind == "pairwise":
        n1, n2, dims = case["n1"], case["n2"], case["dims"]
        out = _empty((n1, n2), "float64")
        state.update(args=[_array(rnd.uniform(0.0, 1.0, (n, dims), "float64"))
                           for n in (n1, n2)] + [out],
                     grid=(n1, n2), out=_tensor(out))
    else:
        m, n, k, dtype = case["m"], case["n"], case["k"], case["dtype"]
        a = _array(rnd.normal((k, m) if case["ta"] else (m, k), dtype))
        b = _array(rnd.normal((n, k) if case["tb"] else (k, n), dtype))
        out = _empty((m, n), dtype)
        state.update(args=[a.T if case["ta"] else a, b.T if case["tb"] else b, out],
                     out=_tensor(out))
    torch.cuda.synchronize()
    return state


def run(state):
    kind = state["kind"]
    if kind == "launch":
        _small_kernel[state["n"], kapi.DEFAULT_LOCAL_SIZE](*state["args"])
        return state["out"]
    if kind == "add":
        return _tensor((_scaled_add if state["scale"] else _add)(state["a"], state["b"]))
    if kind == "black_scholes":
        (ops.black_scholes if state["fused"] else _black_scholes)(*state["args"])
        return state["out"]
    if kind == "sum":
        return _tensor((_sum_columns if state["axis"] == 0 else _sum_rows)(state["x"]))
    if kind == "norm":
        return _norm(state["x"])
    if kind == "pairwise":
        _pairwise[state["grid"], kapi.DEFAULT_LOCAL_SIZE](*state["args"])
        return state["out"]
    _dot(*state["args"])
    return state["out"]


def work(case):
    kind = case["kind"]
    size = np.dtype(_NUMPY[case.get("dtype", "float32")]).itemsize
    if kind == "launch":
        return {"bytes": 24 * case["n"], "flops": 2 * case["n"]}
    if kind == "add":
        full = case["rows"] * case["cols"]
        return {"bytes": size * (2 * full + (case["cols"] if case["broadcast"] else full)),
                "flops": full}
    if kind == "black_scholes":
        return {"bytes": 20 * case["n"], "flops": 60 * case["n"]}
    if kind == "sum":
        kept = case["cols"] if case["axis"] == 0 else case["rows"]
        result = 8 if case["dtype"].startswith("int") else size
        full = case["rows"] * case["cols"]
        return {"bytes": size * full + result * kept, "flops": full}
    if kind == "norm":
        return {"bytes": 4 * case["n"] + 4, "flops": 2 * case["n"]}
    if kind == "pairwise":
        n1, n2, dims = case["n1"], case["n2"], case["dims"]
        return {"bytes": 8 * (n1 * n2 + dims * (n1 + n2)), "flops": n1 * n2 * (3 * dims + 1)}
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": size * (m * k + k * n + m * n), "flops": 2 * m * n * k}


def tolerance(case):
    """About four times what the present kernels differ by from the same work in
    float64 (float64 products: from sums over pieces of K).  The error of a
    product of centred values grows with the root of the number of terms:
    1.15e-6 at k = 4096 in float32, 3.1e-15 at k = 8000 in float64."""
    kind, dtype = case["kind"], case.get("dtype", "float32")
    if kind in ("launch", "add") or dtype.startswith("int"):
        return "exact"
    if kind == "black_scholes":         # 8.2e-8, 4.2e-7
        return {"rel": 4e-7, "max": 2e-6}
    if kind == "pairwise":              # the same bits; one place of sum or root
        return {"rel": 4e-16, "max": 1e-15}
    if kind == "norm":                  # 4.8e-8
        return {"rel": 2e-7}
    if kind == "sum":                   # 1.0e-7, 2.7e-16
        return {"rel": 4e-7 if dtype == "float32" else 1e-15}
    root = math.sqrt(case["k"])
    return {"rel": max(1e-6, 7e-8 * root) if dtype == "float32" else
            max(2e-15, 1.4e-16 * root)}
