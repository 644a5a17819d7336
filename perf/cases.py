"""Workloads of the library, as programs that use it call them: iterative sparse products on kept handles, graph
products and triangle counts on R-MAT graphs, dense tensor contractions, and the memref entry points that compiled
programs bind to.  Sizes are those of the benchmark and the tests, and the range between them.

A case names its operation (`op`) and its sizes; everything else is made from the seed."""
import functools
import math

import numpy as np
import torch

from comet_amd import runtime as rt

RMAT = (0.57, 0.19, 0.19)            # quadrant probabilities a, b, c of the graphs
MEAN_ROW, CAP_ROW = 16.0, 4096       # power-law matrices: mean and longest row


def listed():
    return [
        # one step of a two-sided solver (biconjugate gradients: A x and y A) on a small system: the calls are all latency
        {"name": "spmv_small", "op": "spmv", "n": 2_500, "mean": 5.0, "both_sides": True},
        # a product with a system whose vectors do not fit an L2
        {"name": "spmv_large", "op": "spmv", "n": 1_000_000, "mean": 10.0, "both_sides": False},
        # a power-law matrix times a block of vectors of an odd width (graph features, block eigensolvers)
        {"name": "spmm_odd_width", "op": "spmm", "n": 60_001, "width": 33},
        # the headline product
        {"name": "spmm_large", "op": "spmm", "n": 500_000, "width": 64},
        # shortest paths of two steps on a small graph
        {"name": "spgemm_small_min_plus", "op": "spgemm", "n": 1_024, "edge_factor": 8, "reduce": "min", "mult": "plus"},
        # the square of an adjacency matrix, materialised (output sizes in the gigabytes)
        {"name": "spgemm_large", "op": "spgemm", "n": 65_536, "edge_factor": 16, "reduce": "plus", "mult": "times"},
        # common neighbours of every edge, in one call
        {"name": "spgemm_masked", "op": "spgemm_masked", "n": 200_003, "edge_factor": 16},
        # triangles of the benchmark's graph
        {"name": "tricount_large", "op": "tricount", "n": 1 << 20, "edge_factor": 16},
        # a coupled-cluster term as a program runs it once: few outputs, a long sum, the plan made in the call
        {"name": "ttgt_ccsd_t1", "op": "ttgt", "expr": "icmn,mnca->ia", "extents": "i=30,c=61,m=30,n=30,a=61",
         "keep_plan": False},
        # the benchmark's contraction, its plan kept between calls
        {"name": "ttgt_large", "op": "ttgt", "expr": "aebf,dfce->abcd", "extents": "a=64,e=64,b=64,f=64,d=64,c=64",
         "keep_plan": True},
        # attention scores / factor models: a dense product sampled at the entries of a sparse matrix
        {"name": "sddmm", "op": "sddmm", "n": 250_000, "width": 64},
        # what a compiled program calls: everything comes from and goes back to host memory
        {"name": "host_spmm", "op": "host_spmm", "n": 30_011, "width": 32, "index_bits": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["spmv", "spmm", "spgemm", "spgemm_masked", "tricount", "ttgt", "sddmm", "host_spmm", "host_spmv"])
    if op == "spmv":
        n = _log_int(rng, 1_000, 1_200_000)
        return {"op": op, "n": n, "mean": round(rng.uniform(3.0, 10.0), 2), "both_sides": n < 30_000 or rng.random() < 0.5}
    if op in ("spmm", "sddmm"):
        return {"op": op, "n": _log_int(rng, 2_000, 500_000), "width": _log_int(rng, 3, 64)}
    if op == "spgemm":
        reduce, mult = rng.choice([("plus", "times"), ("min", "plus")])
        return {"op": op, "n": _log_int(rng, 300, 65_000), "edge_factor": rng.randint(4, 16), "reduce": reduce,
                "mult": mult}
    if op == "spgemm_masked":
        return {"op": op, "n": _log_int(rng, 500, 260_000), "edge_factor": rng.randint(4, 16)}
    if op == "tricount":
        return {"op": op, "n": _log_int(rng, 1_000, 1 << 20), "edge_factor": rng.randint(4, 16)}
    if op == "ttgt":
        expr = rng.choice(["aebf,dfce->abcd", "cima,mc->ia", "icmn,mnca->ia"])
        labels = sorted(set(expr) - set(",->"))
        return {"op": op, "expr": expr, "extents": ",".join("%s=%d" % (l, _log_int(rng, 6, 62)) for l in labels),
                "keep_plan": rng.random() < 0.5}
    width = 1 if op == "host_spmv" else _log_int(rng, 2, 64)
    return {"op": op, "n": _log_int(rng, 500, 150_000), "width": width, "index_bits": rng.choice([32, 64])}


# ----------------------------------------------------------------------------- inputs
class _Exposed:
    """A device array of the library as torch takes one; `owner` keeps the memory alive."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 3,
                                         "strides": None}


def _view(array):
    return torch.as_tensor(_Exposed(array.ptr, array.shape, array.dtype.str, array), device="cuda")


def _device_array(t):
    out = rt.DeviceArray(tuple(t.shape), np.dtype(str(t.dtype).replace("torch.", "")))
    if t.numel():
        _view(out).copy_(t)
    return out


def _csr_views(c):
    """The arrays of a product the library made; they live as long as the tensors do."""
    rows, _, nnz = c.dims()
    pos, crd, val = c.device_arrays()
    out = {"pos": torch.as_tensor(_Exposed(pos, (rows + 1,), "<i8", c), device="cuda")}
    if nnz:
        out["crd"] = torch.as_tensor(_Exposed(crd, (nnz,), "<i4", c), device="cuda")
        out["val"] = torch.as_tensor(_Exposed(val, (nnz,), "<f8", c), device="cuda")
    return out


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(1_000_003 + int(seed))


def _uniform(g, shape, lo=-1.0, hi=1.0):
    return torch.rand(shape, generator=g, device=_device(), dtype=torch.float64) * (hi - lo) + lo


def _rows_of(g, lengths, ncols):
    """Sorted distinct (row, column) keys: lengths[i] uniform columns in row i, repeats dropped."""
    rows = torch.repeat_interleave(torch.arange(len(lengths), device=_device()), lengths)
    cols = torch.randint(0, ncols, (len(rows),), generator=g, device=_device())
    return torch.unique(rows * ncols + cols)


def _poisson_keys(g, n, mean):
    return _rows_of(g, torch.poisson(torch.full((n,), mean, device=_device()), generator=g).long().clamp_(max=n), n)


def _power_law_keys(g, n):
    """Row lengths with the tail of Zipf(1.5), scaled to the mean and capped."""
    z = torch.rand(n, generator=g, device=_device(), dtype=torch.float64).clamp_(min=1e-9).pow_(-2.0).floor_()
    cap = min(CAP_ROW, n)
    lo, hi = 0.0, 64.0
    for _ in range(40):
        mid = 0.5 * (lo + hi)
        if float(torch.ceil(z * mid).clamp_(1, cap).mean()) < MEAN_ROW:
            lo = mid
        else:
            hi = mid
    return _rows_of(g, torch.ceil(z * hi).clamp_(1, cap).long(), n)


def _graph_keys(g, n, edge_factor):
    """Symmetric R-MAT graph on n vertices without loops or repeated edges."""
    scale = max(1, (n - 1).bit_length())
    a, b, c = RMAT
    m = edge_factor << scale
    u = torch.zeros(m, dtype=torch.int64, device=_device())
    v = torch.zeros(m, dtype=torch.int64, device=_device())
    for _ in range(scale):
        r = torch.rand(m, generator=g, device=_device())
        u.mul_(2).add_(r >= a + b)
        v.mul_(2).add_(((r >= a) & (r < a + b)) | (r >= a + b + c))
    keep = (u != v) & (u < n) & (v < n)
    u, v = u[keep], v[keep]
    return torch.unique(torch.cat([u * n + v, v * n + u]))


def _renumbered(keys, n, row_shift, col_shift):
    """The same pattern with its rows and columns moved round: what another seed gets where the number of stored
    entries belongs to the case."""
    rows = torch.div(keys, n, rounding_mode="floor")
    return torch.sort((rows + row_shift) % n * n + (keys - rows * n + col_shift) % n).values


def _matrix(keys, n, val, read_mode=1):
    rows = torch.div(keys, n, rounding_mode="floor")
    row, col = rows.to(torch.int32), (keys - rows * n).to(torch.int32)
    return rt.CsrMatrix.from_coo_device((n, n), _device_array(row), _device_array(col), _device_array(val), read_mode)


def _extents(case):
    return {k: int(v) for k, v in (t.split("=") for t in case["extents"].split(","))}


def _labels(case):
    operands, out = case["expr"].split("->")
    return (*operands.split(","), out)


def prepare(case, seed):
    rt.init(0)
    op, g = case["op"], _generator(seed)
    state = {"op": op}
    if op == "ttgt":
        a, b, c = _labels(case)
        e = _extents(case)
        state.update(labels=(a, b, c), A=_device_array(_uniform(g, [e[l] for l in a])),
                     B=_device_array(_uniform(g, [e[l] for l in b])), C=rt.DeviceArray([e[l] for l in c]),
                     plan=rt.ttgt_plan(a, b, c, e) if case["keep_plan"] else None)
        state["out"] = _view(state["C"])
        return state
    n = case["n"]
    if op == "spmv":
        keys = _poisson_keys(g, n, case["mean"])
        state.update(A=_matrix(keys, n, _uniform(g, len(keys))), x=_device_array(_uniform(g, n)), y=rt.DeviceArray(n))
        state["out"] = _view(state["y"])
        if case["both_sides"]:
            state.update(w=_device_array(_uniform(g, n)), z=rt.DeviceArray(n))
            state["out"] = (state["out"], _view(state["z"]))
    elif op == "spmm":
        keys, k = _power_law_keys(g, n), case["width"]
        state.update(A=_matrix(keys, n, _uniform(g, len(keys))), B=_device_array(_uniform(g, (n, k))),
                     C=rt.DeviceArray((n, k)))
        state["out"] = _view(state["C"])
    elif op == "sddmm":
        shifts = np.random.default_rng(seed).integers(0, n, 2)
        keys, k = _renumbered(_power_law_keys(_generator(0), n), n, int(shifts[0]), int(shifts[1])), case["width"]
        state.update(S=_matrix(keys, n, _uniform(g, len(keys))), C=_device_array(_uniform(g, (n, k))),
                     D=_device_array(_uniform(g, (k, n))), values=rt.DeviceArray(len(keys)))
        state["out"] = _view(state["values"])
    elif op in ("spgemm", "spgemm_masked"):
        shift = int(np.random.default_rng(seed).integers(0, n))
        keys = _renumbered(_graph_keys(_generator(0), n, case["edge_factor"]), n, shift, shift)
        state["A"] = _matrix(keys, n, 1.0 - _uniform(g, len(keys), 0.0, 1.0))
        if op == "spgemm":
            plain = (case["reduce"], case["mult"]) == ("plus", "times")
            state["semiring"] = None if plain else (case["reduce"], case["mult"])
    elif op == "tricount":
        keys = _graph_keys(g, n, case["edge_factor"])
        ones = torch.ones(len(keys), dtype=torch.float64, device=_device())
        state["L"] = _matrix(keys, n, ones, read_mode=2)           # the strictly lower triangle
    else:       # host_spmm, host_spmv: what a compiled program holds in its memrefs
        keys, k = _power_law_keys(g, n), case["width"]
        index = np.int64 if case["index_bits"] == 64 else np.int32
        rows = torch.div(keys, n, rounding_mode="floor")
        pos = torch.zeros(n + 1, dtype=torch.int64, device=_device())
        pos[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
        shape = (n, k) if op == "host_spmm" else (n,)
        host = {"pos": pos.cpu().numpy().astype(index), "crd": (keys - rows * n).cpu().numpy().astype(index),
                "val": _uniform(g, len(keys)).cpu().numpy(), "B": _uniform(g, shape).cpu().numpy(), "C": np.zeros(shape)}
        dense = rt.memref2d if op == "host_spmm" else rt.memref1d
        state.update(host=host, memrefs=[rt.memref1d(host[k]) for k in ("pos", "crd", "val")] +
                     [dense(host[k]) for k in ("B", "C")],
                     call=getattr(rt.lib(), "_mlir_ciface_comet_hip_%s_csr_f64_i%d" % (op[5:], case["index_bits"])))
    return state


def run(s):
    op = s["op"]
    if op == "spmv":
        rt.spmv(s["A"], s["x"], s["y"], accumulate=False)
        if "w" in s:
            rt.vecmat(s["w"], s["A"], s["z"], accumulate=False)
        return s["out"]
    if op == "spmm":
        rt.spmm(s["A"], s["B"], s["C"], accumulate=False)
        return s["out"]
    if op == "sddmm":
        rt.sddmm(s["S"], s["C"], s["D"], out_values=s["values"])
        return s["out"]
    if op == "spgemm":
        return _csr_views(rt.spgemm(s["A"], s["A"], semiring=s["semiring"]))
    if op == "spgemm_masked":
        return _csr_views(rt.spgemm(s["A"], s["A"], mask=s["A"]))
    if op == "tricount":
        return rt.triangle_count(s["L"])
    if op == "ttgt":
        a, b, c = s["labels"]
        rt.ttgt_contract(a, b, c, s["A"], s["B"], s["C"], plan=s["plan"])
        return s["out"]
    s["host"]["C"].fill(0.0)            # a program fills its output and the product adds into it
    s["call"](*s["memrefs"])
    return s["host"]["C"]


# ----------------------------------------------------------------------------- what a pass cannot do without
@functools.lru_cache(maxsize=64)
def _counts(op, n, size):
    """Entries of the matrix, products, and entries and sum of products of the result, for one graph of this size."""
    g = _generator(0)
    if op == "spmv":
        return {"nnz": len(_poisson_keys(g, n, size))}
    if op == "power_law":
        return {"nnz": len(_power_law_keys(g, n))}
    keys = _graph_keys(g, n, size)
    degree = torch.bincount(torch.div(keys, n, rounding_mode="floor"), minlength=n).double()
    got = {"nnz": len(keys), "products": float((degree * degree).sum())}
    if not torch.cuda.is_available():          # bounds, where no product can be taken
        got.update(out=min(got["products"], float(n) * n), hits=got["nnz"], triangles=got["nnz"])
        return got
    rt.init(0)
    A = _matrix(keys, n, torch.ones(len(keys), dtype=torch.float64, device=_device()))
    if op == "spgemm":
        got["out"] = rt.spgemm_symbolic(A, A)[1]
    else:
        got["hits"] = rt.spgemm_symbolic(A, A, A)[1]
        got["triangles"] = rt.spgemm_masked_sum(A, A, A) / 6
    return got


def work(case):
    op = case["op"]
    if op == "ttgt":
        a, b, c = _labels(case)
        e = _extents(case)
        size = lambda labels: math.prod(e[l] for l in labels)  # noqa: E731
        return {"bytes": 8 * (size(a) + size(b) + size(c)), "flops": 2 * size(set(a + b))}
    n = case["n"]
    if op == "spmv":
        nnz = _counts("spmv", n, case["mean"])["nnz"]
        products = 2 if case["both_sides"] else 1        # both read the one matrix
        return {"bytes": 12 * nnz + 4 * (n + 1) + 16 * n * products, "flops": 2 * nnz * products}
    if op in ("spmm", "sddmm", "host_spmm", "host_spmv"):
        k = case["width"]
        nnz = _counts("power_law", n, 0)["nnz"]
        more = 8 * nnz if op == "sddmm" else 0
        return {"bytes": 12 * nnz + 4 * (n + 1) + 16 * n * k + more, "flops": 2 * nnz * k}
    if op == "spgemm":
        t = _counts(op, n, case["edge_factor"])
        return {"bytes": 12 * (t["nnz"] + t["out"]) + 12 * (n + 1), "flops": 2 * t["products"]}
    t = _counts("masked", n, case["edge_factor"])
    if op == "spgemm_masked":
        return {"bytes": 12 * (t["nnz"] + t["hits"]) + 12 * (n + 1), "flops": 12 * t["triangles"]}
    return {"bytes": 2 * t["nnz"] + 4 * (n + 1), "flops": 2 * t["triangles"]}


def tolerance(case):
    if case["op"] == "tricount" or case.get("reduce") == "min":
        return "exact"                   # whole numbers; the least of sums of two
    return {"rel": 1e-12, "max": 1e-10}  # double precision sums in any order
