"""The calls that stand for what programs have this framework do, with the
inputs, the work and the accuracy each is measured by.

Two front doors are used, as programs use them: tt-lang kernels written with
the drop-in `ttl` / `ttnn` modules (traced once per shape, synchronous like the
reference's), and `ttlhip.kernels`, the functions a program with torch tensors
calls (launched on the current stream, not synchronised).  Outputs go to the
tensor that the caller passes.
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "tt-lang_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ttnn  # noqa: E402
from ttl import ttl  # noqa: E402
from ttlhip import expr as X  # noqa: E402
from ttlhip import kernels as K  # noqa: E402

TILE = 32
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


# --- tt-lang kernels ---------------------------------------------------------
# Every core takes a run of tile rows, one block per row of tiles; the last
# cores take fewer where the rows do not divide.


@ttl.kernel(grid="auto")
def add(a_in, b_in, out):
    tile_rows = a_in.shape[0] // TILE
    width = a_in.shape[1] // TILE
    gh, gw = ttl.grid_size()
    rows_per_core = math.ceil(tile_rows / (gh * gw))
    a_cb = ttl.make_circular_buffer_like(a_in, shape=(1, width), buffer_factor=2)
    b_cb = ttl.make_circular_buffer_like(b_in, shape=(1, width), buffer_factor=2)
    o_cb = ttl.make_circular_buffer_like(out, shape=(1, width), buffer_factor=2)

    @ttl.compute()
    def comp():
        c = ttl.core(dims=1)
        for r in range(c * rows_per_core, min((c + 1) * rows_per_core, tile_rows)):
            with a_cb.wait() as a, b_cb.wait() as b, o_cb.reserve() as o:
                o.store(a + b)

    @ttl.datamovement()
    def reader():
        c = ttl.core(dims=1)
        for r in range(c * rows_per_core, min((c + 1) * rows_per_core, tile_rows)):
            with a_cb.reserve() as a, b_cb.reserve() as b:
                ta = ttl.copy(a_in[r, 0:width], a)
                tb = ttl.copy(b_in[r, 0:width], b)
                ta.wait()
                tb.wait()

    @ttl.datamovement()
    def writer():
        c = ttl.core(dims=1)
        for r in range(c * rows_per_core, min((c + 1) * rows_per_core, tile_rows)):
            with o_cb.wait() as o:
                ttl.copy(o, out[r, 0:width]).wait()


@ttl.kernel(grid="auto")
def exp_row_pipe(a_in, b_row, c_in, out):
    tile_rows = a_in.shape[0] // TILE
    width = a_in.shape[1] // TILE
    gh, gw = ttl.grid_size()
    rows_per_core = math.ceil(tile_rows / (gh * gw))
    a_cb = ttl.make_circular_buffer_like(a_in, shape=(1, width), buffer_factor=2)
    b_cb = ttl.make_circular_buffer_like(b_row, shape=(1, width), buffer_factor=2)
    c_cb = ttl.make_circular_buffer_like(c_in, shape=(1, width), buffer_factor=2)
    o_cb = ttl.make_circular_buffer_like(out, shape=(1, width), buffer_factor=2)

    @ttl.compute()
    def comp():
        c = ttl.core(dims=1)
        for r in range(c * rows_per_core, min((c + 1) * rows_per_core, tile_rows)):
            with a_cb.wait() as ab, b_cb.wait() as bb, c_cb.wait() as cb, o_cb.reserve() as ob:
                ob.store(ttl.math.exp(ab + ttl.math.broadcast(bb, dims=[0])) * cb)

    @ttl.datamovement()
    def reader():
        c = ttl.core(dims=1)
        for r in range(c * rows_per_core, min((c + 1) * rows_per_core, tile_rows)):
            with a_cb.reserve() as ab, b_cb.reserve() as bb, c_cb.reserve() as cb:
                ttl.copy(a_in[r, 0:width], ab).wait()
                ttl.copy(b_row[0, 0:width], bb).wait()
                ttl.copy(c_in[r, 0:width], cb).wait()

    @ttl.datamovement()
    def writer():
        c = ttl.core(dims=1)
        for r in range(c * rows_per_core, min((c + 1) * rows_per_core, tile_rows)):
            with o_cb.wait() as ob:
                ttl.copy(ob, out[r, 0:width]).wait()


def _row_kernel(form):
    @ttl.kernel(grid="auto")
    def rows(x_in, out):
        tile_rows = x_in.shape[0] // TILE
        width = x_in.shape[1] // TILE
        gh, gw = ttl.grid_size()
        rows_per_core = math.ceil(tile_rows / (gh * gw))
        x_cb = ttl.make_circular_buffer_like(x_in, shape=(1, width), buffer_factor=2)
        y_cb = ttl.make_circular_buffer_like(out, shape=(1, width), buffer_factor=2)

        @ttl.compute()
        def comp():
            c = ttl.core(dims=1)
            for r in range(c * rows_per_core, min((c + 1) * rows_per_core, tile_rows)):
                with x_cb.wait() as x, y_cb.reserve() as y:
                    if form == "softmax":
                        m = ttl.math.broadcast(ttl.math.reduce_max(x, 1.0, dims=[1]), y, dims=[1])
                        e = ttl.math.exp(x - m)
                        s = ttl.math.recip(ttl.math.reduce_sum(e, 1.0, dims=[1]))
                        y.store(e * ttl.math.broadcast(s, y, dims=[1]))
                    else:
                        ss = ttl.math.broadcast(ttl.math.reduce_sum(x * x, 1.0, dims=[1]), y,
                                                dims=[1])
                        y.store(x * ttl.math.rsqrt(ss * (1.0 / (width * TILE)) + 1e-5))

        @ttl.datamovement()
        def reader():
            c = ttl.core(dims=1)
            for r in range(c * rows_per_core, min((c + 1) * rows_per_core, tile_rows)):
                with x_cb.reserve() as x:
                    ttl.copy(x_in[r, 0:width], x).wait()

        @ttl.datamovement()
        def writer():
            c = ttl.core(dims=1)
            for r in range(c * rows_per_core, min((c + 1) * rows_per_core, tile_rows)):
                with y_cb.wait() as y:
                    ttl.copy(y, out[r, 0:width]).wait()

    return rows


ROWS = {"softmax": _row_kernel("softmax"), "rms": _row_kernel("rms")}


# --- the cases ---------------------------------------------------------------


def listed():
    return [
        # the eltwise example at its own size: a tile program's smallest call, all latency
        {"name": "add_f32_256", "kind": "add", "rows": 256, "cols": 256, "dtype": "f32"},
        # the fused broadcast / exp pipe at the benchmark's size: a streaming store of a large
        # tensor
        {"name": "exp_pipe_4096", "kind": "pipe", "rows": 4096, "cols": 4096, "dtype": "bf16"},
        # row softmax of attention scores or logits, rows that are no power of two
        {"name": "softmax_2016x2880", "kind": "rows", "form": "softmax", "rows": 2016,
         "cols": 2880},
        # column sums of a gradient (a bias gradient): the reduction over rows
        {"name": "col_sums_4096", "kind": "reduce", "op": "sum", "dims": "0", "rows": 4096,
         "cols": 4096},
        # one tile of rows (a decode step's batch) times a projection's weights
        {"name": "matmul_32x11008x4096", "kind": "matmul", "dtype": "bf16", "m": 32, "k": 11008,
         "n": 4096},
        # an ordinary product whose tiles divide nothing
        {"name": "matmul_1056x992x1504", "kind": "matmul", "dtype": "bf16", "m": 1056, "k": 992,
         "n": 1504},
        # the benchmark's large product
        {"name": "matmul_4096", "kind": "matmul", "dtype": "bf16", "m": 4096, "k": 4096,
         "n": 4096},
        # fp32 tensors, the dtype of the matmul examples
        {"name": "matmul_f32_2048", "kind": "matmul", "dtype": "f32", "m": 2048, "k": 2048,
         "n": 2048},
        # block-float weights: a decode step and a prefill over the same MLP weights
        {"name": "bfp8_32x4096x11008", "kind": "block", "bits": 8, "m": 32, "k": 4096,
         "n": 11008},
        {"name": "bfp8_4096x4096x11008", "kind": "block", "bits": 8, "m": 4096, "k": 4096,
         "n": 11008},
        # the benchmark's attention
        {"name": "sdpa_4x32x4096x128", "kind": "sdpa", "b": 4, "h": 32, "s": 4096, "d": 128,
         "causal": False},
        # a prompt's causal attention, its length a whole number of tiles and no more
        {"name": "sdpa_causal_1x32x2016x128", "kind": "sdpa", "b": 1, "h": 32, "s": 2016,
         "d": 128, "causal": True},
    ]


def _tiles(rng, lo, hi):
    """A multiple of 32 in [lo, hi], spread over its logarithm."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(lo, min(hi, int(round(n / TILE)) * TILE))


def draw(rng):
    kind = rng.choice(["add", "pipe", "rows", "reduce", "matmul", "matmul", "matmul", "block",
                       "block", "sdpa", "sdpa"])
    if kind in ("add", "pipe"):
        return {"kind": kind, "rows": _tiles(rng, 64, 4096), "cols": _tiles(rng, 64, 4096),
                "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "rows":
        return {"kind": kind, "form": rng.choice(["softmax", "rms"]),
                "rows": _tiles(rng, 64, 4096), "cols": _tiles(rng, 128, 8192)}
    if kind == "reduce":
        return {"kind": kind, "op": rng.choice(["sum", "sum", "max"]),
                "dims": rng.choice(["0", "0", "1", "01"]), "rows": _tiles(rng, 64, 8192),
                "cols": _tiles(rng, 64, 8192)}
    if kind == "matmul" and rng.random() < 0.3:
        return {"kind": kind, "dtype": "f32", "m": _tiles(rng, 64, 2048),
                "k": _tiles(rng, 64, 2048), "n": _tiles(rng, 64, 2048)}
    if kind == "matmul":
        return {"kind": kind, "dtype": "bf16", "m": _tiles(rng, 32, 4096),
                "k": _tiles(rng, 256, 11008), "n": _tiles(rng, 256, 11008)}
    if kind == "block":
        return {"kind": kind, "bits": rng.choice([8, 8, 4]), "m": _tiles(rng, 32, 4096),
                "k": _tiles(rng, 512, 4096), "n": _tiles(rng, 512, 11008)}
    s = _tiles(rng, 64, 4096)
    return {"kind": kind, "b": rng.choice([1, 1, 2, 4]), "h": rng.choice([8, 16, 32]), "s": s,
            "d": rng.choice([64, 128, 128]), "causal": rng.random() < 0.5}


# --- inputs ------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(g, shape, lo, hi, dtype):
    x = torch.rand(shape, generator=g, device="cuda", dtype=torch.float32)
    return (x * (hi - lo) + lo).to(dtype)


def _normal(g, shape, std, dtype):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (x * std).to(dtype)


def _inputs(case, seed):
    """The input tensors of a case, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("add", "pipe"):
        dt, shape = DTYPES[case["dtype"]], (case["rows"], case["cols"])
        a = _uniform(g, shape, -2, 2, dt)
        b = _uniform(g, shape if kind == "add" else (1, shape[1]), -2, 2, dt)
        return (a, b) if kind == "add" else (a, b, _uniform(g, shape, -2, 2, dt))
    if kind in ("rows", "reduce"):
        if case.get("dims") == "01":  # a total of positive terms (a loss, a norm)
            return (_uniform(g, (case["rows"], case["cols"]), 0, 1, torch.bfloat16),)
        return (_normal(g, (case["rows"], case["cols"]), 1.0, torch.bfloat16),)
    if kind == "matmul":
        dt = DTYPES[case["dtype"]]
        return (_normal(g, (case["m"], case["k"]), 1.0, dt),
                _normal(g, (case["k"], case["n"]), case["k"] ** -0.5, dt))
    if kind == "block":
        return (_normal(g, (case["m"], case["k"]), 1.0, torch.bfloat16),
                _normal(g, (case["k"], case["n"]), case["k"] ** -0.5, torch.float32))
    shape = (case["b"], case["h"], case["s"], case["d"])
    return tuple(_normal(g, shape, 1.0, torch.bfloat16) for _ in range(3))


def prepare(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    st = {"case": case}
    if kind in ("add", "pipe", "rows"):
        st["out"] = torch.zeros_like(x[0])
        st["args"] = [ttnn.Tensor(t, layout=ttnn.TILE_LAYOUT) for t in (*x, st["out"])]
        st["kernel"] = {"add": add, "pipe": exp_row_pipe}.get(kind) or ROWS[case["form"]]
    elif kind == "reduce":
        dims = [int(d) for d in case["dims"]]
        st["x"], st["dims"] = x[0], dims
        st["prog"] = X.compile_expr(X.Leaf(0, torch.bfloat16))
        st["operands"] = [K.OperandMap(x[0])]
        st["out"] = torch.zeros(1 if 0 in dims else case["rows"], 1 if 1 in dims else case["cols"],
                                dtype=torch.float32, device="cuda")
    elif kind == "matmul":
        st["a"], st["b"] = x
        st["out"] = torch.zeros(case["m"], case["n"], dtype=x[0].dtype, device="cuda")
    elif kind == "block":
        pack = K.bfp8_pack_host if case["bits"] == 8 else K.bfp4_pack_host
        st["a"], st["q"] = x[0], pack(x[1]).cuda()
        st["out"] = torch.zeros(case["m"], case["n"], dtype=torch.bfloat16, device="cuda")
    else:
        st["qkv"] = x
        st["out"] = torch.zeros_like(x[0])
        st["scale"] = 1.0 / math.sqrt(case["d"])
    return st


def run(st):
    case = st["case"]
    kind, out = case["kind"], st["out"]
    if kind in ("add", "pipe", "rows"):
        st["kernel"](*st["args"])
    elif kind == "reduce":
        K.reduce(st["prog"], st["operands"], case["op"], st["dims"], out,
                 (0, 0, case["rows"], case["cols"]))
    elif kind == "matmul":
        K.matmul(st["a"], st["b"], out)
    elif kind == "block":
        (K.matmul_bfp8w if case["bits"] == 8 else K.matmul_bfp4w)(st["a"], st["q"], out)
    else:
        q, k, v = st["qkv"]
        K.sdpa_fwd(q, k, v, out, st["scale"], causal=case["causal"])
    return out


# --- work and accuracy -------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("add", "pipe"):
        n, size = case["rows"] * case["cols"], 2 if case["dtype"] == "bf16" else 4
        return {"bytes": 3 * n * size + (case["cols"] * size if kind == "pipe" else 0),
                "flops": n * (1 if kind == "add" else 3)}
    if kind == "rows":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n, "flops": (5 if case["form"] == "softmax" else 3) * n}
    if kind == "reduce":
        n = case["rows"] * case["cols"]
        res = {"0": case["cols"], "1": case["rows"], "01": 1}[case["dims"]]
        return {"bytes": 2 * n + 4 * res, "flops": n}
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": (m * k + k * n + m * n) * (2 if case["dtype"] == "bf16" else 4),
                "flops": 2 * m * k * n}
    if kind == "block":
        m, k, n = case["m"], case["k"], case["n"]
        weights = k * n * case["bits"] // 8 + k * n // 16
        return {"bytes": 2 * m * k + weights + 2 * m * n, "flops": 2 * m * k * n}
    n = case["b"] * case["h"] * case["s"] * case["d"]
    # two products of S x S x D per head; under the causal mask their lower triangles
    return {"bytes": 8 * n,
            "flops": 4 * n * ((case["s"] + 1) / 2 if case["causal"] else case["s"])}


def tolerance(case):
    kind = case["kind"]
    if kind == "add" or (kind == "reduce" and case["op"] == "max"):
        return "exact"  # one rounding of one exact operation, or a selection
    if kind == "pipe":
        # every op rounds to the tensors' dtype; exp differs by an ulp between implementations
        return {"rel": 8e-3, "max": 3e-2} if case["dtype"] == "bf16" else {"rel": 1e-6, "max": 4e-6}
    if kind == "rows":
        return {"rel": 1e-2, "max": 4e-2}  # bf16 roundings of each op of the chain
    if kind == "reduce":
        return {"rel": 4e-6, "max": 2e-5}  # fp32 sums that cancel
    if kind == "matmul" and case["dtype"] == "f32":
        return {"rel": 4e-6}
    if kind == "sdpa":
        return {"rel": 1.2e-2}
    return {"rel": 7e-3}  # fp32 sums rounded once to bf16


def _block_values(w, bits):
    """The float64 values of fp32 weights in block-float form: 16 consecutive
    columns share the largest one's exponent, `bits` with the sign, rounded
    half to even and saturated."""
    rows, cols = w.shape
    g = w.double().view(rows, cols // 16, 16)
    e = torch.frexp(g.abs().amax(-1, keepdim=True)).exponent.double() - 1
    unit = torch.exp2(e - (bits - 2))
    return (torch.round(g / unit).clamp(-(2 ** (bits - 1) - 1), 2 ** (bits - 1) - 1)
            * unit).view(rows, cols)


def exact(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    if kind == "block":
        return x[0].double() @ _block_values(x[1], case["bits"])
    x = [t.double() for t in x] if kind != "sdpa" else x
    if kind == "add":
        return x[0] + x[1]
    if kind == "pipe":
        return torch.exp(x[0] + x[1]) * x[2]
    if kind == "rows":
        if case["form"] == "softmax":
            return torch.softmax(x[0], 1)
        return x[0] * torch.rsqrt(x[0].square().mean(1, keepdim=True) + 1e-5)
    if kind == "reduce":
        dims = [int(d) for d in case["dims"]]
        return x[0].sum(dims, keepdim=True) if case["op"] == "sum" else x[0].amax(dims, True)
    if kind == "matmul":
        return x[0] @ x[1]
    q, k, v = (t.flatten(0, 1) for t in x)
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    scale = 1.0 / math.sqrt(case["d"])
    hidden = torch.ones(case["s"], case["s"], dtype=torch.bool, device=q.device).triu_(1)
    for i in range(q.shape[0]):
        p = (q[i].double() @ k[i].double().t().contiguous()) * scale
        if case["causal"]:
            p.masked_fill_(hidden, -math.inf)
        out[i] = torch.softmax(p, 1) @ v[i].double()
    return out.view(x[0].shape)
