"""The work that users of the package have it do, as cases that can be timed.

A case is one call (or one training pass) through the package's public entry
points on seeded synthetic inputs.  The kinds, by ``op``:

- ``spmm``       CSR × dense (``kernels.spmm``): fp32, bf16 or fp8-e4m3 dense operand,
                 with or without edge values and the fused GCN epilogue
- ``spmv``       CSR × vector (``kernels.spmv``)
- ``vcsr``       SpMV on the zero-padded 1×4-blocked CSR (``kernels.vcsr_spmv``)
- ``sddmm``      sampled dense × dense on a CSR pattern (``kernels.sddmm``): fp32 or bf16
- ``spgemm``     sparse × sparse into a dense matrix (``kernels.spgemm_dense``)
- ``transpose``  CSR → CSC (``kernels.csr_transpose``)
- ``coo``        unordered triplets → canonical CSR (``kernels.coo_to_csr``)
- ``max``        max aggregation, forward and backward (``op.SPMMMaxFunction``)
- ``layer``      a GCN layer, forward and backward (``op.GCNConv``)
- ``step``       a GCN training step (``gcn.train_step``, or ``gcn.GraphedStep`` when
                 ``graphed``)

Matrices: ``uniform`` (every position equally likely), ``rmat`` (a = .57,
b = c = .19, d = .05, as the benchmark's: hub rows and columns, many empty rows)
and ``power`` (a symmetric power-law graph with self loops, as the GCN's).
"""
import math

import torch

from armsparse_amd import gcn, kernels, op

DEV = "cuda"


# --------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest everyday product (the reference driver's 4096² at 1%, 64 columns): latency
        dict(name="spmm_4096_n64", op="spmm", kind="uniform", rows=4096, cols=4096, nnz=167_772, n=64, dtype="f32",
             values=True, epilogue=False),
        # the benchmark's headline product: a million-row R-MAT times 128 fp32 columns
        dict(name="spmm_rmat1m_n128", op="spmm", kind="rmat", rows=1 << 20, cols=1 << 20, nnz=1 << 24, n=128,
             dtype="f32", values=True, epilogue=False),
        # a GCN aggregation in bf16 on a mid-size graph: odd node count, rows that are not whole cache
        # lines, normalisation, bias and ReLU fused
        dict(name="spmm_graph_bf16_n100", op="spmm", kind="power", rows=200_003, cols=200_003, nnz=5_000_003, n=100,
             dtype="bf16", values=True, epilogue=True),
        # power iteration / ranking on the same million-row matrix
        dict(name="spmv_rmat1m", op="spmv", kind="rmat", rows=1 << 20, cols=1 << 20, nnz=1 << 24),
        # the reference's own SpMV format, bit-exact order
        dict(name="vcsr_rmat1m", op="vcsr", kind="rmat", rows=1 << 20, cols=1 << 20, nnz=1 << 24),
        # attention scores / edge gradients: 128-wide dot products on the edges
        dict(name="sddmm_rmat1m_k128", op="sddmm", kind="rmat", rows=1 << 20, cols=1 << 20, nnz=1 << 24, n=128,
             dtype="f32"),
        # the reference driver's sparse × sparse product
        dict(name="spgemm_4096", op="spgemm", kind="uniform", rows=4096, cols=4096, nnz=167_772),
        # building a graph's reverse adjacency
        dict(name="transpose_rmat1m", op="transpose", kind="rmat", rows=1 << 20, cols=1 << 20, nnz=1 << 24,
             values=True),
        # building a matrix from an edge list as it is loaded: unordered, with repeated edges
        dict(name="coo_rmat300k", op="coo", kind="rmat", rows=300_007, cols=300_007, nnz=6_000_001, values=True,
             drop=False),
        # max-pool neighbourhood aggregation with its gradient
        dict(name="max_rmat131k_n64", op="max", kind="rmat", rows=1 << 17, cols=1 << 17, nnz=1 << 21, n=64,
             values=False),
        # a hidden GCN layer of a mid-size graph, with the gradients of x, W and b
        dict(name="layer_170k_128_256_bf16", op="layer", nodes=170_000, pairs=1_200_000, fin=128, fout=256,
             precision="bf16"),
        # the reference script's training step at its PubMed size, as the package replays it
        dict(name="step_pubmed_bf16", op="step", nodes=19_717, pairs=44_324, fin=500, hidden=64, classes=3,
             precision="bf16", graphed=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A feature width: any number, or (half of the time) a multiple of 8 as layers are usually sized."""
    n = _log_int(rng, lo, hi)
    return max(8, n // 8 * 8) if rng.random() < 0.5 else n


def _matrix(rng, max_rows=1 << 20, max_nnz=1 << 24):
    kind = rng.choice(["uniform", "rmat", "power"])
    rows = _log_int(rng, 1 << 10, max_rows)
    if rng.random() < 0.3:
        rows = 1 << int(math.log2(rows))
    nnz = min(max_nnz, int(rows * math.exp(rng.uniform(math.log(3), math.log(40)))), rows * rows // 16)
    cols = rows if kind != "uniform" or rng.random() < 0.5 else _log_int(rng, rows // 4, rows)
    return dict(kind=kind, rows=rows, cols=cols, nnz=nnz)


def draw(rng):
    what = rng.choice(["spmm", "spmm", "spmm", "spmv", "vcsr", "sddmm", "sddmm", "spgemm", "transpose", "coo", "max",
                       "layer", "step"])
    if what == "spmm":
        n = _width(rng, 1, 256)
        c = _matrix(rng, min(1 << 20, (1 << 27) // n), min(1 << 24, (1 << 31) // n))
        return dict(c, op=what, n=n, dtype=rng.choice(["f32", "f32", "bf16", "fp8"]), values=rng.random() < 0.7,
                    epilogue=rng.random() < 0.3)
    if what in ("spmv", "vcsr"):
        return dict(_matrix(rng), op=what)
    if what == "sddmm":
        n = _width(rng, 8, 256)
        c = _matrix(rng, min(1 << 20, (1 << 27) // n), min(1 << 24, (1 << 31) // n))
        return dict(c, op=what, n=n, dtype=rng.choice(["f32", "bf16"]))
    if what == "spgemm":
        rows = _log_int(rng, 256, 4096)
        return dict(op=what, kind=rng.choice(["uniform", "rmat"]), rows=rows, cols=rows,
                    nnz=int(rows * rows * rng.uniform(0.002, 0.01)))
    if what == "transpose":
        return dict(_matrix(rng), op=what, values=rng.random() < 0.7)
    if what == "coo":
        return dict(_matrix(rng, 300_007, 6_000_001), op=what, values=rng.random() < 0.7, drop=rng.random() < 0.3)
    if what == "max":
        n = _width(rng, 4, 128)
        c = _matrix(rng, 1 << 17, min(1 << 21, (1 << 27) // n))
        return dict(c, op=what, n=n, values=rng.random() < 0.5)
    if what == "layer":
        nodes = _log_int(rng, 2_000, 170_000)
        return dict(op=what, nodes=nodes, pairs=int(nodes * rng.uniform(2, 7)), fin=_width(rng, 16, 160),
                    fout=_width(rng, 4, 256), precision=rng.choice(["bf16", "bf16", "fp32"]))
    nodes = _log_int(rng, 2_000, 30_000)
    return dict(op=what, nodes=nodes, pairs=int(nodes * rng.uniform(2, 5)), fin=_width(rng, 32, 600),
                hidden=8 * rng.randint(2, 16), classes=rng.randint(3, 40), precision=rng.choice(["bf16", "bf16", "fp32"]),
                graphed=rng.random() < 0.5)


# -------------------------------------------------------------------- inputs
def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed(seed * 64 + stream)


def _uniform(shape, seed, stream, lo=-1.0, hi=1.0):
    return torch.rand(shape, generator=_gen(seed, stream), device=DEV).mul_(hi - lo).add_(lo)


def _positions(kind, rows, cols, count, g):
    """`count` (row, column) positions of the kind, in no order, repeats among them."""
    if kind == "uniform":
        return (torch.randint(rows, (count,), generator=g, device=DEV),
                torch.randint(cols, (count,), generator=g, device=DEV))
    if kind == "power":  # endpoint weights (i + 1)^-1/2: the degrees' exponent is 3
        r = (torch.rand(count, generator=g, device=DEV, dtype=torch.float64).square_() * rows).long()
        c = (torch.rand(count, generator=g, device=DEV, dtype=torch.float64).square_() * cols).long()
        return r, c
    r = torch.zeros(count, dtype=torch.int64, device=DEV)
    c = torch.zeros(count, dtype=torch.int64, device=DEV)
    for _ in range(max(1, (max(rows, cols) - 1).bit_length())):
        u = torch.rand(count, generator=g, device=DEV)
        r.mul_(2).add_(u >= 0.76)
        c.mul_(2).add_(((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    inside = (r < rows) & (c < cols)
    return r[inside], c[inside]


def _keys(kind, rows, cols, nnz, seed):
    """nnz distinct sorted row·cols + column keys."""
    g = _gen(seed, 1)
    keys = torch.empty(0, dtype=torch.int64, device=DEV)
    more = nnz
    while keys.numel() < nnz:
        r, c = _positions(kind, rows, cols, more + more // 3 + 64, g)
        keys = torch.unique(torch.cat([keys, r * cols + c]))
        more = max(nnz - keys.numel(), nnz // 8)
    if keys.numel() > nnz:
        keep = torch.randperm(keys.numel(), generator=g, device=DEV)[:nnz]
        keys = keys[torch.sort(keep).values]
    return keys


def _to_csr(keys, rows, cols):
    r = torch.div(keys, cols, rounding_mode="floor")
    rowptr = torch.zeros(rows + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(torch.bincount(r, minlength=rows), 0, out=rowptr[1:])
    return rowptr.int(), (keys - r * cols).int()


def _csr(c, seed):
    rp, ci = _to_csr(_keys(c["kind"], c["rows"], c["cols"], c["nnz"], seed), c["rows"], c["cols"])
    return rp, ci, _uniform(ci.numel(), seed, 2) if c.get("values", True) else None


def _graph(nodes, pairs, seed):
    """(rowptr, colind) of a symmetric power-law graph with self loops."""
    r, c = _positions("power", nodes, nodes, pairs, _gen(seed, 3))
    loops = torch.arange(nodes, device=DEV)
    return _to_csr(torch.unique(torch.cat([r * nodes + c, c * nodes + r, loops * (nodes + 1)])), nodes, nodes)


def _dense(c, seed):
    """(operand, per-row fp8 scale or None) of c["n"] columns, in the case's type."""
    b = _uniform((c["cols"], c["n"]), seed, 4)
    if c["dtype"] == "bf16":
        return b.to(torch.bfloat16), None
    if c["dtype"] == "fp8":
        return kernels.quantize_fp8_rows(b)
    return b, None


def prepare(case, seed):
    what = case["op"]
    if what == "step":
        torch.manual_seed(seed)
        task = gcn.make_task(precision=case["precision"], seed=seed % (1 << 31), n=case["nodes"], pairs=case["pairs"],
                             features=case["fin"], hidden=case["hidden"], classes=case["classes"])
        return dict(op=what, task=task, step=gcn.GraphedStep(task) if case["graphed"] else None)
    if what == "layer":
        torch.manual_seed(seed)
        rp, ci = _graph(case["nodes"], case["pairs"], seed)
        w = torch.ones(ci.numel(), device=DEV)
        conv = op.GCNConv(case["fin"], case["fout"], cached=True, precision=case["precision"]).to(DEV)
        with torch.no_grad():
            conv.weight.copy_(_uniform(conv.weight.shape, seed, 5, -0.1, 0.1))
            conv.bias.copy_(_uniform(conv.bias.shape, seed, 6, -0.1, 0.1))
        dt = torch.bfloat16 if case["precision"] == "bf16" else torch.float32
        x = torch.relu(_uniform((case["nodes"], case["fin"]), seed, 7)).to(dt).requires_grad_(True)
        gy = _uniform((case["nodes"], case["fout"]), seed, 8)
        return dict(op=what, conv=conv, x=x, gy=gy, graph=(rp, ci, rp, ci, w, w))
    if what == "coo":  # an edge list in no order; one edge in ten is a repeat, one in a hundred an explicit zero
        nnz, cols, g = case["nnz"], case["cols"], _gen(seed, 9)
        once = _keys(case["kind"], case["rows"], cols, nnz - nnz // 10, seed)
        once = once[torch.randperm(once.numel(), generator=g, device=DEV)]
        keys = torch.cat([once, once[torch.randint(once.numel() // 2, (nnz // 10,), generator=g, device=DEV)]])
        v = _uniform(nnz, seed, 2)
        v[once.numel() - nnz // 100:once.numel()] = 0.0
        at = torch.randperm(nnz, generator=g, device=DEV)
        r = torch.div(keys, cols, rounding_mode="floor")
        return dict(op=what, args=(r[at].int(), (keys - r * cols)[at].int(), v[at] if case["values"] else None,
                                   case["rows"], cols, case["drop"]))
    rp, ci, va = _csr(case, seed)
    s = dict(op=what, a=(rp, ci, va))
    if what == "spmm":
        s["b"], s["scale"] = _dense(case, seed)
        s["more"] = {}
        if case["epilogue"]:
            deg = (rp[1:] - rp[:-1]).float()
            s["more"] = dict(row_scale=deg.clamp_(min=1).rsqrt_(), bias=_uniform(case["n"], seed, 6), relu=True)
    elif what == "spmv":
        s["x"] = _uniform(case["cols"], seed, 4)
    elif what == "vcsr":
        s["a"] = kernels.csr_to_vcsr(rp, ci, va, case["cols"])
        s["x"] = _uniform((case["cols"] + 3) // 4 * 4, seed, 4)
        s["y"] = _uniform(case["rows"], seed, 6)
    elif what == "sddmm":
        dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
        s["u"] = torch.randn((case["rows"], case["n"]), generator=_gen(seed, 4), device=DEV).to(dt)
        s["v"] = torch.randn((case["cols"], case["n"]), generator=_gen(seed, 5), device=DEV).to(dt)
    elif what == "spgemm":
        s["b"] = _csr(case, seed + (1 << 30))
        s["c"] = _uniform((case["rows"], case["cols"]), seed, 4)
    elif what == "transpose":
        s["cols"] = case["cols"]
    elif what == "max":
        s["x"] = _uniform((case["cols"], case["n"]), seed, 4).requires_grad_(True)
        s["g"] = _uniform((case["rows"], case["n"]), seed, 5)
    return s


# --------------------------------------------------------------------- a pass
def run(state):
    what = state["op"]
    if what == "spmm":
        return kernels.spmm(*state["a"], state["b"], dense_scale=state["scale"], **state["more"])
    if what == "spmv":
        return kernels.spmv(*state["a"], state["x"])
    if what == "vcsr":
        return kernels.vcsr_spmv(*state["a"], state["x"], state["y"])
    if what == "sddmm":
        rp, ci, va = state["a"]
        return kernels.sddmm(rp, ci, state["u"], state["v"], scale=va)
    if what == "spgemm":
        return kernels.spgemm_dense(state["a"], state["b"], state["c"])
    if what == "transpose":
        return kernels.csr_transpose(*state["a"], state["cols"])
    if what == "coo":
        return kernels.coo_to_csr(*state["args"])
    if what == "max":
        rp, ci, va = state["a"]
        x = state["x"]
        x.grad = None
        y = op.SPMMMaxFunction.apply(rp, ci, x, va)
        y.backward(state["g"])
        return y.detach(), x.grad
    if what == "layer":
        conv, x = state["conv"], state["x"]
        x.grad = conv.weight.grad = conv.bias.grad = None
        y = conv(x, *state["graph"])
        y.backward(state["gy"])
        return y.detach(), x.grad, conv.weight.grad, conv.bias.grad
    task, step = state["task"], state["step"]
    loss = step.replay() if step is not None else gcn.train_step(task, sync=False)
    return [loss] + [p.grad for p in task.model.parameters()]  # a replayed step's loss is read off it when wanted


# --------------------------------------------------------------- floor of a pass
def work(case):
    what, esz = case["op"], {"bf16": 2, "fp8": 1}.get(case.get("dtype"), 4)
    if what in ("layer", "step"):
        m, e = case["nodes"], 2 * case["pairs"] + case["nodes"]
        half = case["precision"] == "bf16"
        dims = ([(case["fin"], case["fout"])] if what == "layer" else
                [(case["fin"], case["hidden"]), (case["hidden"], case["classes"])])
        b = f = 0
        for i, (k, n) in enumerate(dims):
            dx = what == "layer" or i > 0  # the first layer of a model needs no gradient of x
            b += (2 if half else 4) * m * k * (2 if dx else 1)  # x, and its gradient
            b += 2 * 4 * m * n  # y, and its gradient
            b += 2 * (4 * (m + 1) + 8 * e)  # the graph, forward and backward
            b += 4 * (k * n + n) * (2 if what == "layer" else 7)  # W and b, their gradients, Adam's state
            f += 2 * m * k * n * (3 if dx else 2) + 2 * 2 * e * n
        return dict(bytes=b, flops=f)
    m, k, e = case["rows"], case["cols"], case["nnz"]
    a = 4 * (m + 1) + (8 if case.get("values", True) else 4) * e
    if what == "spmm":
        return dict(bytes=a + esz * k * case["n"] + (4 * k if esz == 1 else 0) + 4 * m * case["n"],
                    flops=2 * e * case["n"])
    if what == "spmv":
        return dict(bytes=a + 4 * k + 4 * m, flops=2 * e)
    if what == "vcsr":  # nearly every nonzero is alone in its block: four values and the first's column
        return dict(bytes=4 * (m + 1) + 20 * e + 4 * k + 8 * m, flops=8 * e)
    if what == "sddmm":
        return dict(bytes=a + 4 * e + esz * (m + k) * case["n"], flops=2 * e * case["n"])
    if what == "spgemm":
        return dict(bytes=2 * a + 8 * m * k, flops=2 * e * e // max(k, 1))
    if what == "transpose":
        return dict(bytes=2 * a + 4 * (k - m), flops=0)
    if what == "coo":
        w = 12 if case["values"] else 8
        return dict(bytes=w * e + a - (w - 4) * (e // 10), flops=0)
    # max: x and the gradient of y read, y and the gradient of x written
    return dict(bytes=a + 8 * (m + k) * case["n"], flops=2 * e * case["n"])


# ----------------------------------------------------------- 64-bit references
def _rows_of(rp):
    n = rp.numel() - 1
    return torch.repeat_interleave(torch.arange(n, device=rp.device), (rp[1:] - rp[:-1]).long())


def _product64(r, c, v, b, m):
    """A·b in float64, 16 columns at a time; A by its entries' rows, columns and values."""
    out = torch.empty((m, b.shape[1]), dtype=torch.float64, device=b.device)
    for lo in range(0, b.shape[1], 16):
        part = b[:, lo:lo + 16].double()
        acc = torch.zeros((m, part.shape[1]), dtype=torch.float64, device=b.device)
        for at in range(0, r.numel(), 1 << 22):
            s = slice(at, at + (1 << 22))
            t = part[c[s]]
            acc.index_add_(0, r[s], t if v is None else t.mul_(v[s].double().unsqueeze(1)))
        out[:, lo:lo + 16] = acc
    return out


def exact(case, seed):
    what = case["op"]
    if what == "step":
        return None
    s = prepare(case, seed)
    if what == "layer":
        rp, ci = s["graph"][:2]
        r, c, m = _rows_of(rp), ci.long(), case["nodes"]
        norm = (rp[1:] - rp[:-1]).double().rsqrt_().unsqueeze(1)
        x, w = s["x"].detach().double(), s["conv"].weight.detach().double()
        y = _product64(r, c, None, norm * (x @ w), m) * norm + s["conv"].bias.detach().double()
        dh = _product64(r, c, None, norm * s["gy"].double(), m) * norm  # the graph is symmetric
        return y, dh @ w.t(), x.t() @ dh, s["gy"].double().sum(0)
    if what == "coo":
        r, c, v, rows, cols, drop = s["args"]
        if v is None:
            return None
        keys, at = torch.unique(r.long() * cols + c.long(), return_inverse=True)
        sums = torch.zeros(keys.numel(), dtype=torch.float64, device=DEV).index_add_(0, at, v.double())
        if drop:  # which sums are zero is decided in 32 bits
            return None
        return None, None, sums
    rp, ci, va = s["a"]
    if what == "vcsr":  # the padded blocks' zeros add nothing
        keep = va != 0
        y = s["y"].double()
        return y.index_add_(0, _rows_of(rp)[keep], va[keep].double() * s["x"].double()[ci[keep].long()])
    r, c = _rows_of(rp), ci.long()
    if what == "spmm":
        b = s["b"]
        if case["dtype"] == "fp8":
            b = b.view(torch.float8_e4m3fn).float().double() * s["scale"].double().unsqueeze(1)
        out = _product64(r, c, va, b, case["rows"])
        if case["epilogue"]:
            out = torch.relu(out * s["more"]["row_scale"].double().unsqueeze(1) + s["more"]["bias"].double())
        return out
    if what == "spmv":
        return torch.zeros(case["rows"], dtype=torch.float64, device=DEV).index_add_(
            0, r, va.double() * s["x"].double()[c])
    if what == "sddmm":
        out = torch.empty(ci.numel(), dtype=torch.float64, device=DEV)
        for at in range(0, ci.numel(), 1 << 20):
            t = slice(at, at + (1 << 20))
            out[t] = (s["u"][r[t]].double() * s["v"][c[t]].double()).sum(1) * va[t].double()
        return out
    if what == "spgemm":
        def full(rp, ci, va, n):
            d = torch.zeros((rp.numel() - 1, n), dtype=torch.float64, device=DEV)
            d[_rows_of(rp), ci.long()] = va.double()
            return d
        return s["c"].double() + full(rp, ci, va, case["cols"]) @ full(*s["b"], case["cols"])
    if what == "transpose":
        if va is None:
            return None
        return None, None, va[torch.sort(c * case["rows"] + r).indices].double()
    # max: the last of the largest 32-bit products wins
    x, g, n = s["x"].detach(), s["g"], case["n"]
    prod = x[c] if va is None else x[c] * va.unsqueeze(1)
    rn = r.unsqueeze(1).expand(-1, n)
    y = torch.full((case["rows"], n), float(kernels.MAX_INIT), device=DEV).scatter_reduce_(0, rn, prod, "amax")
    at = torch.where(prod == y[r], torch.arange(ci.numel(), device=DEV).unsqueeze(1), -1)
    win = torch.full((case["rows"], n), -1, device=DEV).scatter_reduce_(0, rn, at, "amax")
    gr = torch.where(win >= 0, g.double(), 0.0) if va is None else \
        torch.where(win >= 0, g.double() * va.double()[win.clamp(min=0)], 0.0)
    gx = torch.zeros((case["cols"], n), dtype=torch.float64, device=DEV)
    gx.scatter_add_(0, c[win.clamp(min=0)], gr)
    return y.double(), gx
