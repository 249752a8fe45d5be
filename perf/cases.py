"""What this package is timed on: the message-passing work of a graph network's
user, through the public entry points (`dgl.graph`, `update_all`, `dgl.ops`),
on GPU tensors.

`listed` names the cases, `draw` gives further ones of the same ranges;
`prepare` makes a case's inputs from a seed, `run` is one pass, `exact` the
same results in float64 from plain torch, `work` the bytes and operations a
pass cannot do without, `tolerance` how far another correct implementation at
the same precision can be off.
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "mojo-dgl_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import mojodgl as dgl  # noqa: E402
import mojodgl.function as fn  # noqa: E402
import mojodgl.ops as ops  # noqa: E402

# ---------------------------------------------------------------- the cases


def listed():
    return [
        # the smallest calls: two message-passing rounds on a toy graph, where
        # latency and launches count
        {"name": "update_all_small", "kind": "update_all", "n": 2000, "e": 20000, "f": 64},
        # the reference's own precision and benchmark shape: every family of
        # op once in float64
        {"name": "messages_f64", "kind": "messages_f64", "n": 200000, "e": 1000000, "f": 32,
         "heads": 8},
        # the largest: inference of an attention layer on a power-law graph
        {"name": "gat_forward", "kind": "gat", "n": 2500000, "e": 60000000, "heads": 8, "d": 32,
         "train": False},
        # an attention layer's training step, fewer and narrower heads
        {"name": "gat_train", "kind": "gat", "n": 300000, "e": 6000000, "heads": 4, "d": 16,
         "train": True},
        # first-layer aggregation of wide raw features on a dense graph whose
        # node ids follow its communities, one weight per edge
        {"name": "gcn_forward", "kind": "gcn", "n": 230000, "e": 114000000, "f": 602,
         "local": True, "train": False},
        # last-layer aggregation to an odd number of classes, trained
        {"name": "gcn_train", "kind": "gcn", "n": 1000000, "e": 20000000, "f": 47,
         "local": False, "train": True},
        # max pooling over neighbours, trained (the gradient follows the
        # selected edges)
        {"name": "pool_max_train", "kind": "pool", "n": 500000, "e": 5000000, "f": 100},
        # link scoring: one dot product per edge
        {"name": "link_score", "kind": "link", "n": 1000000, "e": 20000000, "f": 128,
         "train": False},
        # graph-level readout over ragged segments
        {"name": "readout", "kind": "readout", "s": 1000000, "mean_len": 20, "f": 16,
         "train": False},
        # a relation-typed transform of every edge's features, inference
        {"name": "gather_mm", "kind": "typed_mm", "n": 10000000, "k": 128, "m": 128, "r": 64,
         "by": "gather", "dtype": "float32", "train": False},
        # the same over rows sorted by relation, odd widths, trained
        {"name": "segment_mm_train", "kind": "typed_mm", "n": 2500000, "k": 100, "m": 47, "r": 24,
         "by": "segment", "dtype": "float32", "train": True},
        # a sampled mini-batch: a new graph for every step, one mean
        # aggregation forward and backward
        {"name": "minibatch", "kind": "minibatch", "n": 150001, "e": 400003, "f": 100},
    ]


def _between(rng, lo, hi):
    """A whole number, its logarithm spread evenly over [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["update_all", "messages_f64", "gat", "gat", "gcn", "gcn", "pool", "link",
                       "readout", "typed_mm", "typed_mm", "minibatch"])
    if kind == "update_all":
        n = _between(rng, 500, 10000)
        return {"kind": kind, "n": n, "e": n * rng.randint(4, 16) + rng.randint(0, 63),
                "f": _between(rng, 16, 128)}
    if kind == "messages_f64":
        n = _between(rng, 20000, 500000)
        return {"kind": kind, "n": n, "e": n * rng.randint(4, 16) + rng.randint(0, 63),
                "f": _between(rng, 8, 128), "heads": rng.choice([1, 2, 4, 8])}
    if kind == "gat":
        train = rng.random() < 0.5
        n = _between(rng, 50000, 800000 if train else 1700000)
        return {"kind": kind, "n": n, "e": n * rng.randint(6, 24) + rng.randint(0, 63),
                "heads": rng.choice([1, 2, 3, 4, 6, 8]), "d": rng.choice([7, 8, 16, 25, 32]),
                "train": train}
    if kind == "gcn":
        train = rng.random() < 0.5
        f = rng.choice([_between(rng, 3, 64), _between(rng, 64, 602)])
        local = rng.random() < 0.5
        n = _between(rng, 20000, 1000000)
        # edges times columns, for about the time of the largest listed case
        most = 6e9 if train else 6e10 if local and n <= 230000 else 1.5e10
        e = int(min(n * rng.randint(4, 200), 114e6, most / f)) + rng.randint(0, 63)
        return {"kind": kind, "n": n, "e": e, "f": f, "local": local, "train": train}
    if kind == "pool":
        n = _between(rng, 20000, 500000)
        return {"kind": kind, "n": n, "e": n * rng.randint(4, 12) + rng.randint(0, 63),
                "f": _between(rng, 16, 128)}
    if kind == "link":
        train = rng.random() < 0.5
        n = _between(rng, 20000, 1000000)
        return {"kind": kind, "n": n, "e": n * rng.randint(4, 12 if train else 20),
                "f": _between(rng, 16, 256 if not train else 100), "train": train}
    if kind == "readout":
        train = rng.random() < 0.5
        s = _between(rng, 1000, 1000000)
        mean = min(_between(rng, 4, 200), 20000000 // s)
        f = min(_between(rng, 1, 256), max(1, 320000000 // (s * mean)))
        return {"kind": kind, "s": s, "mean_len": mean, "f": f, "train": train}
    if kind == "typed_mm":
        train = rng.random() < 0.5
        k, m = _between(rng, 16, 256), _between(rng, 16, 256)
        if rng.random() < 0.5:  # layer widths are often powers of two
            k, m = rng.choice([16, 32, 64, 128, 256]), rng.choice([16, 32, 64, 128, 256])
        dtype = rng.choice(["float32", "float32", "float32", "float64"])
        most = 10000000 * 128 // max(k, m) // (3 if train else 1) // (2 if dtype == "float64" else 1)
        return {"kind": kind, "n": _between(rng, 20000, max(40000, most)), "k": k, "m": m,
                "r": _between(rng, 4, 200), "by": rng.choice(["gather", "segment"]),
                "dtype": dtype, "train": train}
    n = _between(rng, 5000, 300000)
    return {"kind": kind, "n": n, "e": n * rng.randint(2, 8) + rng.randint(0, 63),
            "f": _between(rng, 16, 256)}


# ---------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape, dtype=torch.float32):
    return torch.randn(*shape, device="cuda", generator=gen, dtype=dtype)


def _ids(gen, hi, count):
    return torch.randint(0, hi, (count,), device="cuda", generator=gen)


def _power_law(gen, n, e, exponent=2.1, cap=20000):
    """Destinations with expected degrees ~ Zipf(exponent), about `cap` at
    most, in random edge order; sources uniform."""
    x = torch.rand(n, device="cuda", generator=gen, dtype=torch.float64)
    z = (1.0 - x).pow(-1.0 / (exponent - 1.0)).floor()
    z.clamp_(max=max(2.0, float(cap) * n * 5.0 / e))
    ends = z.cumsum(0)
    at = torch.rand(e, device="cuda", generator=gen, dtype=torch.float64) * ends[-1]
    v = torch.searchsorted(ends, at, right=True).clamp_(max=n - 1)
    return _ids(gen, n, e), v


def _communities(gen, n, e, blocks=50, intra=0.95):
    """Edges inside equal blocks of neighbouring ids, the rest anywhere."""
    size = max(1, n // blocks)
    u, v = _ids(gen, n, e), _ids(gen, n, e)
    inside = torch.rand(e, device="cuda", generator=gen) < intra
    near = torch.clamp(v // size * size + u % size, max=n - 1)
    return torch.where(inside, near, u), v


def _lengths(gen, count, rows):
    """Lengths of `rows` rows dealt to segments one by one: near Poisson."""
    return torch.bincount(_ids(gen, count, rows), minlength=count)


def _relation_lengths(gen, n, r):
    """Relation sizes as ragged as a knowledge graph's: n rows dealt by
    weights that differ by orders of magnitude."""
    w = torch.rand(r, device="cuda", generator=gen, dtype=torch.float64).pow(3) + 1e-3
    ends = (w.cumsum(0) / w.sum() * n).round().to(torch.int64)
    ends[-1] = n
    return torch.diff(ends, prepend=torch.zeros(1, dtype=torch.int64, device="cuda"))


def _inputs(case, seed):
    """The input tensors of a case, from the seed alone."""
    gen = _gen(seed)
    kind = case["kind"]
    x = {}
    if kind in ("update_all", "minibatch", "pool", "messages_f64", "link"):
        x["u"], x["v"] = _ids(gen, case["n"], case["e"]), _ids(gen, case["n"], case["e"])
    if kind == "update_all":
        x["h"] = _normal(gen, case["n"], case["f"])
        x["w"] = torch.rand(case["e"], case["f"], device="cuda", generator=gen)
    elif kind == "messages_f64":
        x["h"] = _normal(gen, case["n"], case["f"], dtype=torch.float64)
        x["w"] = torch.rand(case["e"], case["f"], device="cuda", generator=gen,
                            dtype=torch.float64)
        x["s"] = _normal(gen, case["e"], case["heads"], 1, dtype=torch.float64)
    elif kind == "gat":
        x["u"], x["v"] = _power_law(gen, case["n"], case["e"])
        x["el"] = _normal(gen, case["n"], case["heads"], 1)
        x["er"] = _normal(gen, case["n"], case["heads"], 1)
        x["h"] = _normal(gen, case["n"], case["heads"], case["d"])
        if case["train"]:
            x["gz"] = _normal(gen, case["n"], case["heads"], case["d"])
    elif kind == "gcn":
        n, e = case["n"], case["e"]
        if case["local"]:
            x["u"], x["v"] = _communities(gen, n, e)
        else:
            x["u"], x["v"] = _power_law(gen, n, e)
        du = torch.bincount(x["u"], minlength=n).float()
        dv = torch.bincount(x["v"], minlength=n).float()
        x["w"] = (du[x["u"]] * dv[x["v"]]).rsqrt().unsqueeze(1)
        x["h"] = _normal(gen, n, case["f"])
        if case["train"]:
            x["gz"] = _normal(gen, n, case["f"])
    elif kind in ("pool", "minibatch"):
        x["h"] = _normal(gen, case["n"], case["f"])
        x["gz"] = _normal(gen, case["n"], case["f"])
    elif kind == "link":
        scale = case["f"] ** -0.5
        x["h"] = _normal(gen, case["n"], case["f"]) * scale
        x["k"] = _normal(gen, case["n"], case["f"]) * scale
        if case["train"]:
            x["gs"] = _normal(gen, case["e"], 1)
    elif kind == "readout":
        rows = case["s"] * case["mean_len"]
        x["seglen"] = _lengths(gen, case["s"], rows)
        x["x"] = _normal(gen, rows, case["f"])
        if case["train"]:
            x["gs"] = _normal(gen, case["s"], case["f"])
            x["ga"] = _normal(gen, rows, case["f"])
    elif kind == "typed_mm":
        dtype = getattr(torch, case["dtype"])
        n, k, m, r = case["n"], case["k"], case["m"], case["r"]
        x["a"] = _normal(gen, n, k, dtype=dtype)
        x["b"] = _normal(gen, r, k, m, dtype=dtype) * k ** -0.5
        if case["by"] == "gather":
            x["idx"] = _ids(gen, r, n)
        else:
            x["seglen"] = _relation_lengths(gen, n, r)
        if case["train"]:
            x["gz"] = _normal(gen, n, m, dtype=dtype)
    return x


#: What a training step differentiates by.
_LEAVES = {"gat": ("h", "el", "er"), "gcn": ("h",), "pool": ("h",), "link": ("h", "k"),
           "readout": ("x",), "typed_mm": ("a", "b"), "minibatch": ("h",)}


def prepare(case, seed):
    x = _inputs(case, seed)
    if case.get("train", case["kind"] in ("pool", "minibatch")):
        for name in _LEAVES[case["kind"]]:
            x[name].requires_grad_(True)
    x["case"] = case
    if "u" in x and case["kind"] != "minibatch":  # a mini-batch's graph is the step's own
        g = dgl.graph((x.pop("u"), x.pop("v")), num_nodes=case["n"])
        if "h" in x:
            g.ndata["h"] = x["h"]
        if "w" in x:
            g.edata["w"] = x["w"]
        x["g"] = g
    return x


# ---------------------------------------------------------------- one pass


def run(x):
    case = x["case"]
    return _RUN[case["kind"]](x, case)


def _run_update_all(x, case):
    g = x["g"]
    g.update_all(fn.u_mul_e("h", "w", "m"), fn.sum("m", "sum"))
    g.update_all(fn.copy_u("h", "m"), fn.max("m", "max"))
    return {"sum": g.ndata["sum"], "max": g.ndata["max"]}


def _run_messages_f64(x, case):
    g = x["g"]
    g.update_all(fn.u_mul_e("h", "w", "m"), fn.sum("m", "sum"))
    g.update_all(fn.u_add_e("h", "w", "m"), fn.mean("m", "mean"))
    g.update_all(fn.copy_u("h", "m"), fn.max("m", "max"))
    return {"sum": g.ndata["sum"], "mean": g.ndata["mean"], "max": g.ndata["max"],
            "mul": ops.u_mul_v(g, x["h"], x["h"]), "a": ops.edge_softmax(g, x["s"])}


def _run_gat(x, case):
    g = x["g"]
    e = ops.u_add_v(g, x["el"], x["er"])
    e = torch.nn.functional.leaky_relu(e, 0.2)
    a = ops.edge_softmax(g, e)
    z = ops.u_mul_e_sum(g, x["h"], a)
    if not case["train"]:
        return {"z": z, "a": a}
    dh, del_, der = torch.autograd.grad(z, (x["h"], x["el"], x["er"]), x["gz"])
    return {"z": z, "dh": dh, "del": del_, "der": der}


def _run_gcn(x, case):
    g = x["g"]
    g.update_all(fn.u_mul_e("h", "w", "m"), fn.sum("m", "z"))
    z = g.ndata["z"]
    if not case["train"]:
        return {"z": z}
    dh, = torch.autograd.grad(z, x["h"], x["gz"])
    return {"z": z, "dh": dh}


def _run_pool(x, case):
    g = x["g"]
    g.update_all(fn.copy_u("h", "m"), fn.max("m", "z"))
    z = g.ndata["z"]
    dh, = torch.autograd.grad(z, x["h"], x["gz"])
    return {"z": z, "dh": dh}


def _run_link(x, case):
    s = ops.u_dot_v(x["g"], x["h"], x["k"])
    if not case["train"]:
        return {"s": s}
    dh, dk = torch.autograd.grad(s, (x["h"], x["k"]), x["gs"])
    return {"s": s, "dh": dh, "dk": dk}


def _run_readout(x, case):
    a = ops.segment_softmax(x["seglen"], x["x"])
    total = ops.segment_reduce(x["seglen"], x["x"], "sum")
    most = ops.segment_reduce(x["seglen"], x["x"], "max")
    if not case["train"]:
        return {"a": a, "sum": total, "max": most}
    dx, = torch.autograd.grad((a, total, most), x["x"], (x["ga"], x["gs"], x["gs"]))
    return {"a": a, "sum": total, "max": most, "dx": dx}


def _run_typed_mm(x, case):
    if case["by"] == "gather":
        z = ops.gather_mm(x["a"], x["b"], idx_b=x["idx"])
    else:
        z = ops.segment_mm(x["a"], x["b"], x["seglen"])
    if not case["train"]:
        return {"z": z}
    da, db = torch.autograd.grad(z, (x["a"], x["b"]), x["gz"])
    return {"z": z, "da": da, "db": db}


def _run_minibatch(x, case):
    g = dgl.graph((x["u"], x["v"]), num_nodes=case["n"])
    g.ndata["h"] = x["h"]
    g.update_all(fn.copy_u("h", "m"), fn.mean("m", "z"))
    z = g.ndata["z"]
    dh, = torch.autograd.grad(z, x["h"], x["gz"])
    return {"z": z, "dh": dh}


_RUN = {"update_all": _run_update_all, "messages_f64": _run_messages_f64, "gat": _run_gat,
        "gcn": _run_gcn, "pool": _run_pool, "link": _run_link, "readout": _run_readout,
        "typed_mm": _run_typed_mm, "minibatch": _run_minibatch}

# ---------------------------------------------------------------- in float64


def _chunks(count, width):
    """Slices of `count` rows of `width` float64 values, about 4 GB each."""
    step = max(1, 500_000_000 // max(1, width))
    return [slice(i, min(count, i + step)) for i in range(0, count, step)]


def _sum_rows(index, rows, value):
    """out[index[i]] += value(i) over all i, `value` giving a slice's rows."""
    out = None
    for s in _chunks(index.numel(), value.width):
        part = value(s)
        if out is None:
            out = torch.zeros((rows,) + tuple(part.shape[1:]), dtype=torch.float64, device="cuda")
        out.index_add_(0, index[s], part)
    return out


class _Rows:
    def __init__(self, width, make):
        self.width, self.make = width, make

    def __call__(self, s):
        return self.make(s)


def _softmax_by(index, rows, x):
    ix = index.view((-1,) + (1,) * (x.dim() - 1)).expand_as(x)
    top = torch.full((rows,) + tuple(x.shape[1:]), -math.inf, dtype=torch.float64, device="cuda")
    top.scatter_reduce_(0, ix, x, "amax")
    p = torch.exp(x - top[index])
    total = torch.zeros_like(top).index_add_(0, index, p)
    return p / total[index]


def _max_by(index, rows, rows_of):
    """Maxima per row of `index` (0 where there is none) and the first entry
    reaching each (-1: none); `rows_of(c)` gives column c's values."""
    count = index.numel()
    number = torch.arange(count, device="cuda")
    best, first = [], []
    for x in rows_of:
        top = torch.full((rows,), -math.inf, dtype=torch.float64, device="cuda")
        top.scatter_reduce_(0, index, x, "amax")
        hit = torch.where(x == top[index], number, torch.full_like(number, count))
        at = torch.full((rows,), count, dtype=torch.int64, device="cuda")
        at.scatter_reduce_(0, index, hit, "amin")
        best.append(torch.where(torch.isinf(top), torch.zeros_like(top), top))
        first.append(torch.where(at == count, torch.full_like(at, -1), at))
    return torch.stack(best, 1), torch.stack(first, 1)


def exact(case, seed):
    x = {k: v.double() if v.is_floating_point() else v for k, v in _inputs(case, seed).items()}
    return _EXACT[case["kind"]](x, case)


def _exact_update_all(x, case):
    n, f, u, v, h, w = case["n"], case["f"], x["u"], x["v"], x["h"], x["w"]
    most, _ = _max_by(v, n, (h[u, c] for c in range(f)))
    return {"sum": _sum_rows(v, n, _Rows(f, lambda s: h[u[s]] * w[s])), "max": most}


def _exact_messages_f64(x, case):
    n, f, u, v, h, w = case["n"], case["f"], x["u"], x["v"], x["h"], x["w"]
    most, _ = _max_by(v, n, (h[u, c] for c in range(f)))
    deg = torch.bincount(v, minlength=n).clamp(min=1).unsqueeze(1)
    return {"sum": _sum_rows(v, n, _Rows(f, lambda s: h[u[s]] * w[s])),
            "mean": _sum_rows(v, n, _Rows(f, lambda s: h[u[s]] + w[s])) / deg, "max": most,
            "mul": h[u] * h[v], "a": _softmax_by(v, n, x["s"])}


def _exact_gat(x, case):
    n, width, u, v, h = case["n"], case["heads"] * case["d"], x["u"], x["v"], x["h"]
    t = x["el"][u] + x["er"][v]
    slope = torch.where(t > 0, 1.0, 0.2).double()
    t *= slope
    a = _softmax_by(v, n, t)
    del t
    z = _sum_rows(v, n, _Rows(width, lambda s: h[u[s]] * a[s]))
    if not case["train"]:
        return {"z": z, "a": a}
    gz = x["gz"]
    dh = _sum_rows(u, n, _Rows(width, lambda s: gz[v[s]] * a[s]))
    da = torch.cat([(h[u[s]] * gz[v[s]]).sum(-1, keepdim=True)
                    for s in _chunks(u.numel(), width)])
    dt = a * (da - torch.zeros_like(x["er"]).index_add_(0, v, a * da)[v]) * slope
    return {"z": z, "dh": dh, "del": torch.zeros_like(x["el"]).index_add_(0, u, dt),
            "der": torch.zeros_like(x["er"]).index_add_(0, v, dt)}


def _exact_gcn(x, case):
    n, f, u, v, h, w = case["n"], case["f"], x["u"], x["v"], x["h"], x["w"]
    out = {"z": _sum_rows(v, n, _Rows(f, lambda s: h[u[s]] * w[s]))}
    if case["train"]:
        out["dh"] = _sum_rows(u, n, _Rows(f, lambda s: x["gz"][v[s]] * w[s]))
    return out


def _exact_pool(x, case):
    n, f, u, v, h = case["n"], case["f"], x["u"], x["v"], x["h"]
    most, first = _max_by(v, n, (h[u, c] for c in range(f)))
    dh = torch.zeros_like(h)
    for c in range(f):
        some = first[:, c] >= 0
        dh[:, c].index_add_(0, u[first[some, c]], x["gz"][some, c])
    return {"z": most, "dh": dh}


def _exact_link(x, case):
    n, f, u, v, h, k = case["n"], case["f"], x["u"], x["v"], x["h"], x["k"]
    out = {"s": torch.cat([(h[u[s]] * k[v[s]]).sum(1, keepdim=True)
                           for s in _chunks(u.numel(), f)])}
    if case["train"]:
        out["dh"] = _sum_rows(u, n, _Rows(f, lambda s: k[v[s]] * x["gs"][s]))
        out["dk"] = _sum_rows(v, n, _Rows(f, lambda s: h[u[s]] * x["gs"][s]))
    return out


def _exact_readout(x, case):
    s, f, val = case["s"], case["f"], x["x"]
    of = torch.repeat_interleave(torch.arange(s, device="cuda"), x["seglen"])
    a = _softmax_by(of, s, val)
    total = torch.zeros(s, f, dtype=torch.float64, device="cuda").index_add_(0, of, val)
    most, first = _max_by(of, s, (val[:, c] for c in range(f)))
    out = {"a": a, "sum": total, "max": most}
    if case["train"]:
        ga = x["ga"]
        dx = a * (ga - torch.zeros_like(total).index_add_(0, of, a * ga)[of]) + x["gs"][of]
        for c in range(f):
            some = first[:, c] >= 0
            dx[first[some, c], c] += x["gs"][some, c]
        out["dx"] = dx
    return out


def _exact_typed_mm(x, case):
    a, b, r = x["a"], x["b"], case["r"]
    if case["by"] == "gather":
        groups = [torch.nonzero(x["idx"] == i).view(-1) for i in range(r)]
    else:
        ends = x["seglen"].cumsum(0).tolist()
        groups = [slice(ends[i - 1] if i else 0, ends[i]) for i in range(r)]
    z = torch.empty(case["n"], case["m"], dtype=torch.float64, device="cuda")
    da, db = torch.empty_like(a), torch.empty_like(b)
    for i, rows in enumerate(groups):
        z[rows] = a[rows] @ b[i]
        if case["train"]:
            da[rows] = x["gz"][rows] @ b[i].t().contiguous()
            db[i] = a[rows].t().contiguous() @ x["gz"][rows]
    return {"z": z, "da": da, "db": db} if case["train"] else {"z": z}


def _exact_minibatch(x, case):
    n, f, u, v, h = case["n"], case["f"], x["u"], x["v"], x["h"]
    deg = torch.bincount(v, minlength=n).clamp(min=1).unsqueeze(1).double()
    gz = x["gz"] / deg
    return {"z": _sum_rows(v, n, _Rows(f, lambda s: h[u[s]])) / deg,
            "dh": _sum_rows(u, n, _Rows(f, lambda s: gz[v[s]]))}


_EXACT = {"update_all": _exact_update_all, "messages_f64": _exact_messages_f64,
          "gat": _exact_gat, "gcn": _exact_gcn, "pool": _exact_pool, "link": _exact_link,
          "readout": _exact_readout, "typed_mm": _exact_typed_mm,
          "minibatch": _exact_minibatch}

# ---------------------------------------------------------------- bounds


def work(case):
    """Each input read once and each output written once; the products and
    sums of the definition."""
    kind = case["kind"]
    n, e, f = case.get("n", 0), case.get("e", 0), case.get("f", 0)
    if kind == "update_all":
        return {"bytes": 4 * (n * f + e * f + 2 * n * f) + 8 * e, "flops": 3 * e * f}
    if kind == "messages_f64":
        k = case["heads"]
        return {"bytes": 8 * (n * f + e * f + 3 * n * f + e * f + 2 * e * k) + 8 * e,
                "flops": 6 * e * f + 4 * e * k}
    if kind == "gat":
        k, d = case["heads"], case["d"]
        b = 4 * (2 * n * k + 2 * n * k * d) + 8 * e
        if not case["train"]:
            return {"bytes": b + 4 * e * k, "flops": 2 * e * k * d + 6 * e * k}
        return {"bytes": b + 4 * (2 * n * k + 2 * n * k * d),
                "flops": 6 * e * k * d + 14 * e * k}
    if kind == "gcn":
        passes = 2 if case["train"] else 1
        return {"bytes": passes * 4 * 2 * n * f + 12 * e, "flops": passes * 2 * e * f}
    if kind == "pool":
        return {"bytes": 4 * 4 * n * f + 8 * e, "flops": e * f + n * f}
    if kind == "link":
        b = 4 * (2 * n * f + e) + 8 * e
        if not case["train"]:
            return {"bytes": b, "flops": 2 * e * f}
        return {"bytes": b + 4 * (2 * n * f + e), "flops": 6 * e * f}
    if kind == "readout":
        rows, s = case["s"] * case["mean_len"], case["s"]
        b = 4 * f * (2 * rows + 2 * s) + 8 * s
        if case["train"]:
            b += 4 * f * (2 * rows + s)
        return {"bytes": b, "flops": (12 if case["train"] else 6) * rows * f}
    if kind == "typed_mm":
        size = 8 if case["dtype"] == "float64" else 4
        k, m, r = case["k"], case["m"], case["r"]
        ids = n if case["by"] == "gather" else r
        b = size * (n * (k + m) + r * k * m) + 8 * ids
        if case["train"]:
            b += size * (n * (k + m) + r * k * m)
        return {"bytes": b, "flops": (6 if case["train"] else 2) * n * k * m}
    return {"bytes": 4 * 4 * n * f + 16 * e, "flops": 2 * e * f + 2 * n * f}


def tolerance(case):
    """About four times the largest error against `exact` over the ranges:
    sums of float32 (float64) terms in one order or another; the relation
    weights' gradients add up thousands of rows."""
    double = case["kind"] == "messages_f64" or case.get("dtype") == "float64"
    if case["kind"] == "typed_mm":
        return {"rel": 4e-14, "max": 5e-13} if double else {"rel": 5e-6, "max": 1e-4}
    return {"rel": 1e-15, "max": 1e-14} if double else {"rel": 2e-6, "max": 3e-5}
