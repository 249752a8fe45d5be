"""Edge-wise kernels at the widths where their lanes end, values moved by a
planned permutation, and graphs made from GPU endpoints."""

import numpy as np
import pytest
import torch

import mojodgl as dgl
import mojodgl.ops as ops
import oracle
from mojodgl import DGLError, heterograph

pytestmark = pytest.mark.gpu


def small_graph(seed, n=70, e=900):
    rng = np.random.default_rng(seed)
    u, v = rng.integers(0, n, e), rng.integers(0, n, e)
    return u, v, n


def shifted(a):
    """A GPU copy that starts one element into its buffer."""
    buf = torch.empty(a.size + 1, dtype=torch.from_numpy(a).dtype, device="cuda")
    view = buf[1:].view(a.shape)
    view.copy_(torch.from_numpy(a))
    return view


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("ls,rs", [((w,), (w,)) for w in (1, 2, 3, 5, 7, 31, 33, 66, 67, 130, 257)]
                         + [((5, 7), (5, 1)), ((8, 25), (8, 1)), ((3, 2), (3, 1)), ((1,), (9,)),
                            ((4, 1), (1, 6)), ((2, 3, 5), (2, 1, 5))])
def test_gsddmm_any_width(dtype, ls, rs):
    """One operation per element, so equal bit for bit, whatever the targets."""
    u, v, n = small_graph(sum(ls))
    rng = np.random.default_rng(len(ls))
    g = dgl.graph((u, v), num_nodes=n)
    rows = {"u": u, "v": v, "e": np.arange(u.size)}
    for lt, rt in (("u", "v"), ("e", "u"), ("v", "e")):
        x = rng.normal(size=((u.size if lt == "e" else n),) + ls).astype(dtype)
        y = rng.normal(size=((u.size if rt == "e" else n),) + rs).astype(dtype)
        for op, f in (("add", np.add), ("sub", np.subtract), ("mul", np.multiply),
                      ("div", np.divide)):
            got = ops.gsddmm(g, op, shifted(x), shifted(y), lhs_target=lt, rhs_target=rt)
            np.testing.assert_array_equal(got.cpu().numpy(), f(x[rows[lt]], y[rows[rt]]))
        got = ops.gsddmm(g, "copy_lhs", shifted(x), None, lhs_target=lt)
        np.testing.assert_array_equal(got.cpu().numpy(), x[rows[lt]])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(1,), (2,), (3,), (4,), (5,), (9,), (19,), (67,), (129,), (255,),
                                   (257,), (515,), (3, 7), (4, 25), (2, 300)])
def test_dot_any_width(dtype, shape):
    """A dot of k products in any order: k eps of their magnitudes; an infinite
    element reaches its own edges as IEEE products give it."""
    u, v, n = small_graph(sum(shape))
    rng = np.random.default_rng(7)
    g = dgl.graph((u, v), num_nodes=n)
    x = rng.normal(size=(n,) + shape).astype(dtype)
    y = rng.normal(size=(n,) + shape).astype(dtype)
    x[3, ..., -1] = np.inf
    x[4, ..., 0] = np.nan
    got = ops.u_dot_v(g, shifted(x), shifted(y)).cpu().numpy().astype(np.float64)
    with np.errstate(invalid="ignore"):
        terms = x.astype(np.float64)[u] * y.astype(np.float64)[v]
        ref = terms.sum(-1, keepdims=True)
    fine = np.isfinite(ref)
    np.testing.assert_array_equal(fine, np.isfinite(got))
    np.testing.assert_array_equal(got[~fine & ~np.isnan(ref)], ref[~fine & ~np.isnan(ref)])
    bound = 2 * shape[-1] * np.finfo(dtype).eps * np.abs(terms).sum(-1, keepdims=True)
    assert (np.abs(got - ref)[fine] <= bound[fine] + 1e-300).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("e", [1, 2000, 16383, 16384, 16385, 70000])
def test_planned_order_equals_the_gather(dtype, e, monkeypatch):
    """The two-pass move of one value per edge, both ways, and a scalar edge
    weight before and after the plan is there."""
    monkeypatch.setattr(heterograph, "VALUE_ORDER_MIN", 1)
    monkeypatch.setattr(heterograph, "VALUE_ORDER_CALLS", 2)
    monkeypatch.setattr(ops.spmm, "CSR_ORDER_MIN_EDGES", 0)
    n = max(2, e // 9)
    u, v, n = small_graph(e, n, e)
    g = dgl.graph((u, v), num_nodes=n)
    w = torch.randn(e, 1, device="cuda", dtype=torch.float64).to(dtype)
    x = torch.randn(n, 12, device="cuda", dtype=torch.float64).to(dtype)
    code = 0 if dtype == torch.float32 else 1
    csr = g._device_csr("in")
    for order, index in ((csr.edge_values(), csr.eid), (csr.slot_values(), csr.slot_of_eid())):
        for _ in range(2):
            assert not order.planned()
        assert torch.equal(order(w, code), w[index.long()])
        assert order.planned()
        assert torch.equal(order(w, code), w[index.long()])
    h = dgl.graph((u, v), num_nodes=n)
    results = [ops.u_mul_e_sum(h, x, w) for _ in range(4)]
    assert h._device_csr("in").edge_values()._plan is not None
    assert all(torch.equal(r, results[0]) for r in results)
    np.testing.assert_array_equal(
        results[0].cpu().numpy(),
        oracle.gspmm(u, v, n, "mul", "sum", x.cpu().numpy(), w.cpu().numpy(),
                     np.float32 if code == 0 else np.float64))


@pytest.mark.parametrize("e", [1, 255, 257, 131073, 400003])
def test_graph_from_gpu_endpoints(e, monkeypatch):
    """int64 GPU endpoints in one pass: the same graph as from host arrays and
    from int32 tensors, the range checked with the same error."""
    u, v, n = small_graph(e, max(1, e // 3), e)
    ud, vd = torch.from_numpy(u).cuda(), torch.from_numpy(v).cuda()
    host = dgl.graph((u, v), num_nodes=n)
    (du, dv), lo, hi = heterograph._ingest_coo(ud, vd)
    assert torch.equal(du.long(), ud) and torch.equal(dv.long(), vd)
    assert (lo, hi) == (min(u.min(), v.min()), max(u.max(), v.max()))
    calls = []
    ingest = heterograph._ingest_coo
    monkeypatch.setattr(heterograph, "_ingest_coo", lambda *a: calls.append(1) or ingest(*a))
    dgl.graph((ud, vd), num_nodes=n)
    assert calls  # int64 tensors on this GPU take it
    for g in (dgl.graph((ud, vd), num_nodes=n), dgl.graph((ud.int(), vd.int()), num_nodes=n),
              dgl.graph((ud.repeat_interleave(2)[::2], vd), num_nodes=n)):
        for kind in ("in", "out"):
            a, b = g._device_csr(kind), host._device_csr(kind)
            assert torch.equal(a.indptr, b.indptr) and torch.equal(a.indices, b.indices)
            assert torch.equal(a.eid, b.eid)
            np.testing.assert_array_equal(a.host_indptr, b.host_indptr)
    assert dgl.graph((ud, vd)).number_of_nodes() == int(max(u.max(), v.max())) + 1
    for at, bad in ((0, -1), (e - 1, n), (e // 2, 1 << 40)):
        x = ud.clone()
        x[at] = bad
        with pytest.raises(DGLError, match="node ids must be in"):
            dgl.graph((x, vd), num_nodes=n)
        with pytest.raises(DGLError, match="node ids must be in"):
            dgl.graph((vd, x), num_nodes=n)
