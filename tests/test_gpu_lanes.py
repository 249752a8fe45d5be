"""gspmm's lane layouts at the widths where they can go wrong: runs of columns
that no lane width divides (their last lane shares columns with the one before
it), one to 64 lanes per row and several slabs, rows that end inside, at and
just past a batch of ids, misaligned operands and results; and the fused
backward pass of attention over runs of any length. Sums fold in the oracle's
order, so whole rows are equal bit for bit."""

import ctypes

import numpy as np
import pytest
import torch

import mojodgl as dgl
import mojodgl.ops as ops
import oracle
from mojodgl import _lib, heterograph

# 1 to 64 lanes of 4, 2 or 1 columns, remainders on both sides, 2 to 5 slabs
WIDTHS = [1, 2, 3, 4, 5, 7, 9, 15, 16, 17, 31, 33, 47, 63, 66, 97, 127, 130, 255, 257, 258, 515]


def ragged_graph(seed, n=160, most=40):
    """In-degrees 0, 1, 2, ... `most`, then random, and a hub of 700."""
    rng = np.random.default_rng(seed)
    deg = np.concatenate([np.arange(most + 1), rng.integers(0, most, n - most - 2), [700]])
    v = np.repeat(np.arange(n), deg)
    v = v[rng.permutation(v.size)]
    return rng.integers(0, n, v.size), v, n


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", WIDTHS)
def test_any_width(dtype, d, monkeypatch):
    """copy, a weight per edge and an edge row per edge, sum / mean / max /
    min with args, operands one element off a 16-byte boundary, against the
    oracle bit for bit (no row split)."""
    from mojodgl import heterograph

    monkeypatch.setattr(heterograph, "CHUNK_LEN", 1 << 20)
    u, v, n = ragged_graph(d)
    rng = np.random.default_rng(d + 1)
    g = dgl.graph((u, v), num_nodes=n)

    def off(a):  # a GPU copy that starts one element into its buffer
        buf = torch.empty(a.size + 1, dtype=torch.from_numpy(a).dtype, device="cuda")
        view = buf[1:].view(a.shape)
        view.copy_(torch.from_numpy(a))
        return view

    x = rng.normal(size=(n, d)).astype(dtype)
    for op, y in (("copy_lhs", None), ("mul", (rng.random((u.size, 1)) + 0.5).astype(dtype)),
                  ("add", rng.normal(size=(u.size, d)).astype(dtype))):
        for red in ("sum", "mean", "max", "min"):
            got, (au, ae) = ops.spmm._gspmm(g, op, red, off(x), None if y is None else off(y))
            what = "{} {} d={}".format(op, red, d)
            if red in ("max", "min"):
                want, ru, re_ = oracle.gspmm(u, v, n, op, red, x, y, dtype, with_arg=True)
                np.testing.assert_array_equal(au.cpu().numpy(), ru, err_msg=what)
                np.testing.assert_array_equal(ae.cpu().numpy(), re_, err_msg=what)
            else:
                want = oracle.gspmm(u, v, n, op, red, x, y, dtype)
            np.testing.assert_array_equal(got.cpu().numpy(), want, err_msg=what)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("heads,d", [(1, 7), (2, 5), (8, 25), (3, 10), (6, 7), (4, 3), (5, 2),
                                     (3, 33), (2, 130)])
def test_heads_of_any_width(dtype, heads, d):
    """One weight per head: no lane straddles two heads. The same graph split
    into chunks of 16 slots folds in another order (within tolerance)."""
    u, v, n = ragged_graph(heads * 100 + d)
    rng = np.random.default_rng(d)
    x = rng.normal(size=(n, heads, d)).astype(dtype)
    y = rng.normal(size=(u.size, heads, 1)).astype(dtype)
    keep = v != n - 1  # without the hub no row is split
    g = dgl.graph((u[keep], v[keep]), num_nodes=n)
    np.testing.assert_array_equal(
        ops.u_mul_e_sum(g, x, y[keep]),
        oracle.gspmm(u[keep], v[keep], n, "mul", "sum", x, y[keep], dtype))
    g = dgl.graph((u, v), num_nodes=n)
    from mojodgl.ops import spmm

    got = spmm._run(g, "mul", "sum", torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda(),
                    narrow_split=16)[0].cpu().numpy()
    ref = oracle.gspmm(u, v, n, "mul", "sum", x, y, np.float64)
    bound = oracle.gspmm(u, v, n, "mul", "sum", np.abs(x), np.abs(y), np.float64)
    # a sum of k terms in another order: at most k * eps of the terms' magnitudes
    assert (np.abs(got - ref) <= 700 * np.finfo(dtype).eps * bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("heads,d", [(1, 7), (8, 7), (4, 25), (3, 10), (2, 100), (1, 126),
                                     (8, 33)])
def test_fused_dot_over_any_run(dtype, heads, d):
    """Both gradients of u_mul_e_sum in one pass, runs that no power of two of
    lanes covers exactly: dX equals the separate gspmm bit for bit, dY the
    separate dot to rounding (a sum of d products: d * eps of their
    magnitudes)."""
    from mojodgl.ops import spmm

    u, v, n = ragged_graph(7 * heads + d)
    g = dgl.graph((u, v), num_nodes=n)
    gen = torch.Generator(device="cuda").manual_seed(d)
    G = torch.randn(n, heads, d, device="cuda", generator=gen, dtype=torch.float64).to(dtype)
    X = torch.randn(n, heads, d, device="cuda", generator=gen, dtype=torch.float64).to(dtype)
    Y = torch.randn(u.size, heads, 1, device="cuda", generator=gen, dtype=torch.float64).to(dtype)
    fused = spmm._mul_sum_dot(g, G, Y, X)
    assert fused is not None
    dx = spmm._run(g, "mul", "sum", G, Y, kind="out")[0]
    assert torch.equal(fused[0], dx.reshape(X.shape))
    ud, vd = torch.from_numpy(u).cuda(), torch.from_numpy(v).cuda()
    t = X.double()[ud] * G.double()[vd]
    off = (fused[1].double() - t.sum(-1, keepdim=True)).abs()
    assert bool((off <= 2 * d * torch.finfo(dtype).eps * t.abs().sum(-1, keepdim=True)).all())


def test_layout_covers_every_column():
    """mdgl_gspmm_layout with any alignment allowed: lanes of `vec` columns,
    enough of them for every run, at most 64 to a slab (no launch)."""
    lib = _lib.lib()
    for dt in (0, 1):
        for heads, d in [(1, w) for w in WIDTHS] + [(8, 25), (4, 3), (6, 7), (3, 130)]:
            vec, group, lanes = ctypes.c_int64(), ctypes.c_int64(), ctypes.c_int64()
            ls, rs = (ctypes.c_int64 * 2)(heads, d), (ctypes.c_int64 * 2)(heads, 1)
            rc = lib.mdgl_gspmm_layout(_lib.BINARY_OPS["mul"], heads * d, heads, heads * d, 2, ls,
                                       rs, 4, 4, _lib.ANY_ALIGNMENT, dt, ctypes.byref(vec),
                                       ctypes.byref(group), ctypes.byref(lanes))
            assert rc == 0
            run = d if heads > 1 or d > 1 else 1
            assert vec.value <= max(run, 1) and lanes.value * vec.value >= heads * d
            assert lanes.value == heads * -(-run // vec.value)
            assert group.value in (16, 32, 64)
            assert group.value >= min(lanes.value, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("d", [1, 3, 16, 47, 100, 130, 258])
@pytest.mark.parametrize("op", ["copy_lhs", "add", "sub"])
def test_selected_sum_is_the_max_gradient(dtype, d, op):
    """The gradient of max / min in the node operand alone, without the
    per-edge gradients: equal bit for bit to the path through them (taken when
    the edge operand's gradient is asked for too), duplicate edges, equal
    messages and nodes without edges among the inputs."""
    u, v, n = ragged_graph(d + 5)
    u = np.concatenate([u, u[:200]])  # the same edge twice: the first one wins
    v = np.concatenate([v, v[:200]])
    g = dgl.graph((u, v), num_nodes=n)
    gen = torch.Generator(device="cuda").manual_seed(d)
    x = torch.randn(n, d, device="cuda", generator=gen, dtype=torch.float64).to(dtype)
    x[:, 0] = torch.round(x[:, 0])  # equal messages
    y = torch.randn(u.size, d, device="cuda", generator=gen, dtype=torch.float64).to(dtype)
    G = torch.randn(n, d, device="cuda", generator=gen, dtype=torch.float64).to(dtype)
    x.requires_grad_(True)
    for red in ("max", "min"):
        if op == "copy_lhs":
            dx, = torch.autograd.grad(ops.gspmm(g, op, red, x, None), x, G)
            with torch.no_grad():
                _, (_, ae) = ops.spmm._gspmm(g, op, red, x.detach(), None)
            from mojodgl.ops import _autograd

            M = _autograd._edge_grad(g, G, ae, False, 1.0)
            want = _autograd._node_reduce(g, M, "u")
        else:
            dx, = torch.autograd.grad(ops.gspmm(g, op, red, x, y), x, G)
            yy = y.clone().requires_grad_(True)
            want, _ = torch.autograd.grad(ops.gspmm(g, op, red, x, yy), (x, yy), G)
        assert torch.equal(dx, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(64,), (100,), (3, 67)])
@pytest.mark.parametrize("swap", [False, True])
def test_edge_dot_in_slot_order(dtype, shape, swap, monkeypatch):
    """u_dot_v / v_dot_u computed slot by slot of the in-CSR equal the same
    dots taken edge by edge, bit for bit; the first call on a graph without a
    CSR does not build one."""
    from mojodgl.ops import sddmm

    monkeypatch.setattr(sddmm, "DOT_SLOT_MIN_EDGES", 1)
    u, v, n = ragged_graph(sum(shape))
    g = dgl.graph((torch.from_numpy(u).cuda(), torch.from_numpy(v).cuda()), num_nodes=n)
    gen = torch.Generator(device="cuda").manual_seed(3)
    x, y = (torch.randn(n, *shape, device="cuda", generator=gen, dtype=torch.float64).to(dtype)
            for _ in range(2))
    dot = ops.v_dot_u if swap else ops.u_dot_v
    first = dot(g, x, y)
    assert g._current_csr("in") is None
    second = dot(g, x, y)
    assert g._current_csr("in") is not None and g._current_csr("in")._slot_of_eid is not None
    assert first.shape == second.shape and torch.equal(first, second)


@pytest.mark.gpu
def test_rows_past_one_launch():
    """16 lanes a row are 2**32 work-items at 2**28 rows, more than HIP launches
    at once: the rows beyond are reduced too (every 2**20th row and the last
    two hold one edge, the others none)."""
    n = (1 << 28) + 4097
    filled = torch.cat([torch.arange(0, n, 1 << 20, device="cuda"),
                        torch.tensor([n - 2, n - 1], device="cuda")])
    E = filled.numel()
    indptr = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    indptr[filled + 1] = 1
    indptr = torch.cumsum(indptr, 0, dtype=torch.int32)
    index = torch.arange(E, dtype=torch.int32, device="cuda")
    x = torch.arange(1, E + 1, dtype=torch.float32, device="cuda")
    out = torch.full((n,), -1.0, device="cuda")
    _lib.check(_lib.lib().mdgl_gspmm(
        indptr.data_ptr(), index.data_ptr(), index.data_ptr(), x.data_ptr(), None, out.data_ptr(),
        n, _lib.OP_COPY_LHS, 1, 1, 1, 0, None, 0, None, None, None, None, None, None, 0, 0, None,
        None, 0, None, 0, _lib.ANY_ALIGNMENT, 0, _lib.stream()), "gspmm")
    want = torch.zeros(n, device="cuda")
    want[filled] = x
    assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,widths", [(np.float32, (23, 24, 25)), (np.float64, (11, 12, 13))])
def test_edge_rows_either_side_of_streaming(dtype, widths, monkeypatch):
    """Edge rows of 96 bytes or more are read past the caches: the same bits on
    both sides, with the node operand consecutive, one value per row, and
    absent."""
    monkeypatch.setattr(heterograph, "CHUNK_LEN", 1 << 20)  # no row split
    u, v, n = ragged_graph(widths[0])
    g = dgl.graph((u, v), num_nodes=n)
    rng = np.random.default_rng(6)
    for d in widths:
        w = rng.normal(size=(u.size, d)).astype(dtype)
        wt = torch.from_numpy(w).cuda()
        for red in ("sum", "max"):
            want = oracle.gspmm(u, v, n, "copy_rhs", red, None, w, dtype)
            got = ops.gspmm(g, "copy_rhs", red, None, wt)
            np.testing.assert_array_equal(got.cpu().numpy(), want)
            for dl in (d, 1):
                h = rng.normal(size=(n, dl)).astype(dtype)
                got = ops.gspmm(g, "mul", red, torch.from_numpy(h).cuda(), wt)
                want = oracle.gspmm(u, v, n, "mul", red, np.broadcast_to(h, (n, d)).copy(), w,
                                    dtype)
                np.testing.assert_array_equal(got.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [1, 2, 3, 5, 8, 9, 16, 17, 31, 33])
@pytest.mark.parametrize("lanes", [_lib.ROW_LANES_2, _lib.ROW_LANES_4])
def test_rows_of_few_lanes(dtype, d, lanes, monkeypatch):
    """Rows that take only the lanes they need, each lane loading its row's ids:
    the oracle's bits for whole rows of 0 to 40 edges and a hub, and the same
    bits as 16 lanes a row for split rows and the backward passes' kernels."""
    u, v, n = ragged_graph(d)
    rng = np.random.default_rng(d + 7)
    x = rng.normal(size=(n, d)).astype(dtype)
    w = (rng.random((u.size, 1)) + 0.5).astype(dtype)
    e = rng.normal(size=(u.size, d)).astype(dtype)
    operands = (("copy_lhs", x, None), ("copy_rhs", None, e), ("mul", x, w), ("add", x, e),
                ("div", x[:, :1].copy(), e))

    def gpu(a):
        return None if a is None else torch.from_numpy(a).cuda()

    with monkeypatch.context() as m:
        m.setattr(ops.spmm, "_row_lanes", lambda *counts: lanes)
        m.setattr(heterograph, "CHUNK_LEN", 1 << 20)
        g = dgl.graph((u, v), num_nodes=n)
        for op, a, b in operands:
            wide = None if a is None else np.ascontiguousarray(np.broadcast_to(a, (n, d)))
            for red in ("sum", "mean", "max", "min"):
                got, (au, ae) = ops.spmm._gspmm(g, op, red, gpu(a), gpu(b))
                what = "{} {}".format(op, red)
                if red in ("max", "min"):
                    want, ru, re_ = oracle.gspmm(u, v, n, op, red, wide, b, dtype, with_arg=True)
                    if op != "copy_rhs":
                        np.testing.assert_array_equal(au.cpu().numpy(), ru, err_msg=what)
                    if op != "copy_lhs":
                        np.testing.assert_array_equal(ae.cpu().numpy(), re_, err_msg=what)
                else:
                    want = oracle.gspmm(u, v, n, op, red, wide, b, dtype)
                np.testing.assert_array_equal(got.cpu().numpy(), want, err_msg=what)

    def backward(fewest):
        with monkeypatch.context() as m:
            m.setattr(ops.spmm, "_row_lanes", lambda *counts: fewest)
            g = dgl.graph((u, v), num_nodes=n)
            out = []
            for op, a, b in operands:
                leaves = [gpu(t).requires_grad_(True) for t in (a, b) if t is not None]
                for red in ("sum", "max"):
                    z = ops.gspmm(g, op, red, *((None,) if a is None else ()), *leaves,
                                  *((None,) if b is None else ()))
                    G = torch.cos(torch.arange(z.numel(), device="cuda").reshape(z.shape)).to(z)
                    out += [z.detach(), *torch.autograd.grad(z, leaves, G)]
                if op in ("copy_lhs", "add"):  # the node operand alone
                    z = ops.gspmm(g, op, "max", leaves[0], None if b is None else gpu(b))
                    out += torch.autograd.grad(z, leaves[:1], G)
            return out

    for got, want in zip(backward(lanes), backward(0)):
        assert torch.equal(got, want)
