"""The orders a CSR keeps for moving edge values (heterograph._ValueOrder),
their lifetime on CPU index tensors, and what is left where the GPU's memory
has no room for them."""

import gc
import weakref

import numpy as np
import pytest
import torch

import mojodgl as dgl
import mojodgl.heterograph as hg
import mojodgl.ops as ops
from mojodgl import _lib


@pytest.fixture
def csr(monkeypatch):
    monkeypatch.setattr(_lib, "settle", lambda: None)
    monkeypatch.setattr(hg, "_inverse_permutation",
                        lambda p: torch.argsort(p.long()).to(torch.int32))
    indptr = torch.tensor([0, 2, 3, 5], dtype=torch.int32)
    indices = torch.tensor([0, 1, 2, 1, 0], dtype=torch.int32)
    eid = torch.tensor([3, 0, 4, 2, 1], dtype=torch.int32)
    return [hg._DeviceCSR(hg._RawCSR(indptr, indices, eid), 512)]


def test_orders_do_not_outlive_their_csr(csr):
    """The CSR (and with it the graph's GPU memory) goes with its last
    reference, whichever orders were made: nothing waits for the cyclic
    collector."""
    one = csr.pop()
    edge, slot = one.edge_values(), one.slot_values()
    assert slot._gather.tolist() == one.slot_of_eid().tolist() == [1, 4, 3, 0, 2]
    assert edge._gather is one.eid
    gone = weakref.ref(one)
    gc.collect()
    gc.disable()
    try:
        del one, edge, slot
        assert gone() is None
    finally:
        gc.enable()


def test_a_plan_without_room_is_given_up(csr, monkeypatch):
    """The call that would build the plan gathers instead, and no later call
    tries again."""
    monkeypatch.setattr(hg, "VALUE_ORDER_MIN", 1)
    monkeypatch.setattr(hg, "VALUE_ORDER_CALLS", 1)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    order = csr[0].edge_values()
    tried = []

    def build():
        tried.append(1)
        raise torch.OutOfMemoryError("no room")

    monkeypatch.setattr(order, "_build", build)
    assert [order.planned() for _ in range(4)] == [False] * 4
    assert len(tried) == 1


@pytest.mark.gpu
def test_a_move_without_room_for_its_second_buffer_gathers(monkeypatch):
    monkeypatch.setattr(hg, "VALUE_ORDER_MIN", 1)
    monkeypatch.setattr(hg, "VALUE_ORDER_CALLS", 0)
    rng = np.random.default_rng(3)
    g = dgl.graph((rng.integers(0, 500, 40001), rng.integers(0, 500, 40001)), num_nodes=500)
    csr = g._device_csr("in")
    order = csr.edge_values()
    w = torch.rand(40001, 1, device="cuda")
    assert order.planned()
    real, made = torch.empty_like, []

    def empty_like(t):
        made.append(1)
        if len(made) == 2:
            raise torch.OutOfMemoryError("no room")
        return real(t)

    monkeypatch.setattr(torch, "empty_like", empty_like)
    got = order(w, 0)
    monkeypatch.setattr(torch, "empty_like", real)
    assert len(made) == 2
    assert torch.equal(got, w[csr.eid.long()]) and torch.equal(order(w, 0), got)


@pytest.mark.gpu
def test_a_dot_without_room_for_the_slot_order_goes_edge_by_edge(monkeypatch):
    from mojodgl.ops import sddmm

    monkeypatch.setattr(sddmm, "DOT_SLOT_MIN_EDGES", 1)
    rng = np.random.default_rng(4)
    g = dgl.graph((rng.integers(0, 90, 3000), rng.integers(0, 90, 3000)), num_nodes=90)
    x = torch.randn(90, 40, device="cuda")
    want = ops.gsddmm(g, "dot", x, x)  # the first dot of a graph: edge by edge
    tried = []

    def slot_dot(*args):
        tried.append(1)
        raise torch.OutOfMemoryError("no room")

    monkeypatch.setattr(sddmm, "_slot_dot", slot_dot)
    for _ in range(3):
        assert torch.equal(ops.gsddmm(g, "dot", x, x), want)
    assert len(tried) == 1


@pytest.mark.parametrize("n,plans", [(2_000_000, False), (3_000_000, False), (8_000_000, True)])
def test_a_plan_is_built_only_where_its_moves_are_faster(n, plans, monkeypatch):
    """A gather of 2M values takes 23 us and a planned move 26; the build at 3M
    costs 30 moves' savings, at 8M nine."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    order = hg._ValueOrder(torch.empty(n, dtype=torch.int32))
    monkeypatch.setattr(order, "_build", lambda: (None,) * 3)
    assert not any(order.planned() for _ in range(hg.VALUE_ORDER_CALLS))
    assert order.planned() == plans


@pytest.mark.gpu
def test_scalar_weights_of_packed_rows_replay_until_the_plan(monkeypatch):
    """Rows packed several to a wavefront read a scalar weight by edge id until
    its order is planned: such calls replay their launch, count towards the
    plan, and take the full path from then on, with the same bits."""
    from mojodgl.ops import spmm

    monkeypatch.setattr(hg, "VALUE_ORDER_MIN", 1)
    monkeypatch.setattr(hg, "VALUE_ORDER_CALLS", 4)
    monkeypatch.setattr(spmm, "CSR_ORDER_MIN_EDGES", 1)
    rng = np.random.default_rng(5)
    n, e = 300, 20000
    g = dgl.graph((rng.integers(0, n, e), rng.integers(0, n, e)), num_nodes=n)
    h, w = torch.randn(n, 24, device="cuda"), torch.rand(e, 1, device="cuda")
    want = ops.u_mul_e_sum(g, h, w)
    assert len(g._launches) == 1
    order = next(iter(g._launches.values())).order
    for _ in range(3):
        assert torch.equal(ops.u_mul_e_sum(g, h, w), want)
    assert order._plan is None
    for _ in range(3):
        assert torch.equal(ops.u_mul_e_sum(g, h, w), want)
    assert order._plan is not None and order is g._device_csr("in").edge_values()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,d,slots", [(torch.float32, 256, True), (torch.float32, 257, False),
                                           (torch.float64, 128, True), (torch.float64, 129, False)])
def test_dots_too_wide_for_the_slot_kernel_build_no_csr(dtype, d, slots, monkeypatch):
    """64 lanes of 16 bytes hold a destination's row; a wider dot goes edge by
    edge and asks for neither the in-CSR nor a second buffer."""
    from mojodgl.ops import sddmm

    monkeypatch.setattr(sddmm, "DOT_SLOT_MIN_EDGES", 1)
    rng = np.random.default_rng(d)
    u, v = rng.integers(0, 50, 700), rng.integers(0, 50, 700)
    g = dgl.graph((u, v), num_nodes=50)
    x, y = (torch.randint(-8, 9, (50, d), device="cuda").to(dtype) for _ in range(2))
    for _ in range(3):  # whole numbers: exact in any order
        got = ops.u_dot_v(g, x, y)
        assert torch.equal(got, (x[u] * y[v]).sum(-1, keepdim=True))
    assert (g._current_csr("in") is not None) == slots


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,d", [(torch.float32, 32), (torch.float64, 16)])
def test_dots_of_one_line_go_slot_by_slot_on_even_graphs_only(dtype, d, monkeypatch):
    """Rows of 128 bytes: slot by slot from 16 edges a row on when no row has more
    than four times that; one column more takes the slot order in any case. The
    results are the same bits either way."""
    from mojodgl.ops import sddmm

    monkeypatch.setattr(sddmm, "DOT_SLOT_MIN_EDGES", 1)
    calls = []
    real = sddmm._slot_dot
    monkeypatch.setattr(sddmm, "_slot_dot", lambda *a: calls.append(1) or real(*a))
    rng = np.random.default_rng(d)
    n = 60
    even = np.repeat(np.arange(n), 20)
    hub = np.concatenate([even, np.full(400, 7)])
    few = np.repeat(np.arange(n), 15)
    for v, slots in ((even, True), (hub, False), (few, False)):
        u = rng.integers(0, n, v.size)
        for width in (d, d + 1):
            g = dgl.graph((u, v), num_nodes=n)
            x, y = (torch.randn(n, width, device="cuda", dtype=dtype) for _ in range(2))
            want = ops.u_dot_v(g, x, y)  # the first dot of a graph: edge by edge
            del calls[:]
            for _ in range(2):
                assert torch.equal(ops.u_dot_v(g, x, y), want)
            assert bool(calls) == (slots or width > d)
