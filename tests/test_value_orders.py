"""The orders a CSR keeps for moving edge values (heterograph._ValueOrder),
host side: their lifetime, on CPU index tensors."""

import gc
import weakref

import pytest
import torch

import mojodgl.heterograph as hg
from mojodgl import _lib


@pytest.fixture
def csr(monkeypatch):
    monkeypatch.setattr(_lib, "settle", lambda: None)
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
