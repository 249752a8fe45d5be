"""gsddmm and its generated variants (reference python/mojodgl/ops/sddmm.py).

Same entry points, argument meaning and errors as the reference, with two
differences: operands broadcast with NumPy's rules (the reference accepts
1-D and 2-D features only, widening a width-1 operand by copying it,
sddmm.py:50-68), and the result keeps the operands' float32/float64 dtype.
"""

from __future__ import annotations

import math
import sys
from itertools import product

import numpy as np
import torch

from .. import _lib
from .._lib import BINARY_OPS, OP_COPY_LHS, OP_COPY_RHS, TARGETS
from ..base import DGLError
from . import _autograd

__all__ = ["gsddmm", "copy_u", "copy_v", "copy_e"]


def _shape(a):
    if isinstance(a, (np.ndarray, torch.Tensor, _lib.Feat)):
        return tuple(a.shape)
    return tuple(np.shape(a))


def reshape_lhs_rhs(lhs_data, rhs_data):
    r"""Expand dims so that there will be no broadcasting issues with different
    number of dimensions. For example, given two shapes (N, 3, 1), (E, 5, 3, 4)
    that are valid broadcastable shapes, change them to (N, 1, 3, 1) and
    (E, 5, 3, 4).

    The padding goes right after the first (node / edge) axis
    (reference sddmm.py:24-47); numpy arrays and tensors are reshaped as views.
    """
    lhs_shape, rhs_shape = _shape(lhs_data), _shape(rhs_data)
    if len(lhs_shape) != len(rhs_shape):
        nd = max(len(lhs_shape), len(rhs_shape))
        new_l = (lhs_shape[0],) + (1,) * (nd - len(lhs_shape)) + lhs_shape[1:]
        new_r = (rhs_shape[0],) + (1,) * (nd - len(rhs_shape)) + rhs_shape[1:]
        lhs_data = _reshape(lhs_data, new_l)
        rhs_data = _reshape(rhs_data, new_r)
    return lhs_data, rhs_data


def _reshape(a, shape):
    if isinstance(a, _lib.Feat):
        return _lib.Feat(a.data.reshape(shape), a.is_torch, a.device)
    if isinstance(a, (np.ndarray, torch.Tensor)):
        return a.reshape(shape)
    return np.reshape(a, shape)


def feat_shape(shape):
    """Feature shape of an operand; a 1-D operand is read as (n, 1)."""
    shape = tuple(shape)
    return shape[1:] if len(shape) > 1 else (1,)


def width(shape) -> int:
    w = 1
    for x in feat_shape(shape):
        w *= int(x)
    return w


def out_feat_shape(lshape, rshape, dot=False):
    """Broadcast feature shape of two padded operands (dot: last axis contracted)."""
    lf, rf = feat_shape(lshape), feat_shape(rshape)
    if dot:
        if lf[-1] != rf[-1]:
            raise DGLError("dot needs matching feature widths, {} vs {}".format(lf[-1], rf[-1]))
        lf, rf = lf[:-1], rf[:-1]
    if lf == rf:
        return lf + ((1,) if dot else ())
    try:
        out = tuple(np.broadcast_shapes(lf, rf))
    except ValueError:
        raise DGLError("operands are not broadcastable: {} and {}".format(lshape, rshape))
    return out + ((1,) if dot else ())


_SHAPE_ARGS = {}


def shape_ptrs(lshape, rshape):
    """(nd, lhs feature shape, rhs feature shape, their addresses, key) for
    the C ABI: int64 host arrays, kept per shape pair (they are only read),
    their data pointers, which the caller passes while it holds the arrays,
    and the pair of feature-shape tuples they hold."""
    key = (feat_shape(lshape), feat_shape(rshape))
    got = _SHAPE_ARGS.get(key)
    if got is None:
        lf = np.ascontiguousarray(key[0], dtype=np.int64)
        rf = np.ascontiguousarray(key[1], dtype=np.int64)
        assert lf.size == rf.size
        lf.flags.writeable = False
        rf.flags.writeable = False
        got = (int(lf.size), lf, rf, lf.ctypes.data, rf.ctypes.data, key)
        if len(_SHAPE_ARGS) < 4096:
            _SHAPE_ARGS[key] = got
    return got


def _check_rows(a, want: int, what: str) -> None:
    """Reject an operand whose row count is not the one its target implies
    (reference sddmm.py:71-80; the kernels index without bounds checks)."""
    if a.shape[0] != want:
        raise DGLError("{} data must have {} rows, got {}".format(what, want, a.shape[0]))


def gsddmm(g, op, lhs_data, rhs_data, lhs_target="u", rhs_target="v"):
    r"""Generalized Sampled-Dense-Dense Matrix Multiplication interface.
    It computes edge features by :attr:`op` lhs features and rhs features.

    .. math::

        x_{e} = \phi(x_{lhs}, x_{rhs}), \forall (u,e,v)\in \mathcal{G}

    Parameters
    ----------
    g : DGLGraph
        The input graph.
    op : str
        ``add``, ``sub``, ``mul``, ``div``, ``dot``, ``copy_lhs`` or ``copy_rhs``.
    lhs_data, rhs_data : numpy array, torch tensor or None
        The operands (None when the op does not read it).
    lhs_target, rhs_target : str
        ``u`` (source), ``v`` (destination) or ``e`` (edge).

    Returns
    -------
    Edge features of shape ``(E,) + broadcast feature shape`` (``(E, ..., 1)``
    for dot), a numpy array or, when an operand is a tensor, a tensor (which
    takes part in autograd when an operand requires grad).
    """
    num_edges = g.number_of_edges()
    num_nodes = g.number_of_nodes()
    if lhs_target not in TARGETS or rhs_target not in TARGETS:
        raise DGLError("lhs_target/rhs_target must be one of 'u', 'v', 'e'")
    if _autograd.needs_grad(lhs_data, rhs_data):
        return _autograd.GSDDMM.apply(g, op, lhs_data, rhs_data, lhs_target, rhs_target)
    L = R = None
    if op == "copy_lhs":
        L = _lib.feature(lhs_data)
        fshape = feat_shape(L.shape)
        code = OP_COPY_LHS
    elif op == "copy_rhs":
        R = _lib.feature(rhs_data)
        fshape = feat_shape(R.shape)
        code = OP_COPY_RHS
    else:
        if op not in BINARY_OPS:
            raise DGLError("op {} not recognized".format(op))
        L, R = reshape_lhs_rhs(_lib.feature(lhs_data), _lib.feature(rhs_data))
        fshape = out_feat_shape(L.shape, R.shape, dot=(op == "dot"))
        code = BINARY_OPS[op]
    if L is not None:
        _check_rows(L, num_edges if lhs_target == "e" else num_nodes,
                    "edge" if lhs_target == "e" else "node")
    if R is not None:
        _check_rows(R, num_edges if rhs_target == "e" else num_nodes,
                    "edge" if rhs_target == "e" else "node")
    dtype = _lib.common_dtype(L, R)
    as_torch = _lib.wants_torch(L, R)
    dev = _lib.out_device(L, R)
    dout = int(math.prod(fshape[:-1] if op == "dot" else fshape))
    if num_edges == 0 or dout == 0:
        empty = np.zeros((num_edges,) + tuple(fshape), dtype=dtype)
        return torch.from_numpy(empty).to(dev) if as_torch else empty
    lt = L if L is not None else R
    rt = R if R is not None else L
    dl, dr = width(lt.shape), width(rt.shape)
    if code in (OP_COPY_LHS, OP_COPY_RHS):
        nd, lsp, rsp = 0, None, None
    else:
        # the arrays stay referenced (here and in the cache) through the call
        nd, _lsa, _rsa, lsp, rsp, _ = shape_ptrs(L.shape, R.shape)
    lhs = _lib.on_device(L, dtype) if L is not None else None
    rhs = _lib.on_device(R, dtype) if R is not None else None
    if op == "dot" and num_edges >= DOT_SLOT_MIN_EDGES and L.shape[1:] == R.shape[1:] \
            and {lhs_target, rhs_target} == {"u", "v"} \
            and _slot_row(dtype.itemsize * dl // dout, num_edges, num_nodes):
        try:
            csr = g._dot_csr()
            if csr is not None and dtype.itemsize * dl <= DOT_SLOT_MIN_ROW * dout \
                    and csr.longest * num_nodes > DOT_SLOT_EVEN * num_edges:
                csr = None
            out = None if csr is None else _slot_dot(
                csr, *((lhs, rhs) if lhs_target == "u" else (rhs, lhs)), num_edges, num_nodes, dl,
                dout, tuple(fshape), dtype)
        except torch.OutOfMemoryError:
            # no room for the CSR, its slot order or the second set of results:
            # edge by edge below, which needs none of them, from now on
            g._dots, out = -1, None
        if out is not None:
            return _lib.give_back(out, as_torch, dev)
    uids, vids = g._device_coo()
    # allocated in its final shape: the same row-major bytes as (E, dout)
    out = torch.empty((num_edges,) + tuple(fshape), dtype=_lib.torch_dtype(dtype),
                      device=_lib.device())
    rc = _lib.lib().mdgl_gsddmm(
        _lib.ptr(uids), _lib.ptr(vids), _lib.ptr(lhs), _lib.ptr(rhs), out.data_ptr(), num_edges,
        TARGETS[lhs_target], TARGETS[rhs_target], code, dl, dr, dout, nd, lsp, rsp,
        _lib.dtype_code(dtype), _lib.stream())
    _lib.check(rc, "gsddmm")
    return _lib.give_back(out, as_torch, dev)


# an edge-wise dot between the endpoints runs in CSR slot order from this many
# edges on, when a dot's rows have more than this many bytes: a destination's row
# then stays in registers, one gathered row per edge less, for the results'
# move into edge-id order (128 columns, 20M edges: 3,119 us edge by edge, 1,484
# slot by slot and 107 for the planned move, 370 until that is planned
# (_ValueOrder); 2,658 us with the destinations' rows read again from cache for
# every slot). The most is what 64 lanes of 16 bytes hold: wider rows go edge by
# edge, which is decided before the in-CSR would be built for them.
# Rows of a single 128-byte line gain on graphs of many edges a row and even
# degrees only. us edge by edge and slot by slot, rows of 128 and of 256 bytes,
# random destinations: 2 edges a row 365 565, 713 663; 8 a row 599 620, 1,322
# 792; 16 a row 590 453, 1,141 671; power law: 4 a row 264 500, 555 590; 20 a row
# 163 214, 330 286; 24 a row (60M edges) 2,002 2,316, 4,278 3,249
DOT_SLOT_MIN_EDGES = 1 << 20
DOT_SLOT_MIN_ROW = 128
DOT_SLOT_MAX_ROW = 1024
DOT_SLOT_MEAN = 16  # edges a row on average, for rows of DOT_SLOT_MIN_ROW bytes
DOT_SLOT_EVEN = 4   # times that average: the longest row, for the same


def _slot_row(row, num_edges, num_nodes):
    """Whether dots over rows of `row` bytes may run in slot order."""
    return DOT_SLOT_MIN_ROW < row <= DOT_SLOT_MAX_ROW or (
        row == DOT_SLOT_MIN_ROW and num_edges >= DOT_SLOT_MEAN * num_nodes)


def _slot_dot(csr, x, y, num_edges, num_nodes, d, dout, fshape, dtype):
    """The dot of every edge between its source's row of `x` and its
    destination's of `y` (mdgl_gspmm_row_dot: the same sums, and so the same
    bits, as edge by edge) in edge-id order. Rows are split as short as the
    backward passes' (a slot's dot is its own: nothing to fold), so that the rows
    of a wavefront end together (20 edges a row, power law, 64 columns: 366 us
    with 512 slots a unit, 286 with 64)."""
    lib, code, st = _lib.lib(), _lib.dtype_code(dtype), _lib.stream()
    tdt, gdev = _lib.torch_dtype(dtype), _lib.device()
    sched = csr.chunks
    if _autograd.NARROW_SPLIT < sched.chunk_len:
        sched = csr.chunks_for(_autograd.NARROW_SPLIT)
    tmp = torch.empty((num_edges, dout), dtype=tdt, device=gdev)
    _lib.check(lib.mdgl_gspmm_row_dot(
        csr.indptr.data_ptr(), csr.indices.data_ptr(), x.data_ptr(), y.data_ptr(), tmp.data_ptr(),
        num_nodes, d, dout, _lib.ptr(sched.chunk_row), _lib.ptr(sched.chunk_start),
        sched.num_chunks, sched.chunk_len, _lib.ANY_ALIGNMENT, code, st), "gspmm_row_dot")
    if dout == 1:
        order = csr.slot_values()
        order.planned()
        return order(tmp, code).reshape((num_edges,) + fshape)
    out = torch.empty((num_edges,) + fshape, dtype=tdt, device=gdev)
    _lib.check(lib.mdgl_gather_rows(tmp.data_ptr(), csr.slot_of_eid().data_ptr(), out.data_ptr(),
                                    num_edges, dout, code, st), "gather_rows")
    return out


def _gen_sddmm_func(lhs_target, rhs_target, binary_op):
    name = "{}_{}_{}".format(lhs_target, binary_op, rhs_target)
    where = {"u": "source node", "e": "edge", "v": "destination node"}

    def func(g, x, y):
        return gsddmm(g, binary_op, x, y, lhs_target=lhs_target, rhs_target=rhs_target)

    func.__name__ = name
    func.__qualname__ = name
    func.__doc__ = (
        "Generalized SDDMM function: edge features by {op} of the {l} features `x` and the "
        "{r} features `y`. Feature shapes broadcast with NumPy's rules.\n\n"
        "Parameters\n----------\ng : DGLGraph\nx : {l} features\ny : {r} features\n\n"
        "Returns\n-------\nThe edge features.\n").format(
            op=binary_op, l=where[lhs_target], r=where[rhs_target])
    return func


def _register_sddmm_func():
    for lhs, rhs in product("uve", "uve"):
        if lhs != rhs:
            for binary_op in ("add", "sub", "mul", "div", "dot"):
                func = _gen_sddmm_func(lhs, rhs, binary_op)
                setattr(sys.modules[__name__], func.__name__, func)
                __all__.append(func.__name__)


def copy_u(g, x):
    """Source node features copied to every edge: ``out[e] = x[u[e]]``."""
    return gsddmm(g, "copy_lhs", x, None)


def copy_v(g, x):
    """Destination node features copied to every edge: ``out[e] = x[v[e]]``."""
    return gsddmm(g, "copy_rhs", None, x)


def copy_e(g, x):
    """Edge features as edge features: returns `x` itself (as the reference)."""
    return x


_register_sddmm_func()
