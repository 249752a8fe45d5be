"""segment_mm / gather_mm and their gradients at the widths where the kernels'
tiles end: K around the 16-deep chunks and the 4-float pieces, N around the
column blocks, groups that are empty, of one row and just past a tile, rows
that start on any 4-byte boundary, and rows with inf or NaN beside ordinary
ones."""

import numpy as np
import pytest
import torch

import mojodgl.ops as ops

pytestmark = pytest.mark.gpu

KS = [1, 3, 4, 5, 6, 7, 15, 16, 17, 20, 31, 32, 33, 47, 64, 66, 97, 100, 127, 128, 130, 192, 255,
      256, 257]
NS = [1, 2, 15, 16, 17, 32, 33, 47, 64, 65, 100, 128, 129, 200, 256]


def groups(seed, r=9):
    """Lengths with empty groups, single rows and just past 32, 128 and 256."""
    rng = np.random.default_rng(seed)
    seg = np.array([0, 1, 33, 129, 0, 257, 31, 128, 100 + rng.integers(0, 50)])[:r]
    return seg, np.repeat(np.arange(r), seg)


def inputs(k, n, dtype, seed, lengths):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rows = int(lengths.sum())

    def draw(*shape):
        return torch.randn(*shape, device="cuda", generator=gen, dtype=torch.float64).to(dtype)

    return draw(rows, k), draw(len(lengths), k, n), draw(rows, n)


def product(a, b, group):
    return torch.bmm(a.unsqueeze(1), b[group]).squeeze(1)


def within(got, ref, bound, terms, dtype):
    # a sum of `terms` products in any order: terms * eps of their magnitudes,
    # and the three smallest part products left out (2^-24) for float32
    tol = (terms + 4) * torch.finfo(dtype).eps
    off = (got.double() - ref).abs()
    assert bool((off <= tol * bound + 1e-300).all()), float((off / (bound + 1e-300)).max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("k,n", [(k, NS[(i * 7 + j * 4) % len(NS)]) for i, k in enumerate(KS)
                                 for j in range(3)] + [(64, n) for n in NS] + [(16, n) for n in NS]
                         # four column blocks of a narrow K, each length of a
                         # row's last piece; gradient tiles of 3, 5, 6 and 7
                         # blocks whole and cut
                         + [(47, 100), (17, 66), (50, 131), (5, 257), (48, 15), (80, 47), (79, 33),
                            (96, 64), (95, 18), (112, 49), (111, 16)])
def test_products_and_gradients(dtype, k, n):
    seg, grp = groups(k * 1000 + n)
    a, b, G = inputs(k, n, dtype, k * 1000 + n, seg)
    rng = np.random.default_rng(k + n)
    order = rng.permutation(grp.size)
    for by in ("segment", "gather"):
        ids = grp if by == "segment" else grp[order]
        group = torch.from_numpy(ids).cuda()
        a.requires_grad_(True)
        b.requires_grad_(True)
        z = (ops.segment_mm(a, b, seg) if by == "segment"
             else ops.gather_mm(a, b, idx_b=group))
        da, db = torch.autograd.grad(z, (a, b), G)
        a, b = a.detach(), b.detach()
        A, B, D = a.double(), b.double(), G.double()
        within(z.detach(), product(A, B, group), product(A.abs(), B.abs(), group), k, dtype)
        bt = B.transpose(1, 2).contiguous()
        within(da, product(D, bt, group), product(D.abs(), bt.abs(), group), n, dtype)
        ref = torch.zeros_like(B)
        bound = torch.zeros_like(B)
        for r in range(len(seg)):
            rows = (group == r).nonzero().view(-1)
            ref[r] = A[rows].t().contiguous() @ D[rows]
            bound[r] = A[rows].abs().t().contiguous() @ D[rows].abs()
        within(db, ref, bound, int(seg.max()), dtype)


# Every instance of the forward kernels with more tiles than workgroups: column
# blocks by LDS depth by the number of 16-deep chunks of a row, which leaves every
# remainder in the ring of chunks in flight; float64 in two, four and eight blocks.
MANY = ([(torch.float32, k, n) for k, n in (
    (12, 20), (20, 30), (40, 17), (60, 32), (70, 9), (90, 31), (100, 20), (120, 5), (140, 24),
    (250, 16), (10, 47), (30, 64), (44, 33), (64, 50), (72, 40), (92, 64), (100, 47), (127, 60),
    (130, 40), (160, 70), (250, 100), (9, 100), (25, 66), (47, 100), (63, 128), (66, 100),
    (85, 129), (103, 70), (121, 90))]
    + [(torch.float64, k, n) for k, n in ((16, 32), (48, 20), (128, 17), (32, 64), (112, 40),
                                          (64, 100))])


@pytest.mark.parametrize("dtype,k,n", MANY)
def test_several_tiles_per_workgroup(dtype, k, n):
    """2,600 groups of 0 to 260 rows: a workgroup goes from tile to tile within a
    group and over group ends (its block of b kept, or loaded again), in segments
    and gathered, forward and both gradients."""
    rng = np.random.default_rng(k * n)
    seg = rng.choice([0, 1, 5, 31, 32, 33, 127, 128, 129, 260], 2600)
    ids = np.repeat(np.arange(seg.size), seg)
    a, b, G = inputs(k, n, dtype, k + n, seg)
    a.requires_grad_(True)
    b.requires_grad_(True)
    for by in ("segment", "gather"):
        group = torch.from_numpy(ids if by == "segment" else rng.permutation(ids)).cuda()
        z = ops.segment_mm(a, b, seg) if by == "segment" else ops.gather_mm(a, b, idx_b=group)
        da, db = torch.autograd.grad(z, (a, b), G)
        B = b.detach().double()
        bt = B.transpose(1, 2).contiguous()
        ref, bound = torch.zeros_like(B), torch.zeros_like(B)
        step = max(1, (1 << 25) // (k * n))
        for lo in range(0, group.numel(), step):
            at = slice(lo, lo + step)
            g, x, y = group[at], a.detach()[at].double(), G[at].double()
            within(z.detach()[at], product(x, B, g), product(x.abs(), B.abs(), g), k, dtype)
            within(da[at], product(y, bt, g), product(y.abs(), bt.abs(), g), n, dtype)
            pairs = x.unsqueeze(2) * y.unsqueeze(1)
            ref.index_add_(0, g, pairs)
            bound.index_add_(0, g, pairs.abs())
        within(db, ref, bound, int(seg.max()), dtype)


@pytest.mark.parametrize("by", ["segment", "gather"])
@pytest.mark.parametrize("k,n", [(16, 16), (17, 32), (20, 250), (33, 129), (47, 100), (64, 64),
                                 (100, 47), (100, 20), (128, 33), (130, 200), (199, 61), (250, 250),
                                 (256, 32)])
def test_split_products_are_no_further_off_than_float32_ones(k, n, by):
    """The part products left out cost less than the roundings saved: the result
    is no further from 64 bits than that of float32 MFMAs, which a value of b out
    of the split's range (times a zero of a, so that the sums are the same) sends
    the same call to."""
    rows, r = 40000, 5
    gen = torch.Generator(device="cuda").manual_seed(k * n)
    a = torch.randn(rows, k, device="cuda", generator=gen)
    a[:, 0] = 0
    b = torch.randn(r, k, n, device="cuda", generator=gen)
    group = torch.randint(0, r, (rows,), device="cuda", generator=gen).sort()[0]
    seg = torch.bincount(group, minlength=r).cpu()
    ref = torch.empty(rows, n, device="cuda", dtype=torch.float64)
    for i in range(r):
        at = (group == i).nonzero().view(-1)
        ref[at] = a[at].double() @ b[i].double()

    def off(b):
        z = ops.segment_mm(a, b, seg) if by == "segment" else ops.gather_mm(a, b, idx_b=group)
        return float((z.double() - ref).norm() / ref.norm())

    plain = b.clone()
    plain[:, 0] = 1e30
    assert 0 < off(b) <= off(plain)


def gradient_of_b(a, G, group, r):
    """a^T G per group in float64, and the sum of the products' magnitudes."""
    ref = torch.zeros(r, a.shape[1], G.shape[1], dtype=torch.float64, device="cuda")
    bound = torch.zeros_like(ref)
    for i in range(r):
        rows = (group == i).nonzero().view(-1)
        x, y = a[rows].double(), G[rows].double()
        ref[i] = x.t().contiguous() @ y
        bound[i] = x.abs().t().contiguous() @ y.abs()
    return ref, bound


# float32 gradients of b: widths that fill tiles of 128 x 128 (whole, cut, several,
# just under), register tiles of every width along the second axis, both at and
# off a 16-byte boundary
@pytest.mark.parametrize("k,n", [(128, 128), (120, 124), (128, 112), (112, 124), (108, 128),
                                 (256, 128), (124, 256), (252, 244), (512, 120), (100, 100),
                                 (80, 80), (64, 80), (144, 144), (160, 160), (200, 200), (72, 176)])
@pytest.mark.parametrize("shift", [0, 1])
def test_gradient_tiles(k, n, shift):
    seg, grp = groups(k + n)
    rng = np.random.default_rng(k * n)
    a, b, G = inputs(k, n, torch.float32, k * n, seg)

    def off(x):  # a copy that starts `shift` elements into its buffer
        buf = torch.empty(x.numel() + shift, device="cuda")
        view = buf[shift:].view(x.shape)
        return view.copy_(x)

    a, G = off(a), off(G)
    b.requires_grad_(True)
    for by in ("segment", "gather"):
        group = torch.from_numpy(grp if by == "segment" else grp[rng.permutation(grp.size)]).cuda()
        z = ops.segment_mm(a, b, seg) if by == "segment" else ops.gather_mm(a, b, idx_b=group)
        db, = torch.autograd.grad(z, (b,), G)
        ref, bound = gradient_of_b(a, G, group, len(seg))
        within(db, ref, bound, int(seg.max()), torch.float32)


@pytest.mark.parametrize("dtype,k,n,r", [(torch.float32, 12, 20, 3), (torch.float32, 128, 128, 5),
                                         (torch.float32, 40, 72, 200), (torch.float64, 32, 64, 3),
                                         (torch.float64, 48, 33, 7)])
@pytest.mark.parametrize("by", ["segment", "gather"])
def test_gradient_over_longer_chunks(dtype, k, n, r, by):
    """More than 524,288 rows: a workgroup sums 512 rows or more."""
    rows = 600011
    gen = torch.Generator(device="cuda").manual_seed(k)
    a = torch.randn(rows, k, device="cuda", generator=gen, dtype=dtype)
    G = torch.randn(rows, n, device="cuda", generator=gen, dtype=dtype)
    b = torch.randn(r, k, n, device="cuda", generator=gen, dtype=dtype).requires_grad_(True)
    group = torch.randint(0, r, (rows,), device="cuda", generator=gen)
    if by == "segment":
        group = group.sort()[0]
        z = ops.segment_mm(a, b, torch.bincount(group, minlength=r).cpu())
    else:
        z = ops.gather_mm(a, b, idx_b=group)
    db, = torch.autograd.grad(z, (b,), G)
    ref, bound = gradient_of_b(a, G, group, r)
    # a chunk's chain, the streams, then the group's chunks
    within(db, ref, bound, 4096 + rows // 512, dtype)


@pytest.mark.parametrize("k,n", [(4, 5), (7, 17), (18, 33), (47, 64), (100, 47), (61, 20),
                                 (130, 40), (255, 100)])
def test_inf_and_nan_stay_in_their_rows(k, n):
    """inf, NaN, zero and huge values: their rows as IEEE products give them,
    the others as without them; the same for a block of b that holds them."""
    seg, grp = groups(k)
    a, b, _ = inputs(k, n, torch.float32, k, seg)
    group = torch.from_numpy(grp).cuda()
    clean = ops.segment_mm(a, b, seg)
    for spot, value in ((0, float("inf")), (k - 1, float("nan")), (k - 1, -float("inf")),
                        (k // 2, 1e38)):
        x = a.clone()
        x[5, spot] = value
        got = ops.segment_mm(x, b, seg)
        want = product(x.double(), b.double(), group).float()
        keep = torch.ones(a.shape[0], dtype=torch.bool, device="cuda")
        keep[5] = False
        assert torch.equal(torch.isnan(got[5]), torch.isnan(want[5]))
        assert torch.equal(torch.isinf(got[5]), torch.isinf(want[5]))
        # rows that shared its wavefront may take the float32 path: same to rounding
        bound = product(a.double().abs(), b.double().abs(), group)
        within(got[keep], clean[keep].double(), bound[keep], 2 * k, torch.float32)
    y = b.clone()
    y[5, k - 1, n - 1] = float("inf")
    got = ops.segment_mm(a, y, seg)
    want = product(a.double(), y.double(), group)
    rows = (group == 5).nonzero().view(-1)
    assert torch.equal(torch.isinf(got), torch.isinf(want))
    assert bool(torch.isinf(got[rows, n - 1]).all())
