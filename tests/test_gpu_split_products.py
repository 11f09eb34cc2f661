"""fp32 products on the bf16 matrix instructions (operands split into three bf16 parts): partial
chunks of channels, taps whose entries are neighbours in memory or not, columns at the seam and
at the last pixel of a plane, second levels of a mesh's transposed map, and operands the split
cannot represent."""
import pytest
import torch

import helpers
from helpers import rel_err
from oracle import ops as O

from mappedconvolutions_amd import _C, _lib
from mappedconvolutions_amd.util import synthetic

pytestmark = pytest.mark.gpu


def _grid(h, w, k, dx, dy):
    y, x = torch.meshgrid(torch.arange(h).float(), torch.arange(w).float(), indexing="ij")
    taps = [torch.stack((x + i % 3 - 1 + dx, y + i // 3 - 1 + dy), -1) for i in range(k)]
    return torch.stack(taps, 2).contiguous()


# channels around 8 and 16 (the halves of a chunk), outputs around 64 and 128, widths whose rows
# end inside a tile; 32-bit sums of up to 9 * 40 terms: a few 1e-7 of the result's magnitude,
# 1e-5 allowed like everywhere in these tests
@pytest.mark.parametrize("ci,co", [(1, 1), (7, 5), (8, 64), (9, 65), (11, 6), (13, 27), (15, 128),
                                   (16, 130), (17, 3), (24, 40), (31, 64), (40, 129)])
@pytest.mark.parametrize("interp,dx,dy", [(0, 0.0, 0.0), (1, 0.25, 0.0), (1, 0.4, 0.3),
                                          (2, 0.25, 0.0), (2, -0.3, 0.6)])
def test_split_products_over_images(ci, co, interp, dx, dy, device):
    g = torch.Generator().manual_seed(ci * 1000 + co)
    B, h, w_, k = 2, 5, 37, 9
    smap = _grid(h, w_, k, dx, dy)
    rnd = lambda *s: torch.randn(s, generator=g)
    x, w, b, gy = rnd(B, ci, h, w_), rnd(co, ci, k), rnd(co), rnd(B, co, h, w_)
    y = _C.mapped_conv_forward(x.cuda(), smap.cuda(), w.cuda(), b.cuda(), k, interp)
    assert rel_err(y, O.mapped_conv_forward(x, smap, w, b, k, interp)) < 1e-5
    gx = _C.mapped_conv_backward(gy.cuda(), smap.cuda(), x.cuda(), w.cuda(), b.cuda(), k, interp,
                                 needs=(True, False, False))[0]
    assert rel_err(gx, O.mapped_conv_backward(gy, smap, x, w, b, k, interp)[0]) < 1e-5


@pytest.mark.parametrize("shape", [(1, 1), (1, 2), (2, 1), (3, 2)])
@pytest.mark.parametrize("ci", [5, 7, 12])
def test_split_products_over_the_smallest_planes(ci, shape, device):
    """A plane of one pixel has no neighbour to fetch along; the last pixel has none to its right."""
    g = torch.Generator().manual_seed(3)
    h, w_ = shape
    k, co = 9, 6
    smap = _grid(h, w_, k, 0.25, 0.5)
    x, w, b = (torch.randn(s, generator=g) for s in ((2, ci, h, w_), (co, ci, k), (co,)))
    for interp in (0, 1, 2):
        y = _C.mapped_conv_forward(x.cuda(), smap.cuda(), w.cuda(), b.cuda(), k, interp)
        assert rel_err(y, O.mapped_conv_forward(x, smap, w, b, k, interp)) < 1e-5


@pytest.mark.parametrize("per_cell", [1, 3, 4, 5, 8, 11])
@pytest.mark.parametrize("ci,co", [(16, 64), (20, 128)])
def test_split_products_over_meshes(per_cell, ci, co, device):
    """`per_cell` contributions to every cell of the transposed map: within its first four slots,
    in the second level, beyond it (the overflow list)."""
    g = torch.Generator().manual_seed(per_cell)
    V, k = 300, 3
    idx = (torch.arange(V) // per_cell).view(1, V, 1, 1).expand(1, V, k, 1).float()
    smap = torch.stack((idx, torch.zeros_like(idx)), -1).contiguous()
    iw = torch.rand(1, V, k, 1, generator=g)
    x, w, b, gy = (torch.randn(s, generator=g)
                   for s in ((2, ci, 1, V), (co, ci, k), (co,), (2, co, 1, V)))
    y = _C.weighted_mapped_conv_forward(*[t.cuda() for t in (x, smap, iw, w, b)], k, 0)
    assert rel_err(y, O.weighted_mapped_conv_forward(x, smap, iw, w, b, k, 0)) < 1e-5
    gx = _C.weighted_mapped_conv_backward(*[t.cuda() for t in (gy, smap, iw, x, w, b)], k, 0,
                                          needs=(True, False, False))[0]
    assert rel_err(gx, O.weighted_mapped_conv_backward(gy, smap, iw, x, w, b, k, 0)[0]) < 1e-5


@pytest.mark.parametrize("co", [1, 31, 32, 33, 64, 65, 95, 96, 97, 128, 160, 192, 225])
@pytest.mark.parametrize("mesh", [False, True])
def test_outputs_in_blocks_of_32(co, mesh, device):
    """A workgroup computes one to four blocks of 32 outputs.  32-bit sums of 7 * 21 terms: a few 1e-7
    of the result's magnitude, 1e-5 allowed like everywhere here; a NaN reaches every output of the
    pixels that sample it and no other pixel."""
    g = torch.Generator().manual_seed(co)
    B, ci, k = 2, 21, 7
    rnd = lambda *s: torch.randn(s, generator=g)
    if mesh:
        h, w_ = 1, 150
        smap = torch.stack((torch.randint(w_, (1, w_, k), generator=g).float(),
                            torch.zeros(1, w_, k)), -1).contiguous()
    else:
        h, w_ = 5, 33
        smap = _grid(h, w_, k, 0.25, 0.5)
    interp = 0 if mesh else 1
    x, w, b = rnd(B, ci, h, w_), rnd(co, ci, k), rnd(co)
    want = O.mapped_conv_forward(x, smap, w, b, k, interp)
    y = _C.mapped_conv_forward(x.cuda(), smap.cuda(), w.cuda(), b.cuda(), k, interp)
    assert rel_err(y, want) < 1e-5
    x[1, 4, h // 2, 17] = float("nan")
    got = _C.mapped_conv_forward(x.cuda(), smap.cuda(), w.cuda(), b.cuda(), k, interp).cpu()
    ok = torch.isfinite(O.mapped_conv_forward(x, smap, w, b, k, interp))
    assert torch.equal(torch.isfinite(got), ok) and ok[0].all() and not ok.all()
    assert ((got - want).abs()[ok] <= 1e-5 * want.abs().max()).all()


def _wide_map(kind, h, w_, k, g):
    """Maps whose tiles' boxes do and do not fit a window, at the seam and at both ends of the rows."""
    smap = _grid(h, w_, k, 0.3, 0.4)
    x, y = smap.unbind(-1)
    if kind == "seam":  # columns that go round the image inside a tile
        x = (x + w_ - 11.5) % w_
    elif kind == "spread":  # taps from next to each other to half the image apart, row by row
        x = x + torch.linspace(0, w_ / 2, h)[:, None, None] * (torch.arange(k) % 3 - 1)
    elif kind == "steep":  # rows far apart
        y = y + torch.linspace(-60, 60, w_)[None, :, None]
    elif kind == "random":
        x, y = torch.rand(h, w_, k, generator=g) * w_, torch.rand(h, w_, k, generator=g) * h
    elif kind == "outside":  # tiles of which no tap is inside
        x = torch.where((torch.arange(h) % 8 < 4)[:, None, None], x, x - 4 * w_)
    return torch.stack((x, y), -1).contiguous()


@pytest.mark.parametrize("kind", ["grid", "seam", "spread", "steep", "random", "outside"])
@pytest.mark.parametrize("shape,ci,co,k", [((200, 512), 20, 30, 9), ((98, 1001), 33, 70, 5),
                                           ((402, 250), 17, 9, 4), ((3, 33000), 24, 96, 1),
                                           ((33000, 3), 18, 20, 3)])
@pytest.mark.parametrize("interp,weighted", [(1, False), (2, False), (2, True)])
def test_windows_of_pixels(kind, shape, ci, co, k, interp, weighted, device):
    """Grids of 768 workgroups and more read their taps from a window of the source where they fit one.
    32-bit sums of up to 9 * 33 terms against the oracle's 64-bit ones: a few 1e-7 of the largest result."""
    g = torch.Generator().manual_seed(k)
    h, w_ = shape
    smap = _wide_map(kind, h, w_, k, g)
    rnd = lambda *s: torch.randn(s, generator=g)
    x, w, b, gy = rnd(1, ci, h, w_), rnd(co, ci, k), rnd(co), rnd(1, co, h, w_)
    if weighted:
        smap, iw = smap.unsqueeze(-2).contiguous(), torch.rand(h, w_, k, 1, generator=g)
        fwd, bwd, maps = _C.weighted_mapped_conv_forward, _C.weighted_mapped_conv_backward, (smap, iw)
        want, wbwd = O.weighted_mapped_conv_forward, O.weighted_mapped_conv_backward
    else:
        fwd, bwd, maps = _C.mapped_conv_forward, _C.mapped_conv_backward, (smap,)
        want, wbwd = O.mapped_conv_forward, O.mapped_conv_backward
    cu = lambda *ts: [t.cuda() for t in ts]
    y = fwd(*cu(x, *maps, w, b), k, interp)
    assert rel_err(y, want(x, *maps, w, b, k, interp)) < 1e-5
    gx = bwd(*cu(gy, *maps, x, w, b), k, interp, needs=(True, False, False))[0]
    assert rel_err(gx, wbwd(gy, *maps, x, w, b, k, interp)[0]) < 1e-5


@pytest.mark.parametrize("what", ["x_inf", "x_nan", "w_inf", "overflow", "large"])
def test_operands_without_a_split(what, device):
    """An infinity or NaN among the operands and sums beyond fp32 come out as the fp32
    instructions have them: infinite or NaN exactly where the sum over the taps is, finite values
    unchanged.  (Values of 3e38 round up to an infinite bf16.)"""
    g = torch.Generator().manual_seed(1)
    B, ci, co, h, w_, k = 1, 16, 64, 6, 40, 9
    smap = _grid(h, w_, k, 0.25, 0.25)
    x, w, b = (torch.randn(s, generator=g) for s in ((B, ci, h, w_), (co, ci, k), (co,)))
    if what == "x_inf":
        x[0, 3, 2, 7] = float("inf")
    elif what == "x_nan":
        x[0, 0, 5, 39] = float("nan")
    elif what == "w_inf":
        w[5, 3, 4], x = float("-inf"), x.abs()
    elif what == "overflow":
        x[0, :, 3, 20], w = 3e38, w.abs()
    else:
        x[0, 2, 3, 20], w = 3.4e38, w * 1e-3
    y = _C.mapped_conv_forward(x.cuda(), smap.cuda(), w.cuda(), b.cuda(), k, 1).cpu()
    want = O.mapped_conv_forward(x, smap, w, b, k, 1)
    if what == "w_inf":
        # one output channel has the infinity, or NaN where it meets a corner of weight zero; the
        # others are what they are without it
        assert not torch.isfinite(y[:, 5]).any()
        y, want = (torch.cat((t[:, :5], t[:, 6:]), 1) for t in (y, want))
    ok = torch.isfinite(want)
    assert ok.any() and torch.equal(torch.isfinite(y), ok)
    assert ((y - want).abs()[ok] <= 1e-5 * want.abs()[ok].max()).all()


def _like(got, want, tol=1e-5):
    """Finite, infinite and NaN in the same places, finite values within `tol` of the largest."""
    got, ok = got.cpu(), torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), ok) and ok.any() and not ok.all()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert ((got - want).abs()[ok] <= tol * want.abs()[ok].max()).all()


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("interp,planned", [(0, False), (0, True), (1, False), (1, True)])
def test_not_finite_operands_over_images(value, interp, planned, device):
    """The fp32 form takes over in the forward and in the input gradient of both convolutions.
    (No tap leaves the image beside the element that is not finite, so no weight of zero meets
    it.)"""
    g = torch.Generator().manual_seed(11)
    B, ci, co, h, w_, k = 2, 20, 40, 12, 70, 9
    smap = _grid(h, w_, k, 0.25, 0.25)
    x, w, b, gy = (torch.randn(s, generator=g)
                   for s in ((B, ci, h, w_), (co, ci, k), (co,), (B, co, h, w_)))
    x[1, 3, 5, 44] = value
    gy[0, 7, 6, 12] = value
    xd, sd, wd, bd, gd = (t.cuda() for t in (x, smap, w, b, gy))
    plan = _C.conv_map_plan(sd, None, h, w_, interp) if planned else None
    _like(_C.mapped_conv_forward(xd, sd, wd, bd, k, interp, plan=plan),
          O.mapped_conv_forward(x, smap, w, b, k, interp))
    gx = _C.mapped_conv_backward(gd, sd, xd, wd, bd, k, interp, plan=plan,
                                 needs=(True, False, False))[0]
    _like(gx, O.mapped_conv_backward(gy, smap, x, w, b, k, interp)[0])
    # transposed: gy goes forward (co channels in), x comes back as the output's gradient
    bt = torch.randn(ci, generator=g)
    y = _C.mapped_transposed_conv_forward(gd, sd, wd, bt.cuda(), h, w_, k, interp, plan=plan)
    _like(y, O.mapped_transposed_conv_forward(gy, smap, w, bt, h, w_, k, interp))
    gt = _C.mapped_transposed_conv_backward(xd, sd, gd, wd, bt.cuda(), k, interp, plan=plan,
                                            needs=(True, False, False))[0]
    _like(gt, O.mapped_transposed_conv_backward(x, smap, gy, w, bt, k, interp)[0])


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("per_cell", [3, 5, 11])
def test_not_finite_operands_over_meshes(value, planned, per_cell, device):
    """Likewise over vertices: the fp32 form overwrites the destination and its second level is
    added onto that; the overflow list's share comes once."""
    g = torch.Generator().manual_seed(per_cell)
    V, k, ci, co = 700, 3, 20, 130
    idx = (torch.arange(V) // per_cell).view(1, V, 1, 1).expand(1, V, k, 1).float()
    smap = torch.stack((idx, torch.zeros_like(idx)), -1).contiguous()
    iw = torch.rand(1, V, k, 1, generator=g) + 0.5
    x, w, b, gy = (torch.randn(s, generator=g)
                   for s in ((2, ci, 1, V), (co, ci, k), (co,), (2, co, 1, V)))
    x[1, 3, 0, 17] = value
    gy[0, 7, 0, 333] = value
    d = [t.cuda() for t in (x, smap, iw, w, b, gy)]
    plan = _C.conv_map_plan(d[1], d[2], 1, V, 0) if planned else None
    _like(_C.weighted_mapped_conv_forward(*d[:5], k, 0, plan=plan),
          O.weighted_mapped_conv_forward(x, smap, iw, w, b, k, 0))
    gx = _C.weighted_mapped_conv_backward(d[5], *d[1:3], d[0], *d[3:5], k, 0, plan=plan,
                                          needs=(True, False, False))[0]
    _like(gx, O.weighted_mapped_conv_backward(gy, smap, iw, x, w, b, k, 0)[0])


def test_only_the_tiles_with_a_value_that_is_not_finite_are_computed_again(device):
    """Pixels far from a NaN keep the bits they have without it."""
    g = torch.Generator().manual_seed(12)
    B, ci, co, h, w_, k = 2, 16, 64, 32, 128, 9
    smap = _grid(h, w_, k, 0.25, 0.25).cuda()
    x, w, b = (torch.randn(s, generator=g).cuda() for s in ((B, ci, h, w_), (co, ci, k), (co,)))
    clean = _C.mapped_conv_forward(x, smap, w, b, k, 1)
    x[0, 3, 9, 40] = float("nan")
    y = _C.mapped_conv_forward(x, smap, w, b, k, 1)
    assert torch.isnan(y[0]).any()
    # (tiles are 4 x 32 pixels, taps reach two pixels)
    far = torch.ones(h, w_, dtype=torch.bool)
    far[4:16, 32 - 32:64 + 32] = False
    assert torch.equal(y[1], clean[1]) and torch.equal(y[0][:, far], clean[0][:, far])


# (x = 2^p * u, w = 2^q * v with u, v of ordinary size: the result is 2^(p + q) times the one
# for u and v, to the last bit, wherever fp32 holds the operands in full: |x| >= 2^-126.  The
# split's own range ends at operands of 2^104 and results of 2^80, where the fp32 form takes
# over: another order of summation, a few 2^-24 of the result's size.)
@pytest.mark.parametrize("p,q,bits", [(0, 0, True), (-108, 60, True), (-112, 100, True),
                                      (-118, 100, True), (-124, 30, True), (60, -112, True),
                                      (100, -124, True), (30, -124, True), (-60, -60, True),
                                      (110, -110, False), (-110, 110, False), (45, 45, False)])
@pytest.mark.parametrize("mesh", [False, True])
def test_operands_of_every_magnitude_count_in_full(p, q, bits, mesh, device):
    g = torch.Generator().manual_seed(13)
    B, ci, co, h, w_, k = 1, 24, 40, 9, 40, 9
    if mesh:
        h, w_ = 1, 360
        idx = torch.randint(w_, (1, w_, k), generator=g).float()
        smap = torch.stack((idx, torch.zeros_like(idx)), -1).contiguous()
    else:
        smap = _grid(h, w_, k, 0.0, 0.0)
    interp = 0 if mesh else 1  # (whole rows and columns: interpolation weights of one)
    unit = lambda *s: (1 + torch.rand(s, generator=g)) * (1 - 2 * torch.randint(2, s, generator=g))
    u, v, gu = unit(B, ci, h, w_), unit(co, ci, k), unit(B, co, h, w_)
    b = torch.zeros(co)
    run = lambda x, w: _C.mapped_conv_forward(x.cuda(), smap.cuda(), w.cuda(), b.cuda(), k, interp)
    y = run(u * 2.0 ** p, v * 2.0 ** q).double().cpu() * 2.0 ** -(p + q)
    if bits:
        assert torch.equal(y, run(u, v).double().cpu())
    want = O.mapped_conv_forward(u.double(), smap.double(), v.double(), b.double(), k, interp)
    assert ((y - want).norm() / want.norm()).item() < 1e-6
    # the input gradient (slots of the transposed map are filled in any order: not the same bits)
    gx = _C.mapped_conv_backward((gu * 2.0 ** p).cuda(), smap.cuda(), u.cuda(),
                                 (v * 2.0 ** q).cuda(), b.cuda(), k, interp,
                                 needs=(True, False, False))[0].double().cpu() * 2.0 ** -(p + q)
    want = O.mapped_conv_backward(gu.double(), smap.double(), u.double(), v.double(), b.double(),
                                  k, interp)[0]
    assert ((gx - want).norm() / want.norm()).item() < 1e-6


def _forward_both(x, smap, w, b, k, interp):
    """Through the split products, and (a byte of workspace short of their room) through the fp32
    matrix instructions."""
    lib = _lib.load()
    B, ci, h, w_ = x.shape
    co, (oh, ow) = w.shape[0], smap.shape[:2]
    sizes = (B, ci, co, h, w_, oh, ow, k, 0)
    need = lib.mcx_conv_forward_workspace(*sizes, _lib.MCX_F32)
    ws = torch.empty(need, dtype=torch.uint8, device=x.device)
    out = []
    for given in (need, need - 1):
        y = torch.empty(B, co, oh, ow, device=x.device)
        rc = lib.mcx_conv_forward(x.data_ptr(), smap.data_ptr(), None, w.data_ptr(), b.data_ptr(),
                                  y.data_ptr(), ws.data_ptr(), given, *sizes, interp,
                                  _lib.MCX_F32, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        out.append(y.double().cpu())
    return out


@pytest.mark.parametrize("c", [1, 2, 3, 5, 6, 8, 9, 10, 11, 16, 17, 24, 33, 64, 128])
@pytest.mark.parametrize("interp,shift", [(0, 0.0), (1, 0.0), (1, 0.3)])
def test_accuracy_is_not_below_fp32(c, interp, shift, device):
    """Distance from the 64-bit result in 2-norm, dense operands: the forward's is no larger than
    that of the fp32 matrix instructions on the same operands, which serve it themselves where the
    split products' would be (few channels).  (2 % are allowed for: at nine and ten channels the two
    are equal.)"""
    g = torch.Generator().manual_seed(9)
    h, w_, k, co = 32, 64, 9, 64
    smap = synthetic.latitude_map(h, w_, 1) + shift
    x, w, b = (torch.randn(s, generator=g) for s in ((1, c, h, w_), (co, c, k), (co,)))
    split, fp32 = _forward_both(x.cuda(), smap.cuda(), w.cuda(), b.cuda(), k, interp)
    want = O.mapped_conv_forward(x.double(), smap.double(), w.double(), b.double(), k, interp)
    far = lambda y: ((y - want).norm() / want.norm()).item()
    assert torch.equal(split, fp32) == (c <= 5)
    assert far(split) <= 1.02 * far(fp32), (far(split), far(fp32))


@pytest.mark.parametrize("f,shift", [(2, 0.0), (3, 0.0), (2, 0.4)])
@pytest.mark.parametrize("ci,co,k", [(20, 18, 9), (9, 33, 9), (16, 17, 1), (32, 40, 1), (20, 30, 25)])
def test_taps_whose_boxes_are_larger_than_windows(f, shift, ci, co, k, device):
    """Maps of every second and third pixel, whose tiles' boxes are two windows and more: the rest of the
    taps reads memory; and one tap, of one block of outputs, always does.  32-bit sums of up to 25 * 40 terms."""
    g = torch.Generator().manual_seed(ci + k)
    h, w_ = 150, 330
    smap = synthetic.latitude_map(f * h, f * w_, 2)[::f, ::f, :k].contiguous()
    smap[..., 1] = (smap[..., 1] + shift).clamp(0, f * h - 1)
    rnd = lambda *s: torch.randn(s, generator=g)
    x, w, b, gy = rnd(2, co, f * h, f * w_), rnd(ci, co, k), rnd(ci), rnd(2, ci, h, w_)
    cu = lambda *ts: [t.cuda() for t in ts]
    y = _C.mapped_conv_forward(*cu(x, smap, w, b), k, 1)
    assert rel_err(y, O.mapped_conv_forward(x, smap, w, b, k, 1)) < 1e-5
    gx = _C.mapped_conv_backward(*cu(gy, smap, x, w, b), k, 1, needs=(True, False, False))[0]
    assert rel_err(gx, O.mapped_conv_backward(gy, smap, x, w, b, k, 1)[0]) < 1e-5
