"""fp64 convolutions over channel-last records against the CPU oracle, at the edges of their
tiles: channel counts around the widths a pass of lanes covers (2, 4 and 8 lanes of two
channels; 1, 4 and 16 outputs), more channels and taps than one pass takes, locations around a
workgroup's share, weighted taps, and the call without a workspace (the scalar kernels)."""
import ctypes

import pytest
import torch

import helpers
from helpers import rel_err
from oracle import ops as O

from mappedconvolutions_amd import _C, _lib
from mappedconvolutions_amd.util import synthetic

pytestmark = pytest.mark.gpu

# (Ci, Co, K, map height, map width, P): sums of up to a few hundred terms in 64 bits differ by
# some 1e-15 of the result with their order; 1e-12 is what the fp64 tests beside this one allow
SHAPES = [(1, 1, 1, 1, 1, 0), (2, 1, 9, 5, 7, 0), (3, 4, 6, 4, 32, 0), (4, 5, 9, 8, 17, 0),
          (5, 16, 10, 3, 43, 0), (8, 17, 9, 9, 15, 0), (9, 2, 5, 16, 16, 3), (16, 3, 9, 4, 33, 0),
          (17, 9, 4, 6, 11, 6), (33, 20, 11, 5, 13, 0)]


# Enough locations (of two images) for the weight gradient's records, too: tiles that end ragged,
# more than one tile a workgroup; one channel, whose forward takes records from 196 608 on
LARGER = [(1, 1, 1, 32, 32, 0), (2, 1, 9, 31, 67, 0), (3, 4, 6, 32, 33, 0), (5, 16, 10, 30, 43, 0),
          (8, 17, 9, 29, 45, 0), (9, 2, 5, 48, 48, 3), (16, 3, 9, 34, 33, 0), (17, 9, 4, 36, 31, 6),
          (33, 20, 3, 45, 53, 0), (1, 3, 9, 320, 308, 0)]


# few channels scattered into many: planes that are added to before the product (16 destination
# channels a workgroup, 128 or 256 locations)
PLANES = [(6, 1, 9, 4, 32, 0), (7, 1, 1, 5, 7, 0), (13, 2, 9, 9, 15, 0), (16, 1, 5, 16, 16, 3),
          (17, 1, 9, 31, 67, 0), (20, 3, 10, 8, 17, 0), (33, 4, 3, 29, 45, 6), (40, 1, 64, 3, 43, 0)]


# the same with locations enough for planes to pay: more for fewer channels
MANY = [(64, 1, 9, 17, 43, 0), (40, 1, 64, 17, 43, 0), (33, 1, 3, 31, 67, 6), (16, 1, 5, 48, 48, 3),
        (13, 1, 9, 45, 53, 0), (7, 1, 10, 72, 70, 0), (20, 3, 9, 72, 70, 0)]


@pytest.mark.parametrize("ci,co,k,mh,mw,p", SHAPES + LARGER + PLANES + MANY)
@pytest.mark.parametrize("interp", [0, 1, 2])
def test_fp64_products(ci, co, k, mh, mw, p, interp, device):
    g = torch.Generator().manual_seed(ci * 100 + co)
    B, ih, iw_ = 2, 6, 9
    smap, wts = helpers.random_map(g, mh, mw, k, p, ih, iw_, torch.float64,
                                   integer=interp == 1 and k == 9)
    rnd = lambda *s: torch.randn(s, generator=g, dtype=torch.float64)
    cuda = lambda t: None if t is None else t.cuda()
    pre = "weighted_" if p else ""
    maps = [smap] + ([wts] if p else [])
    x, w, b, gy = rnd(B, ci, ih, iw_), rnd(co, ci, k), rnd(co), rnd(B, co, mh, mw)
    for name, args in ((pre + "mapped_conv_forward", [x, *maps, w, b, k, interp]),
                       (pre + "mapped_conv_backward", [gy, *maps, x, w, b, k, interp])):
        want = getattr(O, name)(*args)
        got = getattr(_C, name)(*[cuda(a) if torch.is_tensor(a) else a for a in args])
        for i, (a, c) in enumerate(zip(*[v if isinstance(v, (list, tuple)) else [v]
                                         for v in (got, want)])):
            assert rel_err(a, c) < 1e-12, (name, i)
    # the transposed convolution: the map's locations are the input's pixels
    xt, wt, bt, gt = rnd(B, ci, mh, mw), rnd(ci, co, k), rnd(co), rnd(B, co, ih, iw_)
    for name, args in (
            (pre + "mapped_transposed_conv_forward", [xt, *maps, wt, bt, ih, iw_, k, interp]),
            (pre + "mapped_transposed_conv_backward", [gt, *maps, xt, wt, bt, k, interp])):
        want = getattr(O, name)(*args)
        got = getattr(_C, name)(*[cuda(a) if torch.is_tensor(a) else a for a in args])
        for i, (a, c) in enumerate(zip(*[v if isinstance(v, (list, tuple)) else [v]
                                         for v in (got, want)])):
            assert rel_err(a, c) < 1e-12, (name, i)


@pytest.mark.parametrize("interp", [0, 1, 2])
def test_infinite_weights_reach_what_is_added_to(interp, device):
    """A product weight that is infinite makes a destination pixel infinite where a tap lands on it
    and leaves it alone where none does, also where the sums are taken before the product.
    (Positive operands: no two infinities of different signs meet.)"""
    g = torch.Generator().manual_seed(22)
    B, ci, co, k, h, w_ = 2, 12, 1, 9, 9, 20
    smap = torch.rand(h, w_, k, 2, generator=g, dtype=torch.float64) * 4 + 2.25
    smap[..., 0] += torch.arange(k) % 3  # (other pixels under every tap)
    w = torch.rand(co, ci, k, generator=g, dtype=torch.float64) + 0.1
    w[0, 5, 4] = float("inf")
    x, gy, b = (torch.rand(s, generator=g, dtype=torch.float64) + 0.1
                for s in ((B, ci, h, w_), (B, co, h, w_), (co,)))
    got = _C.mapped_conv_backward(*[t.cuda() for t in (gy, smap, x, w, b)], k, interp,
                                  needs=(True, False, False))[0].cpu()
    assert not torch.isnan(got).any() and (got[:, 5] == 0).any()
    w[0, 5, 4] = 1.0
    hit = torch.zeros_like(w)
    hit[0, 5, 4] = 1.0
    reached = O.mapped_conv_backward(gy, smap, x, hit, b, k, interp)[0] != 0
    assert torch.equal(torch.isinf(got), reached)
    want = O.mapped_conv_backward(gy, smap, x, w, b, k, interp)[0]
    assert ((got - want).abs()[~reached] <= 1e-12 * want.abs().max()).all()


@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("weight", [float("inf"), float("nan")])
def test_minus_zeros_are_added_too(weight, interp, device):
    """A pixel that only zeros of negative sign were added to is still one that was added to: an infinite
    weight makes it NaN, as does a weight that is NaN."""
    g = torch.Generator().manual_seed(23)
    B, ci, co, k, h, w_ = 2, 64, 1, 9, 21, 20
    smap = torch.rand(h, w_, k, 2, generator=g, dtype=torch.float64) * 4 + 2.25
    smap[..., 0] += torch.arange(k) % 3
    w = torch.rand(co, ci, k, generator=g, dtype=torch.float64) + 0.1
    w[0, 5, 4] = weight
    x, b = torch.zeros(B, ci, h, w_, dtype=torch.float64), torch.zeros(co, dtype=torch.float64)
    gy = torch.full((B, co, h, w_), -0.0, dtype=torch.float64)
    got = _C.mapped_conv_backward(*[t.cuda() for t in (gy, smap, x, w, b)], k, interp,
                                  needs=(True, False, False))[0].cpu()
    want = O.mapped_conv_backward(gy, smap, x, w, b, k, interp)[0]
    assert torch.isnan(want).any() and torch.equal(torch.isnan(got), torch.isnan(want))


@pytest.mark.parametrize("share", [1.0, 0.8, 0.2, 0.02])
def test_planes_with_less_scratch(share, device):
    """Sums taken before the product ask for more scratch than records; with less, records run, and
    with less than those the scalar kernels."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(24)
    B, ci, co, k, h, w_ = 2, 16, 1, 25, 48, 60
    smap, _ = helpers.random_map(g, h, w_, k, 0, h, w_, torch.float64)
    x, w, b, gy = (torch.randn(s, generator=g, dtype=torch.float64)
                   for s in ((B, ci, h, w_), (co, ci, k), (co,), (B, co, h, w_)))
    size = (B, ci, co, h, w_, h, w_, k, 0)
    need = int(share * lib.mcx_conv_backward_workspace(*size, _lib.MCX_F64))
    gyd, sd, xd, wd, gx = *(t.cuda() for t in (gy, smap, x, w)), torch.empty(B, ci, h, w_, device="cuda",
                                                                          dtype=torch.float64)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    rc = lib.mcx_conv_backward(gyd.data_ptr(), sd.data_ptr(), None, xd.data_ptr(), wd.data_ptr(),
                               gx.data_ptr(), None, None, ws.data_ptr(), need, *size, 1, _lib.MCX_F64,
                               torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert rel_err(gx, O.mapped_conv_backward(gy, smap, x, w, b, k, 1)[0]) < 1e-12


@pytest.mark.parametrize("interp", [0, 1, 2])
def test_infinite_interpolation_weights_at_the_border(interp, device):
    """A tap that lies partly outside the image, or on whole rows and columns, has corners that do
    not count; an infinite weight of such a tap makes its sample infinite, not NaN.  (Positive
    operands: no two infinities of different signs meet.)"""
    g = torch.Generator().manual_seed(21)
    B, ci, co, k, p, h, w_ = 2, 5, 3, 9, 2, 32, 34
    smap, wts = helpers.random_map(g, h, w_, k, p, h, w_, torch.float64)
    smap.clamp_(-0.4, 33.25)                          # (no tap lies outside altogether)
    smap[..., 1].clamp_(max=31.25)
    smap[1] = smap[1].round().clamp_(0, 31)
    for n in range(0, h * w_, 23):
        wts.view(h * w_, k, p)[n, n % k, n % p] = float("inf")
    x, w, b, gy = (torch.rand(s, generator=g, dtype=torch.float64) + 0.1
                   for s in ((B, ci, h, w_), (co, ci, k), (co,), (B, co, h, w_)))
    dev = [t.cuda() for t in (x, smap, wts, w, b, gy)]
    got = [_C.weighted_mapped_conv_forward(*dev[:5], k, interp)]
    got += _C.weighted_mapped_conv_backward(dev[5], *dev[1:3], dev[0], *dev[3:5], k, interp)
    want = [O.weighted_mapped_conv_forward(x, smap, wts, w, b, k, interp)]
    want += O.weighted_mapped_conv_backward(gy, smap, wts, x, w, b, k, interp)
    assert torch.isinf(want[0]).any() and not torch.isinf(want[0]).all()
    assert not torch.isnan(want[0]).any()
    for i, (a, c) in enumerate(zip(got, want)):
        # (the oracle's input gradient adds corners of weight zero too: NaN)
        a, c = a.cpu()[~torch.isnan(c)], c[~torch.isnan(c)]
        ok = torch.isfinite(c)
        assert torch.equal(torch.isinf(a), torch.isinf(c)) and not torch.isnan(a).any(), i
        assert not ok.any() or ((a - c).abs()[ok] <= 1e-12 * c.abs()[ok].max()).all(), i


# (S, D, K, map rows, columns, P): both sides of the rules that let the map decide (for the scatter
# 2^20 taps of up to eight source channels; for the gather, from D channels into S, 196 608
# locations of 3 * 2^20 samples at one tap, or at two for up to sixteen outputs), under maps that
# are coherent, that are not, and half of whose neighbours are
@pytest.mark.parametrize("s,d,k,mh,mw,p", [(1, 10, 9, 241, 242, 0), (2, 3, 9, 241, 241, 0),
                                           (1, 17, 9, 241, 242, 2), (8, 9, 9, 241, 242, 0),
                                           (9, 9, 9, 241, 242, 0), (3, 16, 1, 314, 314, 0),
                                           (3, 15, 1, 314, 314, 0), (16, 16, 2, 314, 314, 2),
                                           (17, 16, 2, 314, 314, 0)])
@pytest.mark.parametrize("kind", ["coherent", "shuffled", "half"])
def test_fp64_products_where_the_map_decides(s, d, k, mh, mw, p, kind, device):
    g = torch.Generator().manual_seed(mh + s)
    B, interp, np = 2, 1, max(p, 1)
    at = torch.arange(mh * mw)
    if kind == "shuffled":
        at = torch.randperm(mh * mw, generator=g)
    elif kind == "half":
        at = torch.where(at // 2 % 2 == 0, at, at.flip(0))
    base = torch.stack((at % mw, at // mw), -1).double().view(mh, mw, 1, 1, 2)
    step = torch.randint(-2, 3, (1, 1, k, np, 2), generator=g)
    smap = (base + step + 0.3).contiguous()
    smap = smap if p else smap[:, :, :, 0].contiguous()
    wts = torch.rand(mh, mw, k, p, generator=g, dtype=torch.float64) if p else None
    rnd = lambda *size: torch.randn(size, generator=g, dtype=torch.float64)
    # a transposed convolution: s channels scattered into d, and d gathered into s
    x, w, b, gy = rnd(B, s, mh, mw), rnd(s, d, k), rnd(d), rnd(B, d, mh, mw)
    pre, maps = ("weighted_", (smap, wts)) if p else ("", (smap,))
    dm = [t.cuda() for t in maps]
    y = getattr(_C, pre + "mapped_transposed_conv_forward")(x.cuda(), *dm, w.cuda(), b.cuda(), mh,
                                                            mw, k, interp)
    want = getattr(O, pre + "mapped_transposed_conv_forward")(x, *maps, w, b, mh, mw, k, interp)
    assert rel_err(y, want) < 1e-12
    gx = getattr(_C, pre + "mapped_transposed_conv_backward")(gy.cuda(), *dm, x.cuda(), w.cuda(),
                                                              b.cuda(), k, interp,
                                                              needs=(True, False, False))[0]
    want = getattr(O, pre + "mapped_transposed_conv_backward")(gy, *maps, x, w, b, k, interp)[0]
    assert rel_err(gx, want) < 1e-12


def _every_call(lib, workspace):
    """The six products of both convolutions through the C ABI, fp64; `workspace(bytes)` gives the
    (pointer, size) that each call is handed.  [(what, bytes asked for, result, oracle's)]."""
    g = torch.Generator().manual_seed(5)
    B, ci, co, k, h, w_ = 2, 5, 3, 9, 33, 40
    smap, _ = helpers.random_map(g, h, w_, k, 0, h, w_, torch.float64)
    x, w, b, gy = (torch.randn(s, generator=g, dtype=torch.float64)
                   for s in ((B, ci, h, w_), (co, ci, k), (co,), (B, co, h, w_)))
    wt, bt = w.transpose(0, 1).contiguous(), b            # [ci, co, k] of the transposed one
    dx, dm, dw, db, dg, dwt = (t.cuda() for t in (x, smap, w, b, gy, wt))
    ptr = lambda t: None if t is None else t.data_ptr()
    size, tail = (B, ci, co, h, w_, h, w_, k, 0), (1, _lib.MCX_F64,
                                                    torch.cuda.current_stream().cuda_stream)
    new = lambda t: torch.full(t.shape, float("nan"), dtype=torch.float64, device="cuda")
    out = []

    def forward(name, weight, weight_d, want):
        need = getattr(lib, "mcx_%s_forward_workspace" % name)(*size, _lib.MCX_F64)
        y = new(want)
        rc = getattr(lib, "mcx_%s_forward" % name)(ptr(dx), ptr(dm), None, ptr(weight_d), ptr(db),
                                                   ptr(y), *workspace(need), *size, *tail)
        assert rc == 0
        out.append((name, need, y, want))

    def backward(name, weight_d, want):
        need = getattr(lib, "mcx_%s_backward_workspace" % name)(*size, _lib.MCX_F64)
        for i in range(3):                                # one gradient a call
            grads = [new(t) if i == j else None for j, t in enumerate(want)]
            rc = getattr(lib, "mcx_%s_backward" % name)(ptr(dg), ptr(dm), None, ptr(dx),
                                                        ptr(weight_d), *map(ptr, grads),
                                                        *workspace(need), *size, *tail)
            assert rc == 0
            out.append((name, need, grads[i], want[i]))

    forward("conv", w, dw, O.mapped_conv_forward(x, smap, w, b, k, 1))
    backward("conv", dw, O.mapped_conv_backward(gy, smap, x, w, b, k, 1))
    forward("tconv", wt, dwt, O.mapped_transposed_conv_forward(x, smap, wt, bt, h, w_, k, 1))
    backward("tconv", dwt, O.mapped_transposed_conv_backward(gy, smap, x, wt, bt, k, 1))
    return out


@pytest.mark.parametrize("given", ["all", "one byte less", "none"])
def test_fp64_without_a_workspace(given, device):
    """Every product asks for a workspace at this size and does without one, or with less: the
    scalar kernels."""
    lib, kept = _lib.load(), []

    def workspace(need):
        if given == "none":
            return None, 0
        kept.append(torch.empty(need, dtype=torch.uint8, device=device))
        return kept[-1].data_ptr(), need - (given != "all")

    for name, need, got, want in _every_call(lib, workspace):
        assert need > 0, name
        assert rel_err(got, want) < 1e-12, name


def test_fp64_where_no_memory_is_left_for_a_workspace(device):
    """The layers' ops go through without the records' copy of an operand: what the process may
    hold is limited to the tensors, the results and 16 MB."""
    g = torch.Generator(device="cuda").manual_seed(8)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=torch.float64)
    B, ci, co, k, h, w_ = 1, 64, 2, 9, 256, 512
    torch.cuda.empty_cache()                              # (no blocks of earlier tests to reuse)
    smap = synthetic.latitude_map(h, w_, 1, dtype=torch.float64).cuda()
    x, w, b, gy = rnd(B, ci, h, w_), rnd(co, ci, k), rnd(co), rnd(B, co, h, w_)
    xt, wt, bt = gy, w, rnd(ci)                           # transposed: co channels in, ci out
    calls = [(lambda: [_C.mapped_conv_forward(x, smap, w, b, k, 1)], gy),
             (lambda: _C.mapped_conv_backward(gy, smap, x, w, b, k, 1), x),
             (lambda: [_C.mapped_transposed_conv_forward(xt, smap, wt, bt, h, w_, k, 1)], x),
             (lambda: _C.mapped_transposed_conv_backward(x, smap, xt, wt, bt, k, 1), xt)]
    total = torch.cuda.get_device_properties(0).total_memory
    for call, like in calls:
        torch.cuda.empty_cache()
        want = call()
        torch.cuda.empty_cache()
        room = torch.cuda.memory_reserved() + like.numel() * 8 + (16 << 20)
        ooms = torch.cuda.memory_stats()["num_ooms"]
        torch.cuda.set_per_process_memory_fraction(room / total)
        try:
            got = call()
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert torch.cuda.memory_stats()["num_ooms"] > ooms
        for a, c in zip(got, want):
            assert rel_err(a, c) < 1e-12
        del got, want, a, c


@pytest.mark.parametrize("n", [1 << 13, (1 << 13) + 1, 100003])
def test_bias_gradient_of_one_channel(n, device):
    """The sum's two stages set in at 2^14 values of a channel."""
    g = torch.Generator().manual_seed(n)
    gy = torch.randn(2, 1, 1, n, generator=g, dtype=torch.float64)
    smap = torch.zeros(1, n, 1, 2, dtype=torch.float64)
    x, w, b = torch.zeros(2, 1, 2, 2).double(), torch.zeros(1, 1, 1).double(), torch.zeros(1).double()
    gb = _C.mapped_conv_backward(gy.cuda(), smap.cuda(), x.cuda(), w.cuda(), b.cuda(), 1, 1)[2]
    want = gy.sum().item()
    # n terms of magnitude one in 64 bits: at most n * 2^-53 * sum|gy| apart, far less in practice
    assert abs(gb.item() - want) <= 1e-12 * gy.abs().sum().item()


@pytest.mark.parametrize("ci,co,k,p", [(3, 1, 9, 0), (4, 1, 5, 2), (7, 1, 10, 0), (10, 1, 9, 0),
                                       (17, 1, 11, 0), (1, 1, 4, 0), (2, 2, 4, 0), (8, 4, 9, 0), (9, 3, 1, 3),
                                       (17, 4, 8, 0), (6, 5, 3, 0)])
@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("few", [False, True])
def test_weight_gradient_of_several_taps_a_workgroup(ci, co, k, p, interp, few, device):
    """From 98 304 locations (65 536 with two to four outputs) a workgroup takes several taps: below and
    above, taps that fill no whole group, channels around a pass of lanes.  Sums of 100 000 terms in 64 bits
    differ by some 1e-14 of the result with their order; 1e-12 is allowed like everywhere here."""
    g = torch.Generator().manual_seed(ci * 100 + k)
    B, ih, iw_ = 2, 60, 90
    mh, mw = (180, 181) if few else (221, 223)
    smap, wts = helpers.random_map(g, mh, mw, k, p, ih, iw_, torch.float64)
    x, gy, w, b = (torch.randn(s, generator=g, dtype=torch.float64)
                   for s in ((B, ci, ih, iw_), (B, co, mh, mw), (co, ci, k), (co,)))
    maps = [smap] + ([wts] if p else [])
    name = ("weighted_" if p else "") + "mapped_conv_backward"
    got = getattr(_C, name)(*[t.cuda() for t in (gy, *maps, x, w, b)], k, interp,
                            needs=(False, True, False))[1]
    assert rel_err(got, getattr(O, name)(gy, *maps, x, w, b, k, interp)[1]) < 1e-12


@pytest.mark.parametrize("ci,co,k,locations", [
    # one output
    (10, 1, 9, 196607), (10, 1, 9, 196608), (6, 1, 8, 196608), (10, 1, 7, 196608), (16, 1, 17, 196608),
    (10, 1, 10, 196608), (3, 1, 5, 131072), (3, 1, 9, 131071), (3, 1, 9, 131072), (4, 1, 14, 131074),
    # groups of three taps, filled and not, on either side of 65 536 and 196 608
    (10, 1, 6, 65535), (10, 1, 6, 65536), (3, 1, 8, 65537), (2, 1, 7, 65539), (2, 1, 5, 196611), (12, 1, 10, 196608),
    (16, 1, 4, 196609), (1, 1, 25, 65536),
    # two to four: 65 536 locations, with more than nine taps 131 072, groups of three
    (4, 2, 8, 65535), (4, 2, 8, 65536), (4, 2, 7, 65536), (10, 4, 9, 65539),
    (5, 3, 17, 131071), (5, 3, 17, 131072), (5, 3, 25, 131073)])
def test_weight_gradient_around_the_rule_for_several_taps(ci, co, k, locations, device):
    """Locations and taps on either side of where a workgroup takes several taps.  Sums of 200 000
    terms of both signs in 64 bits: up to some 1e-14 of the result with their order, 1e-12 allowed."""
    g = torch.Generator().manual_seed(ci + 31 * k)
    ih, iw_ = 20, 33
    smap, _ = helpers.random_map(g, 1, locations, k, 0, ih, iw_, torch.float64)
    x, gy, w, b = (torch.randn(s, generator=g, dtype=torch.float64)
                   for s in ((1, ci, ih, iw_), (1, co, 1, locations), (co, ci, k), (co,)))
    got = _C.mapped_conv_backward(*[t.cuda() for t in (gy, smap, x, w, b)], k, 1,
                                  needs=(False, True, False))[1]
    assert rel_err(got, O.mapped_conv_backward(gy, smap, x, w, b, k, 1)[1]) < 1e-12
