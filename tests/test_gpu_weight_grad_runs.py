"""fp32 weight gradients over runs of neighbouring pixels: groups of eight pixels and strips of eight
groups that end inside a row, blocks of 16 gathered and 64 plain channels, passes of nine taps, runs
that wrap at the seam, leave the image or are two pixels apart, maps without runs, and operands
that the split cannot represent."""
import pytest
import torch

from helpers import rel_err
from oracle import ops as O

from mappedconvolutions_amd import _C
from mappedconvolutions_amd.util import synthetic

pytestmark = pytest.mark.gpu


def _grid(h, w, k, dx, dy, step=1):
    y, x = torch.meshgrid(torch.arange(h).float(), torch.arange(w).float(), indexing="ij")
    side = max(1, round(k ** 0.5))
    taps = [torch.stack((step * x + i % side - side // 2 + dx, step * y + i // side - side // 2 + dy), -1)
            for i in range(k)]
    return torch.stack(taps, 2).contiguous()


def _check(B, ci, co, ih, iw, smap, interp, weights=None, seed=0):
    g = torch.Generator().manual_seed(seed)
    oh, ow, k = smap.shape[:3]
    x, gy = torch.randn(B, ci, ih, iw, generator=g), torch.randn(B, co, oh, ow, generator=g)
    w, b = torch.randn(co, ci, k, generator=g), torch.randn(co, generator=g)
    if weights is None:
        got = _C.mapped_conv_backward(gy.cuda(), smap.cuda(), x.cuda(), w.cuda(), b.cuda(), k, interp,
                                      needs=(False, True, True))
        want = O.mapped_conv_backward(gy, smap, x, w, b, k, interp)
    else:
        got = _C.weighted_mapped_conv_backward(
            *[t.cuda() for t in (gy, smap, weights, x, w, b)], k, interp, needs=(False, True, True))
        want = O.weighted_mapped_conv_backward(gy, smap, weights, x, w, b, k, interp)
    # 32-bit sums of some thousand terms: a few 1e-7 of the result's magnitude, 1e-5 allowed as
    # everywhere in these tests
    assert rel_err(got[1], want[1]) < 1e-5 and rel_err(got[2], want[2]) < 1e-5


@pytest.mark.parametrize("h,w", [(2, 1), (2, 7), (3, 8), (4, 9), (3, 63), (2, 64), (5, 65), (3, 72),
                                 (7, 130), (33, 69)])
@pytest.mark.parametrize("interp,dx,dy", [(0, 0.0, 0.0), (1, 0.25, 0.0), (1, -0.4, 0.3),
                                          (2, 0.25, 0.0), (2, -0.3, 0.6)])
def test_rows_that_end_inside_a_group_or_a_strip(h, w, interp, dx, dy, device):
    _check(2, 17, 5, h, w, _grid(h, w, 9, dx, dy), interp)


@pytest.mark.parametrize("ci,co", [(1, 1), (3, 64), (15, 65), (16, 16), (17, 130), (33, 63)])
@pytest.mark.parametrize("k", [1, 2, 3, 9, 10, 25])
def test_channels_and_taps(ci, co, k, device):
    _check(2, ci, co, 6, 40, _grid(6, 40, k, 0.3, 0.4), 2)


@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("step,h,w", [(1, 24, 48), (2, 12, 24), (2, 5, 17), (3, 6, 20)])
def test_seams_poles_and_steps(interp, step, h, w, device):
    """Columns wrap inside a group, rows are clamped at the poles; every second or third column."""
    smap = synthetic.latitude_map(step * h, step * w, 1)[::step, ::step].contiguous()
    _check(1, 20, 24, step * h, step * w, smap, interp)
    _check(2, 20, 24, step * h, step * w, _grid(h, w, 9, 0.25, 0.5, step), interp)


@pytest.mark.parametrize("part", [0.0, 0.01, 0.03, 0.05, 0.1, 0.5, 1.0])
def test_maps_with_pixels_out_of_place(part, device):
    """A share of the pixels samples anywhere: their groups are read corner by corner, and with
    many of them the whole map goes to the general kernel."""
    g = torch.Generator().manual_seed(7)
    h, w, k = 16, 64, 9
    smap = _grid(h, w, k, 0.3, 0.2)
    away = torch.rand(h, w, k, 1, generator=g) < part / 8
    anywhere = torch.rand(h, w, k, 2, generator=g) * torch.tensor([w + 4.0, h + 4.0]) - 2
    for interp in (1, 2):
        _check(2, 20, 24, h, w, torch.where(away, anywhere, smap), interp)


@pytest.mark.parametrize("interp", [1, 2])
@pytest.mark.parametrize("h,w", [(2, 130), (3, 33), (4, 32), (5, 33), (9, 72)])
@pytest.mark.parametrize("k", [1, 9, 10])
@pytest.mark.parametrize("weighted", [False, True])
def test_whole_rows_without_runs(interp, h, w, k, weighted, device):
    """Mirrored rows: no runs, two corners a tap, which the general kernel reads from a table made by
    the launch that found no runs; tiles of one and of four rows that end ragged."""
    smap = _grid(h, w, k, 0.25, 0.0)
    smap[..., 0] = w - 1 - smap[..., 0]
    weights = None
    if weighted:
        weights = torch.rand(h, w, k, 1, generator=torch.Generator().manual_seed(3)) - 0.5
        smap = smap.unsqueeze(3).contiguous()
    _check(2, 20, 70, h, w, smap, interp, weights)


@pytest.mark.parametrize("B,ci,co,h,w,k,interp,planned", [
    (1, 20, 24, 6, 40, 2, 0, False), (2, 33, 70, 9, 40, 4, 0, False),   # one corner a tap: few launches
    (16, 300, 130, 12, 136, 1, 2, False),                              # one tap of many channels
    (2, 128, 128, 32, 64, 9, 2, True), (2, 128, 128, 32, 64, 9, 1, True)])  # a plan for less than a round
@pytest.mark.parametrize("dy", [0.0, 0.4])
def test_calls_that_the_general_kernel_serves_sooner(B, ci, co, h, w, k, interp, planned, dy, device):
    """Maps of runs all the same: the sizes decide."""
    g = torch.Generator().manual_seed(4)
    smap = _grid(h, w, k, 0.0 if interp == 0 else 0.25, dy)
    x, gy = torch.randn(B, ci, h, w, generator=g), torch.randn(B, co, h, w, generator=g)
    wt, b = torch.zeros(co, ci, k), torch.zeros(co)
    dev = [t.cuda() for t in (gy, smap, x, wt, b)]
    plan = _C.conv_map_plan(dev[1], None, h, w, interp, torch.float32) if planned else None
    got = _C.mapped_conv_backward(*dev, k, interp, plan=plan, needs=(False, True, True))
    want = O.mapped_conv_backward(gy, smap, x, wt, b, k, interp)
    assert rel_err(got[1], want[1]) < 1e-5 and rel_err(got[2], want[2]) < 1e-5


@pytest.mark.parametrize("interp", [0, 1])
def test_one_weighted_point_per_tap(interp, device):
    g = torch.Generator().manual_seed(8)
    weights = torch.rand(9, 33, 9, 1, generator=g)
    smap = _grid(9, 33, 9, 0.25, 0.4).unsqueeze(3).contiguous()
    _check(2, 20, 24, 9, 33, smap, interp, weights)


@pytest.mark.parametrize("what", ["x_inf", "x_nan", "gy_inf", "large"])
def test_operands_without_a_split(what, device):
    """Infinite, NaN and very large operands end as the fp32 instructions have them."""
    g = torch.Generator().manual_seed(9)
    B, ci, co, h, w, k = 1, 16, 20, 6, 40, 9
    smap = _grid(h, w, k, 0.25, 0.25)
    x, gy = torch.rand(B, ci, h, w, generator=g) + 0.5, torch.rand(B, co, h, w, generator=g) + 0.5
    wt, b = torch.zeros(co, ci, k), torch.zeros(co)
    if what == "large":
        x[0, 3] *= 3e37
    elif what == "gy_inf":
        gy[0, 7, 2, 9] = float("inf")
    else:
        x[0, 3, 2, 9] = float("inf" if what == "x_inf" else "nan")
    gw = _C.mapped_conv_backward(gy.cuda(), smap.cuda(), x.cuda(), wt.cuda(), b.cuda(), k, 1,
                                 needs=(False, True, False))[1].cpu()
    want = O.mapped_conv_backward(gy, smap, x, wt, b, k, 1)[1]
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(gw), ok) and torch.equal(torch.isnan(gw), torch.isnan(want))
    scale = want.abs().masked_fill(~ok, 0).amax((0, 2), keepdim=True)
    assert (((gw - want).abs() <= 1e-5 * scale) | ~ok).all()


@pytest.mark.parametrize("p,q", [(0, 0), (-110, 60), (-124, 30), (60, -112), (100, -100)])
def test_operands_of_every_magnitude_count_in_full(p, q, device):
    g = torch.Generator().manual_seed(10)
    B, ci, co, h, w, k = 1, 20, 24, 8, 40, 9
    smap = _grid(h, w, k, 0.0, 0.0)
    unit = lambda *s: (1 + torch.rand(s, generator=g)) * (1 - 2 * torch.randint(2, s, generator=g))
    u, v = unit(B, ci, h, w), unit(B, co, h, w)
    wt, b = torch.zeros(co, ci, k), torch.zeros(co)
    gw = _C.mapped_conv_backward((v * 2.0 ** q).cuda(), smap.cuda(), (u * 2.0 ** p).cuda(), wt.cuda(),
                                 b.cuda(), k, 1, needs=(False, True, False))[1]
    got = gw.double().cpu() * 2.0 ** -(p + q)
    want = O.mapped_conv_backward(v.double(), smap.double(), u.double(), wt.double(), b.double(), k, 1)[1]
    assert ((got - want).norm() / want.norm()).item() < 1e-6


@pytest.mark.parametrize("B,h,w,bar", [(1, 64, 128, 2.2e-7), (4, 128, 256, 3e-7)])
def test_what_the_sums_lose_does_not_add_up(B, h, w, bar, device):
    """The matrix instruction rounds downwards; over many pixels that would show as an error of one
    sign, larger than the fp32 instructions' (which were 2.2e-7 and 3.7e-7 off in 2-norm here)."""
    g = torch.Generator(device="cuda").manual_seed(11)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    smap = synthetic.latitude_map(h, w, 1).cuda()
    x, gy, wt, b = rnd(B, 16, h, w), rnd(B, 64, h, w), rnd(64, 16, 9), rnd(64)
    grad = lambda t: _C.mapped_conv_backward(*[a.to(t) for a in (gy, smap, x, wt, b)], 9, 1,
                                             needs=(False, True, False))[1].double()
    want = grad(torch.float64)
    err = grad(torch.float32) - want
    assert (err.norm() / want.norm()).item() < bar
    assert (err.mean().abs() / err.std()).item() < 0.1


# (in 2-norm and units of 1e-7, what the fp32 instructions were off here)
@pytest.mark.parametrize("B,h,w,normal,positive,relu", [
    (1, 4, 16, 1.46, 1.23, 0.72), (1, 8, 16, 1.49, 0.93, 0.61), (1, 16, 16, 1.53, 0.71, 0.55),
    (1, 16, 32, 2.11, 0.95, 0.64), (1, 16, 64, 2.09, 0.74, 0.55), (1, 32, 64, 2.14, 0.60, 0.51)])
def test_short_sums_are_as_near_to_64_bits_as_fp32_sums(B, h, w, normal, positive, relu, device):
    """One to eight tiles of 128 pixels, operands of either sign, positive ones, and half zeros."""
    g = torch.Generator(device="cuda").manual_seed(12)
    smap = synthetic.latitude_map(h, w, 1).cuda()
    wt, b = torch.zeros(64, 16, 9, device="cuda"), torch.zeros(64, device="cuda")
    for kind, bar in ((lambda t: t, normal), (torch.abs, positive), (lambda t: t.clamp_min(0), relu)):
        x, gy = (kind(torch.randn(B, c, h, w, generator=g, device="cuda")) for c in (16, 64))
        grad = lambda t: _C.mapped_conv_backward(*[a.to(t) for a in (gy, smap, x, wt, b)], 9, 2,
                                                 needs=(False, True, False))[1].double()
        want = grad(torch.float64)
        assert ((grad(torch.float32) - want).norm() / want.norm()).item() < bar * 1e-7


@pytest.mark.parametrize("runs", [True, False])
def test_the_timed_kernel_is_the_one_that_does_the_work(runs, device):
    """A weight gradient's timing request covers the kernel over runs or, for maps without, the
    general one: the larger part of the call, whichever it is."""
    B, ci, co, h, w = 2, 64, 64, 128, 256
    smap = (synthetic.latitude_map(h, w, 1) if runs else synthetic.pixel_shuffle_map(h, w)).cuda()
    x, gy = torch.randn(B, ci, h, w, device="cuda"), torch.randn(B, co, h, w, device="cuda")
    wt, b = torch.randn(co, ci, 9, device="cuda"), torch.randn(co, device="cuda")
    call = lambda: _C.mapped_conv_backward(gy, smap, x, wt, b, 9, 1, needs=(False, True, False))
    (start, end), = _C.make_event_pool(1, device)
    pool = _C.make_event_pool(1, device)
    for _ in range(20):  # (the GPU is behind: what the host takes is not measured)
        call()
    try:
        _C.profile_pool, _C.profile_events = pool, []
        start.record()
        call()
        end.record()
        torch.cuda.synchronize()
        (label, first, last), = _C.profile_events
    finally:
        _C.profile_pool, _C.profile_events = [], None
    assert label == "conv_backward_weight"
    assert first.elapsed_time(last) > 0.3 * start.elapsed_time(end)
