"""Input gradients whose transposed map overfills cells: the list of what is left, by entries and by
images, channel counts around the 16, 32 and 64 lanes of an entry, and lists that overflow as well."""
import pytest
import torch

from helpers import map_contributions, rel_err, transposed_map_overflows
from oracle import ops as O

from mappedconvolutions_amd import _C

pytestmark = pytest.mark.gpu


# (ci is the gradient's channel count; 128 x 64 weights of a tap: images share their reading)
@pytest.mark.parametrize("B", [1, 2, 5])
@pytest.mark.parametrize("ci,co", [(3, 5), (16, 20), (17, 8), (33, 64), (64, 128), (65, 40)])
# (one pixel: what a wave holds for it is added up before the atomics)
@pytest.mark.parametrize("pixels", [1, 6])
@pytest.mark.parametrize("share", [0.1, 0.4, 1.0])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_many_contributions_to_few_pixels(B, ci, co, pixels, share, dtype, device):
    g = torch.Generator().manual_seed(ci + co)
    h, w_, k = 12, 20, 3
    y, x = torch.meshgrid(torch.arange(h).float(), torch.arange(w_).float(), indexing="ij")
    smap = torch.stack((x, y), -1).unsqueeze(2).repeat(1, 1, k, 1)
    crowd = torch.rand(h, w_, k, 1, generator=g) < share  # (these meet in one pixel or in six)
    to = torch.rand(h, w_, k, 2, generator=g) * torch.tensor([2.0, 1.0]) * (pixels > 1) + 3
    smap = torch.where(crowd, to, smap)
    smap = smap.contiguous()
    rnd = lambda *s: torch.randn(s, generator=g).to(dtype).float()
    xs, wt, b, gy = rnd(B, ci, h, w_), rnd(co, ci, k), rnd(co), rnd(B, co, h, w_)
    gx = _C.mapped_conv_backward(gy.cuda().to(dtype), smap.cuda(), xs.cuda().to(dtype),
                                 wt.cuda().to(dtype), b.cuda().to(dtype), k, 1,
                                 needs=(True, False, False))[0]
    want = O.mapped_conv_backward(gy, smap, xs, wt, b, k, 1)[0]
    # (the bars of the other tests: 32-bit sums, and results and samples rounded to bf16)
    assert rel_err(gx.float(), want) < (1e-5 if dtype == torch.float32 else 2e-2)


@pytest.mark.parametrize("ci,co", [(10, 1), (24, 40), (40, 8), (64, 20)])
@pytest.mark.parametrize("pixels", [1, 6])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_long_lists(ci, co, pixels, dtype, device):
    """So many entries and images that every workgroup takes several pieces of the list; its last piece
    is not full, and the next image begins where it ends."""
    g = torch.Generator().manual_seed(ci)
    B, h, w_, k = 100, 12, 20, 7
    y, x = torch.meshgrid(torch.arange(h).float(), torch.arange(w_).float(), indexing="ij")
    smap = torch.stack((x, y), -1).unsqueeze(2).repeat(1, 1, k, 1)
    crowd = torch.rand(h, w_, k, 1, generator=g) < 0.9  # (whole pixels: one contribution each)
    to = (torch.rand(h, w_, k, 2, generator=g) * torch.tensor([3.0, 2.0])).floor() * (pixels > 1) + 3
    smap = torch.where(crowd, to, smap).contiguous()
    cells = map_contributions(smap, None, h, w_, 1)
    spill = (torch.bincount(cells, minlength=h * w_ * k) - 4).clamp_min(0).sum().item()
    assert spill * B // (4 * 64 // (16 if ci <= 16 else 32 if ci <= 32 else 64)) > 2048
    assert not transposed_map_overflows(smap, None, h, w_, 1)
    rnd = lambda *s: torch.randn(s, generator=g).to(dtype).float()
    xs, wt, b, gy = rnd(B, ci, h, w_), rnd(co, ci, k), rnd(co), rnd(B, co, h, w_)
    gx = _C.mapped_conv_backward(gy.cuda().to(dtype), smap.cuda(), xs.cuda().to(dtype),
                                 wt.cuda().to(dtype), b.cuda().to(dtype), k, 1,
                                 needs=(True, False, False))[0]
    want = O.mapped_conv_backward(gy, smap, xs, wt, b, k, 1)[0]
    assert rel_err(gx.float(), want) < (1e-5 if dtype == torch.float32 else 2e-2)
