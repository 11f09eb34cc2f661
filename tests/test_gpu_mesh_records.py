"""fp32 convolutions over vertices (channel-last records that four lanes read together): one to four
points a tap, channel counts around the 16 of a chunk and the 64 and 128 of a workgroup, vertex
counts around a tile's 128, and cells of the transposed map of up to eight contributions and more."""
import pytest
import torch

from helpers import rel_err
from oracle import ops as O

from mappedconvolutions_amd import _C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("points", [1, 2, 3, 4])
@pytest.mark.parametrize("ci,co,v", [(3, 5, 127), (16, 64, 128), (20, 65, 129), (33, 130, 300),
                                     (130, 17, 64)])
@pytest.mark.parametrize("spread", [1.0, 0.2])
def test_weighted_mesh_convolution(points, ci, co, v, spread, device):
    g = torch.Generator().manual_seed(100 * points + ci)
    B, k = 2, 7
    idx = torch.randint(max(1, int(v * spread)), (1, v, k, points), generator=g).float()
    smap = torch.stack((idx, torch.zeros_like(idx)), -1).contiguous()
    iw = torch.rand(1, v, k, points, generator=g)
    iw[torch.rand(iw.shape, generator=g) < 0.2] = 0  # (corners that weigh nothing)
    x, w, b, gy = (torch.randn(s, generator=g)
                   for s in ((B, ci, 1, v), (co, ci, k), (co,), (B, co, 1, v)))
    dev = [t.cuda() for t in (x, smap, iw, w, b, gy)]
    # 32-bit sums of up to some thousand terms: a few 1e-7 of the result's magnitude, 1e-5 allowed
    # as everywhere in these tests
    y = _C.weighted_mapped_conv_forward(*dev[:5], k, 0)
    assert rel_err(y, O.weighted_mapped_conv_forward(x, smap, iw, w, b, k, 0)) < 1e-5
    got = _C.weighted_mapped_conv_backward(dev[5], *dev[1:3], dev[0], *dev[3:5], k, 0)
    want = O.weighted_mapped_conv_backward(gy, smap, iw, x, w, b, k, 0)
    for a, e in zip(got, want):
        assert rel_err(a, e) < 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("points,k", [(1, 7), (2, 7), (3, 8), (4, 1), (4, 7), (4, 9), (4, 10)])
@pytest.mark.parametrize("ci,co,v", [(32, 40, 1030), (33, 129, 1100), (64, 64, 2100), (100, 8, 520),
                                     (256, 64, 1025)])
def test_weight_gradient_over_chunks_of_records(dtype, points, k, ci, co, v, device):
    """Channel groups that share out the XCDs (two, four and eight of them) and others, ranges of tiles that
    are a multiple of eight and not, and taps around the seven and nine of a pass."""
    g = torch.Generator().manual_seed(1000 * points + ci + k)
    B = 2
    idx = torch.randint(v, (1, v, k, points), generator=g).float()
    smap = torch.stack((idx, torch.zeros_like(idx)), -1).contiguous()
    iw = torch.rand(1, v, k, points, generator=g)
    x, gy = (torch.randn(s, generator=g).to(dtype) for s in ((B, ci, 1, v), (B, co, 1, v)))
    w, b = torch.zeros(co, ci, k, dtype=dtype), torch.zeros(co, dtype=dtype)
    got = _C.weighted_mapped_conv_backward(gy.cuda(), smap.cuda(), iw.cuda(), x.cuda(), w.cuda(),
                                           b.cuda(), k, 0, needs=(False, True, True))
    # in 64 bits, tap by tap: [B, ci, v] samples against [B, co, v]
    cols = torch.stack([(x.double()[:, :, 0, idx[0, :, t].long()] * iw[0, :, t].double()).sum(-1)
                        for t in range(k)])
    gw = torch.einsum("bon,kbcn->ock", gy.double()[:, :, 0], cols)
    # fp32: some thousand terms, a few 1e-7; bf16: samples rounded to 2^-9 each and the result once
    tol = 1e-5 if dtype == torch.float32 else 8e-3
    assert rel_err(got[1], gw) < tol
    assert rel_err(got[2], gy.double().sum((0, 2, 3))) < tol


@pytest.mark.parametrize("points,k,ci,co,v", [
    (4, 7, 96, 40, 10922), (4, 7, 96, 40, 10923),  # 2 MB of records, in chunks and whole
    (3, 9, 70, 130, 22000),                        # five groups of channels, two of plain ones
    (4, 1, 160, 8, 6600), (3, 10, 250, 20, 4200),  # ten and sixteen groups
])
def test_bf16_weight_gradient_over_whole_records(points, k, ci, co, v, device):
    """bf16 records of more than 2 MB an image stay whole where the groups of channels are more than four
    and do not share out the XCDs.  Samples are rounded to 2^-9 each and the result once: as above."""
    g = torch.Generator().manual_seed(ci + k)
    B = 2
    idx = torch.randint(v, (1, v, k, points), generator=g).float()
    smap = torch.stack((idx, torch.zeros_like(idx)), -1).contiguous()
    iw = torch.rand(1, v, k, points, generator=g)
    x, gy = (torch.randn(s, generator=g).to(torch.bfloat16) for s in ((B, ci, 1, v), (B, co, 1, v)))
    w, b = torch.zeros(co, ci, k, dtype=torch.bfloat16), torch.zeros(co, dtype=torch.bfloat16)
    got = _C.weighted_mapped_conv_backward(gy.cuda(), smap.cuda(), iw.cuda(), x.cuda(), w.cuda(),
                                           b.cuda(), k, 0, needs=(False, True, False))[1]
    gw = torch.zeros(co, ci, k, dtype=torch.float64)
    for t in range(k):
        col = (x.double()[:, :, 0, idx[0, :, t].long()] * iw[0, :, t].double()).sum(-1)
        gw[:, :, t] = torch.bmm(gy.double()[:, :, 0], col.transpose(1, 2).contiguous()).sum(0)
    assert rel_err(got, gw) < 8e-3
