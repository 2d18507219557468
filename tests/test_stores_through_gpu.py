"""Outputs that are stored through the L2 are the bytes they should be, wherever
they start, and nothing is written in front of them or behind them.

Streaming and wide tiles and first layers go through the L2 where the result starts
at a multiple of 16 bytes and by way of it from 8 bytes or an element further on:
there the comparison is of the two ways.  The other kernels go the same way from
any address - through it, but for depthwise rows of more than 12 MB and fp32 results
of depthwise layers - and what counts is the comparison with conv2d."""
import json

import pytest
import torch

import poplibs_amd as pa
from helpers import make_params
from poplibs_amd import capi

pytestmark = pytest.mark.gpu

TORCH = {pa.FLOAT: torch.float32, pa.HALF: torch.float16}
IGEMM = dict(kernel="igemm", patch=0, pointwise=0, smallTile=0)
STREAMING, RING = "fp32 accumulate)\n", "streamed through an LDS ring"
CASES = [
    # channels that fill a tile's vectors and end inside a tile, one row of
    # pixels more than tiles; K in parts; phases in one launch; groups
    *[(STREAMING, dict(batch=3, field=(11, 12), kernel=(3, 3), ci=24, co=co,
                       pad=1), dict(IGEMM, blockN=bn))
      for co in (8, 72, 136) for bn in (64, 128)],
    # (the parts go to the workspace and their sum through the L2 either way)
    ("summed by a second kernel", dict(
        batch=2, field=(9, 9), kernel=(3, 3), ci=64, co=200, pad=1),
     dict(IGEMM, splitK=3)),
    ("4 phases, one convolution", dict(
        batch=2, field=(9, 9), kernel=(3, 3), ci=32, co=72, pad=1,
        idil=(2, 2)), IGEMM),
    (STREAMING, dict(batch=2, field=(13, 10), kernel=(3, 3), ci=16, co=40,
                     groups=3, pad=1), IGEMM),
    *[("256 x %d x 64" % bn, dict(batch=5, field=(15, 15), kernel=(3, 3),
                                  ci=64, co=co, pad=1),
       dict(blockM=256, blockN=bn)) for co, bn in ((200, 192), (264, 256))],
    *[("small tiles", dict(batch=1, field=(9, 8), kernel=(3, 3), ci=40, co=co,
                           pad=1), dict(smallTile=2)) for co in (4, 36)],
    # pointwise rows that are no whole 64-byte pieces: few bytes of them, and
    # more than 12 MB (a pair of channel blocks to a store)
    *[("pointwise streaming", dict(batch=b, field=(31, 33), kernel=(1, 1),
                                   ci=32, co=co), dict(pointwise=1))
      for b, co in ((2, 40), (40, 168))],
    # first layers: pairs of 16-channel blocks, and an odd number of blocks,
    # which does not go through the L2
    *[("kernel rows as k-steps", dict(batch=2, field=(33, 30), kernel=(7, 7),
                                      ci=3, co=co, pad=3, stride=2),
       dict(thinInput=1)) for co in (32, 64, 48)],
    # depthwise: small workgroups, rings of rows on both sides of 12 MB
    *[("dense row loads, small workgroups", dict(
        batch=2, field=(20, 18), kernel=(3, 3), ci=1, co=1, groups=40, pad=1,
        stride=st), dict(rowRing=0)) for st in (1, 2)],
    *[(RING, dict(batch=b, field=(56, 55), kernel=(3, 3), ci=1, co=1,
                  groups=144, pad=1), dict(rowRing=1)) for b in (1, 13, 14)],
    (RING, dict(batch=3, field=(21, 20), kernel=(5, 5), ci=1, co=1, groups=40,
                pad=2, stride=2), dict(columns=0, rowRing=1)),
]


@pytest.mark.parametrize("out_type", [pa.HALF, pa.FLOAT])
@pytest.mark.parametrize("kernel,kw,constraints", CASES)
def test_same_bytes_through_the_l2(kernel, kw, constraints, out_type):
    p = make_params(pa.HALF, out_type, **kw)
    print("case", p, constraints, flush=True)
    plan = pa.Plan(p, {"planConstraints": json.dumps({"gfx950": constraints})})
    assert kernel in plan.describe(), plan.describe()
    gen = torch.Generator(device="cuda").manual_seed(3)
    dev, s = torch.device("cuda:0"), torch.cuda.current_stream().cuda_stream

    def randoms(n):
        return torch.randn(n, generator=gen, device=dev).half()

    def room(which):
        return torch.empty(max(plan.buffer_bytes(which), 16),
                           dtype=torch.uint8, device=dev)

    taps = p.kernelShape[0] * p.kernelShape[1]
    pixels, out_pixels = p.batchSize, p.batchSize
    for i, o in zip(p.inputFieldShape, p.getOutputFieldShape()):
        pixels, out_pixels = pixels * i, out_pixels * o
    x = randoms(pixels * p.getNumInputChans())
    w = randoms(p.getNumOutputChans() * p.inputChannelsPerConvGroup * taps)
    bias = torch.randn(p.getNumOutputChans(), generator=gen,
                       device=dev).to(TORCH[out_type])
    packed, work = room(capi.BUF_WEIGHTS_PACKED), room(capi.BUF_WORKSPACE)
    plan.pack_weights(w.data_ptr(), packed.data_ptr(), s)
    size = out_pixels * p.getNumOutputChans() * bias.element_size()
    guard = 64
    outs = []
    for off in (0, 8, bias.element_size()):
        buf = torch.full((size + 2 * guard + 8,), 0x5A, dtype=torch.uint8,
                         device=dev)
        assert buf.data_ptr() % 16 == 0
        plan.fwd(x.data_ptr(), packed.data_ptr(),
                 buf.data_ptr() + guard + off, bias.data_ptr(),
                 work.data_ptr(), work.numel(), s)
        torch.cuda.synchronize()
        first, last = guard + off, guard + off + size
        assert bool((buf[:first] == 0x5A).all())
        assert bool((buf[last:] == 0x5A).all())
        outs.append(buf[first:last].clone())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    # fp32 on the CPU, undilated inputs
    if not p.inputTransform.dilation or max(p.inputTransform.dilation) == 1:
        g = p.numConvGroups
        xs = x.float().cpu().reshape(
            p.batchSize, *p.inputFieldShape, -1).permute(0, 3, 1, 2)
        ws = w.float().cpu().reshape(
            p.getNumOutputChans(), p.inputChannelsPerConvGroup,
            *p.kernelShape)
        ref = torch.nn.functional.conv2d(
            xs, ws, bias.float().cpu(), padding=p.kernelShape[0] // 2,
            stride=tuple(p.outputTransform.stride), groups=g)
        got = outs[0].view(TORCH[out_type]).float().cpu().reshape(
            p.batchSize, *p.getOutputFieldShape(), -1).permute(0, 3, 1, 2)
        err = (got - ref).norm() / ref.norm()
        # fp32 sums of halves either way; a half result rounds once
        assert err <= (1e-3 if out_type == pa.HALF else 1e-5), err
