"""Outputs of zero weights are the bias, exactly, in every channel of every
pixel: each kernel's way of reading it, at channel counts that end inside a tile,
from an address that is a multiple of no more than an element's size."""
import json

import numpy as np
import pytest
import torch

import poplibs_amd as pa
from helpers import make_params
from poplibs_amd import capi

pytestmark = pytest.mark.gpu

TORCH = {pa.FLOAT: torch.float32, pa.HALF: torch.float16}
IGEMM = dict(kernel="igemm", patch=0, pointwise=0, smallTile=0)
CASES = [
    # igemmKernel: tiles of 64 and 128 channels, two and four stages; a channel
    # less and more than a tile's; groups; several phases in a launch
    *[("igemm", dict(batch=3, field=(11, 9), kernel=(3, 3), ci=24, co=co,
                     pad=1), dict(IGEMM, blockN=bn, stages=st))
      for co in (1, 63, 65, 130) for bn, st in ((64, 2), (128, 2), (128, 4))],
    ("igemm", dict(batch=2, field=(13, 10), kernel=(3, 3), ci=16, co=40,
                   groups=3, pad=1, stride=2), IGEMM),
    ("igemm", dict(batch=2, field=(9, 9), kernel=(3, 3), ci=32, co=72, pad=1,
                   idil=(2, 2)), IGEMM),
    ("igemm", dict(batch=2, field=(9, 9), kernel=(3, 3), ci=64, co=200, pad=1),
     dict(IGEMM, splitK=3)),
    ("igemm", dict(batch=9, field=(17, 17), kernel=(1, 1), ci=64, co=200),
     dict(blockM=256, blockN=256)),
    # pointwiseKernel: one 64-channel tile to a workgroup, and more
    *[("pointwise", dict(batch=3, field=(15, 14), kernel=(1, 1), ci=ci, co=co),
       dict(pointwise=1)) for ci, co in ((64, 8), (256, 64), (64, 72),
                                         (64, 256), (128, 136), (512, 40))],
    # resident patches
    *[("patch", dict(batch=3, field=(12, 13), kernel=(3, 3), ci=64, co=co,
                     pad=1), dict(patch=mode))
      for mode in (1, 2) for co in (72, 128, 136, 200)],
    # depthwise: rows in rings, strips of columns, tiles
    *[("depthwise", dict(batch=2, field=(20, 18), kernel=(k, k), ci=1, co=1,
                         groups=c, pad=k // 2, stride=s), None)
      for k in (3, 5, 7) for s in (1, 2) for c in (8, 40, 144)],
    # tiles of a few pixels, a first layer
    ("small", dict(batch=1, field=(9, 8), kernel=(3, 3), ci=40, co=33, pad=1),
     dict(smallTile=1)),
    ("thin", dict(batch=2, field=(33, 30), kernel=(7, 7), ci=3, co=48, pad=3,
                  stride=2), dict(thinInput=1)),
]


@pytest.mark.parametrize("out_type", [pa.HALF, pa.FLOAT])
@pytest.mark.parametrize("name,kw,constraints", CASES)
def test_zero_weights_give_the_bias(name, kw, constraints, out_type):
    p = make_params(pa.HALF, out_type, **kw)
    print("case", p, constraints, flush=True)
    options = {"planConstraints": json.dumps({"gfx950": constraints})} \
        if constraints else None
    try:
        plan = pa.Plan(p, options)
    except pa.MxconvError as e:
        pytest.skip(str(e))
    dev = torch.device("cuda:0")
    chans = p.getNumOutputChans()
    gen = torch.Generator(device=dev).manual_seed(7)

    def buf(which):
        return torch.zeros(max(plan.buffer_bytes(which), 16),
                           dtype=torch.uint8, device=dev)

    x = torch.randn(plan.buffer_bytes(capi.BUF_INPUT) // 2, generator=gen,
                    device=dev).half()
    w, packed = buf(capi.BUF_WEIGHTS_EXTERNAL), buf(capi.BUF_WEIGHTS_PACKED)
    bias = torch.randn(chans + 1, generator=gen, device=dev).to(TORCH[out_type])
    n = plan.buffer_bytes(capi.BUF_OUTPUT) // (2 if out_type == pa.HALF else 4)
    y = torch.full((n,), float("nan"), dtype=TORCH[out_type], device=dev)
    ws = buf(capi.BUF_WORKSPACE)
    s = torch.cuda.current_stream().cuda_stream
    plan.pack_weights(w.data_ptr(), packed.data_ptr(), s)
    plan.fwd(x.data_ptr(), packed.data_ptr(), y.data_ptr(),
             bias[1:].data_ptr(), ws.data_ptr(),
             plan.buffer_bytes(capi.BUF_WORKSPACE), s)
    torch.cuda.synchronize()
    want = bias[1:].cpu().numpy()
    np.testing.assert_array_equal(
        y.cpu().numpy().reshape(-1, chans),
        np.broadcast_to(want, (n // chans, chans)))
