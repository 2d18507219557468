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
# what the plan's report says of the kernel
KERNELS = {
    "igemm": "fp32 accumulate)\n",
    "pointwise": "pointwise streaming variant",
    "patch": "input patch resident in LDS",
    "rows": "dense row loads, small workgroups",
    "ring": "input rows streamed through an LDS ring",
    "columns": "strips of columns in registers",
    "tile": "LDS halo tiles",
    "small": "small tiles",
    "thin": "kernel rows as k-steps",
}
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
    # depthwise: small workgroups, strips of columns; rows in rings and tiles,
    # which have to be named at these sizes
    *[(name, dict(batch=2, field=(20, 18), kernel=(k, k), ci=1, co=1,
                  groups=c, pad=k // 2, stride=s), constraints)
      for name, k, constraints in (
          ("rows", 3, None), ("columns", 5, None), ("columns", 7, None),
          ("ring", 3, dict(rowRing=1)), ("ring", 5, dict(columns=0)),
          ("tile", 7, dict(columns=0)))
      for s in (1, 2) for c in (8, 40, 144)],
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
    plan = pa.Plan(p, options)
    kernel = plan.describe().split("Plan (")[1]
    assert KERNELS[name] in kernel, kernel
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


@pytest.mark.parametrize("name,kw,constraints", [
    # one 64-channel tile to a workgroup - the bias enters the sums divided by
    # the scale and is dealt out through LDS - and more of them
    *[("pointwise", dict(batch=3, field=(15, 14), kernel=(1, 1), ci=ci, co=co),
       dict(pointwise=1)) for ci, co in ((64, 8), (128, 72), (512, 64),
                                         (128, 256), (64, 192), (1024, 40))],
    ("igemm", dict(batch=3, field=(11, 9), kernel=(3, 3), ci=32, co=65, pad=1),
     IGEMM),
    ("small", dict(batch=1, field=(9, 8), kernel=(3, 3), ci=64, co=33, pad=1),
     dict(smallTile=1)),
])
@pytest.mark.parametrize("scales", [(0, 0), (-3, 5), (4, 2)])
def test_zero_weights_give_the_bias_of_quarters(name, kw, constraints, scales):
    p = make_params(pa.QUARTER, pa.HALF, **kw)
    print("case", p, constraints, scales, flush=True)
    plan = pa.Plan(p, {"planConstraints": json.dumps({"gfx950": constraints})})
    kernel = plan.describe().split("Plan (")[1]
    assert KERNELS[name] in kernel, kernel
    dev = torch.device("cuda:0")
    chans = p.getNumOutputChans()
    gen = torch.Generator(device=dev).manual_seed(8)

    def buf(which):
        return torch.zeros(max(plan.buffer_bytes(which), 16),
                           dtype=torch.uint8, device=dev)

    x = torch.randn(plan.buffer_bytes(capi.BUF_INPUT), generator=gen,
                    device=dev).to(torch.float8_e4m3fn).view(torch.uint8)
    w, packed = buf(capi.BUF_WEIGHTS_EXTERNAL), buf(capi.BUF_WEIGHTS_PACKED)
    # (halves that stay normal ones when divided by the scale)
    bias = torch.randn(chans + 1, generator=gen, device=dev).half()
    y = torch.full((plan.buffer_bytes(capi.BUF_OUTPUT) // 2,), float("nan"),
                   dtype=torch.float16, device=dev)
    ws = buf(capi.BUF_WORKSPACE)
    s = torch.cuda.current_stream().cuda_stream
    plan.pack_weights(w.data_ptr(), packed.data_ptr(), s)
    plan.fwd_quarter(x.data_ptr(), pa.quarter_metadata(1, scales[0]),
                     packed.data_ptr(), pa.quarter_metadata(1, scales[1]),
                     y.data_ptr(), bias[1:].data_ptr(), ws.data_ptr(),
                     plan.buffer_bytes(capi.BUF_WORKSPACE), s)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(
        y.cpu().numpy().reshape(-1, chans),
        np.broadcast_to(bias[1:].cpu().numpy(), (y.numel() // chans, chans)))
