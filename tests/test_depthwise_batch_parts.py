"""Depthwise layers whose batch goes out as several launches: the parts of a
batch that meets the limit of a launch's offsets exactly (1 GiB of input: a
part of as many bytes would be taken apart again, without end)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import poplibs_amd as pa
from poplibs_amd import capi
from helpers import make_params

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# 2^20 bytes of input to an image, so 1024 of them are the limit
LAYER = dict(field=(64, 64), groups=128)

CALL = """
import sys
sys.path[:0] = [{root!r}, {tests!r}]
import poplibs_amd as pa
from helpers import make_params
plan = pa.Plan(make_params(pa.HALF, batch={batch}, kernel=({k}, {k}),
                           pad={k} // 2, **{layer!r}))
try:
    plan.fwd(4096, 4096, 4096, None, 4096, 1 << 20, 0)
except pa.MxconvError as e:
    print("refused", e)
"""


@pytest.mark.parametrize("k", [3, 5, 7])
@pytest.mark.parametrize("batch", [1023, 1024, 1025, 2048])
def test_parts_come_to_an_end(batch, k):
    """Without a GPU: the first part's launch is refused.  (In a process of its
    own, which endless parts would end; the addresses are nobody's, so not
    where a launch could happen.)"""
    import torch
    if torch.cuda.is_available():
        pytest.skip("a process without a GPU")
    code = CALL.format(root=ROOT, tests=os.path.join(ROOT, "tests"),
                       batch=batch, k=k, layer=LAYER)
    done = subprocess.run([sys.executable, "-c", code], capture_output=True,
                          text=True, timeout=120)
    assert done.returncode == 0, done.returncode
    assert "refused" in done.stdout, done.stdout + done.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("k", [3, 5])
def test_parts_of_a_batch_at_the_limit(oracle, k):
    import torch
    p = make_params(pa.HALF, batch=1024, kernel=(k, k), pad=k // 2, **LAYER)
    print("case", k, flush=True)
    plan = pa.Plan(p)
    dev = torch.device("cuda:0")
    torch.manual_seed(3)
    shape = (1024, 64, 64, 128)
    acts = torch.randint(0, 2, shape, dtype=torch.int8, device=dev).half()
    acts = acts.mul_(2).sub_(1)
    assert acts.numel() * 2 == plan.buffer_bytes(capi.BUF_INPUT) == 1 << 30
    weights = np.random.default_rng(3).choice(
        [-1.0, 1.0], (128, 1, 1, k, k)).astype(np.float16)
    w = torch.from_numpy(weights).to(dev)
    packed = torch.empty(plan.buffer_bytes(capi.BUF_WEIGHTS_PACKED),
                         dtype=torch.uint8, device=dev)
    out = torch.full(shape, float("nan"), dtype=torch.float16, device=dev)
    need = plan.buffer_bytes(capi.BUF_WORKSPACE)
    work = torch.empty(max(need, 16), dtype=torch.uint8, device=dev)
    s = torch.cuda.current_stream().cuda_stream
    plan.pack_weights(w.data_ptr(), packed.data_ptr(), s)
    plan.fwd(acts.data_ptr(), packed.data_ptr(), out.data_ptr(), None,
             work.data_ptr(), need, s)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out).all())
    # the first images, and those around the line between the parts
    at = [0, 511, 1022, 1023]
    one = make_params(pa.HALF, batch=len(at), kernel=(k, k), pad=k // 2,
                      **LAYER)
    want = oracle.convolution(
        one, acts[at].permute(0, 3, 1, 2).cpu().numpy().astype(np.float64),
        weights.astype(np.float64), threads=8)
    # (sums of up to 25 signs: whole numbers that halves hold)
    np.testing.assert_array_equal(
        out[at].permute(0, 3, 1, 2).cpu().numpy().astype(np.float64), want)
