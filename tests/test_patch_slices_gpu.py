"""The resident-patch kernel of 16-pixel blocks beyond whole channel slices
that all fit in LDS (csrc/igemm_patch.hip): a partial last slice, K cut along
its slices, rings of slices, against the CPU oracle."""
import json

import numpy as np
import pytest

import poplibs_amd as pa
from helpers import make_params, random_data, rel_l2

PATCH = "MFMA blocks of 16 pixels"


def _options(parts=1, **more):
    doc = dict(patch=2, **more)
    if parts > 1:
        doc["splitK"] = parts
    return {"planConstraints": json.dumps({"gfx950": doc})}


CASES = [
    # a partial slice alone, behind whole ones, of one vector, of all but one
    (dict(batch=2, field=(9, 11), kernel=(3, 3), ci=8, co=72, pad=1), 1),
    (dict(batch=2, field=(9, 11), kernel=(3, 3), ci=72, co=72, pad=1), 1),
    (dict(batch=2, field=(14, 14), kernel=(3, 3), ci=120, co=136, pad=1), 1),
    # groups: the next group's channels are not this one's
    (dict(batch=2, field=(12, 12), kernel=(3, 3), ci=80, co=72, groups=2,
          pad=1), 1),
    # channels that are no whole vectors go through the padded copy
    (dict(batch=2, field=(12, 12), kernel=(3, 3), ci=77, co=72, pad=1), 1),
    # parts of K: equal, a shorter last one, a slice each
    (dict(batch=2, field=(14, 14), kernel=(3, 3), ci=256, co=136, pad=1), 2),
    (dict(batch=2, field=(14, 14), kernel=(3, 3), ci=200, co=136, pad=1), 2),
    (dict(batch=2, field=(14, 14), kernel=(2, 3), ci=200, co=132, pad=1), 4),
    (dict(batch=2, field=(14, 14), kernel=(3, 3), ci=77, co=72, pad=1), 2),
    # rings of slices: nine taps, two (a k-step of a wave to a slice), three
    (dict(batch=4, field=(28, 28), kernel=(3, 3), ci=520, co=96, pad=1), 1),
    (dict(batch=2, field=(50, 50), kernel=(2, 1), ci=520, co=72), 1),
    (dict(batch=2, field=(50, 50), kernel=(1, 3), ci=648, co=72), 1),
    (dict(batch=4, field=(28, 28), kernel=(3, 3), ci=776, co=96, pad=1), 2),
]


@pytest.mark.gpu
@pytest.mark.parametrize("kw,parts", CASES)
def test_slices_of_signs_are_exact(oracle, kw, parts):
    from gpu_helpers import quantize, run_conv
    p = make_params(pa.HALF, pa.FLOAT, **kw)
    print("case", kw, parts, flush=True)
    acts, weights, biases = random_data(p, 31, "pm1")
    aq, ad = quantize(acts, p.inputType)
    wq, wd = quantize(weights, p.inputType)
    bq, bd = quantize(biases, p.outputType)
    got, plan = run_conv(p, aq, wq, bq, _options(parts), return_plan=True)
    text = plan.describe()
    assert PATCH in text, text
    assert ("K split into parts         %d " % parts in text) == (parts > 1)
    np.testing.assert_array_equal(got, oracle.convolution(p, ad, wd, bd,
                                                          threads=8))


FP8 = [
    (dict(batch=2, field=(12, 12), kernel=(3, 3), ci=80, co=128, pad=1), 1),
    (dict(batch=2, field=(12, 12), kernel=(3, 3), ci=400, co=96, pad=1), 2),
    # rings: the waves bring the slices themselves
    (dict(batch=2, field=(56, 56), kernel=(3, 3), ci=608, co=96, pad=1), 1),
    (dict(batch=2, field=(60, 60), kernel=(2, 1), ci=512, co=96), 1),
]


@pytest.mark.gpu
@pytest.mark.parametrize("kw,parts", FP8)
def test_slices_fp8(oracle, kw, parts):
    from test_fast_gpu import _fp8_case
    p = make_params(pa.QUARTER, pa.HALF, **kw)
    print("case", kw, parts, flush=True)
    got, want, plan = _fp8_case(oracle, p, 32, 1, 1,
                                options=_options(parts, blockM=112))
    assert PATCH in plan.describe(), plan.describe()
    assert rel_l2(got, want) <= 1e-3


@pytest.mark.gpu
def test_channels_behind_the_last_are_not_multiplied(oracle):
    """What stands behind a pixel's last channel - the next pixel's first - may
    be infinite."""
    from gpu_helpers import quantize, run_conv
    p = make_params(pa.HALF, pa.FLOAT, batch=1, field=(6, 7), kernel=(1, 2),
                    ci=72, co=72)
    acts, weights, _ = random_data(p, 33, "pm1")
    acts[0, 0, 2, 3] = np.inf
    aq, _ = quantize(acts, p.inputType)
    wq, wd = quantize(weights, p.inputType)
    got, plan = run_conv(p, aq, wq, None, _options(), return_plan=True)
    assert PATCH in plan.describe()
    bad = np.zeros((6, 6), bool)
    bad[2, 2] = bad[2, 3] = True
    assert np.isfinite(got[0][:, ~bad]).all()
    assert np.isinf(got[0][:, bad]).all()


def test_slice_plans_come_back_from_their_constraints():
    for kw, parts in ((CASES[1][0], 1), (CASES[6][0], 2), (CASES[9][0], 1)):
        p = make_params(pa.HALF, pa.HALF, **kw)
        plan = pa.Plan(p, _options(parts))
        again = pa.Plan(p, {"planConstraints": plan.constraints()})
        assert again.constraints() == plan.constraints()
        assert again.buffer_bytes(4) == plan.buffer_bytes(4)
