"""Depthwise layers with 3 x 3 taps by lanes that walk down strips of output
columns (csrc/depthwise_columns.hip), against the CPU oracle; and the planner's
choice of them."""
import json

import numpy as np
import pytest

import poplibs_amd as pa
from helpers import make_params, random_data, rel_l2

STRIPS = "strips of columns in registers"


def _options(strips):
    return {"planConstraints": json.dumps({"gfx950": {"strips": strips}})}


CASES = [
    # strips: one partial, exact, one column over; bands of one row and more
    dict(batch=2, field=(6, 3), groups=8, pad=1),
    dict(batch=2, field=(9, 8), groups=40, pad=1),
    dict(batch=1, field=(33, 17), groups=72, pad=1),
    dict(batch=3, field=(17, 9), groups=8, stride=2, pad=1),
    dict(batch=2, field=(31, 34), groups=24, stride=2, pad=1),
    # several rounds of waves
    dict(batch=40, field=(30, 30), groups=232, pad=1),
    # unpadded, unevenly padded, rows and columns of the input cut off
    dict(batch=2, field=(3, 3), groups=16),
    dict(batch=2, field=(20, 17), groups=16, stride=2),
    dict(batch=2, field=(9, 12), groups=24, padLower=(2, 0), padUpper=(1, 2)),
    dict(batch=2, field=(15, 14), groups=16, itl=(2, 1), itu=(1, 3), pad=1),
]


@pytest.mark.gpu
@pytest.mark.parametrize("kw", CASES)
@pytest.mark.parametrize("strips", [2, 4])
@pytest.mark.parametrize("out_type", [pa.HALF, pa.FLOAT])
def test_strips_of_signs_are_exact(oracle, kw, strips, out_type):
    from gpu_helpers import quantize, run_conv
    p = make_params(pa.HALF, out_type, kernel=(3, 3), **kw)
    print("case", kw, strips, out_type, flush=True)
    acts, weights, biases = random_data(p, 71, "pm1")
    got, plan = run_conv(p, quantize(acts, pa.HALF)[0],
                         quantize(weights, pa.HALF)[0],
                         quantize(biases, out_type)[0], _options(strips),
                         return_plan=True)
    assert STRIPS in plan.describe()
    np.testing.assert_array_equal(
        got, oracle.convolution(p, acts, weights, biases, threads=8))


@pytest.mark.gpu
@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("strips", [2, 4])
def test_infinities_stay_in_their_windows(oracle, stride, strips):
    from gpu_helpers import run_conv
    p = make_params(pa.HALF, pa.HALF, batch=1, field=(11, 13), kernel=(3, 3),
                    groups=8, pad=1, stride=stride)
    rng = np.random.default_rng(5)
    acts = rng.choice([-1.0, 1.0], (1, 8, 11, 13)).astype(np.float16)
    weights = rng.choice([-1.0, 1.0], (8, 1, 1, 3, 3)).astype(np.float16)
    finite = np.asarray(run_conv(p, acts, weights, None, _options(strips)))
    acts[0, 3, 4, 6] = np.inf
    got = np.asarray(run_conv(p, acts, weights, None, _options(strips)))
    other = np.isfinite(got)
    rows = [y for y in range(got.shape[2]) if abs(y * stride - 4) <= 1]
    cols = [x for x in range(got.shape[3]) if abs(x * stride - 6) <= 1]
    inside = np.zeros_like(other)
    inside[0, 3][np.ix_(rows, cols)] = True
    np.testing.assert_array_equal(~other, inside)
    np.testing.assert_array_equal(got[other], finite[other])


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["acts", "weights", "both"])
@pytest.mark.parametrize("strips", [2, 4])
@pytest.mark.parametrize("stride", [1, 2])
def test_subnormal_halves_are_exact(oracle, stride, strips, which):
    """Subnormals (multiples of 2^-24 below 2^-14) against signs, and against
    each other: the sums are below 2^24 of their unit, which fp32 holds."""
    from gpu_helpers import run_conv
    p = make_params(pa.HALF, pa.FLOAT, batch=2, field=(17, 13), kernel=(3, 3),
                    groups=24, stride=stride, pad=1)
    print("case", stride, strips, which, flush=True)
    acts, weights, _ = random_data(p, 73, "pm1")
    rng = np.random.default_rng(73)

    def small(like):
        return like * rng.integers(1, 256, like.shape) * 2.0 ** -24

    if which != "weights":
        acts = small(acts)
    if which != "acts":
        weights = small(weights)
    got = run_conv(p, acts.astype(np.float16), weights.astype(np.float16),
                   None, _options(strips))
    np.testing.assert_array_equal(
        got, oracle.convolution(p, acts, weights, threads=8))


@pytest.mark.gpu
def test_the_planner_s_own_strips(oracle):
    from gpu_helpers import quantize, run_conv
    p = make_params(pa.HALF, pa.HALF, batch=12, field=(13, 13), kernel=(3, 3),
                    groups=328, pad=1)
    acts, weights, biases = random_data(p, 72, "normal")
    aq, ad = quantize(acts, pa.HALF)
    wq, wd = quantize(weights, pa.HALF)
    bq, bd = quantize(biases, pa.HALF)
    got, plan = run_conv(p, aq, wq, bq, None, return_plan=True)
    assert STRIPS in plan.describe()
    # sums of nine products and a bias, rounded once to half
    assert rel_l2(got, oracle.convolution(p, ad, wd, bd, threads=8)) <= 1e-3


def test_strips_plan_choice():
    kw = dict(batch=12, field=(13, 13), kernel=(3, 3), groups=328, pad=1)
    p = make_params(pa.HALF, **kw)
    plan = pa.Plan(p)
    doc = plan.constraints()
    assert json.loads(doc)["gfx950"]["strips"] in (2, 4)
    assert pa.Plan(p, {"planConstraints": doc}).constraints() == doc
    # named kernels stay: the ring, no strips; a plan saved without the key
    for other in ({"rowRing": 1}, {"rowRing": 0}, {"columns": 0},
                  {"tileH": 4, "tileW": 4}):
        assert STRIPS not in pa.Plan(p, {"planConstraints": json.dumps(
            {"gfx950": other})}).describe().split("Left aside")[0]
    for bad, options in ((dict(kw, kernel=(5, 5), pad=2), _options(2)),
                         (dict(kw, kdil=2), _options(2)),
                         (dict(kw, stride=3), _options(4)),
                         (kw, _options(3)),
                         (kw, {"planConstraints": json.dumps({"gfx950": {
                             "strips": 2, "rowRing": 1}})})):
        with pytest.raises(pa.MxconvError):
            pa.Plan(make_params(pa.HALF, **bad), options)
    with pytest.raises(pa.MxconvError):
        pa.Plan(make_params(pa.FLOAT, **kw), _options(2))


@pytest.mark.parametrize("batch,field,groups,strips", [
    # up to 24 MB of tensors, to 96 MB and beyond; rings that are near or ahead
    (47, 19, 488, True), (13, 19, 912, False), (12, 43, 144, False),
    (43, 26, 336, True), (17, 39, 792, True), (28, 46, 424, False),
    (8, 98, 800, False)])
def test_layers_that_rings_are_faster_for_stay(batch, field, groups, strips):
    plan = pa.Plan(make_params(pa.HALF, batch=batch, field=(field, field),
                               kernel=(3, 3), groups=groups, pad=1))
    named = json.loads(plan.constraints())["gfx950"]
    assert ("strips" in named) == strips, named
    assert named["rowRing"] == (0 if strips else 1)
