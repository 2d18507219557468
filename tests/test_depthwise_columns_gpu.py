"""Depthwise layers of 5 x 5 and 7 x 7 taps by lanes that walk down strips of
output columns (csrc/depthwise_columns.hip), against the CPU oracle; and the
kernels that they took the place of, which a plan can still name."""
import json

import numpy as np
import pytest

import poplibs_amd as pa
from helpers import make_params, random_data, rel_l2

COLUMNS = "strips of columns in registers"


def _options(columns):
    return {"planConstraints": json.dumps({"gfx950": {"columns": columns}})}


CASES = [
    # strips: one partial, exact, one column over; bands of one row and more
    dict(batch=2, field=(6, 3), kernel=(5, 5), groups=8, pad=2),
    dict(batch=2, field=(9, 8), kernel=(7, 7), groups=40, pad=3),
    dict(batch=1, field=(33, 17), kernel=(5, 5), groups=72, pad=2),
    dict(batch=3, field=(17, 9), kernel=(7, 7), groups=8, stride=2, pad=3),
    dict(batch=2, field=(31, 34), kernel=(5, 5), groups=24, stride=2, pad=2),
    # several rounds of waves: bands of many rows
    dict(batch=24, field=(30, 30), kernel=(7, 7), groups=96, pad=3),
    dict(batch=24, field=(45, 45), kernel=(5, 5), groups=88, stride=2, pad=2),
    # unpadded, unevenly padded, padded beyond the kernel's half
    dict(batch=2, field=(7, 7), kernel=(7, 7), groups=16),
    dict(batch=2, field=(20, 17), kernel=(5, 5), groups=16, stride=2),
    dict(batch=2, field=(9, 12), kernel=(7, 7), groups=24, padLower=(5, 0),
         padUpper=(1, 6)),
    # rows and columns of the input cut off
    dict(batch=2, field=(15, 14), kernel=(5, 5), groups=16, itl=(2, 1),
         itu=(1, 3), pad=2),
]


def _run(oracle, kw, out_type, columns, dist):
    from gpu_helpers import quantize, run_conv
    p = make_params(pa.HALF, out_type, **kw)
    print("case", kw, out_type, columns, flush=True)
    acts, weights, biases = random_data(p, 17, dist)
    if dist != "pm1":
        weights = weights * 0.1
    aq, ad = quantize(acts, p.inputType)
    wq, wd = quantize(weights, p.inputType)
    bq, bd = quantize(biases, p.outputType)
    got, plan = run_conv(p, aq, wq, bq, _options(columns), return_plan=True)
    assert (COLUMNS in plan.describe()) == (columns != 0)
    return got, oracle.convolution(p, ad, wd, bd, threads=8)


@pytest.mark.gpu
@pytest.mark.parametrize("kw", CASES)
@pytest.mark.parametrize("columns", [2, 4])
def test_columns_of_signs_are_exact(oracle, kw, columns):
    np.testing.assert_array_equal(
        *_run(oracle, kw, pa.FLOAT, columns, "pm1"))


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [CASES[2], CASES[4], CASES[9]])
@pytest.mark.parametrize("columns", [0, 2, 4])
def test_columns_of_halves(oracle, kw, columns):
    # a half's rounding, 2^-11, and fp32 sums of 49 products
    got, want = _run(oracle, kw, pa.HALF, columns, "normal")
    assert rel_l2(got, want) <= 2.0 ** -11


@pytest.mark.gpu
@pytest.mark.parametrize("columns", [2, 4])
@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("k", [5, 7])
def test_infinities_stay_in_their_windows(oracle, k, stride, columns):
    """An infinity reaches the outputs whose windows hold it and no other (a
    zero tap or column beside a window would make it a NaN there)."""
    from gpu_helpers import run_conv
    p = make_params(pa.HALF, pa.FLOAT, batch=1, field=(19, 23), kernel=(k, k),
                    groups=16, stride=stride, pad=k // 2)
    acts, weights, _ = random_data(p, 5, "pm1")
    acts, weights = acts.astype(np.float16), weights.astype(np.float16)
    finite = run_conv(p, acts, weights, None, _options(columns))
    at = (0, 16 // 2, 9, 11)  # (batch, channel, row, column)
    acts[at] = np.inf
    got = run_conv(p, acts, weights, None, _options(columns))
    rows = [y for y in range(finite.shape[2])
            if 0 <= at[2] + k // 2 - y * stride < k]
    cols = [x for x in range(finite.shape[3])
            if 0 <= at[3] + k // 2 - x * stride < k]
    inside = np.zeros(finite.shape, bool)
    inside[np.ix_([0], [at[1]], rows, cols)] = True
    assert np.isinf(got[inside]).all()
    np.testing.assert_array_equal(got[~inside], finite[~inside])


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["acts", "weights", "both"])
@pytest.mark.parametrize("columns", [2, 4])
@pytest.mark.parametrize("k,stride", [(5, 2), (7, 1)])
def test_subnormal_halves_are_exact(oracle, k, stride, columns, which):
    """Subnormals (multiples of 2^-24 below 2^-14) against signs, and against
    each other: the sums are below 2^24 of their unit, which fp32 holds."""
    from gpu_helpers import run_conv
    p = make_params(pa.HALF, pa.FLOAT, batch=2, field=(17, 13), kernel=(k, k),
                    groups=24, stride=stride, pad=k // 2)
    print("case", k, stride, columns, which, flush=True)
    acts, weights, _ = random_data(p, 23, "pm1")
    rng = np.random.default_rng(23)

    def small(like):
        return like * rng.integers(1, 256, like.shape) * 2.0 ** -24

    if which != "weights":
        acts = small(acts)
    if which != "acts":
        weights = small(weights)
    got = run_conv(p, acts.astype(np.float16), weights.astype(np.float16),
                   None, _options(columns))
    want = oracle.convolution(p, acts, weights, threads=8)
    np.testing.assert_array_equal(got, want)


def test_columns_plan_choice():
    kw = dict(batch=4, field=(30, 30), kernel=(7, 7), groups=48, pad=3)
    plan = pa.Plan(make_params(pa.HALF, **kw))
    assert COLUMNS in plan.describe()
    # a dump names the strip and makes the same plan
    doc = plan.constraints()
    assert json.loads(doc)["gfx950"]["columns"] in (2, 4)
    again = pa.Plan(make_params(pa.HALF, **kw), {"planConstraints": doc})
    assert again.constraints() == doc
    # a tile, the row ring or 0 name other kernels
    for other in ({"tileH": 4, "tileW": 4}, {"columns": 0}):
        text = pa.Plan(make_params(pa.HALF, **kw), {
            "planConstraints": json.dumps({"gfx950": other})}).describe()
        assert COLUMNS not in text
    five = dict(kw, kernel=(5, 5), pad=2)
    assert COLUMNS not in pa.Plan(make_params(pa.HALF, **five), {
        "planConstraints": '{"gfx950": {"rowRing": 1}}'}).describe()
    # what the kernel does not take
    for bad in (dict(kw, kernel=(3, 3), pad=1), dict(kw, kernel=(7, 5)),
                dict(kw, kdil=2), dict(kw, stride=3)):
        assert COLUMNS not in pa.Plan(make_params(pa.HALF, **bad)).describe()
        with pytest.raises(pa.MxconvError):
            pa.Plan(make_params(pa.HALF, **bad), _options(4))
    with pytest.raises(pa.MxconvError):
        pa.Plan(make_params(pa.FLOAT, **kw), _options(2))
    with pytest.raises(pa.MxconvError):
        pa.Plan(make_params(pa.HALF, **kw), _options(5))
