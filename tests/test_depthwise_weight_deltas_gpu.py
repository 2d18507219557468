"""Weight deltas of depthwise layers against the CPU oracle: the sums over the
slices of a pass of many outputs (csrc/depthwise_train.hip), and the kernel that
walks down strips of columns (csrc/depthwise_columns_deltas.hip)."""
import json

import numpy as np
import pytest

import poplibs_amd as pa
from helpers import make_params
from test_weight_update import run_weight_update


def _signs(oracle, kw, out_type=pa.FLOAT, options=None):
    p = make_params(pa.HALF, out_type, **kw)
    print("case", kw, options, flush=True)
    rng = np.random.default_rng(19)
    C = p.numConvGroups
    x = rng.choice([-1.0, 1.0], (p.batchSize, C, *p.inputFieldShape))
    dz = rng.choice([-1.0, 1.0], (p.batchSize, C, *p.getOutputFieldShape()))
    got, plan = run_weight_update(p, x.astype(np.float16),
                                  dz.astype(np.float16), options)
    np.testing.assert_array_equal(got, oracle.weight_deltas(p, x, dz,
                                                            threads=8))
    return plan


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [
    # one slice, fewer than there are parts, and an output past the last
    # workgroup of 32
    dict(batch=1, field=(3, 3), kernel=(3, 3), groups=488, pad=1),
    dict(batch=4, field=(6, 6), kernel=(3, 3), groups=520, pad=1),
    # more than sixteen to a part
    dict(batch=30, field=(13, 13), kernel=(3, 3), groups=1000, pad=1),
])
@pytest.mark.parametrize("out_type", [pa.HALF, pa.FLOAT])
def test_many_outputs_of_signs_are_exact(oracle, kw, out_type):
    # (sums of at most 2048 signs: exact in halves too)
    kw = dict(kw, batch=min(kw["batch"], 12)) if out_type == pa.HALF else kw
    _signs(oracle, kw, out_type)


COLUMNS = "columns walked down in registers"


def _options(columns):
    return {"planConstraints": json.dumps({"gfx950": {"columns": columns}})}


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [
    # strips: one partial, exact, one column over; a channel pair to each slot
    # of four, and as many as a workgroup has threads for
    dict(batch=2, field=(6, 2), kernel=(3, 3), groups=8, pad=1),
    dict(batch=2, field=(9, 8), kernel=(7, 7), groups=40, pad=3),
    dict(batch=1, field=(33, 17), kernel=(5, 5), groups=72, pad=2),
    dict(batch=3, field=(17, 9), kernel=(7, 7), groups=8, stride=2, pad=3),
    dict(batch=2, field=(31, 34), kernel=(5, 5), groups=136, stride=2, pad=2),
    dict(batch=2, field=(10, 11), kernel=(3, 3), groups=264, stride=2, pad=1),
    # a walk over several strips
    dict(batch=2100, field=(5, 5), kernel=(3, 3), groups=256, pad=1),
    # unpadded, unevenly padded, the input cut off
    dict(batch=2, field=(7, 7), kernel=(7, 7), groups=16),
    dict(batch=2, field=(9, 12), kernel=(7, 7), groups=24, padLower=(5, 0),
         padUpper=(1, 6)),
    dict(batch=2, field=(15, 14), kernel=(5, 5), groups=16, itl=(2, 1),
         itu=(1, 3), pad=2),
])
@pytest.mark.parametrize("columns", [2, 4])
def test_columns_of_signs_are_exact(oracle, kw, columns):
    plan = _signs(oracle, kw, options=_options(columns))
    assert COLUMNS in plan.describe()


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["acts", "deltas", "both"])
@pytest.mark.parametrize("columns", [2, 4])
@pytest.mark.parametrize("k,stride", [(3, 1), (5, 2), (7, 1)])
def test_subnormal_halves_are_exact(oracle, k, stride, columns, which):
    """Multiples of 2^-24 below 2^-14 against signs, and against each other:
    sums of 234 products of at most 2^16 units, which fp32 holds."""
    p = make_params(pa.HALF, pa.FLOAT, batch=2, field=(13, 9), kernel=(k, k),
                    groups=16, stride=stride, pad=k // 2)
    print("case", k, stride, columns, which, flush=True)
    rng = np.random.default_rng(29)

    def data(shape, small):
        signs = rng.choice([-1.0, 1.0], shape)
        return signs * rng.integers(1, 256, shape) * 2.0 ** -24 if small \
            else signs

    x = data((2, 16, 13, 9), which != "deltas")
    dz = data((2, 16, *p.getOutputFieldShape()), which != "acts")
    got, plan = run_weight_update(p, x.astype(np.float16),
                                  dz.astype(np.float16), _options(columns))
    assert COLUMNS in plan.describe()
    np.testing.assert_array_equal(got, oracle.weight_deltas(p, x, dz,
                                                            threads=8))


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["acts", "deltas"])
@pytest.mark.parametrize("columns", [2, 4])
@pytest.mark.parametrize("k,stride", [(3, 1), (5, 2), (7, 1)])
def test_infinities_stay_in_their_products(k, stride, columns, where):
    """An infinity at the field's edge reaches the taps that have a product
    with it and no other (a zero opposite it would make a NaN)."""
    p = make_params(pa.HALF, pa.FLOAT, batch=2, field=(13, 15), kernel=(k, k),
                    groups=16, stride=stride, pad=k // 2)
    rng = np.random.default_rng(3)
    x = rng.choice([-1.0, 1.0], (2, 16, 13, 15))
    dz = rng.choice([-1.0, 1.0], (2, 16, *p.getOutputFieldShape()))
    (x if where == "acts" else dz)[1, 5, 0, -1] = np.inf
    want = np.zeros((16, k, k))
    for kh in range(k):
        for kw in range(k):
            ys = [y for y in range(dz.shape[2])
                  if 0 <= y * stride + kh - k // 2 < 13]
            xs = [c for c in range(dz.shape[3])
                  if 0 <= c * stride + kw - k // 2 < 15]
            a = x[:, :, [y * stride + kh - k // 2 for y in ys]]
            a = a[:, :, :, [c * stride + kw - k // 2 for c in xs]]
            want[:, kh, kw] = (a * dz[:, :, ys][:, :, :, xs]).sum((0, 2, 3))
    assert np.isinf(want).any() and np.isfinite(want[5]).any()
    got, _ = run_weight_update(p, x.astype(np.float16), dz.astype(np.float16),
                               _options(columns))
    np.testing.assert_array_equal(got.reshape(want.shape), want)


def test_columns_plan_choice():
    def plan(options=None, dtype=pa.HALF, **kw):
        return pa.WeightUpdatePlan(make_params(dtype, dtype, **kw), options)
    big = dict(batch=16, field=(40, 40), kernel=(5, 5), groups=96, pad=2)
    chosen = plan(**big)
    assert COLUMNS in chosen.describe()
    doc = chosen.constraints()
    assert json.loads(doc)["gfx950"]["columns"] in (2, 4)
    again = plan({"planConstraints": doc}, **big)
    assert again.constraints() == doc
    assert again.workspace_bytes() == chosen.workspace_bytes()
    off = plan(_options(0), **big)
    assert COLUMNS not in off.describe()
    assert COLUMNS not in plan({"planConstraints": off.constraints()},
                               **big).describe()
    # little work, fp32 tensors, other kernels and strides
    small = dict(batch=2, field=(9, 9), kernel=(5, 5), groups=16, pad=2)
    assert COLUMNS not in plan(**small).describe()
    assert COLUMNS in plan(_options(2), **small).describe()
    for bad in (dict(big, dtype=pa.FLOAT), dict(big, kernel=(5, 3)),
                dict(big, stride=3), dict(big, kdil=2)):
        assert COLUMNS not in plan(**bad).describe()
        with pytest.raises(pa.MxconvError):
            plan(_options(4), **bad)


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [
    # walks of four pixels: one slice, a last slice of one pixel
    dict(batch=1, field=(3, 3), kernel=(3, 3), groups=8, pad=1),
    dict(batch=1, field=(29, 7), kernel=(3, 3), groups=24, pad=1),
    # 256 slices of four pixels, and a pixel more: of eight
    dict(batch=2, field=(32, 32), kernel=(3, 3), groups=104, pad=1),
    dict(batch=1, field=(2049, 1), kernel=(3, 3), groups=104, pad=1),
    # of sixteen (more than 2 MB of sums with eight), stride 2, uneven padding
    dict(batch=11, field=(12, 11), kernel=(5, 5), groups=808, stride=2, pad=2),
    dict(batch=9, field=(11, 12), kernel=(3, 3), groups=48, stride=2,
         padLower=(2, 0), padUpper=(0, 1))])
def test_walks_of_small_layers_are_exact(oracle, kw):
    """A slot's walk over the pixels is as short as the number of slices and the
    size of their sums allow (depthwiseWeightDeltaKernel)."""
    _signs(oracle, kw, options=_options(0))
