"""Weight deltas of fp32 layers by the kernel that gathers pixels in registers
(wuWindowFloatKernel in csrc/wu_window.hip), against the CPU oracle."""
import json

import numpy as np
import pytest

import poplibs_amd as pa
from helpers import make_params, rel_l2
from test_weight_window_gpu import CASES, WINDOW, _signs

# the half kernel's edges, and: channels by one around the tiles of 16, 32 and
# 48, groups of odd widths, a layer of one pixel
FLOAT_CASES = CASES + [
    dict(batch=2, field=(6, 9), kernel=(3, 3), ci=15, co=17, pad=1),
    dict(batch=2, field=(6, 9), kernel=(1, 1), ci=31, co=33),
    dict(batch=2, field=(6, 9), kernel=(3, 3), ci=47, co=49, pad=1, stride=2),
    dict(batch=2, field=(6, 9), kernel=(3, 3), ci=3, co=5, groups=7, pad=1),
    dict(batch=1, field=(1, 1), kernel=(1, 1), ci=3, co=3, groups=2),
]


@pytest.mark.gpu
@pytest.mark.parametrize("kw", FLOAT_CASES)
def test_float_window_of_signs_is_exact(oracle, kw):
    from test_weight_update import run_weight_update
    for out_type in (pa.FLOAT, pa.HALF):
        p = make_params(pa.FLOAT, out_type, **kw)
        print("case", kw, out_type, flush=True)
        x, dz = _signs(p, 41)
        want = oracle.weight_deltas(p, x, dz, threads=8)
        got, plan = run_weight_update(p, x.astype(np.float32),
                                      dz.astype(np.float32))
        assert WINDOW in plan.describe(), plan.describe()
        np.testing.assert_array_equal(
            got, want if out_type == pa.FLOAT else
            want.astype(np.float16).astype(np.float64))


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [CASES[4], CASES[5], CASES[16], CASES[21],
                                CASES[24]])
def test_float_window_is_as_close_as_the_convolution(oracle, kw):
    """fp32 sums of N products: no further from the exact ones than a chain of
    N roundings, and not further than the pass's own convolution by more than
    the two differ in the order of their additions."""
    from test_weight_update import run_weight_update
    p = make_params(pa.FLOAT, pa.FLOAT, **kw)
    rng = np.random.default_rng(43)
    x = rng.standard_normal((p.batchSize, p.getNumInputChans(),
                             *p.inputFieldShape)).astype(np.float32)
    dz = rng.standard_normal((p.batchSize, p.getNumOutputChans(),
                              *p.getOutputFieldShape())).astype(np.float32)
    want = oracle.weight_deltas(p, x.astype(np.float64),
                                dz.astype(np.float64), threads=8)
    got, _ = run_weight_update(p, x, dz)
    own, plan = run_weight_update(
        p, x, dz, {"planConstraints": '{"gfx950": {"weightDeltas": 0}}'})
    assert WINDOW not in plan.describe()
    pixels = p.batchSize * np.prod(p.getOutputFieldShape())
    assert rel_l2(got, want) <= 2.0 ** -24 * np.sqrt(pixels)
    assert rel_l2(got, want) <= 1.25 * rel_l2(own, want)


@pytest.mark.gpu
def test_infinities_stay_with_the_taps_that_read_them(oracle):
    from test_weight_update import run_weight_update
    p = make_params(pa.FLOAT, pa.FLOAT, batch=2, field=(6, 11), kernel=(3, 3),
                    ci=16, co=16)
    x, dz = _signs(p, 73)
    dz = np.abs(dz)
    for at, taps in (((0, 3, 0, 0), [(0, 0)]),
                     ((0, 3, 2, 10), [(0, 2), (1, 2), (2, 2)])):
        x[at] = np.inf
        got, plan = run_weight_update(p, x.astype(np.float32),
                                      dz.astype(np.float32))
        assert WINDOW in plan.describe(), plan.describe()
        x[at] = 0.0
        want = oracle.weight_deltas(p, x, dz, threads=8)
        for kh, kw in taps:
            want[..., 3, kh, kw] = np.inf
        np.testing.assert_array_equal(got, want)


def test_float_window_plan_choice():
    kw = dict(batch=4, field=(12, 12), kernel=(3, 3), ci=24, co=40, pad=1)
    p = make_params(pa.FLOAT, pa.FLOAT, **kw)
    plan = pa.WeightUpdatePlan(p)
    assert WINDOW in plan.describe()
    text = plan.constraints()
    assert json.loads(text)["gfx950"]["deltaWindow"] == 1
    again = pa.WeightUpdatePlan(p, {"planConstraints": text})
    assert again.constraints() == text
    assert again.workspace_bytes() == plan.workspace_bytes()
    # what names the pass's own convolution, or a tile of it, keeps it
    for other in ({"deltaWindow": 0}, {"weightDeltas": 0}, {"splitK": 2},
                  {"kernel": "igemm"}, {"smallTile": 0}):
        assert WINDOW not in pa.WeightUpdatePlan(
            p, {"planConstraints": json.dumps({"gfx950": other})}).describe()
    # ... and what the kernel does not take
    for bad in (dict(kw, kernel=(5, 5), pad=2), dict(kw, stride=3),
                dict(kw, kdil=2)):
        assert WINDOW not in pa.WeightUpdatePlan(
            make_params(pa.FLOAT, pa.FLOAT, **bad)).describe()
