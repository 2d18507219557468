"""Weight deltas by the kernel that gathers pixels in registers
(csrc/wu_window.hip) at the edges of its units of eight columns, its tiles of
channels and groups, and its chunks, against the CPU oracle."""
import json

import numpy as np
import pytest

import poplibs_amd as pa
from helpers import make_params, rel_l2

WINDOW = "pixels gathered in registers"
BY_NAME = {"planConstraints": '{"gfx950": {"deltaWindow": 1}}'}

# rows of two columns, of a unit less one, a unit, one more; two units and one
CASES = [dict(batch=3, field=(5, w), kernel=(3, 3), ci=16, co=24, pad=1)
         for w in (2, 7, 8, 9, 17)]
CASES += [
    # stride 2: seventeen columns for eight outputs; rows that end early
    dict(batch=2, field=(9, 33), kernel=(3, 3), ci=32, co=40, pad=1, stride=2),
    dict(batch=2, field=(8, 16), kernel=(1, 1), ci=48, co=16, stride=2),
    dict(batch=3, field=(7, 15), kernel=(2, 3), ci=24, co=32, stride=(3, 1)),
    # 1 x 1, the field as one row: less than a unit, and no whole unit
    dict(batch=1, field=(1, 5), kernel=(1, 1), ci=24, co=16),
    dict(batch=3, field=(7, 7), kernel=(1, 1), ci=72, co=72),
    # tiles: one channel more than 32 and 64, whole ones, odd counts
    dict(batch=2, field=(9, 10), kernel=(3, 3), ci=66, co=34, pad=1),
    dict(batch=2, field=(9, 10), kernel=(3, 3), ci=64, co=128, pad=1),
    dict(batch=2, field=(9, 10), kernel=(3, 3), ci=17, co=19, pad=1),
    # input truncation, padding on one side, all a kernel can meet
    dict(batch=2, field=(12, 14), kernel=(3, 3), ci=16, co=16, itl=(1, 0),
         itu=(0, 2), pad=1),
    dict(batch=2, field=(9, 11), kernel=(3, 3), ci=16, co=16, padLower=(0, 2),
         padUpper=(1, 0)),
    dict(batch=2, field=(6, 6), kernel=(3, 3), ci=16, co=16, pad=2),
    # groups: several to a tile, the last tile with fewer, unlike channels
    dict(batch=3, field=(10, 9), kernel=(3, 3), ci=4, co=4, groups=32, pad=1),
    dict(batch=3, field=(10, 9), kernel=(3, 3), ci=8, co=8, groups=5, pad=1),
    dict(batch=3, field=(10, 9), kernel=(1, 1), ci=16, co=16, groups=32,
         stride=2),
    dict(batch=3, field=(10, 9), kernel=(3, 3), ci=6, co=10, groups=4, pad=1),
    dict(batch=3, field=(10, 9), kernel=(3, 3), ci=40, co=24, groups=3, pad=1),
    # many chunks, summed by the second kernel
    dict(batch=16, field=(28, 28), kernel=(3, 3), ci=24, co=40, pad=1),
    dict(batch=16, field=(28, 28), kernel=(3, 3), ci=8, co=8, groups=16,
         pad=1, stride=2),
    # ... sums of a tap that are no whole vectors
    dict(batch=24, field=(26, 27), kernel=(3, 3), ci=38, co=7, pad=1),
    dict(batch=30, field=(31, 29), kernel=(1, 1), ci=40, co=64),
]


def _signs(p, seed):
    rng = np.random.default_rng(seed)
    x = rng.choice([-1.0, 1.0],
                   (p.batchSize, p.getNumInputChans(), *p.inputFieldShape))
    dz = rng.choice([-1.0, 1.0], (p.batchSize, p.getNumOutputChans(),
                                  *p.getOutputFieldShape()))
    return x, dz


@pytest.mark.gpu
@pytest.mark.parametrize("kw", CASES)
def test_window_weight_deltas_of_signs_are_exact(oracle, kw):
    # +-1 tensors: every product and every partial sum is a small integer
    from test_weight_update import run_weight_update
    p = make_params(pa.HALF, pa.FLOAT, **kw)
    print("case", p, flush=True)
    x, dz = _signs(p, 71)
    got, plan = run_weight_update(p, x.astype(np.float16),
                                  dz.astype(np.float16), BY_NAME)
    assert WINDOW in plan.describe(), plan.describe()
    np.testing.assert_array_equal(
        got, oracle.weight_deltas(p, x, dz, threads=8))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [pa.HALF, pa.FLOAT])
@pytest.mark.parametrize("steps", [7, 8, 9, 16, 17, 25])
def test_waves_with_odd_and_even_counts_of_steps(oracle, dtype, steps):
    """A workgroup's waves (eight, or sixteen or four with fp32 tensors) take a
    chunk's k-steps in turn, two to a round of their loop: none, an even number,
    an odd one, and both in one workgroup."""
    from test_weight_update import run_weight_update
    p = make_params(dtype, pa.FLOAT, batch=1, field=(4 * steps - 1, 8),
                    kernel=(3, 3), ci=256, co=512, pad=1)
    print("case", dtype, steps, flush=True)
    x, dz = _signs(p, 76)
    np_type = np.float16 if dtype == pa.HALF else np.float32
    got, plan = run_weight_update(p, x.astype(np_type), dz.astype(np_type),
                                  BY_NAME if dtype == pa.HALF else {})
    assert WINDOW in plan.describe(), plan.describe()
    assert "chunks of %d k-steps" % steps in plan.describe(), plan.describe()
    np.testing.assert_array_equal(
        got, oracle.weight_deltas(p, x, dz, threads=8))


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [
    # odd channels in groups: copies filled up to whole vectors, of both
    # tensors or of one; groups that stay by themselves, that run as one, a
    # last tile with fewer; one chunk and many
    dict(batch=3, field=(10, 9), kernel=(3, 3), ci=5, co=7, groups=4, pad=1),
    dict(batch=3, field=(10, 9), kernel=(3, 3), ci=5, co=7, groups=8, pad=1),
    dict(batch=3, field=(10, 9), kernel=(3, 3), ci=9, co=16, groups=3, pad=1),
    dict(batch=3, field=(10, 9), kernel=(1, 1), ci=8, co=3, groups=16,
         stride=2),
    dict(batch=2, field=(9, 11), kernel=(3, 3), ci=33, co=17, groups=2, pad=1),
    dict(batch=20, field=(23, 25), kernel=(3, 3), ci=3, co=3, groups=16,
         pad=1),
])
@pytest.mark.parametrize("out_type", [pa.HALF, pa.FLOAT])
def test_odd_channels_in_groups_are_exact(oracle, kw, out_type):
    from test_weight_update import run_weight_update
    p = make_params(pa.HALF, out_type, **kw)
    print("case", p, flush=True)
    x, dz = _signs(p, 74)
    got, plan = run_weight_update(p, x.astype(np.float16),
                                  dz.astype(np.float16), BY_NAME)
    assert WINDOW in plan.describe(), plan.describe()
    want = oracle.weight_deltas(p, x, dz, threads=8)
    np.testing.assert_array_equal(
        got, want if out_type == pa.FLOAT else
        want.astype(np.float16).astype(np.float64))


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [CASES[3], CASES[5], CASES[9], CASES[16],
                                CASES[-4], CASES[-1]])
def test_window_weight_deltas_to_half(oracle, kw):
    from gpu_helpers import quantize
    from test_weight_update import run_weight_update
    p = make_params(pa.HALF, pa.HALF, **kw)
    print("case", p, flush=True)
    rng = np.random.default_rng(72)
    xq, xd = quantize(rng.standard_normal(
        (p.batchSize, p.getNumInputChans(), *p.inputFieldShape)), pa.HALF)
    dq, dd = quantize(rng.standard_normal(
        (p.batchSize, p.getNumOutputChans(), *p.getOutputFieldShape())) * 0.1,
        pa.HALF)
    got, plan = run_weight_update(p, xq, dq, BY_NAME)
    assert WINDOW in plan.describe(), plan.describe()
    # (fp32 sums, rounded once)
    assert rel_l2(got, oracle.weight_deltas(p, xd, dd, threads=8)) <= 5e-4


@pytest.mark.gpu
def test_infinities_stay_with_the_taps_that_read_them(oracle):
    """A unit's columns behind the row's end belong to the next row: an
    infinity there is no part of this row's sums."""
    from test_weight_update import run_weight_update
    p = make_params(pa.HALF, pa.FLOAT, batch=2, field=(6, 11), kernel=(3, 3),
                    ci=16, co=16)
    x, dz = _signs(p, 73)
    dz = np.abs(dz)
    x[0, 3, 0, 0] = np.inf  # read by tap (0, 0) alone
    got, plan = run_weight_update(p, x.astype(np.float16),
                                  dz.astype(np.float16), BY_NAME)
    assert WINDOW in plan.describe(), plan.describe()
    x[0, 3, 0, 0] = 0.0
    want = oracle.weight_deltas(p, x, dz, threads=8)
    want[..., 3, 0, 0] = np.inf
    np.testing.assert_array_equal(got, want)


def test_what_the_window_kernel_does_not_take_is_refused_by_name():
    for kw in (dict(kernel=(5, 5), pad=2), dict(kernel=(3, 3), stride=(1, 3)),
               dict(kernel=(3, 2))):
        p = make_params(pa.HALF, pa.HALF, batch=2, field=(12, 12), ci=16,
                        co=16, **kw)
        assert WINDOW not in pa.WeightUpdatePlan(p).describe()
        with pytest.raises(pa.MxconvError, match="weightDeltas"):
            pa.WeightUpdatePlan(p, BY_NAME)


def test_window_plans_come_back_from_their_constraints():
    for kw in (CASES[9], CASES[16], CASES[-1]):
        p = make_params(pa.HALF, pa.HALF, **kw)
        plan = pa.WeightUpdatePlan(p)
        assert WINDOW in plan.describe(), plan.describe()
        text = plan.constraints()
        assert json.loads(text)["gfx950"]["deltaWindow"] == 1
        again = pa.WeightUpdatePlan(p, {"planConstraints": text})
        assert again.constraints() == text
        assert again.workspace_bytes() == plan.workspace_bytes()
