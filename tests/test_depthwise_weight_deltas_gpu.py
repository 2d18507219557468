"""Weight deltas of depthwise layers against the CPU oracle: the sums over the
slices of a pass of many outputs (csrc/depthwise_train.hip)."""
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
