"""Channels that are no whole vectors under little work: by a chain of products
per thread where it is short, on the matrix cores behind a padded copy where it
is not, against the CPU oracle on both sides of the line."""
import numpy as np
import pytest

import poplibs_amd as pa
from helpers import make_params, random_data

CASES = [
    (pa.HALF, dict(batch=2, field=(3, 3), kernel=(1, 1), ci=63, co=20), True),
    (pa.HALF, dict(batch=2, field=(3, 3), kernel=(1, 1), ci=65, co=20), False),
    (pa.FLOAT, dict(batch=2, field=(3, 3), kernel=(1, 1), ci=62, co=9), True),
    (pa.FLOAT, dict(batch=2, field=(3, 3), kernel=(1, 1), ci=65, co=9), False),
    (pa.HALF, dict(batch=1, field=(8, 8), kernel=(3, 3), ci=4, co=8), True),
    (pa.HALF, dict(batch=1, field=(8, 8), kernel=(3, 3), ci=5, co=8), False),
    (pa.FLOAT, dict(batch=1, field=(5, 5), kernel=(3, 3), ci=5, co=3), False),
    (pa.QUARTER, dict(batch=2, field=(3, 3), kernel=(1, 1), ci=8, co=16),
     True),
    (pa.QUARTER, dict(batch=2, field=(3, 3), kernel=(1, 1), ci=9, co=16),
     False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,kw,generic", CASES)
def test_signs_are_exact(oracle, dtype, kw, generic):
    from gpu_helpers import quantize, run_conv
    out = pa.FLOAT if dtype == pa.FLOAT else pa.HALF
    p = make_params(dtype, out, **kw)
    print("case", dtype, kw, flush=True)
    acts, weights, biases = random_data(p, 7, "pm1")
    aq, ad = quantize(acts, dtype, oracle)
    wq, wd = quantize(weights, dtype, oracle)
    bq, bd = quantize(biases, out)
    got, plan = run_conv(p, aq, wq, bq, return_plan=True)
    assert ("generic direct" in plan.describe()) == generic
    np.testing.assert_array_equal(got, oracle.convolution(p, ad, wd, bd,
                                                          threads=8))
