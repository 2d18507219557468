"""Depthwise layers over an input dilated by two (the backward pass of a strided
depthwise layer): a thread takes a 2 x 2 block of outputs, or two below each other
(depthwiseDilatedBlockKernel in csrc/depthwise_train.hip), against the CPU
oracle.  +-1 data: sums of at most 25 products and a bias, exact in half."""
import numpy as np
import pytest

import poplibs_amd as pa
from helpers import make_params, random_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [
    # one block to a thread: two input elements, two columns of them,
    # output rows and columns that start or end in the middle of a block
    dict(batch=2, field=(2, 2), kernel=(3, 3), groups=8, pad=2),
    dict(batch=3, field=(9, 2), kernel=(3, 3), groups=24, padLower=(0, 2),
         padUpper=(1, 1)),
    dict(batch=2, field=(7, 8), kernel=(3, 3), groups=16, padLower=(2, 1),
         padUpper=(1, 2)),
    # two: rows of blocks that are no whole pairs
    dict(batch=4, field=(62, 63), kernel=(3, 3), groups=64, pad=1),
    dict(batch=4, field=(63, 62), kernel=(3, 3), groups=64, padLower=(2, 0),
         padUpper=(0, 2)),
    dict(batch=1, field=(2, 2), kernel=(5, 5), groups=8, pad=4),
    dict(batch=3, field=(9, 2), kernel=(5, 5), groups=24, pad=3),
    dict(batch=2, field=(7, 8), kernel=(5, 5), groups=16, padLower=(3, 1),
         padUpper=(1, 4))])
@pytest.mark.parametrize("out_type", [pa.HALF, pa.FLOAT])
@pytest.mark.parametrize("biased", [False, True])
def test_blocks_of_a_dilated_input(oracle, kw, out_type, biased):
    from gpu_helpers import quantize, run_conv
    p = make_params(pa.HALF, out_type, idil=2, **kw)
    print("case", p, flush=True)
    acts, weights, biases = random_data(p, 65, "pm1")
    got, plan = run_conv(p, quantize(acts, pa.HALF)[0],
                         quantize(weights, pa.HALF)[0],
                         quantize(biases, out_type)[0] if biased else None,
                         None, return_plan=True)
    assert "dilated input" in plan.describe(), plan.describe()
    want = oracle.convolution(p, acts, weights, biases if biased else None,
                              threads=8)
    np.testing.assert_array_equal(got, want)
