"""wuTapKernel's table of pixels at its edges: chunks that end inside a group of
512 pixels, at one, and beyond what the table holds at a time (2048), against
the oracle."""
import re

import numpy as np
import pytest

import poplibs_amd as pa
from test_weight_update import (DENSE_WU, FORCE_DENSE_WU, make_params, rel_l2,
                                run_weight_update)

# many tiles of channels, so that there are few chunks
TILES = dict(kernel=(3, 3), ci=16 * 128, co=8)


@pytest.mark.gpu
@pytest.mark.parametrize("kw,chunks,pixels", [
    # 64 (a chunk of 256), 512 and 576 pixels
    (dict(batch=1, field=(8, 8), pad=1, **TILES), 1, 256),
    (dict(batch=2, field=(16, 16), pad=1, **TILES), 1, 512),
    (dict(batch=4, field=(12, 12), pad=1, **TILES), 1, 576),
    # three chunks of 1088 pixels, the last one shorter
    (dict(batch=4, field=(56, 57), pad=1, stride=2, **TILES), 3, 1088),
    # one of 3136
    (dict(batch=1, field=(56, 56), pad=1, kernel=(3, 3), ci=3520, co=8), 1,
     3136),
])
def test_long_chunks(oracle, kw, chunks, pixels):
    from gpu_helpers import quantize
    p = make_params(pa.HALF, pa.FLOAT, **kw)
    print("case", p, flush=True)
    rng = np.random.default_rng(91)
    xq, xd = quantize(rng.standard_normal(
        (p.batchSize, p.getNumInputChans(), *p.inputFieldShape)), pa.HALF)
    dq, dd = quantize(rng.standard_normal(
        (p.batchSize, p.getNumOutputChans(), *p.getOutputFieldShape())) * 0.1,
        pa.HALF)
    got, plan = run_weight_update(p, xq, dq, FORCE_DENSE_WU)
    assert DENSE_WU in plan.describe(), plan.describe()
    assert "%d chunks of %d pixels" % (chunks, pixels) in plan.describe(), \
        plan.describe()
    # (fp32 sums of at most 3136 products)
    assert rel_l2(got, oracle.weight_deltas(p, xd, dd, threads=8)) <= 1e-5


@pytest.mark.gpu
def test_what_a_chunk_does_not_have_meets_no_infinity():
    # chunks of an odd count of steps of 64: the one more that rounds them up is
    # read as zeros on both sides, also where the next chunk's deltas are infinite
    n = 81920
    p = make_params(pa.HALF, pa.FLOAT, batch=1, field=(n,), kernel=(1,), ci=16,
                    co=16)
    x = np.ones((1, 16, n), np.float16)
    dz = np.ones((1, 16, n), np.float16)
    dz[0, 3, n // 2:] = np.inf
    got, plan = run_weight_update(p, x, dz, FORCE_DENSE_WU)
    chunk = re.search(r"(\d+) chunks of (\d+) pixels", plan.describe())
    assert int(chunk[1]) > 1 and int(chunk[2]) % 128 == 64, plan.describe()
    got = got.reshape(16, 16)
    assert np.isposinf(got[3]).all()
    np.testing.assert_array_equal(np.delete(got, 3, 0), float(n))
