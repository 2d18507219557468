"""The 256-pixel tiles (csrc/igemm_wide.hip), both widths, against the oracle at
the edges of tiles, k-steps and blocks of workgroups."""
import pytest

import poplibs_amd as pa
from helpers import make_params, rel_l2

pytestmark = pytest.mark.gpu

CASES = [
    # less than a tile; one k-step, an odd and an even number of them
    dict(field=(5, 7), kernel=(1, 1), ci=64, co=24),
    dict(batch=2, field=(12, 12), kernel=(1, 1), ci=128, co=200),
    dict(batch=2, field=(12, 12), kernel=(3, 3), ci=64, co=40, pad=1),
    # five M tiles (a whole block of four and one more), three N tiles
    dict(batch=5, field=(16, 15), kernel=(2, 2), ci=64, co=520, pad=1),
    # channels that fill no k-step, a stride, a dilated kernel, groups
    dict(batch=2, field=(33, 31), kernel=(3, 3), ci=40, co=56, stride=(2, 1),
         pad=2, kdil=(1, 2)),
    dict(batch=2, field=(17, 16), kernel=(3, 3), ci=24, co=72, groups=3,
         pad=1),
    dict(batch=1, field=(6, 7, 8), kernel=(3, 2, 2), ci=16, co=24, pad=1),
    # padded channels, an output field with zeros around, odd outputs
    dict(batch=3, field=(20, 20), kernel=(3, 3), ci=13, co=33, pad=1),
    dict(batch=2, field=(12, 12), kernel=(3, 3), ci=64, co=24, pad=1,
         opl=(1, 0), opu=(0, 2)),
]


def _options(width):
    return {"planConstraints": '{"gfx950": {"kernel": "igemm", "pointwise": 0,'
                               ' "blockM": 256, "blockN": %d}}' % width}


@pytest.mark.parametrize("width", [192, 256])
@pytest.mark.parametrize("kw", CASES)
@pytest.mark.parametrize("out_type", [pa.FLOAT, pa.HALF])
def test_wide_tiles_half(oracle, kw, width, out_type):
    from test_fast_gpu import _run
    p = make_params(pa.HALF, out_type, **kw)
    assert "256 x %d x 64" % width in pa.Plan(p, _options(width)).describe()
    exact = out_type == pa.FLOAT
    _run(oracle, p, 71, 0 if exact else 1e-3, "implicit GEMM",
         dist="pm1" if exact else "normal", options=_options(width))


@pytest.mark.parametrize("in_format", [0, 1])
@pytest.mark.parametrize("w_format", [0, 1])
@pytest.mark.parametrize("width,ci", [(192, 144), (256, 128), (256, 48)])
def test_wide_tiles_quarter(oracle, width, ci, in_format, w_format):
    from test_fast_gpu import _fp8_case
    p = make_params(pa.QUARTER, pa.HALF, batch=2, field=(14, 13),
                    kernel=(3, 3), ci=ci, co=200, pad=1)
    got, want, plan = _fp8_case(oracle, p, 73, in_format, w_format,
                                options=_options(width))
    assert "256 x %d x 128" % width in plan.describe()
    assert rel_l2(got, want) <= 1e-3


def test_planner_takes_wide_tiles_for_products_that_fill_the_chip():
    plan = pa.MatMulPlan(pa.HALF, pa.HALF, 1, 4096, 4096, 4096)
    assert "block M x N x K            256 x 256 x 64" in plan.describe()
    again = pa.Plan(pa.matMulParams(pa.HALF, pa.HALF, 1, 4096, 4096, 4096),
                    {"planConstraints": plan.constraints()})
    assert again.packs_like(plan)
    small = pa.MatMulPlan(pa.HALF, pa.HALF, 1, 1024, 1024, 1024)
    assert "256 x 256" not in small.describe()


# Rows of outputs that start at any element: whole vectors at every offset and
# the channels behind the last one, in tiles of every width, with groups (whose
# channels start inside a vector) and with input channels that are padded in a
# copy at every offset.
RAGGED = [
    dict(batch=2, field=(11, 12), kernel=(1, 1), ci=64, co=7),
    dict(batch=2, field=(11, 12), kernel=(3, 3), ci=33, co=67, pad=1),
    dict(batch=2, field=(9, 9), kernel=(1, 1), ci=71, co=131),
    dict(batch=1, field=(13, 12), kernel=(1, 1), ci=64, co=301),
    dict(batch=2, field=(8, 9), kernel=(3, 3), ci=19, co=13, groups=3, pad=1),
]


@pytest.mark.parametrize("tile", [(128, 64), (128, 128), (256, 192),
                                  (256, 256)])
@pytest.mark.parametrize("kw", RAGGED)
@pytest.mark.parametrize("out_type", [pa.FLOAT, pa.HALF])
def test_rows_of_no_whole_vectors(oracle, kw, tile, out_type):
    from test_fast_gpu import _run
    p = make_params(pa.HALF, out_type, **kw)
    options = {"planConstraints": '{"gfx950": {"kernel": "igemm", "patch": 0, '
                                  '"pointwise": 0, "blockM": %d, "blockN": '
                                  '%d}}' % tile}
    assert "%d x %d x 64" % tile in pa.Plan(p, options).describe()
    exact = out_type == pa.FLOAT
    _run(oracle, p, 72, 0 if exact else 1e-3, "implicit GEMM",
         dist="pm1" if exact else "normal", options=options)
