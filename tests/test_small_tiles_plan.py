"""When the planner takes the small tiles (csrc/igemm_small.hip): by estimates
for few tiles to a CU and for many.  Planning only; no GPU needed."""
import json

import pytest

import poplibs_amd as pa
from helpers import make_params


def _small_tile(p):
    return json.loads(pa.Plan(p).constraints())["gfx950"].get("smallTile", 0)


@pytest.mark.parametrize("dtype,kw", [
    # a tile or less per CU, a deep layer, a product's few rows
    (pa.FLOAT, dict(batch=1, field=(32, 32), kernel=(3, 3), ci=16, co=16,
                    pad=1)),
    (pa.HALF, dict(batch=1, field=(14, 14), kernel=(3, 3), ci=256, co=256,
                   pad=1)),
    (pa.HALF, dict(batch=16, field=(1, 1), kernel=(1, 1), ci=4096, co=4096)),
    # thousands of them: 8 or 32 channels out, 43.2 us for 58, 10 for 12
    (pa.HALF, dict(batch=7, field=(172, 172), kernel=(3, 3), ci=8, co=8,
                   pad=1)),
    (pa.HALF, dict(batch=10, field=(126, 126), kernel=(3, 3), ci=8, co=32,
                   pad=1)),
    (pa.FLOAT, dict(batch=13, field=(118, 118), kernel=(1, 1), ci=16, co=8,
                    groups=16)),
])
def test_small_tiles_are_taken(dtype, kw):
    assert _small_tile(make_params(dtype, **kw)) != 0


@pytest.mark.parametrize("dtype,kw", [
    # thousands of tiles where 128-pixel ones are faster, us with and without:
    # 50.5 / 19.1, 13.0 / 7.2, 49.9 / 36.9
    (pa.HALF, dict(batch=31, field=(87, 87), kernel=(3, 3), ci=4, co=14,
                   groups=4, pad=1)),
    (pa.HALF, dict(batch=5, field=(41, 41), kernel=(3, 3), ci=16, co=80,
                   groups=4, pad=1)),
    (pa.HALF, dict(batch=34, field=(46, 46), kernel=(5, 5), ci=4, co=44,
                   groups=8, stride=2, pad=2)),
    # fp8: 156 / 94, 25.3 / 14.4, 44.7 / 30.5
    (pa.QUARTER, dict(batch=58, field=(125, 125), kernel=(1, 1), ci=16, co=40,
                      groups=8, stride=2)),
    (pa.QUARTER, dict(batch=36, field=(15, 15), kernel=(3, 3), ci=80, co=16,
                      groups=16, pad=1)),
    (pa.QUARTER, dict(batch=4, field=(241, 241), kernel=(1, 1), ci=16, co=64,
                      groups=8, stride=2)),
])
def test_small_tiles_are_left(dtype, kw):
    out = pa.HALF if dtype == pa.QUARTER else dtype
    assert _small_tile(make_params(dtype, out, **kw)) == 0


@pytest.mark.parametrize("batch", [1, 4, 16, 64])
@pytest.mark.parametrize("dtype", [pa.HALF, pa.FLOAT])
def test_the_constraints_name_the_tile(dtype, batch):
    # (whichever estimates picked it)
    p = make_params(dtype, batch=batch, field=(40, 40), kernel=(3, 3), ci=16,
                    co=24, pad=1)
    plan = pa.Plan(p)
    again = pa.Plan(p, {"planConstraints": plan.constraints()})
    assert again.constraints() == plan.constraints()
    assert again.packs_like(plan)
