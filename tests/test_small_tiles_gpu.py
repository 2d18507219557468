"""The small-tile kernel (csrc/igemm_small.hip), every tile forced, against the
oracle at the edges of its tiles, k-steps and waves."""
import pytest

import poplibs_amd as pa
from helpers import make_params, rel_l2

pytestmark = pytest.mark.gpu

SMALL = "small tiles"
HALF_CASES = [
    # one output pixel, one k-step half filled
    dict(field=(1, 1), kernel=(1, 1), ci=8, co=8),
    # pixels and channels just over a tile of 64 x 32, K just over 16 waves
    # of one group of four steps
    dict(field=(13, 5), kernel=(1, 1), ci=2056, co=40),
    dict(batch=3, field=(5, 13), kernel=(3, 3), ci=24, co=33, pad=1),
    # more tiles than CUs, two groups of loads and more
    dict(batch=2, field=(40, 40), kernel=(3, 3), ci=72, co=50, pad=1),
    dict(batch=1, field=(9, 7), kernel=(5, 3), ci=136, co=17, pad=2,
         stride=(2, 1), kdil=(1, 2)),
    # truncated and unevenly padded windows, strided 1 x 1
    dict(batch=2, field=(9, 8), kernel=(2, 3), ci=16, co=20, padLower=(0, 2),
         padUpper=(3, 0)),
    dict(batch=2, field=(9, 8), kernel=(1, 1), ci=16, co=20, stride=2),
    # zero-stuffed inputs, groups, output padding, padded channels
    dict(batch=2, field=(6, 5), kernel=(3, 3), ci=16, co=24, idil=2, pad=1),
    dict(batch=2, field=(6, 5), kernel=(3, 3), ci=16, co=24, idil=3,
         stride=2, pad=2),
    dict(batch=2, field=(6, 5), kernel=(3, 3), ci=32, co=20, groups=3, pad=1),
    dict(batch=2, field=(9, 8), kernel=(3, 3), ci=64, co=24, pad=1,
         opl=(1, 0), opu=(0, 2)),
    dict(batch=2, field=(30, 30), kernel=(3, 3), ci=13, co=60, pad=1),
    dict(batch=3, field=(40,), kernel=(3,), ci=16, co=10, flipK=True),
]


def _options(tile):
    return {"planConstraints": '{"gfx950": {"kernel": "igemm", '
                               '"smallTile": %d}}' % tile}


@pytest.mark.parametrize("tile", [1, 2, 3, 4])
@pytest.mark.parametrize("kw", HALF_CASES)
def test_small_tiles_half(oracle, kw, tile):
    from test_fast_gpu import _run
    p = make_params(pa.HALF, pa.FLOAT, **kw)
    assert SMALL in pa.Plan(p, _options(tile)).describe()
    _run(oracle, p, 61, 0, "implicit GEMM", dist="pm1",
         options=_options(tile))


@pytest.mark.parametrize("tile", [1, 2, 3, 4])
@pytest.mark.parametrize("kw", [HALF_CASES[2], HALF_CASES[4], HALF_CASES[7]])
def test_small_tiles_float_and_bias(oracle, kw, tile):
    from test_fast_gpu import _run
    p = make_params(pa.FLOAT, pa.FLOAT, **kw)
    _run(oracle, p, 62, 2e-6, "implicit GEMM", wscale=0.1,
         options=_options(tile))


@pytest.mark.parametrize("in_format", [0, 1])
@pytest.mark.parametrize("w_format", [0, 1])
@pytest.mark.parametrize("tile", [1, 3, 4])
def test_small_tiles_quarter(oracle, tile, in_format, w_format):
    from test_fast_gpu import _fp8_case
    p = make_params(pa.QUARTER, pa.HALF, batch=2, field=(9, 8), kernel=(3, 3),
                    ci=48, co=21, pad=1)
    got, want, plan = _fp8_case(oracle, p, 63, in_format, w_format,
                                options=_options(tile))
    assert SMALL in plan.describe()
    assert rel_l2(got, want) <= 1e-3


def test_small_tiles_share_a_launch(oracle):
    """Several of them in a multi-convolution give what each gives alone."""
    import torch
    from poplibs_amd import capi
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(3)
    plans, ins, ws, outs, biases, want, keep = [], [], [], [], [], [], []
    for kw in (dict(field=(9, 8), kernel=(3, 3), ci=24, co=33, pad=1),
               dict(batch=2, field=(5, 5), kernel=(3, 3), ci=16, co=40),
               dict(batch=3, field=(12, 4), kernel=(2, 3), ci=32, co=8)):
        plan = pa.Plan(make_params(pa.HALF, **kw), _options(3))
        bufs = [torch.randn(max(plan.buffer_bytes(b) // 2, 8), generator=g,
                            device=dev).half()
                for b in (capi.BUF_INPUT, capi.BUF_WEIGHTS_PACKED,
                          capi.BUF_OUTPUT, capi.BUF_OUTPUT, capi.BUF_BIAS)]
        x, w, alone, shared, bias = bufs
        plan.fwd(x.data_ptr(), w.data_ptr(), alone.data_ptr(),
                 bias.data_ptr())
        plans.append(plan)
        ins.append(x.data_ptr())
        ws.append(w.data_ptr())
        outs.append(shared.data_ptr())
        biases.append(bias.data_ptr())
        want.append((alone, shared))
        keep.append(bufs)
    pa.multi_fwd(plans, ins, ws, outs, biases=biases)
    torch.cuda.synchronize()
    for alone, shared in want:
        assert torch.equal(alone, shared)
