"""Weight packing (csrc/pack_weights.hip) where its layouts have edges: several
phases in a launch, selected taps, fused groups, half-filled vectors
and blocks; +-1 data, exact against the oracle."""
import json

import pytest

import poplibs_amd as pa
from helpers import make_params

pytestmark = pytest.mark.gpu

CASES = [
    # six phases; phases without taps
    (dict(batch=2, field=(6, 5), kernel=(4, 3), ci=16, co=40, idil=(2, 3),
          pad=3),
     dict(kernel="igemm", smallTile=0), 0),
    (dict(batch=2, field=(6, 5), kernel=(2, 1), ci=24, co=130, idil=(2, 4),
          pad=(1, 0)), dict(kernel="igemm", smallTile=0), 0),
    # padded input channels, phases of a fused group
    (dict(batch=2, field=(7, 9), kernel=(3, 3), ci=13, co=5, idil=2, pad=1),
     dict(kernel="igemm", smallTile=0), 0),
    (dict(batch=2, field=(7, 6), kernel=(3, 3), ci=4, co=12, groups=8, idil=2,
          pad=1), dict(kernel="igemm", smallTile=0), 4),
    # resident patch, both orders: channels beyond a block, selected taps
    (dict(batch=2, field=(14, 14), kernel=(3, 3), ci=64, co=40, pad=1,
          flipK=True), dict(kernel="igemm", patch=1, blockM=64), 0),
    (dict(batch=2, field=(14, 14), kernel=(2, 3), ci=128, co=200, pad=1),
     dict(kernel="igemm", patch=2, blockM=112), 0),
]


@pytest.mark.parametrize("kw,gfx,groups", CASES)
def test_packed_weights(oracle, kw, gfx, groups):
    from test_fast_gpu import _run
    doc = {"gfx950": gfx}
    if groups:
        doc["convGroupsPerGroup"] = groups
    p = make_params(pa.HALF, pa.FLOAT, **kw)
    _run(oracle, p, 71, 0, "implicit GEMM", dist="pm1",
         options={"planConstraints": json.dumps(doc)})


@pytest.mark.parametrize("kw", [
    dict(field=(5, 6, 7), kernel=(2, 3, 1), ci=3, co=9, groups=2),
    dict(field=(9, 9), kernel=(1, 1), ci=70, co=65),
    dict(field=(9,), kernel=(5,), ci=1, co=1, groups=33)])
@pytest.mark.parametrize("dtype", [pa.HALF, pa.FLOAT, pa.QUARTER])
def test_transpose_chans_flip(kw, dtype):
    import torch
    p = make_params(dtype, pa.HALF if dtype == pa.QUARTER else dtype, **kw)
    elem = {pa.HALF: torch.float16, pa.FLOAT: torch.float32,
            pa.QUARTER: torch.uint8}[dtype]
    g, co, ci = kw.get("groups", 1), kw["co"], kw["ci"]
    w = torch.arange(g * co * ci * 30, device="cuda")[
        :g * co * ci * int(torch.tensor(kw["kernel"]).prod())]
    w = (w % 251).to(elem).reshape(g, co, ci, *kw["kernel"])
    out = torch.empty(g, ci, co, *kw["kernel"], dtype=elem, device="cuda")
    pa.weightsTransposeChansFlipXY(p, w.data_ptr(), out.data_ptr())
    axes = list(range(3, w.dim()))
    want = w.cpu().transpose(1, 2).flip(axes)
    assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("gfx", [dict(smallTile=2), dict(patch=1),
                                 dict(patch=2), dict(patch=0, blockN=64),
                                 dict(patch=0, blockN=128, splitK=2)])
@pytest.mark.parametrize("groups", [2, 8])
def test_packed_weights_end_with_their_buffer(gfx, groups):
    # groups taken as one: the buffer is the fused groups' packed weights and
    # nothing behind them is written
    import torch
    from poplibs_amd import capi
    p = make_params(pa.HALF, pa.HALF, batch=2, field=(14, 14), kernel=(3, 3),
                    ci=64 // groups, co=24, groups=16, pad=1)
    plan = pa.Plan(p, {"planConstraints": json.dumps(
        {"convGroupsPerGroup": groups, "gfx950": dict(gfx, kernel="igemm")})})
    assert "conv groups per group      %d" % groups in plan.describe()
    n = plan.buffer_bytes(capi.BUF_WEIGHTS_PACKED)
    fused = 16 // groups * (64 * 9) * (24 * groups) * 2
    assert fused <= n <= fused * 8 // 3  # (channels to whole tiles)
    w = torch.randn(16 * 24 * 64 // groups * 9, device="cuda").half()
    packed = torch.full((n + 4096,), 0xa5, dtype=torch.uint8, device="cuda")
    plan.pack_weights(w.data_ptr(), packed.data_ptr())
    torch.cuda.synchronize()
    assert bool((packed[n:] == 0xa5).all())
    assert int((packed[:n].view(torch.int16) != 0).sum()) == w.numel() - int(
        (w == 0).sum())
