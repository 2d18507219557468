"""Tiles of 128 to 256 pixels x 64 to 256 channels (csrc/igemm_flex.hip), every
shape at the edges of tiles, of k-steps and of taps, against the oracle.  +-1
data: sums of at most 2 048 products and a bias are exact in half."""
import json

import pytest

import poplibs_amd as pa
from helpers import make_params

TILES = [(m, n, 1) for m in (128, 192, 256) for n in range(64, 257, 32)
         if (m, n) != (256, 64)]
TILES += [(128, 64, 2), (128, 96, 2), (128, 128, 2), (128, 160, 2),
          (192, 64, 2), (192, 96, 2)]


def _options(tile):
    m, n, flex = tile
    return {"planConstraints": json.dumps({"gfx950": {
        "kernel": "igemm", "patch": 0, "blockM": m, "blockN": n,
        "flex": flex}})}


def _exact(oracle, tile, kw, idil_phases=0):
    from test_fast_gpu import _run
    p = make_params(pa.HALF, **kw)
    print("case", tile, p, flush=True)
    text = pa.Plan(p, _options(tile)).describe()
    assert "%d x %d x 64" % tile[:2] in text, text
    assert ("two workgroups per CU" in text) == (tile[2] == 2), text
    if idil_phases:
        assert "%d phases" % idil_phases in text, text
    _run(oracle, p, 91, 0, "implicit GEMM", dist="pm1",
         options=_options(tile))


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
def test_every_tile_at_its_edges(oracle, tile):
    m, n, _ = tile
    # five M tiles (a block of four and one more), the last of one pixel; two N
    # tiles, the last of one channel; seven k-steps, more than any stages
    _exact(oracle, tile, dict(batch=1, field=(4 * m + 1,), kernel=(1,), ci=448,
                              co=n + 1))
    # a whole tile and a part, taps that share a k-step, images within a tile
    _exact(oracle, tile, dict(batch=3, field=(11, m // 16), kernel=(3, 3),
                              ci=8, co=n - 8, pad=1))


FORMS = [
    # fewer k-steps than stages: half of one, one, two
    dict(field=(9, 15), kernel=(1, 1), ci=32, co=72),
    dict(field=(9, 15), kernel=(1, 1), ci=64, co=72),
    dict(field=(9, 15), kernel=(1, 1), ci=72, co=72),
    # a chunk of 8 channels to a tap, and taps that straddle k-steps
    dict(batch=2, field=(13, 12), kernel=(5, 6), ci=8, co=40, pad=2),
    dict(batch=2, field=(13, 12), kernel=(3, 3), ci=40, co=130, pad=1),
    # strides, a dilated kernel, groups, a depth, a truncated input
    dict(batch=2, field=(33, 31), kernel=(3, 3), ci=72, co=200, stride=2,
         pad=1),
    dict(batch=2, field=(23, 21), kernel=(3, 3), ci=24, co=72, groups=3,
         stride=(1, 2), kdil=(2, 1), pad=(2, 1)),
    dict(batch=2, field=(6, 7, 8), kernel=(3, 2, 2), ci=16, co=24, pad=1),
    dict(batch=2, field=(19, 21), kernel=(3, 3), ci=64, co=40,
         itl=(1, 0), itu=(0, 3), padLower=(0, 2), padUpper=(2, 0)),
    # channels filled up in a copy, odd rows of outputs, zeros around the field
    dict(batch=3, field=(20, 20), kernel=(3, 3), ci=13, co=33, pad=1),
    dict(batch=2, field=(12, 12), kernel=(3, 3), ci=64, co=24, pad=1,
         opl=(1, 0), opu=(0, 2)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [(128, 64, 1), (128, 96, 2), (128, 160, 1),
                                  (192, 96, 2), (192, 256, 1), (256, 224, 1)])
@pytest.mark.parametrize("kw", FORMS)
def test_forms_of_layers(oracle, tile, kw):
    _exact(oracle, tile, kw)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("parts,kw", [
    # parts of three k-steps, the last of one; of one each; of two, the last of
    # none; taps that a part's first chunk starts in the middle of
    (3, dict(field=(9, 31), kernel=(1, 1), ci=448, co=260)),
    (7, dict(batch=2, field=(9, 15), kernel=(1, 1), ci=448, co=36)),
    (5, dict(field=(5, 15), kernel=(1, 1), ci=448, co=68)),
    (4, dict(batch=3, field=(9, 11), kernel=(3, 3), ci=40, co=136, pad=1,
             stride=(1, 2)))])
def test_k_in_parts(oracle, tile, parts, kw):
    from test_fast_gpu import _run
    options = _options(tile)
    named = json.loads(options["planConstraints"])
    named["gfx950"]["splitK"] = parts
    options = {"planConstraints": json.dumps(named)}
    p = make_params(pa.HALF, **kw)
    print("case", tile, parts, p, flush=True)
    assert "parts         %d" % parts in pa.Plan(p, options).describe()
    for bias in (True, False):
        _run(oracle, p, 93, 0, "implicit GEMM", dist="pm1", bias=bias,
             options=options)


@pytest.mark.gpu
def test_channels_filled_up_behind_the_parts_sums(oracle):
    """Ragged channels, whose copy lies behind the parts' sums in the
    workspace."""
    from test_fast_gpu import _run
    p = make_params(pa.HALF, batch=6, field=(16, 15), kernel=(3, 3), ci=845,
                    co=132, pad=1)
    options = {"planConstraints": '{"gfx950": {"kernel": "igemm", "patch": 0, '
                                  '"blockM": 192, "blockN": 160, "flex": 1, '
                                  '"splitK": 20}}'}
    assert "845 -> 848" in pa.Plan(p, options).describe()
    _run(oracle, p, 94, 1e-3, "implicit GEMM", wscale=0.05, options=options)


@pytest.mark.gpu
@pytest.mark.parametrize("p,filled", [
    (pa.matMulParams(pa.HALF, pa.HALF, 1, 133, 4872, 2744), None),
    (pa.matMulParams(pa.HALF, pa.HALF, 1, 480, 2407, 1040), "2407 -> 2408"),
    (make_params(pa.HALF, batch=8, field=(28, 33), kernel=(3, 3), ci=515,
                 co=144, pad=1), "515 -> 520")])
def test_the_planner_s_own_parts(oracle, p, filled):
    """K in parts as the planner itself cuts it, channels filled up in a copy
    among them."""
    from test_fast_gpu import _run
    plan = pa.Plan(p)
    print("case", p, flush=True)
    named = json.loads(plan.constraints())["gfx950"]
    assert named["flex"] == 1 and named["splitK"] > 1, named
    assert ("input channels padded" in plan.describe()) == bool(filled)
    assert not filled or filled in plan.describe(), plan.describe()
    _run(oracle, p, 95, 1e-3, "implicit GEMM", wscale=0.05)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [(128, 160, 2), (192, 96, 2), (256, 160, 1)])
@pytest.mark.parametrize("kw,phases", [
    (dict(batch=2, field=(14, 15), kernel=(3, 3), ci=40, co=72, idil=2,
          padLower=(1, 1), padUpper=(2, 1)), 4),
    # a phase of which no tap meets an input element
    (dict(batch=2, field=(9, 9), kernel=(1, 1), ci=64, co=136, idil=2), 4)])
def test_phases_in_one_launch(oracle, tile, kw, phases):
    _exact(oracle, tile, kw, phases)


@pytest.mark.gpu
def test_the_planner_s_own_phases(oracle):
    """A backward pass whose channels fill tiles of 128 badly."""
    p = make_params(pa.HALF, batch=35, field=(17, 18), kernel=(3, 3), ci=16,
                    co=136, idil=2, padLower=(1, 1), padUpper=(2, 1))
    assert "128 x 160 x 64" in pa.Plan(p).describe()
    from test_fast_gpu import _run
    _run(oracle, p, 92, 0, "implicit GEMM", dist="pm1")


@pytest.mark.gpu
@pytest.mark.parametrize("tile,parts,co", [
    *[(tile, 1, co) for tile in ((128, 96, 2), (192, 160, 1), (256, 256, 1))
      for co in (33, 72, 268)],
    ((128, 128, 1), 3, 72), ((128, 128, 1), 3, 268)])
def test_results_and_biases_anywhere(tile, parts, co):
    """A result that starts at a multiple of 16 bytes leaves through the L2 in
    rows of whole vectors, from 8 bytes or an element further on as whole vectors
    by way of it; a bias may start at any element.  The same bytes each time,
    nothing in front or behind."""
    import torch
    from poplibs_amd import capi
    options = _options(tile)
    named = json.loads(options["planConstraints"])
    named["gfx950"]["splitK"] = parts
    p = make_params(pa.HALF, batch=3, field=(11, 12), kernel=(3, 3), ci=72,
                    co=co, pad=1)
    print("case", tile, parts, co, flush=True)
    plan = pa.Plan(p, {"planConstraints": json.dumps(named)})
    dev, s = torch.device("cuda:0"), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=dev).manual_seed(8)

    def randoms(n):
        return torch.randn(n, generator=gen, device=dev).half()
    x, w = randoms(3 * 11 * 12 * 72), randoms(co * 72 * 9)
    bias = randoms(co)
    packed = torch.empty(plan.buffer_bytes(capi.BUF_WEIGHTS_PACKED),
                         dtype=torch.uint8, device=dev)
    work = torch.empty(max(plan.buffer_bytes(capi.BUF_WORKSPACE), 16),
                       dtype=torch.uint8, device=dev)
    plan.pack_weights(w.data_ptr(), packed.data_ptr(), s)
    size, guard, outs = 3 * 11 * 12 * co * 2, 64, []
    for off in (0, 8, 2):
        for first in (0, 1):
            moved = torch.zeros(co + 1, device=dev).half()
            moved[first:first + co] = bias
            buf = torch.full((size + 2 * guard + 8,), 0x5A, dtype=torch.uint8,
                             device=dev)
            assert buf.data_ptr() % 16 == 0 and moved.data_ptr() % 16 == 0
            plan.fwd(x.data_ptr(), packed.data_ptr(),
                     buf.data_ptr() + guard + off, moved.data_ptr() + 2 * first,
                     work.data_ptr(), work.numel(), s)
            torch.cuda.synchronize()
            assert bool((buf[:guard + off] == 0x5A).all())
            assert bool((buf[guard + off + size:] == 0x5A).all())
            outs.append(buf[guard + off:guard + off + size].clone())
    for other in outs[1:]:
        assert torch.equal(outs[0], other)
    ref = torch.nn.functional.conv2d(
        x.float().cpu().reshape(3, 11, 12, 72).permute(0, 3, 1, 2),
        w.float().cpu().reshape(co, 72, 3, 3), bias.float().cpu(), padding=1)
    got = outs[0].view(torch.float16).float().cpu().reshape(
        3, 11, 12, co).permute(0, 3, 1, 2)
    # fp32 sums of halves, rounded once
    assert (got - ref).norm() <= 1e-3 * ref.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [(128, 64, 1), (192, 96, 2)])
def test_an_input_beyond_two_gigabytes(tile):
    """Offsets count from the first image that a tile reads: every image of such
    a batch as it comes out alone."""
    import torch
    from poplibs_amd import capi
    kw = dict(field=(512, 512), kernel=(3, 3), ci=256, co=16, pad=1)
    plans = [pa.Plan(make_params(pa.HALF, batch=b, **kw), _options(tile))
             for b in (17, 1)]
    assert plans[0].buffer_bytes(capi.BUF_INPUT) > 2 ** 31
    print("case", tile, flush=True)
    dev, s = torch.device("cuda:0"), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=dev).manual_seed(9)
    x = torch.randn((17, 512, 512, 256), generator=gen, device=dev,
                    dtype=torch.float16)
    w = torch.randn((16, 256, 3, 3), generator=gen, device=dev,
                    dtype=torch.float16) * 0.02

    def run(plan, images):
        packed, out = (torch.empty(plan.buffer_bytes(b), dtype=torch.uint8,
                                   device=dev)
                       for b in (capi.BUF_WEIGHTS_PACKED, capi.BUF_OUTPUT))
        plan.pack_weights(w.data_ptr(), packed.data_ptr(), s)
        plan.fwd(images.data_ptr(), packed.data_ptr(), out.data_ptr(), None,
                 None, 0, s)
        torch.cuda.synchronize()
        return out.view(torch.float16).view(-1, 512, 512, 16)

    got = run(plans[0], x)
    for image in (0, 7, 8, 15, 16):
        assert torch.equal(got[image], run(plans[1], x[image])[0]), image
    assert torch.isfinite(got).all() and got.abs().max() > 0


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [False, True])
def test_a_multi_convolution_in_one_launch(bias):
    """Two layers in one tile shape share a launch, a third in another shape has
    its own: as one by one."""
    import torch
    from poplibs_amd import capi
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(5)
    s = torch.cuda.current_stream().cuda_stream
    plans, ins, packed, biases, outs, want = [], [], [], [], [], []
    for tile, kw in [((128, 96, 2), dict(batch=2, field=(13, 12), ci=40,
                                         co=96)),
                     ((128, 96, 2), dict(batch=3, field=(9, 9), ci=72,
                                         co=200)),
                     ((192, 96, 2), dict(batch=1, field=(9, 9), ci=64,
                                         co=33))]:
        p = make_params(pa.HALF, kernel=(3, 3), pad=1, **kw)
        plan = pa.Plan(p, _options(tile))

        def values(which):
            n = plan.buffer_bytes(which) // 2
            return torch.randn(n, generator=gen, device=dev).half()
        x, w = values(capi.BUF_INPUT), values(capi.BUF_WEIGHTS_EXTERNAL)
        pk = values(capi.BUF_WEIGHTS_PACKED)
        plan.pack_weights(w.data_ptr(), pk.data_ptr(), s)
        b = torch.randn(p.getNumOutputChans(), generator=gen, device=dev)
        biases.append(b.half())
        outs.append(values(capi.BUF_OUTPUT)), want.append(outs[-1].clone())
        plan.fwd(x.data_ptr(), pk.data_ptr(), want[-1].data_ptr(),
                 biases[-1].data_ptr() if bias else None, None, 0, s)
        plans.append(plan), ins.append(x), packed.append(pk)
    pa.multi_fwd(plans, [x.data_ptr() for x in ins],
                 [w.data_ptr() for w in packed], [o.data_ptr() for o in outs],
                 biases=[b.data_ptr() for b in biases] if bias else None,
                 stream=s)
    torch.cuda.synchronize()
    for got, expected in zip(outs, want):
        assert torch.equal(got, expected)


@pytest.mark.gpu
@pytest.mark.parametrize("layers,shared", [
    # (batch, field, kernel, channels, stride): K in parts in front of tiles of 128
    # x 64 and behind them; in two shapes of its own; beside too many tiles to gain
    # by it, or by enough
    ([(15, 22, 5, 248, 168, 1), (15, 22, 5, 248, 48, 1)], True),
    ([(15, 22, 5, 248, 48, 1), (15, 22, 5, 248, 168, 1)], True),
    ([(7, 22, 5, 392, 312, 1), (6, 21, 5, 392, 264, 1)], True),
    # (weights packed in 288 columns, read in 320)
    ([(11, 30, 3, 424, 288, 2), (12, 36, 3, 376, 196, 2)], True),
    ([(7, 22, 5, 392, 312, 1), (15, 22, 5, 248, 168, 1)], False),
    ([(19, 13, 5, 464, 280, 1), (8, 22, 5, 472, 200, 1)], False),
    ([(15, 22, 5, 248, 168, 1), (22, 27, 3, 352, 56, 1)], False)])
def test_k_in_parts_shares_a_launch(layers, shared):
    """Sums of K in parts are rounded elsewhere than those of K whole: the bytes
    tell which of the two ran."""
    import torch
    from poplibs_amd import capi
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(6)
    s = torch.cuda.current_stream().cuda_stream

    def run(plan, x, w, bias, out, work):
        packed = torch.empty(plan.buffer_bytes(capi.BUF_WEIGHTS_PACKED),
                             dtype=torch.uint8, device=dev)
        plan.pack_weights(w.data_ptr(), packed.data_ptr(), s)
        plan.fwd(x.data_ptr(), packed.data_ptr(), out.data_ptr(),
                 bias.data_ptr(), work.data_ptr(), work.numel(), s)
        return packed

    plans, ins, packed, biases, outs, works = [], [], [], [], [], []
    own, whole, flexible = [], [], []
    for batch, field, kernel, ci, co, stride in layers:
        p = make_params(pa.HALF, batch=batch, field=(field, field),
                        kernel=(kernel, kernel), ci=ci, co=co, stride=stride,
                        pad=kernel // 2)
        plan = pa.Plan(p)
        named = json.loads(plan.constraints())["gfx950"]
        flexible.append(bool(named.get("flex")) and named["splitK"] > 1)

        def values(which):
            n = plan.buffer_bytes(which) // 2
            return torch.randn(n, generator=gen, device=dev).half()
        x, w = values(capi.BUF_INPUT), values(capi.BUF_WEIGHTS_EXTERNAL)
        bias = torch.randn(co, generator=gen, device=dev).half()
        out = values(capi.BUF_OUTPUT)
        work = torch.empty(max(plan.buffer_bytes(capi.BUF_WORKSPACE), 16),
                           dtype=torch.uint8, device=dev)
        own.append(out.clone()), whole.append(out.clone())
        packed.append(run(plan, x, w, bias, own[-1], work))
        run(pa.Plan(p, {"planConstraints": json.dumps({"gfx950": dict(
            kernel="igemm", patch=0, pointwise=0, blockM=128, blockN=64,
            splitK=1)})}), x, w, bias, whole[-1], work)
        plans.append(plan), ins.append(x), biases.append(bias)
        outs.append(out), works.append(work)
    assert any(flexible)
    pa.multi_fwd(plans, [x.data_ptr() for x in ins],
                 [w.data_ptr() for w in packed], [o.data_ptr() for o in outs],
                 biases=[b.data_ptr() for b in biases],
                 workspaces=[w.data_ptr() for w in works],
                 workspace_bytes=[w.numel() for w in works], stream=s)
    torch.cuda.synchronize()
    for got, alone, k_whole, parts in zip(outs, own, whole, flexible):
        assert torch.equal(got, k_whole if shared else alone)
        assert not parts or not torch.equal(alone, k_whole)


@pytest.mark.parametrize("m,k,n", [(133, 4872, 5488), (450, 7416, 1400)])
def test_packed_weights_of_parts_are_the_tile_s(m, k, n):
    from poplibs_amd import capi
    p = pa.matMulParams(pa.HALF, pa.HALF, 1, m, k, n)
    plan = pa.Plan(p)
    again = pa.Plan(p, {"planConstraints": plan.constraints()})
    named = json.loads(plan.constraints())["gfx950"]
    assert named["splitK"] > 1
    rows = plan.buffer_bytes(capi.BUF_WEIGHTS_PACKED) // (-(-k // 64) * 128)
    assert rows == -(-n // named["blockN"]) * named["blockN"]
    assert again.packs_like(plan)


def test_plans_name_the_tile_and_come_back():
    p = make_params(pa.HALF, batch=25, field=(57, 57), kernel=(3, 3), ci=136,
                    co=200, pad=1)
    plan = pa.Plan(p)
    named = json.loads(plan.constraints())["gfx950"]
    assert named["flex"] in (1, 2)
    again = pa.Plan(p, {"planConstraints": plan.constraints()})
    assert again.constraints() == plan.constraints()
    assert again.packs_like(plan)
    without = pa.Plan(p, {"planConstraints": '{"gfx950": {"flex": 0}}'})
    assert "flex" not in without.constraints()


@pytest.mark.parametrize("m,k,n", [
    # taken from tiles of 256 x 256 of the other kernel, from 128 x 128; parts,
    # of few rows too
    (4096, 4096, 4096), (1026, 1080, 4604), (450, 7416, 1400),
    (97, 44912, 18728)])
def test_the_estimate_shown_is_the_call_s(m, k, n):
    """... and not the share of it that the choice was made by: the same for the
    plan made again from its constraints, which weighs nothing."""
    p = pa.matMulParams(pa.HALF, pa.HALF, 1, m, k, n)
    plan = pa.Plan(p)
    assert json.loads(plan.constraints())["gfx950"]["flex"]
    again = pa.Plan(p, {"planConstraints": plan.constraints()})
    (cycles, _), (expected, _) = plan.estimated_costs(), again.estimated_costs()
    assert abs(cycles - expected) <= 1


@pytest.mark.parametrize("asked", [
    dict(blockM=64, blockN=64, flex=1), dict(blockM=128, blockN=48, flex=1),
    dict(blockM=256, blockN=64, flex=1), dict(blockM=192, blockN=128, flex=2),
    dict(blockM=128, flex=1), dict(blockM=128, blockN=96, flex=3)])
def test_tiles_that_are_not_there_are_refused(asked):
    p = make_params(pa.HALF, batch=2, field=(9, 9), kernel=(3, 3), ci=64,
                    co=64, pad=1)
    with pytest.raises(pa.MxconvError, match="flex|tile"):
        pa.Plan(p, {"planConstraints": json.dumps({"gfx950": asked})})


@pytest.mark.parametrize("kw", [
    dict(dtype=pa.FLOAT, kernel=(3, 3)),
    dict(dtype=pa.QUARTER, out_dtype=pa.HALF, kernel=(3, 3)),
    dict(dtype=pa.HALF, out_dtype=pa.FLOAT, kernel=(3, 3)),
    dict(dtype=pa.HALF, kernel=(6, 6))])
def test_layers_it_does_not_take_are_refused(kw):
    p = make_params(batch=2, field=(9, 9), ci=64, co=64, pad=2, **kw)
    with pytest.raises(pa.MxconvError, match="flex"):
        pa.Plan(p, _options((128, 64, 1)))


@pytest.mark.parametrize("m,k,n", [(133, 4872, 5488), (298, 3528, 3712),
                                   (450, 7416, 1400), (2048, 8192, 1024)])
def test_parts_leave_room_in_the_static_scratch(m, k, n):
    """Callers that bring no workspace have 32 MB of it: products that ran
    without any before K was cut run in it still."""
    from poplibs_amd import capi
    plan = pa.MatMulPlan(pa.HALF, pa.HALF, 1, m, k, n)
    assert plan.buffer_bytes(capi.BUF_WORKSPACE) <= 32 << 20


@pytest.mark.parametrize("m,k,n,parts", [
    # more than 260 tiles of 128 x 64, in a part empty round of 128 x 128 with K
    # whole; more than 800; fewer than 192 channels
    (388, 6240, 5568, True), (1088, 6408, 2576, True),
    (3000, 6408, 2576, False), (32000, 2400, 128, False)])
def test_parts_of_sums_over_more_outputs(m, k, n, parts):
    from poplibs_amd import capi
    plan = pa.MatMulPlan(pa.HALF, pa.HALF, 1, m, k, n)
    chosen = [line for line in plan.describe().split("\n")
              if line.strip().startswith("*")]
    assert ("parts" in chosen[0]) == parts
    assert plan.buffer_bytes(capi.BUF_WORKSPACE) <= 32 << 20


@pytest.mark.parametrize("batch,field,ci,co,flexible", [
    # many input channels, tensors of 116, 110 and 153 MB; of 41 and 390; fewer
    # channels; a large product of few rows
    (101, (49, 14), 408, 432, False), (109, (26, 26), 432, 312, False),
    (88, (31, 31), 432, 472, False), (27, (32, 30), 416, 464, True),
    (112, (28, 52), 448, 744, True), (81, (45, 32), 280, 504, True),
    (1, (6972,), 464, 9976, True)])
def test_large_pointwise_layers_stay_with_their_kernel(batch, field, ci, co,
                                                       flexible):
    p = make_params(pa.HALF, batch=batch, field=field, kernel=(1,) * len(field),
                    ci=ci, co=co)
    named = json.loads(pa.Plan(p).constraints())["gfx950"]
    assert ("flex" in named) == flexible, named
    assert bool(named["pointwise"]) != flexible


@pytest.mark.parametrize("kw,parts", [
    # up to 128 channels: many pixels of a large input, planned with K whole or
    # in parts; fewer of them, a smaller input; more channels
    (dict(batch=9, field=(45, 30), kernel=(3, 3), ci=616, co=120, pad=1), False),
    (dict(batch=7, field=(35, 35), kernel=(5, 5), ci=520, co=104, pad=2), False),
    (dict(batch=6, field=(31, 31), kernel=(5, 5), ci=696, co=80, pad=2), True),
    (dict(batch=15, field=(35, 25), kernel=(5, 5), ci=312, co=72, pad=2), True),
    (dict(batch=9, field=(32, 32), kernel=(5, 5), ci=576, co=136, pad=2), True)])
def test_parts_of_windows_on_many_pixels(kw, parts):
    named = json.loads(pa.Plan(make_params(pa.HALF, **kw)).constraints())["gfx950"]
    assert ("flex" in named and named["splitK"] > 1) == parts, named


@pytest.mark.parametrize("batch,field,ci,co,shared", [
    # 242 and 49 MB of input; 13 and 37
    (99, 61, 328, 40, False), (99, 27, 336, 24, False),
    (18, 61, 96, 48, True), (28, 50, 264, 56, True)])
def test_two_narrow_tiles_to_a_cu_want_a_small_input(batch, field, ci, co,
                                                     shared):
    p = make_params(pa.HALF, batch=batch, field=(field, field), kernel=(5, 5),
                    ci=ci, co=co, pad=2)
    named = json.loads(pa.Plan(p).constraints())["gfx950"]
    assert (named.get("flex") == 2) == shared, named


def test_parts_want_whole_vectors():
    p = make_params(pa.HALF, batch=2, field=(9, 9), kernel=(3, 3), ci=64,
                    co=66, pad=1)
    with pytest.raises(pa.MxconvError, match="flex"):
        pa.Plan(p, {"planConstraints": json.dumps({"gfx950": {
            "kernel": "igemm", "patch": 0, "blockM": 128, "blockN": 96,
            "flex": 1, "splitK": 2}})})


@pytest.mark.parametrize("m,k,n", [
    # columns that tiles of 128 fill to the last and wider ones of their own do
    # not, whose packed weights would be 2^31 bytes and more
    (128, 32768, 32640), (16, 70272, 15136), (300, 376192, 2816),
    (128, 62016, 17272), (200, 89152, 12000), (512, 524096, 2048),
    # ... and the last a buffer reaches in tiles of 128
    (128, 16320, 65408), (4096, 8128, 130944)])
def test_packed_weights_stay_within_a_buffer_s_reach(m, k, n):
    from poplibs_amd import capi
    plan = pa.MatMulPlan(pa.HALF, pa.HALF, 1, m, k, n)
    assert "implicit GEMM" in plan.describe()
    assert plan.buffer_bytes(capi.BUF_WEIGHTS_PACKED) < 2 ** 31


@pytest.mark.parametrize("width,fits", [(128, True), (192, False)])
def test_a_named_tile_whose_weights_no_buffer_reaches_is_refused(width, fits):
    p = make_params(pa.HALF, batch=1, field=(16,), kernel=(1,), ci=32960,
                    co=32512)
    assert (-(-32512 // width) * width * 32960 * 2 < 2 ** 31) == fits
    if fits:
        pa.Plan(p, _options((128, width, 1)))
    else:
        with pytest.raises(pa.MxconvError, match="flex"):
            pa.Plan(p, _options((128, width, 1)))


@pytest.mark.parametrize("m,k,n,parts", [
    # the weights' way from memory is the time: tiles of 128 x 128 and 64, K whole
    # or in parts, fill the chip
    (12, 2384, 31152, False), (99, 4096, 23768, False), (77, 2240, 16232, False),
    (35, 6784, 9688, False),
    # so do tiles of 128 x 96, of which only a longer sum leaves
    (26, 4048, 20192, False), (14, 25184, 18648, True),
    # ... and do not
    (34, 10088, 5712, True), (97, 44912, 18728, True), (117, 2288, 4552, True)])
def test_parts_of_few_rows(m, k, n, parts):
    plan = pa.MatMulPlan(pa.HALF, pa.HALF, 1, m, k, n)
    chosen = [line for line in plan.describe().split("\n")
              if line.strip().startswith("*")]
    flexible = "flexible" in chosen[0] and "parts" in chosen[0]
    assert flexible == parts, chosen
