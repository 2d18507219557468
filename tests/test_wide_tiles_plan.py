"""Which convolutions get tiles of 256 pixels (csrc/igemm_wide.hip): the images
that a tile's pixels lie in have to stay within the kernel's 32-bit offsets.
Planning only; no GPU needed."""
import pytest

import poplibs_amd as pa
from helpers import make_params

H = pa.HALF
WIDE = {"planConstraints": '{"gfx950": {"kernel": "igemm", "pointwise": 0, '
                           '"blockM": 256, "blockN": 256}}'}


def _tile(plan):
    line, = [l for l in plan.describe().splitlines() if "block M" in l]
    return line.split("K  ")[1].strip()


@pytest.mark.parametrize("kw", [
    # 64 pixels of a 562 MB image: 128 of them lie in 3 images (1.69e9 bytes),
    # 256 in 5 (2.81e9)
    dict(batch=32, field=(1048, 1048), kernel=(1, 1), ci=256, co=8192,
         stride=131),
    # 16 pixels of a 143 MB image: 9 images (1.28e9), 17 images (2.43e9)
    dict(batch=128, field=(528, 528), kernel=(5, 5), ci=256, co=4096,
         stride=131),
])
def test_a_tile_never_spans_more_than_it_can_address(kw):
    p = make_params(H, **kw)
    assert _tile(pa.Plan(p)).startswith("128 x ")
    with pytest.raises(pa.MxconvError, match="blockM 256"):
        pa.Plan(p, WIDE)
    # (the same channels, 256 pixels of two images at most: 134 MB each)
    near = make_params(H, **dict(kw, field=(512, 512), stride=31))
    assert _tile(pa.Plan(near, WIDE)) == "256 x 256 x 64"


def test_a_product_of_many_groups_at_the_limit():
    # rows of groups x 4 KB, 256 + 1 of them (a row is an image)
    def product(groups):
        return pa.matMulParams(H, H, groups, 512, 2048, 128)
    assert 257 * 2038 * 4096 < 2 ** 31 - 2 ** 20 < 257 * 2040 * 4096
    assert _tile(pa.Plan(product(2038), WIDE)) == "256 x 256 x 64"
    for groups in (2040, 2100):
        with pytest.raises(pa.MxconvError, match="blockM 256"):
            pa.Plan(product(groups), WIDE)
        assert _tile(pa.Plan(product(groups))).startswith("128 x ")


@pytest.mark.parametrize("kw", [
    dict(batch=2, field=(9, 9), kernel=(6, 6), ci=64, co=64, pad=2),
    # every second output of a 1 x 1 layer's backward pass meets no input
    dict(batch=2, field=(9, 9), kernel=(1, 1), ci=64, co=64, idil=2),
])
def test_a_named_tile_the_kernel_cannot_run_is_refused_by_the_plan(kw):
    with pytest.raises(pa.MxconvError, match="blockM 256"):
        pa.Plan(make_params(H, **kw), WIDE)


@pytest.mark.parametrize("kw", [
    # a short K under large outputs: us in 256-pixel and in 128-pixel tiles
    dict(batch=15, field=(57, 57), kernel=(1, 1), ci=192, co=960),  # 51.1 36.4
    dict(batch=114, field=(38, 38), kernel=(1, 1), ci=144, co=960,
         stride=2),                                                 # 45.8 35.1
    dict(batch=32, field=(56, 56), kernel=(1, 1), ci=256, co=512,
         stride=2),                                                 # 17.4 15.8
])
def test_a_short_sum_keeps_narrow_tiles(kw):
    assert _tile(pa.Plan(make_params(H, **kw))) == "128 x 128 x 64"


def test_products_that_fill_the_chip_keep_it():
    plan = pa.MatMulPlan(H, H, 1, 4096, 4096, 4096)
    assert _tile(plan) == "256 x 256 x 64"


@pytest.mark.parametrize("co,batch,pointwise", [
    # 155 MB of output in rows of 1232 bytes, of whole 64-byte pieces, and less
    (616, 40, False), (608, 40, True), (616, 32, True)])
def test_large_outputs_in_odd_rows_leave_the_pointwise_kernel(co, batch,
                                                              pointwise):
    p = make_params(H, batch=batch, field=(56, 56), kernel=(1, 1), ci=40,
                    co=co)
    text = pa.Plan(p).describe()
    assert ("pointwise streaming" in text) == pointwise, text
    asked = {"planConstraints": '{"gfx950": {"pointwise": 1}}'}
    assert "pointwise streaming" in pa.Plan(p, asked).describe()


@pytest.mark.parametrize("in_type,ci,co,pointwise", [
    # more than 128 bytes of input to a pixel, 150 MB of output and more: pairs
    # of channel tiles write whole lines and stay where they are
    (pa.QUARTER, 160, 368, True), (pa.QUARTER, 144, 488, True),
    (pa.QUARTER, 160, 440, False), (pa.QUARTER, 128, 368, False),
    (H, 80, 456, False), (H, 96, 456, True), (H, 104, 400, False)])
def test_pairs_of_channel_tiles_in_odd_rows_stay(in_type, ci, co, pointwise):
    p = make_params(in_type, H, batch=64, field=(64, 64), kernel=(1, 1), ci=ci,
                    co=co)
    text = pa.Plan(p).describe()
    assert ("pointwise streaming" in text) == pointwise, text
