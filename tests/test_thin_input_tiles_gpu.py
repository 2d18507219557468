"""Tiles and workgroups of the kernel for inputs of 1 to 4 channels
(chooseThinInputTiles in csrc/thin_input.hip), against the CPU oracle."""
import re

import numpy as np
import pytest

import poplibs_amd as pa
from helpers import make_params, random_data


def _shape(plan):
    """(output rows of a tile, workgroups, tiles)"""
    text = plan.describe()
    rows = re.search(r"tiles of (\d+) output rows of one image", text)
    groups = re.search(r"(\d+) persistent \(4 waves\) taking (\d+) tiles",
                       text)
    return int(rows[1]), int(groups[1]), int(groups[2])


CASES = [
    # more tiles than places, of three and of two workgroups to a CU
    dict(batch=1300, field=(16, 20), kernel=(3, 3), ci=3, co=16, pad=1),
    dict(batch=600, field=(16, 16), kernel=(7, 7), ci=3, co=64, pad=3),
    # more than two workgroups to a CU in one round
    dict(batch=40, field=(100, 100), kernel=(3, 3), ci=3, co=16, pad=1),
    # tiles of any number of rows, the last one of an image with fewer
    dict(batch=33, field=(138, 138), kernel=(7, 7), ci=3, co=16, pad=3),
    dict(batch=8, field=(75, 91), kernel=(5, 5), ci=3, co=48, pad=2, stride=2),
]


@pytest.mark.gpu
@pytest.mark.parametrize("kw", CASES)
def test_tiles_of_signs_are_exact(oracle, kw):
    from gpu_helpers import quantize, run_conv
    p = make_params(pa.HALF, pa.FLOAT, **kw)
    print("case", kw, flush=True)
    acts, weights, biases = random_data(p, 13, "pm1")
    aq, ad = quantize(acts, pa.HALF)
    wq, wd = quantize(weights, pa.HALF)
    bq, bd = quantize(biases, pa.FLOAT)
    got, _ = run_conv(p, aq, wq, bq, return_plan=True)
    np.testing.assert_array_equal(got, oracle.convolution(p, ad, wd, bd,
                                                          threads=8))


def test_tiles_fill_the_last_round():
    def shape(kw):
        return _shape(pa.Plan(make_params(pa.HALF, pa.HALF, **kw)))
    for kw, places in ((CASES[0], 768), (CASES[1], 512)):
        rows, groups, tiles = shape(kw)
        assert tiles > groups == places
    for kw, least in ((CASES[2], 512), (CASES[3], 512)):
        rows, groups, tiles = shape(kw)
        assert least < tiles == groups <= 1024
    # few images: a row to a tile while that spreads over the chip
    rows, groups, tiles = shape(dict(batch=1, field=(68, 68), kernel=(3, 3),
                                     ci=3, co=32, pad=1, stride=2))
    assert (rows, tiles) == (1, 34)
