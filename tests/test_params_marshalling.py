"""The short ways of a call made on every training step: parameters marshalled
as one record, and weightsTransposeChansFlipXY's check of parameters without
building the class."""
from ctypes import byref

import numpy as np
import pytest

import poplibs_amd as pa
from poplibs_amd.capi import Status


def _random_params(rng):
    n = int(rng.integers(0, 4))

    def ints(lo, hi):
        return [int(v) for v in rng.integers(lo, hi, n)]

    p = pa.ConvParams(pa.HALF, pa.FLOAT, 2, ints(0, 9), ints(0, 5), 3, 4, 2)
    for t in (p.inputTransform, p.kernelTransform):
        t.truncationLower = ints(0, 2) if rng.random() < .3 else [0] * n
        t.truncationUpper = ints(0, 2) if rng.random() < .3 else [0] * n
        t.dilation = ints(0, 4) if rng.random() < .3 else [1] * n
        t.paddingLower, t.paddingUpper = ints(0, 3), ints(0, 3)
        t.flip = [bool(v) for v in ints(0, 2)]
    o = p.outputTransform
    o.truncationLower = ints(0, 3) if rng.random() < .3 else [0] * n
    o.truncationUpper = ints(0, 2) if rng.random() < .3 else [0] * n
    o.stride = ints(0, 4) if rng.random() < .3 else [1] * n
    o.paddingLower, o.paddingUpper = ints(0, 3), ints(0, 2)
    return p


@pytest.mark.parametrize("seed", range(4))
def test_records_and_checks_agree_with_the_long_way(seed):
    rng = np.random.default_rng(seed)
    L = pa.lib()
    seen = set()
    for _ in range(500):
        p = _random_params(rng)
        c = p.to_c()
        assert bytes(c) == bytes(p._to_c_by_field(len(p.inputFieldShape)))
        valid = L.mxconv_params_validate(byref(c))
        got = L.mxconv_weights_transpose_chans_flip_xy(byref(c), None, None,
                                                       None)
        empty = 0 in p.kernelShape
        seen.add(valid)
        # (valid ones go on to ask for the tensors, unless there is nothing
        # to do)
        assert got == (valid if valid != Status.OK else
                       Status.OK if empty else Status.NULL_ARGUMENT), p
    assert len(seen) == 2


@pytest.mark.parametrize("seed", range(4, 8))
def test_the_record_and_the_class_are_held_to_the_same_rules(seed):
    """mxconv_params_validate reads the C record, canonicalisation asks the
    class: same status, same words."""
    rng = np.random.default_rng(seed)
    L = pa.lib()
    seen = set()
    for _ in range(500):
        c = _random_params(rng).to_c()
        valid = L.mxconv_params_validate(byref(c))
        words = L.mxconv_last_error()
        assert L.mxconv_params_canonicalize(byref(c), byref(type(c)())) == valid
        if valid != Status.OK:
            assert L.mxconv_last_error() == words
        seen.add(words)
    assert len(seen) > 5


def test_every_count_of_dimensions_is_one_record():
    for n in range(pa.capi.MAX_FIELD_DIMS + 1):
        size = list(range(3, 3 + n))
        p = pa.ConvParams(pa.FLOAT, pa.HALF, 7, size, size[::-1], 5, 6, 2)
        p.inputTransform.flip = [d % 2 == 0 for d in range(n)]
        p.outputTransform.paddingUpper = size
        assert bytes(p.to_c()) == bytes(p._to_c_by_field(n))
    p = pa.ConvParams(pa.HALF, pa.HALF, 1, [4, 4], [3, 3], 8, 8)
    p.kernelTransform.dilation = [1]
    with pytest.raises(pa.MxconvError, match="kernel dilation"):
        p.to_c()


def test_lists_of_other_lengths_are_refused():
    for change in ("stride", "paddingUpper"):
        p = pa.ConvParams(pa.HALF, pa.HALF, 1, [4, 4], [3, 3], 8, 8)
        getattr(p.outputTransform, change).append(1)
        p.outputTransform.truncationLower.pop()
        with pytest.raises(pa.MxconvError):
            p.to_c()
