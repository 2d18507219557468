"""The rearrangement kernels behind mxconv_acts_to_internal / _to_external and
mxconv_transpose_grouped_matrix: every size class and its edges, bit for bit."""
import pytest
import torch

import poplibs_amd as pa

pytestmark = pytest.mark.gpu

TYPES = {pa.QUARTER: torch.uint8, pa.HALF: torch.int16, pa.FLOAT: torch.int32}


@pytest.mark.parametrize("groups,rows,cols", [
    (1, 64, 64), (3, 65, 63), (2, 8, 200), (2, 200, 8), (5, 7, 300),
    (1, 1000, 257), (70000, 9, 10),
    # few on one side: around a workgroup's pixels, odd counts
    (2, 3, 2048), (3, 3, 2049), (2, 3, 4097), (2, 2, 5001), (2, 4, 4095),
    (2, 2047, 3), (2, 2049, 3), (1, 6001, 2), (1, 8193, 4),
    (4, 3, 130), (4, 1, 77), (4, 77, 1), (1, 5, 5),
    # ... and in numbers that fill the chip, with workgroups of one wave
    # (up to 512 Ki elements to a side's vector of 16 bytes) and of four
    (43, 3, 2049), (70, 2, 2047), (1, 4, 65537), (19, 4097, 4),
    (1, 100001, 3), (131, 3, 4097), (300, 2, 4095), (2, 4, 299999),
    (270, 4097, 3),
])
@pytest.mark.parametrize("t", TYPES)
def test_transpose(groups, rows, cols, t):
    x = torch.randint(-128 if t else 0, 127, (groups, rows, cols),
                      dtype=torch.int32).to(TYPES[t]).cuda()
    y = torch.full((groups, cols, rows), 99, dtype=TYPES[t], device="cuda:0")
    pa.transposeGroupedMatrix(t, groups, rows, cols, x.data_ptr(),
                              y.data_ptr())
    torch.cuda.synchronize()
    assert torch.equal(y, x.transpose(1, 2))


@pytest.mark.parametrize("g,m,c", [(3, 5, 8), (4, 6, 7), (1, 9, 16),
                                   (16, 1, 24), (5, 130, 64)])
def test_group_shuffle(g, m, c):
    plan = pa.MatMulPlan(pa.HALF, pa.HALF, g, m, c, c)
    x = torch.randint(-9, 9, (g, m, c), dtype=torch.int16).cuda()
    y, z = torch.empty_like(x), torch.empty_like(x)
    plan.lhs_to_internal(x.data_ptr(), y.data_ptr())
    plan.out_to_external(y.data_ptr(), z.data_ptr())
    torch.cuda.synchronize()
    assert torch.equal(y.view(m, g, c), x.transpose(0, 1))
    assert torch.equal(z, x)
