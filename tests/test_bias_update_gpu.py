"""The bias update's two kernels at the edges of their splits, vectors and
row lanes, against a double-precision sum."""
import numpy as np
import pytest
import torch

import poplibs_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,chans", [
    (1, 8),              # one row, one vector
    (63, 40), (64, 40), (65, 40),  # around one split
    (16383, 16), (16385, 16),      # around 256 splits, uneven last split
    (700, 8 * 65),       # two blocks of channels, an odd vector each
    (700, 8 * 64 + 4),   # whole vectors of float, not of half
    (5000, 3), (333, 1), (4097, 144),
    # the last row that goes in one launch; around its row lanes' passes
    (4096, 144), (1024, 33), (1025, 33), (2047, 40), (2049, 24), (256, 32), (257, 31),
    (2048, 144), (2049, 144), (4096, 64), (4096, 32), (4097, 64), (4097, 32),
    (3200, 144), (3201, 144), (3200, 168),
    # workgroups in pairs: one short of 16, 16, one more, the last one partial
    (300, 15 * 32), (300, 16 * 32), (300, 17 * 32), (300, 31 * 32 + 8),
    (300, 33 * 32 - 1), (2048, 32 * 32),
])
@pytest.mark.parametrize("dt,bt", [(pa.HALF, pa.HALF), (pa.HALF, pa.FLOAT),
                                   (pa.FLOAT, pa.FLOAT)])
def test_bias_update_edges(rows, chans, dt, bt):
    types = {pa.HALF: torch.float16, pa.FLOAT: torch.float32}
    g = torch.Generator().manual_seed(rows * 7 + chans)
    z = torch.randn(rows, chans, generator=g).to(types[dt])
    b = torch.randn(chans, generator=g).to(types[bt])
    zd, bd = z.to("cuda:0"), b.to("cuda:0")
    n = pa.bias_update_workspace_bytes(rows, chans)
    ws = torch.full((n,), 0xff, dtype=torch.uint8, device="cuda:0")
    pa.convolutionBiasUpdate(dt, zd.data_ptr(), rows, chans, bt,
                             bd.data_ptr(), 0.25, ws.data_ptr(), n)
    torch.cuda.synchronize()
    want = b.double() + 0.25 * z.double().sum(0)
    tol = 1e-3 if bt == pa.HALF else 1e-5
    np.testing.assert_allclose(bd.cpu().double().numpy(), want.numpy(),
                               rtol=tol, atol=tol * want.abs().max().item())
