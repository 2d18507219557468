"""The last sums of weight deltas and bias updates where their offsets do not fit
31 bits (csrc/depthwise_train.hip, csrc/layout.hip).  +-1 data: exact."""
import pytest

import poplibs_amd as pa
from helpers import make_params


def _signs(shape, seed):
    import torch
    gen = torch.Generator(device="cuda:0").manual_seed(seed)
    return torch.randint(0, 2, shape, generator=gen, device="cuda:0",
                         dtype=torch.int8).mul_(2).sub_(1).half()


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 3])
def test_depthwise_weight_deltas_of_many_channels(batch):
    import torch
    C = 1500008
    p = make_params(pa.HALF, pa.FLOAT, batch=batch, field=(3, 3), kernel=(3, 3),
                    groups=C, pad=1)
    print("case", batch, C, flush=True)
    plan = pa.WeightUpdatePlan(p)
    x, dz = _signs((batch, 3, 3, C), 1), _signs((batch, 3, 3, C), 2)
    dw = torch.full((C, 3, 3), 99.0, device="cuda:0")
    ws = torch.empty(max(plan.workspace_bytes(), 16), dtype=torch.uint8,
                     device="cuda:0")
    # (offsets of one slice and the 40 beyond it that eight parts may ask for)
    assert 41 * 9 * C * 4 >= 2 ** 31
    plan.calculate_weight_deltas(dz.data_ptr(), x.data_ptr(), dw.data_ptr(),
                                 ws.data_ptr(), ws.numel(),
                                 torch.cuda.current_stream().cuda_stream)
    xs, dzs = (torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1)), dz)
    for kh in range(3):
        for kw in range(3):
            want = (xs[:, kh:kh + 3, kw:kw + 3] * dzs).sum(
                (0, 1, 2), dtype=torch.float32)
            assert torch.equal(dw[:, kh, kw], want), (kh, kw)


@pytest.mark.gpu
# (offsets of 31 bits end between the two)
@pytest.mark.parametrize("channels", [2097151, 2097153])
def test_bias_update_of_many_channels(channels):
    import torch
    rows = 1030  # more than one launch takes of ragged rows
    print("case", rows, channels, flush=True)
    dz = _signs((rows, channels), 3)
    bias = torch.arange(channels, device="cuda:0").remainder_(64).float()
    want = bias - 2.0 * dz.sum(0, dtype=torch.float32)
    n = pa.bias_update_workspace_bytes(rows, channels)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda:0")
    pa.convolutionBiasUpdate(pa.HALF, dz.data_ptr(), rows, channels, pa.FLOAT,
                             bias.data_ptr(), -2.0, ws.data_ptr(), n,
                             torch.cuda.current_stream().cuda_stream)
    assert torch.equal(bias, want)
