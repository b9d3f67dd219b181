"""Half-precision outputs of whole tiles at the ends of their types: scores that overflow to infinities, subnormal ones and zeros, with
and without a bias that does so itself, two outputs a conversion."""
import pytest
import torch

from test_gpu_parity import hip, ops  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", [128, 12864, 64, 6432])
def test_cast_of_the_float_scores(hip, ops, tile, dtype, bias):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    torch.manual_seed(5)
    dense = torch.nn.Linear(256, 256, bias=bias).cuda()
    with torch.no_grad():
        dense.weight.mul_(torch.logspace(0, 4, 256, device="cuda")[:, None])
        if bias:
            dense.bias.copy_(torch.logspace(-9, 5.5, 256, device="cuda") * torch.where(torch.arange(256, device="cuda") % 2 == 0, 1.0, -1.0))
    layer = BSIQuantizedLinear(dense, 2, 0.5)
    x = (torch.randn(128, 256, device="cuda") * torch.logspace(-2, 4, 128, device="cuda")[:, None]).to(dtype)
    hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, tile), "tile")
    try:
        with torch.no_grad():
            got = layer(x)
            scores = ops.linear_cuda(x, layer._bsi_keys_cuda, 2)
    finally:
        hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, 0), "tile")
    want = scores.to(dtype) + layer.bias.to(dtype) if bias else scores.to(dtype)
    assert (dtype == torch.float16) == bool(torch.isinf(want).any())
    torch.testing.assert_close(got, want, rtol=0.0, atol=0.0, equal_nan=True)  # an infinite score and the other infinite bias: NaN
