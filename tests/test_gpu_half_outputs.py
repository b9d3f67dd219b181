"""Linear layers whose half-precision output and bias come out of the dot's epilogue: the bits of the float32 scores cast
to the type plus the bias cast to it, on every kernel that has that epilogue, on whole tiles and ragged ones."""
import pytest
import torch

from test_gpu_parity import hip, ops  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Q,d,R,tile", [(1, 256, 16, 0), (3, 512, 70, 0), (4, 1024, 16400, 0), (5, 256, 48, 0), (17, 1024, 100, 0),
                                        (32, 64, 40, 0)] +
                         [shape + (tile,) for tile in (0, 128, 1284, 12864, 64, 6432)
                          for shape in ((33, 512, 64), (64, 192, 136), (128, 512, 256), (200, 320, 133), (256, 256, 384))])
def test_half_output_is_the_cast_of_the_float_one(hip, ops, Q, d, R, tile, dtype, bias):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    torch.manual_seed(Q + d + R)
    layer = BSIQuantizedLinear(torch.nn.Linear(d, R, bias=bias).cuda(), 2, 0.5)
    x = (torch.randn(Q, d, device="cuda") * 3).to(dtype)
    hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, tile), "tile")
    try:
        with torch.no_grad():
            got = layer(x)
            scores = ops.linear_cuda(x, layer._bsi_keys_cuda, 2)
    finally:
        hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, 0), "tile")
    assert scores.dtype == torch.float32 and got.dtype == dtype
    want = scores.to(dtype) + layer.bias.to(dtype) if bias else scores.to(dtype)
    assert torch.equal(got, want)


def test_half_output_of_a_split_launch(hip, ops):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    torch.manual_seed(1)
    layer = BSIQuantizedLinear(torch.nn.Linear(16384, 256).cuda(), 2, 0.5)
    x = torch.randn(64, 16384, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        got = layer(x)
        scores = ops.linear_cuda(x, layer._bsi_keys_cuda, 2)
    assert ops._split_shapes[(x.device.index, 64, 256, 256)]  # the launcher splits this shape
    assert torch.equal(got, scores.to(torch.bfloat16) + layer.bias.to(torch.bfloat16))
