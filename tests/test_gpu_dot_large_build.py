"""The build of a large layer that writes the images in units itself: the bits of the chain on rows of odd lengths and addresses, at the
edges of the chunks a wave holds, values beyond the float32 quantiser; and a pass without a build behind it, on the image it left."""
import pytest
import torch

from test_gpu_parity import hip, ops  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,d,R", [(512, 255, 300), (515, 1021, 256), (600, 4095, 260), (513, 4096, 40), (530, 4300, 256), (512, 16383, 130), (700, 2048, 511)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_same_bits_as_the_chain(hip, ops, Q, d, R, dtype):
    from bsipytorch_amd.linear import BSIQuantizedLinear

    gen = torch.Generator(device="cuda").manual_seed(Q + d + R)
    layer = BSIQuantizedLinear(torch.nn.Linear(d, R).cuda(), 2, 0.5)
    for wide in (False, True):
        x = torch.randn(Q, d, generator=gen, device="cuda") * torch.exp(torch.randn(Q, 1, generator=gen, device="cuda"))
        x[:, torch.rand(d, generator=gen, device="cuda") < 0.002] *= 20.0
        x[1] = 0
        if wide and dtype != torch.float16:
            x[2] *= 1.0e6
        x = x.to(dtype)
        odd = torch.cat([x.new_zeros(1), x.view(-1)])[1:].view(Q, d)  # one element past an aligned address
        outs = {}
        for tile in (256, 128):
            hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, tile), "tile")
            try:
                with torch.no_grad():
                    outs[tile] = layer(x), layer(x), layer(odd)  # the second on the image that the first has left
            finally:
                hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, 0), "tile")
        for got, want in zip(outs[256], outs[128]):
            assert torch.equal(got, want)
