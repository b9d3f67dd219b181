"""Small layers in one launch that has more workgroups than tiles, the others there for the build: the bits of the build and dot in
launches of their own, in both kernels and all kinds of scales and grids, also where workgroups build the shares they wait for."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

PATIENCE = 6  # BSI_OPT_COOP_PATIENCE


@pytest.mark.parametrize("Q,d,R", [(33, 256, 256), (33, 768, 768), (64, 1536, 1030), (512, 512, 300), (1000, 256, 256), (180, 1024, 577),  # chunk scales
                                   (6, 2304, 256), (32, 4096, 257), (1, 300, 271), (24, 2048, 1024),  # the few-rows kernel
                                   (40, 320, 320), (500, 320, 300), (128, 1600, 512), (200, 100, 259), (31, 1000, 400)])  # row scales
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("patience", [2000, 0])
def test_same_bits_as_two_launches(ops, monkeypatch, Q, d, R, dtype, patience):
    from bsipytorch_amd import _native
    from bsipytorch_amd.linear import BSIQuantizedLinear

    gen = torch.Generator(device="cuda").manual_seed(Q + d + R)
    layer = BSIQuantizedLinear(torch.nn.Linear(d, R).cuda(), 2, 0.5)
    keys = layer._bsi_keys_cuda
    layout = keys.layout if Q <= 32 else 2  # BSI_LAYOUT_INT8
    assert ops.lib.bsi_hip_linear_coop_serves(Q, d, R, 2, 7, layout, keys.Sb) == 1
    ops.lib.bsi_hip_set_option(PATIENCE, patience)
    try:
        with torch.no_grad():
            for i in range(3):
                x = torch.randn(Q, d, generator=gen, device="cuda") * torch.exp(torch.randn(Q, 1, generator=gen, device="cuda"))
                x[:, torch.rand(d, generator=gen, device="cuda") < 0.01] *= 20.0
                if i == 2:
                    x[Q // 2] *= 3.0e6  # beyond the float32 quantiser
                x = x.to(dtype)
                layer(x)
                got = _native.linear(layer.__dict__, x)
                assert got is not None
                with monkeypatch.context() as m:
                    m.setenv("BSI_QUERY_CACHE", "0")  # the Python path: build, then dot
                    assert torch.equal(got, layer(x))
    finally:
        ops.lib.bsi_hip_set_option(PATIENCE, 2000)
        ops.linear_cuda_forget()


@pytest.mark.parametrize("Q, d, R, served", [(48, 2048, 2048, 1), (128, 2048, 2048, 0), (33, 4096, 1024, 0), (256, 768, 3072, 1), (512, 512, 512, 1), (128, 1536, 1536, 0), (256, 1024, 1024, 0), (64, 2048, 2048, 1), (200, 1024, 1024, 1), (100, 1536, 1536, 1),
                                             (512, 512, 4096, 0), (128, 1600, 512, 1), (128, 1600, 1600, 0), (300, 704, 256, 1), (300, 704, 255, 0)])
def test_where_the_rule_lies(ops, Q, d, R, served):
    assert ops.lib.bsi_hip_linear_coop_serves(Q, d, R, 2, 7, 2, 6) == served
