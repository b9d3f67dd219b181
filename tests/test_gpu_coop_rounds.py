"""Small layers in one launch whose few workgroups build up to four rounds of chunks: the bits of the build and dot in launches of their
own, in both kernels, also where workgroups build the shares they wait for themselves."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

PATIENCE = 6  # BSI_OPT_COOP_PATIENCE


@pytest.mark.parametrize("Q,d,R", [(33, 1024, 2048), (41, 512, 1024), (60, 512, 1024), (150, 512, 1536), (128, 1024, 2048), (100, 1023, 3072), (30, 2048, 1024),
                                   (48, 768, 2000)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
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
                    x[Q // 2] *= 3.0e6 if dtype != torch.float16 else 100.0  # beyond the float32 quantiser
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
