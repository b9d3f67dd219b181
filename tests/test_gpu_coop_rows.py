"""Small layers in one launch whose waves build a row of several chunks each: the bits of the build and dot in launches of their own
at the edges of the rule and of a row (one chunk and eight, a remainder of one quad), in both kernels, for rows a quad can be loaded
from and rows whose address does not allow it, values beyond the float32 quantiser, and where workgroups build the shares they wait
for themselves."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

PATIENCE = 6  # BSI_OPT_COOP_PATIENCE


@pytest.mark.parametrize("Q,d,R", [(24, 704, 704), (24, 1600, 1600), (32, 1924, 2000), (31, 260, 1024), (77, 1600, 4800), (70, 1980, 4000), (37, 704, 9728),
                                   (250, 100, 8192), (100, 320, 2000), (33, 1860, 2048),
                                   (60, 704, 1024), (200, 448, 700), (90, 900, 1000), (150, 192, 768)])
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
                if i == 2:
                    x[Q // 2] *= 3.0e6 if dtype != torch.float16 else 100.0
                x = x.to(dtype)
                if i == 1:
                    x = torch.cat([x.new_zeros(1), x.view(-1)])[1:].view(Q, d)  # one element past an aligned address
                layer(x)
                got = _native.linear(layer.__dict__, x)
                assert got is not None
                with monkeypatch.context() as m:
                    m.setenv("BSI_QUERY_CACHE", "0")  # the Python path: build, then dot
                    assert torch.equal(got, layer(x))
    finally:
        ops.lib.bsi_hip_set_option(PATIENCE, 2000)
        ops.linear_cuda_forget()
