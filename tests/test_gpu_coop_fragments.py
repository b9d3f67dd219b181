"""The query build inside the few-rows launch, whose copies lie in the order of the kernel's operands: the bits of the build and
the dot in launches of their own at the edges of that order (full and short groups of 16 rows, one chunk and as many as the copy
and the chunk accumulators hold, one and two key tiles a workgroup)."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,d,R", [(15, 256, 4096), (16, 256, 300), (17, 256, 4096), (31, 768, 2048), (32, 8192, 4096), (16, 16384, 4096),
                                   (20, 6400, 16400), (32, 2304, 16416), (18, 1000, 2000), (16, 100, 2100)])
def test_same_bits_as_two_launches(ops, monkeypatch, Q, d, R):
    from bsipytorch_amd import _native
    from bsipytorch_amd.linear import BSIQuantizedLinear

    gen = torch.Generator(device="cuda").manual_seed(Q + d + R)
    layer = BSIQuantizedLinear(torch.nn.Linear(d, R).cuda(), 2, 0.5)
    keys = layer._bsi_keys_cuda
    assert ops.lib.bsi_hip_linear_coop_serves(Q, d, R, 2, 7, keys.layout, keys.Sb) == 1
    with torch.no_grad():
        for i in range(3):  # another magnitude for every row and a wide spread along it: scales that differ everywhere
            x = torch.randn(Q, d, generator=gen, device="cuda") * torch.exp(torch.randn(Q, 1, generator=gen, device="cuda"))
            x *= torch.exp(torch.randn((d + 255) // 256, generator=gen, device="cuda")).repeat_interleave(256)[:d]
            layer(x)
            got = _native.linear(layer.__dict__, x)
            assert got is not None
            with monkeypatch.context() as m:
                m.setenv("BSI_QUERY_CACHE", "0")  # the Python path: build, then dot
                assert torch.equal(got, layer(x))
    ops.linear_cuda_forget()
