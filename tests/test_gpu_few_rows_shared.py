"""Layers of two to four rows on either side of the rule between a build in every workgroup and one that an XCD's workgroups share."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,d,R,shares", [(2, 2304, 16384, 0), (2, 4096, 16384, 1), (2, 5120, 5120, 1), (3, 4096, 5120, 1), (4, 4096, 4096, 0), (4, 8192, 2048, 1),
                                          (1, 8192, 8192, 0), (4, 1024, 77, 0), (3, 8186, 1024, 1), (2, 5110, 5120, 1)])  # the last two: rows that no quad can be loaded from
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_same_bits(ops, monkeypatch, Q, d, R, shares, dtype):
    from bsipytorch_amd import _native
    from bsipytorch_amd.linear import BSIQuantizedLinear

    assert ops.lib.bsi_hip_linear_few_rows_shares(Q, d, R) == shares
    gen = torch.Generator(device="cuda").manual_seed(Q + d + R)
    layer = BSIQuantizedLinear(torch.nn.Linear(d, R).cuda(), 2, 0.5)
    with torch.no_grad():
        for i in range(3):
            x = torch.randn(Q, d, generator=gen, device="cuda") * (3.0e6 if i == 2 else 1.0)
            x[:, ::50] *= 20.0
            x = x.to(dtype)
            layer(x)
            builds = layer.build_calls
            got = _native.linear(layer.__dict__, x)
            assert got is not None and layer.build_calls == builds  # in the dot's launch on either side
            with monkeypatch.context() as m:
                m.setenv("BSI_FUSED_LINEAR", "0")
                m.setenv("BSI_QUERY_CACHE", "0")
                ops._reset_flag_cache()
                want = layer(x)
            ops._reset_flag_cache()
            assert torch.equal(got, want)
    ops.linear_cuda_forget()
