"""Grids of 128 x 128 tiles that are a round and a half: three rounds of 128 x 64 write the same bits, on either side of the rule."""
import ctypes

import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,d,R,tile", [(768, 520, 8192, 12864), (769, 512, 8192, 128), (1281, 1024, 2946, 12864), (530, 600, 8191, 12864), (768, 512, 8192, 128), (768, 1025, 8192, 128),
                                        (768, 256, 8192, 128), (1024, 512, 4096, 128)])
def test_same_bits(ops, Q, d, R, tile):
    from bsipytorch_amd import _lib

    got, segments = ctypes.c_int(), ctypes.c_int()
    _lib.check(_lib.lib.bsi_hip_dot_split_plan(R, Q, (d + 63) // 64, ctypes.byref(got), ctypes.byref(segments)), "plan")
    assert (got.value, segments.value) == (tile, 1)
    gen = torch.Generator(device="cuda").manual_seed(Q + R)
    keys = ops.build_bsi_keys_cuda(torch.randn(R, d, generator=gen, device="cuda") * 0.02, 2, 0.5)[0]
    queries = ops.build_bsi_queries_cuda_batch_packed(torch.randn(Q, d, generator=gen, device="cuda"), 2, 0.5)
    outs = []
    try:
        for option in (0, 128, 64):
            assert _lib.lib.bsi_hip_set_option(1, option) == 0
            outs.append(ops.batch_dot_product_multiquery_cuda_batch_caps(queries, keys)[0])
    finally:
        _lib.lib.bsi_hip_set_option(1, 0)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("Q,d,R,tile", [(768, 512, 8192, 12864), (530, 1000, 8192, 12864), (1281, 700, 2946, 12864), (768, 256, 8192, 128), (768, 1025, 8192, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layers(ops, Q, d, R, tile, dtype):
    """The tile that a layer takes by itself, from two chunks on, and the bits of it and of each tile asked for; some of them the oracle's."""
    from bsipytorch_amd import _lib
    from bsipytorch_amd.linear import BSIQuantizedLinear
    from oracle import bsi_oracle

    plan, streamed = ctypes.c_int(), ctypes.c_int()
    _lib.check(_lib.lib.bsi_hip_linear_plan(Q, d, R, R, _lib.DTYPE_F32, ctypes.byref(plan), ctypes.byref(streamed)), "plan")
    assert (plan.value, streamed.value) == (tile, 0)
    gen = torch.Generator(device="cuda").manual_seed(Q + R)
    dense = torch.nn.Linear(d, R, device="cuda")
    layer = BSIQuantizedLinear(dense, 2, 0.5)
    x = torch.randn(Q, d, generator=gen, device="cuda").to(dtype)
    outs = []
    try:
        for option in (0, 128, 12864, 64):
            assert _lib.lib.bsi_hip_set_option(1, option) == 0
            with torch.no_grad():
                outs.append(layer(x.clone()))
    finally:
        _lib.lib.bsi_hip_set_option(1, 0)
    assert all(torch.equal(outs[0], o) for o in outs[1:])
    if dtype == torch.float32:
        rows, keys = [0, 63, 64, 127, 128, Q - 1], [0, 1, 63, 127, 128, R - 2, R - 1]
        qb = bsi_oracle.build_queries(x[rows].cpu().numpy())
        kb = bsi_oracle.build_keys(dense.weight.detach()[keys].cpu().numpy())
        want = bsi_oracle.dot_fixed(qb["words"], qb["scales"], kb["words"], kb["scales"], bsi_oracle.scale_inv(2, 2))[1]
        want = want + dense.bias.detach()[keys].cpu().numpy()
        assert (outs[0][rows][:, keys].cpu().numpy() == want).all()
