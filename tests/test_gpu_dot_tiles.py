"""The matrix-core dot on grids of more than one round (a workgroup takes several tiles): the bits of the launch that stores
its integers and takes one tile a workgroup, over chunk counts that change the ring's phase, ragged edges and row scales."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,R,d,relu", [(2050, 2181, 64, False), (2100, 2177, 256, False), (2049, 2300, 512, True), (4100, 2177, 700, False),
                                        (1100, 4800, 1280, False), (8192, 768, 300, True), (129, 16640, 512, False), (33, 40000, 256, False)])
@pytest.mark.parametrize("tile", [0, 128, 12864])
def test_same_bits_as_one_tile_a_workgroup(ops, Q, R, d, relu, tile):
    gen = torch.Generator(device="cuda").manual_seed(Q + R + d)
    x = torch.randn(Q, d, generator=gen, device="cuda")
    x[:, ::97] *= 30.0
    keys = ops.build_bsi_keys_cuda(torch.randn(R, d, generator=gen, device="cuda") * 0.02, 2, 0.5)[0]
    queries = ops.build_bsi_queries_cuda_batch_packed(torch.relu(x) if relu else x, 2, 0.5)
    bias = torch.randn(R, generator=gen, device="cuda")
    want = ops.debug_chunk_ints(queries, keys, "mfma")[1]
    ops.lib.bsi_hip_set_option(1, tile)
    try:
        for _ in range(3):
            assert torch.equal(ops.batch_dot_product_multiquery_cuda_batch_caps(queries, keys)[0], want)
        got = ops.batch_dot_product_multiquery_cuda_batch_caps(queries, keys, bias)[0]
    finally:
        ops.lib.bsi_hip_set_option(1, 0)
    assert torch.equal(got, want + bias)
