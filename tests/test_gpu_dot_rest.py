"""Grids whose last round is done as halves or quarters of its tiles: the bits of smaller tiles all over, with key and query tiles that
are cut off, in either order of the tiles, and nothing written beside the outputs."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,d,R", [(530, 3072, 8192), (281, 3100, 12483), (1100, 4096, 4000), (257, 3072, 11100), (3594, 6144, 1536), (768, 6150, 8192),
                                   (2049, 3072, 4030), (640, 3071, 8130)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_same_bits(ops, Q, d, R, dtype):
    from bsipytorch_amd import _lib
    from bsipytorch_amd.linear import BSIQuantizedLinear

    n = -(-Q // 128) * -(-R // 128)
    assert n > 256 and 0 < n % 256 <= (64 if d < 6000 else 128)
    gen = torch.Generator(device="cuda").manual_seed(Q + R)
    layer = BSIQuantizedLinear(torch.nn.Linear(d, R, device="cuda"), 2, 0.5)
    x = torch.randn(Q, d, generator=gen, device="cuda").to(dtype)
    got = []
    try:
        for tile in (128, 64):
            assert _lib.lib.bsi_hip_set_option(1, tile) == 0
            with torch.no_grad():
                got.append(layer(x.clone()))
    finally:
        _lib.lib.bsi_hip_set_option(1, 0)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("Q,R,stride", [(530, 8192, 8192), (281, 12483, 12490)])
def test_nothing_beside_the_outputs(ops, Q, R, stride):
    from bsipytorch_amd import _lib

    d, L = 3072, _lib.lib
    keys = ops.build_bsi_keys_cuda(torch.randn(R, d, device="cuda") * 0.02, 2, 0.5)[0]
    qb = ops.build_bsi_queries_cuda_batch_packed(torch.randn(Q, d, device="cuda"), 2, 0.5)
    out = torch.full((Q + 1, stride), float("nan"), device="cuda")
    rc = L.bsi_hip_dot(qb.words.data_ptr(), qb.ints8.data_ptr(), qb.chunk_scales.data_ptr(), d // 256, 7, d // 64, keys.ints8.data_ptr(),
                       _lib.LAYOUT_INT8, keys.slice_weights.data_ptr(), 6, R, Q, 1e-4, stride, out.data_ptr(), None, _lib.CORE_AUTO, None, 0,
                       torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert not torch.isnan(out[:Q, :R]).any() and torch.isnan(out[:Q, R:]).all() and torch.isnan(out[Q:]).all()
