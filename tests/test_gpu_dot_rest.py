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


@pytest.mark.parametrize("Q,d,R,tile", [(3276, 8192, 4096, 256), (2555, 6144, 5120, 256), (1287, 5120, 9472, 256), (600, 4096, 8192, 128), (1100, 8192, 4096, 128),
                                        (768, 6150, 8192, 128)])
def test_the_tile_a_layer_takes_by_itself(ops, Q, d, R, tile):
    """Layers whose last round would be parts: where the integer sums cost less, and where they do not; the bits of small tiles, and the
    oracle's in tiles of the first and the last round."""
    import ctypes

    from bsipytorch_amd import _lib
    from bsipytorch_amd.linear import BSIQuantizedLinear
    from oracle import bsi_oracle

    plan, streamed = ctypes.c_int(), ctypes.c_int()
    _lib.check(_lib.lib.bsi_hip_linear_plan(Q, d, R, R, _lib.DTYPE_F32, ctypes.byref(plan), ctypes.byref(streamed)), "plan")
    n = -(-Q // 128) * -(-R // 128)
    assert plan.value == tile and 0 < n % 256 <= 128
    gen = torch.Generator(device="cuda").manual_seed(Q + R)
    dense = torch.nn.Linear(d, R, device="cuda")
    layer = BSIQuantizedLinear(dense, 2, 0.5)
    x = torch.randn(Q, d, generator=gen, device="cuda")
    x[:, torch.rand(d, generator=gen, device="cuda") < 0.001] *= 20.0
    got = []
    try:
        for option in (0, 64):
            assert _lib.lib.bsi_hip_set_option(1, option) == 0
            with torch.no_grad():
                got.append(layer(x.clone()))
    finally:
        _lib.lib.bsi_hip_set_option(1, 0)
    assert torch.equal(got[0], got[1])
    rows, keys = [0, 1, Q // 2, Q - 65, Q - 64, Q - 1], [0, 65, R // 2, R - 129, R - 65, R - 64, R - 1]
    qb = bsi_oracle.build_queries(x[rows].cpu().numpy())
    kb = bsi_oracle.build_keys(dense.weight.detach()[keys].cpu().numpy())
    want = bsi_oracle.dot_fixed(qb["words"], qb["scales"], kb["words"], kb["scales"], bsi_oracle.scale_inv(2, 2))[1]
    assert (got[0][rows][:, keys].cpu().numpy() == want + dense.bias.detach()[keys].cpu().numpy()).all()


@pytest.mark.parametrize("Q,d,R", [(530, 3072, 8192), (281, 3100, 12483), (768, 6150, 8190)])  # the last: a part past the last key
@pytest.mark.parametrize("tiled", [False, True])
def test_tiled_key_images_and_the_next_layers_keys(ops, Q, d, R, tiled):
    from bsipytorch_amd import _lib

    L = _lib.lib
    gen = torch.Generator(device="cuda").manual_seed(Q)
    keys = ops.build_bsi_keys_cuda(torch.randn(R, d, generator=gen, device="cuda") * 0.02, 2, 0.5)[0]
    x = torch.randn(Q, d, generator=gen, device="cuda")
    bias = torch.randn(R, generator=gen, device="cuda")
    ws = torch.empty(int(L.bsi_hip_linear_workspace_bytes(Q, d, 7)), dtype=torch.uint8, device="cuda")
    image, layout = keys.ints8, _lib.LAYOUT_INT8
    if tiled:  # blocks of 64 keys x 128 elements
        chunks = (d + 255) // 256
        padded = torch.zeros((R + 63) // 64 * 64, chunks * 256, dtype=torch.int8, device="cuda")
        padded[:R] = image.view(torch.int8).reshape(R, chunks * 256)
        image = padded.view(-1, 64, chunks * 2, 128).transpose(1, 2).contiguous()
        layout = _lib.LAYOUT_INT8_TILED

    def run(option, warm):
        out = torch.full((Q, R), float("nan"), device="cuda")
        assert L.bsi_hip_set_option(1, option) == 0
        try:
            rc = L.bsi_hip_linear_out(x.data_ptr(), _lib.DTYPE_F32, Q, d, 2, 7, 1, ws.data_ptr(), ws.numel(), image.data_ptr(), layout,
                                      keys.slice_weights.data_ptr(), 6, R, 1e-4, R, bias.data_ptr(), out.data_ptr(), _lib.DTYPE_F32, _lib.CORE_AUTO,
                                      image.data_ptr() if warm else None, image.numel() if warm else 0, torch.cuda.current_stream().cuda_stream)
        finally:
            L.bsi_hip_set_option(1, 0)
        assert rc == 0
        return out

    want = run(64, False)
    assert not torch.isnan(want).any()
    for warm in (False, True):
        assert torch.equal(run(128, warm), want)
