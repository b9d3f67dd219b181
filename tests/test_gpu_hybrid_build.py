"""The query build that measures its streams: same streams, offsets, scales and weights as the build and the codec's own
passes, at the edges of its chunks, held registers, row scales and the emit pass's groups."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,d,threshold", [(1, 1, 0.5), (1, 256, 0.5), (3, 2048, 0.0), (5, 2047, 1.0), (9, 8192, 0.5), (2, 8448, 0.5),
                                           (3, 8500, 0.4), (7, 1600, 0.5), (300, 512, 0.5), (1170, 300, 0.5), (1, 65536, 0.5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_same_as_build_and_encode(ops, Q, d, threshold, dtype):
    from bsipytorch_amd import _native

    gen = torch.Generator(device="cuda").manual_seed(Q + d)
    x = torch.randn(Q, d, generator=gen, device="cuda").to(dtype)
    x[::2] = x[::2].relu()
    x[0, : d // 2] = 0
    if Q > 2:
        x[1] *= 3.0e6  # beyond the float32 quantiser
    ops._flags()
    got = _native.hybrid(x, 2, threshold)
    assert got is not None
    streams, off, lens, flags, scales, weights = got
    b = ops._build_query_batch(x, 2, want_ints8=False)
    want = ops.ewah_compress_slices(b.words.view(-1, b.words.shape[2]), threshold)
    for mine, theirs in zip((streams, off, lens, flags), want):
        assert torch.equal(mine, theirs)
    if weights is None:
        assert torch.equal(scales, b.chunk_scales)
    else:
        assert torch.equal(scales, b.row_scales) and torch.equal(weights, b.slice_weights)
    h = ops.build_bsi_queries_cuda_batch_hybrid(x, 2, threshold)
    assert torch.equal(h.comp_words, streams) and torch.equal(h.slice_weights, b.slice_weights)


def test_beyond_its_limits(ops):
    from bsipytorch_amd import _native

    ops._flags()
    for shape in ((1171, 64), (1, 65537)):
        x = torch.randn(*shape, device="cuda")
        assert _native.hybrid(x, 2, 0.5) is None
        h = ops.build_bsi_queries_cuda_batch_hybrid(x, 2, 0.5)
        assert h.comp_words.numel() == int(h.comp_len.sum())
