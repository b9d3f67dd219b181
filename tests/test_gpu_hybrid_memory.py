"""The streams of a hybrid batch: the tensors hold what the streams need and no more, call after call, whatever share of the batch
compresses."""
import io

import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kept", [0.0, 0.02, 0.5, 1.0])
def test_streams_own_their_bytes(ops, kept):
    from bsipytorch_amd import _native

    gen = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn(40, 4096, generator=gen, device="cuda")
    x *= (torch.arange(4096, device="cuda") < kept * 4096)
    ops._flags()
    again = []
    for _ in range(3):  # the memory of one call is the next one's
        streams, off, lens, flags, scales, _ = _native.hybrid(x, 2, 0.5)
        again.append((streams, off, lens))
    b = ops._build_query_batch(x, 2, want_ints8=False)
    want = ops.ewah_compress_slices(b.words.view(-1, b.words.shape[2]), 0.5)
    for streams, off, lens in again:
        assert torch.equal(streams, want[0]) and torch.equal(off, want[1]) and torch.equal(lens, want[2])
        assert streams.is_contiguous() and streams.untyped_storage().nbytes() == streams.numel() * 8
    file = io.BytesIO()
    torch.save(streams, file)
    assert len(file.getvalue()) < streams.numel() * 8 + 4096
