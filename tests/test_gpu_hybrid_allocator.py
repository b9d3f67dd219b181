"""What a hybrid batch takes of the allocator: the streams' own bytes, in its granularity, and besides them, while the call runs, the
planes and what the lengths come in."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


def rounded(nbytes):
    return (nbytes + 511) // 512 * 512


@pytest.mark.parametrize("kind", ["normal", "relu", "zeros", "first tenth"])
@pytest.mark.parametrize("Q, d", [(64, 2048), (300, 4096)])
def test_bytes_kept_and_bytes_at_most(ops, kind, Q, d):
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(Q, d, generator=gen, device="cuda")
    if kind == "relu":
        x = x.relu()
    elif kind == "zeros":
        x.zero_()
    elif kind == "first tenth":
        x[Q // 10:] = 0
    held = ops.build_bsi_queries_cuda_batch_hybrid(x, 2, 0.5)  # what is made once: flags, constants
    del held
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    held = ops.build_bsi_queries_cuda_batch_hybrid(x, 2, 0.5)
    S = Q * held.Sa
    small = 3 * rounded(S * 8) + rounded(Q * (d + 255) // 256 * 4 + 4) + 512  # offsets, lengths, flags, scales
    streams = rounded(held.comp_words.numel() * 8)
    kept, most = torch.cuda.memory_allocated() - before, torch.cuda.max_memory_allocated() - before
    assert kept <= streams + small
    assert most <= streams + small + rounded(S * held.W * 8)
