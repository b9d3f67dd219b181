"""What a hybrid batch asks of the allocator: the streams' own bytes, and besides them, while the call runs, the planes and what the
lengths come in.  (Bytes asked for: what a request is given depends on the blocks that earlier tests have left, up to 1 MiB more.)"""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


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
    before = torch.cuda.memory_stats()["requested_bytes.all.current"]
    held = ops.build_bsi_queries_cuda_batch_hybrid(x, 2, 0.5)
    S, streams = Q * held.Sa, held.comp_words.numel() * 8
    small = S * (8 + 4 + 4) + Q * (d // 256) * 4  # offsets, lengths, flags; scales
    stats = torch.cuda.memory_stats()
    assert stats["requested_bytes.all.current"] - before <= streams + small
    assert stats["requested_bytes.all.peak"] - before <= streams + small + S * held.W * 8
