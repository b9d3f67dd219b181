"""The build that measures its streams, asked for the lengths of slices and of rows, and the stream decoder where a block of literals
ends inside, at and beyond the window of 64 words that it holds."""
import numpy as np
import pytest
import torch

from test_gpu_parity import dev, hip, ops  # noqa: F401  (fixtures and helpers)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,d,bits", [(1, 64, 2), (3, 300, 7), (65, 512, 8), (2, 65536, 7)])
def test_lengths_of_slices_and_of_rows(ops, Q, d, bits):
    from bsipytorch_amd import _lib

    x = torch.randn(Q, d, generator=torch.Generator(device="cuda").manual_seed(Q), device="cuda")
    x[:, d // 3:] = 0
    W, chunks = (d + 63) // 64, (d + 255) // 256
    chunked, got = W % 4 == 0, []
    for entry, n in ((_lib.lib.bsi_hip_build_measure, Q * bits), (_lib.lib.bsi_hip_build_measure_rows, Q)):
        words = torch.zeros(Q * bits, W, dtype=torch.int64, device="cuda")
        scales = torch.zeros(Q * chunks, device="cuda")
        weights = torch.zeros(Q * bits, device="cuda")
        flags, lens = (torch.zeros(Q * bits, dtype=torch.int32, device="cuda") for _ in range(2))
        host = torch.full((n,), -1, dtype=torch.int32, pin_memory=True)
        rc = entry(x.data_ptr(), _lib.DTYPE_F32, Q, d, 2, bits, int(chunked), 0.5, words.data_ptr(), scales.data_ptr(), weights.data_ptr(),
                   flags.data_ptr(), lens.data_ptr(), host.data_ptr(), torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        torch.cuda.synchronize()
        got.append([t.cpu() for t in (words, scales, weights, flags, lens)] + [host.clone()])
    for a, b in zip(got[0][:5], got[1][:5]):
        assert torch.equal(a, b)
    assert torch.equal(got[0][5], got[0][4]) and torch.equal(got[1][5], got[0][4].view(Q, bits).sum(1, dtype=torch.int32))


@pytest.mark.parametrize("W", [1, 62, 63, 64, 65, 127, 128, 190])
def test_literals_around_the_window(ops, W):
    rng = np.random.default_rng(W)
    words = rng.integers(1, 2**63, size=(6, W), dtype=np.uint64)
    words[1, : W // 2] = 0            # a run, then literals
    words[2, W // 3:] = 2**64 - 1     # literals, then a run
    words[3, ::2] = 0                 # a marker every other word
    words[4, max(0, W - 64):] = 0
    words[5] = 0
    comp, off, lens, _ = ops.ewah_compress_slices(dev(words), 1.0)  # all of them run-length coded
    out = torch.empty(6, W, dtype=torch.int64, device="cuda")
    from bsipytorch_amd import _lib

    assert _lib.lib.bsi_hip_ewah_decompress_batch(comp.data_ptr(), off.data_ptr(), lens.data_ptr(), 6, W, out.data_ptr(),
                                                  torch.cuda.current_stream().cuda_stream) == 0
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint64), words)


@pytest.mark.parametrize("Q,d,R", [(8, 2048, 300), (9, 2048, 300), (16, 1600, 77), (17, 257, 40), (32, 2048, 130), (3, 8192, 50), (4, 8192, 50)])
def test_decode_inside_the_dot_and_ahead_of_it(ops, Q, d, R):
    from bsipytorch_amd import _lib

    gen = torch.Generator(device="cuda").manual_seed(Q + d)
    x = torch.randn(Q, d, generator=gen, device="cuda").relu()
    keys = ops.build_bsi_keys_cuda(torch.randn(R, d, generator=gen, device="cuda") * 0.02, 2, 0.5)[0]
    h = ops.build_bsi_queries_cuda_batch_hybrid(x, 2, 0.5)
    planes, layout = keys.words, keys.layout
    assert layout == _lib.LAYOUT_TILED16
    scales = h.chunk_scales if h.chunk_scales is not None else h.row_scales
    stride = scales.shape[1] if h.chunk_scales is not None else 1
    need, got = int(_lib.lib.bsi_hip_dot_ewah_batch_workspace_bytes(Q, h.W)), []
    for size in (0, need):
        ws = torch.empty(max(size, 16), dtype=torch.uint8, device="cuda")
        out = torch.full((Q, R), float("nan"), device="cuda")
        rc = _lib.lib.bsi_hip_dot_ewah_batch(h.comp_words.data_ptr(), h.comp_off.data_ptr(), h.comp_len.data_ptr(), h.Sa, h.W, scales.data_ptr(),
                                             stride, planes.data_ptr(), layout, keys.slice_weights.data_ptr(), 6, R, Q, float(np.float32(1e-4)),
                                             R, None, out.data_ptr(), None, ws.data_ptr() if size else None, size,
                                             torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        got.append(out.cpu())
    assert torch.equal(got[0], got[1])
    assert torch.equal(got[0], ops.batch_dot_product_multiquery_cuda_batch_caps(h, keys)[0].cpu())
