"""The key build of rows of over 16 chunks read with nontemporal loads: what the build of their parts, which are read plainly,
gives; rows that are read again (large magnitudes, more than 32 chunks) and rows whose last chunk is short among them."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,d,dtype", [(3301, 8192, torch.float32), (12800, 4160, torch.bfloat16), (6609, 8256, torch.float16), (6163, 4352, torch.float32)])
def test_same_as_its_parts(ops, R, d, dtype):
    gen = torch.Generator(device="cuda").manual_seed(R)
    w = torch.randn(R, d, generator=gen, device="cuda") * 0.02
    w[7] *= 300.0
    w[R - 1, d - 1] = 4.0e6 if dtype != torch.float16 else 60000.0
    w = w.to(dtype)
    assert w.numel() * w.element_size() >= 100 << 20
    whole = ops.build_bsi_keys_cuda(w, 2, 0.5)[0]
    half = R // 2 // 16 * 16
    parts = [ops.build_bsi_keys_cuda(p.contiguous(), 2, 0.5)[0] for p in (w[:half], w[half:])]
    for name in ("words", "ints8", "slice_weights", "shifts"):
        assert torch.equal(getattr(whole, name), torch.cat([getattr(p, name) for p in parts])), name
