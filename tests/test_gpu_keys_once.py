"""The key build of matrices read with nontemporal loads (large ones of whole lines): what the build of their parts, which are
read plainly, gives; rows with magnitudes that are read again among them."""
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,d,dtype", [(10240, 4096, torch.bfloat16), (20485, 2048, torch.float16), (5125, 4096, torch.float32), (21000, 1024, torch.float32)])
def test_same_as_its_parts(ops, R, d, dtype):
    gen = torch.Generator(device="cuda").manual_seed(R)
    w = torch.randn(R, d, generator=gen, device="cuda") * 0.02
    w[7] *= 300.0
    w[R - 1, 5] = 4.0e6 if dtype != torch.float16 else 60000.0
    w = w.to(dtype)
    assert w.numel() * w.element_size() >= 80 << 20
    whole = ops.build_bsi_keys_cuda(w, 2, 0.5)[0]
    half = R // 2 // 16 * 16
    parts = [ops.build_bsi_keys_cuda(p.contiguous(), 2, 0.5)[0] for p in (w[:half], w[half:])]
    for name in ("words", "ints8", "slice_weights", "shifts"):
        assert torch.equal(getattr(whole, name), torch.cat([getattr(p, name) for p in parts])), name
