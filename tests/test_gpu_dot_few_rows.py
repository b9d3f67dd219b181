"""The dot of few query rows on an image with its rows one after the other, which the kernel turns round on the way in: row counts
around its groups of 8 and 16 rows, one chunk, fewer chunks than waves, chunks in one pass and in several, one and two key tiles a
workgroup, chunk and row scales, against the oracle on the first and last keys."""
import numpy as np
import pytest
import torch

from oracle import bsi_oracle
from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q", [1, 7, 8, 9, 15, 16, 17, 25, 32])
@pytest.mark.parametrize("d,R", [(256, 40), (8 * 256, 100), (65 * 256, 48), (57 * 256, 4112), (33 * 256, 4112), (300, 4100), (1600, 70),
                                 (3 * 256, 16400), (33 * 256, 16400), (200, 16384)])
def test_outputs_are_the_oracles(ops, Q, d, R):
    gen = torch.Generator(device="cuda").manual_seed(Q * d + R)
    x = torch.randn(Q, d, generator=gen, device="cuda") * torch.exp(torch.randn(Q, 1, generator=gen, device="cuda"))
    x *= torch.exp(torch.randn((d + 255) // 256, generator=gen, device="cuda")).repeat_interleave(256)[:d]
    w = torch.randn(R, d, generator=gen, device="cuda") * 0.02
    keys = ops.build_bsi_keys_cuda(w, 2, 0.5)[0]
    queries = ops.build_bsi_queries_cuda_batch_packed(x, 2, 0.5)
    got = ops.batch_dot_product_multiquery_cuda_batch_caps(queries, keys)[0].cpu().numpy()
    some = np.r_[0:20, R - 20:R]
    qb, kb = bsi_oracle.build_queries(x.cpu().numpy()), bsi_oracle.build_keys(w.cpu().numpy()[some])
    want = bsi_oracle.dot_fixed(qb["words"], qb["scales"], kb["words"], kb["scales"], bsi_oracle.scale_inv(2, 2))[1]
    assert np.array_equal(got[:, some], want)
