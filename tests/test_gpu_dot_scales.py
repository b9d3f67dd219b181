"""Chunk scales of the int8-image dot fetched four chunks at a time: row lengths around the rule's edge and around the groups,
ragged edges, every tile, against the oracle; scales that differ from chunk to chunk and from row to row."""
import numpy as np
import pytest
import torch

from oracle import bsi_oracle
from test_gpu_parity import hip, ops  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [15, 16, 17, 18, 19, 20, 33])
@pytest.mark.parametrize("Q,R", [(33, 70), (128, 130), (129, 192)])
def test_outputs_are_the_oracles(hip, ops, Q, R, chunks):
    gen = torch.Generator(device="cuda").manual_seed(Q * chunks + R)
    d = chunks * 256
    x = torch.randn(Q, d, generator=gen, device="cuda") * torch.exp(2 * torch.randn(Q, chunks, generator=gen, device="cuda")).repeat_interleave(256, 1)
    w = torch.randn(R, d, generator=gen, device="cuda") * 0.02
    keys = ops.build_bsi_keys_cuda(w, 2, 0.5)[0]
    queries = ops.build_bsi_queries_cuda_batch_packed(x, 2, 0.5)
    qb, kb = bsi_oracle.build_queries(x.cpu().numpy()), bsi_oracle.build_keys(w.cpu().numpy())
    want = bsi_oracle.dot_fixed(qb["words"], qb["scales"], kb["words"], kb["scales"], bsi_oracle.scale_inv(2, 2))[1]
    for tile in (0, 128, 12864, 64, 6432):
        hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, tile), "tile")
        try:
            got = ops.batch_dot_product_multiquery_cuda_batch_caps(queries, keys)[0].cpu().numpy()
        finally:
            hip.check(hip.lib.bsi_hip_set_option(hip.OPT_I8_TILE, 0), "tile")
        assert np.array_equal(got, want), tile
