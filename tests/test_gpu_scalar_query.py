"""One query against prebuilt decimal keys on the device-resident route: scores equal to the oracle's exact ones and bytes
equal to the batched builder's, at the edges of its lane groups, LDS staging and slice counts."""
import numpy as np
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,R,scale,negative", [(1, 1, 1.0, True), (63, 5, 1.0, True), (1024, 17, 1.0, False), (1025, 3, 1.0, True),
                                                (2048, 300, 1.0, True), (2049, 33, 1.0, True), (4096, 65, 30.0, True),
                                                (16384, 9, 1.0, True), (300, 7, 2.0e5, True), (16384, 3, 3.0e4, False),
                                                (64, 4, 1.0e12, True), (128, 3, 0.0, True)])
def test_scores_and_bytes(ops, oracle, d, R, scale, negative):
    from bsipytorch_amd import bsi_scalar

    rng = np.random.default_rng(d + R)
    q = (rng.standard_normal(d) * scale).astype(np.float32)
    q = q if negative else np.abs(q)
    # keys small enough that the exact sums stay below 2^53
    K = np.round(rng.standard_normal((R, d)) * (3.0 if scale < 1e6 else 0.02), 2).astype(np.float32)
    K[0] = np.abs(K[0])
    cap = ops.build_bsi_keys(torch.from_numpy(K), 2, 0.3)[0]
    out, total, build_ns, dot_ns, nbytes = ops.batch_dot_product_prebuilt(torch.from_numpy(q).cuda(), cap, 0.4)
    assert out.dtype == torch.float64 and out.device.type == "cpu" and total == build_ns + dot_ns and build_ns > 0 and dot_ns > 0
    np.testing.assert_array_equal(out.numpy(), oracle.scalar_batch_dot_product(q, K, 2))
    sliced = bsi_scalar._Sliced(bsi_scalar._ints_round(torch.from_numpy(q).cuda().unsqueeze(0), 2), 0.4)
    assert nbytes == sliced.mem_bytes()
    raw, _ = bsi_scalar._raw_dot(sliced, cap.sliced)
    assert torch.equal(out, raw[0].cpu() / 1e4)
