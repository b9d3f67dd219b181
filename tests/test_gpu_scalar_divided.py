"""Scores divided on the GPU: the float64 quotients that the host's division gives, for divisors that divide nothing evenly."""
import numpy as np
import pytest
import torch

from test_gpu_parity import ops  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("divisor", [1e4, 3.0, 7.1e-9, 1.7e300, -1e2])
@pytest.mark.parametrize("d,R", [(300, 1), (257, 4200), (2048, 1000)])
def test_quotients(ops, divisor, d, R):
    from bsipytorch_amd import _native

    gen = torch.Generator(device="cuda").manual_seed(R)
    keys = ops.build_bsi_keys(torch.randn(R, d, generator=gen, device="cuda"), 2, 0.5)[0].sliced
    x = torch.randn(d, generator=gen, device="cuda")
    whole = _native.scalar_query(x, keys.words, keys.weights, 2, 0.5, 1.0)[0].numpy()
    assert np.array_equal(whole, np.round(whole)) and np.abs(whole).max() > 0
    got = _native.scalar_query(x, keys.words, keys.weights, 2, 0.5, divisor)[0].numpy()
    np.testing.assert_array_equal(got.view(np.int64), (whole / divisor).view(np.int64))
