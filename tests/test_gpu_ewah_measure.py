"""Flags, lengths, offsets and total of the one-call measuring passes against the separate ones and the oracle's streams, at
slice counts around the scan's runs and block."""
import numpy as np
import pytest
import torch

from test_gpu_parity import dev, hip, ops  # noqa: F401  (fixtures and helpers)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,W", [(1, 1), (3, 64), (7, 65), (63, 130), (1023, 3), (1024, 4), (1025, 5), (4099, 33)])
def test_measure_and_emit(hip, ops, oracle, S, W):
    rng = np.random.default_rng(S * 131 + W)
    words = rng.integers(0, 2**64, size=(S, W), dtype=np.uint64)
    words[rng.random((S, W)) < 0.5] = 0
    words[::3] = 0
    words[1::5] = 2**64 - 1
    flags = oracle.compress_flags(words, 0.4)
    want_words, want_off, want_len = oracle.ewah_encode(words, flags)[:3]
    got_words, got_off, got_len, got_flags = ops.ewah_compress_slices(dev(words), 0.4)
    np.testing.assert_array_equal(got_flags.cpu().numpy(), flags)
    np.testing.assert_array_equal(got_len.cpu().numpy(), want_len)
    np.testing.assert_array_equal(got_off.cpu().numpy(), want_off)
    np.testing.assert_array_equal(got_words.cpu().numpy().view(np.uint64), want_words)
