"""Calls whose threads do not fit one launch (2^32 threads)."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import philox

pytestmark = pytest.mark.gpu


def test_stream_bits(cuda):
    """More than 2^36 bits of a stream (a thread writes 16): the bits at both ends of every 2^35 and the last ones."""

    from hermespy_amd import _lib

    seed, drop, n = 77, 3, (1 << 36) + 37
    bits = torch.full((n,), 7, dtype=torch.uint8, device=cuda)
    _lib.check(_lib.load().hpx_stream_bits(ctypes.c_uint64(seed), drop, _lib.STREAM_BITS, n, _lib.ptr(bits),
                                           _lib.stream_handle()))
    assert int(bits[::4097].max()) <= 1
    for first in (0, (1 << 35) - 128, 1 << 35, (1 << 36) - 128, 1 << 36):
        counter = np.array([[drop, _lib.STREAM_BITS, first >> 7, 0]], dtype=np.uint32)
        words = philox.philox4x32(counter, philox.seed_key(seed)).reshape(-1)
        want = ((words[:, None] >> np.arange(32, dtype=np.uint32)) & 1).reshape(-1).astype(np.uint8)
        got = bits[first:first + 128].cpu().numpy()
        assert np.array_equal(got, want[:got.size])
