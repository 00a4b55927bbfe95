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


def test_lmmse_rows(cuda):
    """2^24 tiles of 64 rows, one pilot and one element: every row is the product of its value and the filter's (a
    complex product in float32: each part within two roundings of its terms)."""

    from hermespy_amd import _lib

    rows, nt = 1 << 28, 4
    g = torch.Generator(device=cuda).manual_seed(9)
    ls = torch.view_as_complex(torch.randn(nt, rows, 2, generator=g, device=cuda))
    filt = torch.view_as_complex(torch.randn(nt, 1, 1, 2, generator=g, device=cuda))
    index = torch.arange(rows, dtype=torch.int32, device=cuda)
    est = torch.full((nt, rows), complex("nan"), dtype=torch.complex64, device=cuda)
    _lib.check(_lib.load().hpx_lmmse_apply(_lib.ptr(ls), nt, rows, 1, _lib.ptr(filt), 1, _lib.ptr(index), rows, _lib.ptr(est),
                                           _lib.stream_handle()))
    for t in range(nt):
        for part in range(0, rows, rows // 8):
            x, got = ls[t, part:part + rows // 8], est[t, part:part + rows // 8]
            error = torch.view_as_real(got - x * filt[t, 0, 0]).abs().amax(dim=-1)
            assert bool((error <= 4 * 2.0**-24 * 2 * x.abs() * filt[t, 0, 0].abs()).all())


# 256 threads a drop, and the library's choice for a launch that fills the GPU many times over
@pytest.mark.parametrize("workgroup,drops", [(256, (1 << 24) + 1000), (0, (1 << 25) + 1000)])
def test_drops(cuda, workgroup, drops):
    """The drops at both ends of a launch of 2^32 threads and more are those of launches of their own."""

    import dataclasses

    from hermespy_amd.configs import siso_64
    from hermespy_amd.simulation import BatchedLink

    link = BatchedLink(dataclasses.replace(siso_64(), workgroup_size=workgroup))
    noise = torch.full((drops,), 0.1, dtype=torch.float64, device=cuda)
    errors = torch.full((drops,), -1, dtype=torch.int32, device=cuda)
    link.run(11, 0, noise, errors)
    assert int(errors.min()) >= 0
    for first in (0, (1 << 24) - 500, drops - 1000):
        alone = torch.full((1000,), -1, dtype=torch.int32, device=cuda)
        link.run(11, first, noise[:1000].contiguous(), alone)
        assert torch.equal(alone, errors[first:first + 1000])
