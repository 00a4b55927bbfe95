"""Both paths of the stage kernels that choose one by size or alignment, at the edges of their pieces."""

import numpy as np
import pytest
import torch

from conftest import rel_err
from oracle import philox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 129, 4096, 5003])
@pytest.mark.parametrize("offset", [0, 1, 16])
def test_stream_bits(cuda, n, offset):
    from hermespy_amd import _lib

    out = torch.full((n + offset + 32,), 7, dtype=torch.uint8, device=cuda)
    _lib.check(_lib.load().hpx_stream_bits(20261202, 17, _lib.STREAM_BITS + 2, n, _lib.ptr(out[offset:]), _lib.stream_handle()))
    got = out.cpu().numpy()
    assert np.array_equal(got[offset:offset + n], philox.stream_bits(20261202, 17, 2, n).astype(np.uint8))
    assert (got[:offset] == 7).all() and (got[offset + n:] == 7).all()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4099, 1 << 20])
@pytest.mark.parametrize("offsets", [(0, 0), (4, 0), (1, 0), (16, 4)])
def test_count_errors(cuda, n, offsets):
    from hermespy_amd import _lib

    rng = np.random.default_rng(n)
    a, b = (rng.integers(0, 2, n + o).astype(np.uint8) for o in offsets)
    ta, tb = (torch.as_tensor(v, device=cuda) for v in (a, b))
    acc = torch.full((1,), 5, dtype=torch.int64, device=cuda)
    _lib.check(_lib.load().hpx_count_errors(_lib.ptr(ta[offsets[0]:]), _lib.ptr(tb[offsets[1]:]), n, _lib.ptr(acc),
                                            _lib.stream_handle()))
    assert int(acc.item()) == 5 + int(np.sum(a[offsets[0]:] != b[offsets[1]:]))


def _terms(rng, paths, terms):
    """(rate, phase, amplitude) of every term; some without amplitude."""

    sos = np.stack([rng.uniform(-2e-4, 2e-4, (paths, terms)), rng.uniform(-np.pi, np.pi, (paths, terms)),
                    rng.uniform(0.1, 1.0, (paths, terms)) / np.sqrt(paths * terms)], axis=-1)
    sos[0, 0, 2] = 0.0
    return sos


# the terms side by side (at most 1536 of them, and room in LDS) and in turn; fewer and more subcarriers than threads
@pytest.mark.parametrize("paths,terms,n,words", [(1, 1, 2, 1), (73, 21, 64, 2), (74, 21, 512, 2), (16, 21, 1024, 3),
                                                 (70, 21, 4096, 1), (5, 400, 256, 1)])
def test_ideal_csi(cuda, paths, terms, n, words):
    from hermespy_amd import _lib

    rng = np.random.default_rng(paths + n)
    cp = n // 4
    sos, delays = _terms(rng, paths, terms), rng.integers(0, cp + 1, paths).astype(np.int32)
    s = rng.standard_normal((2, 1)) + 1j * rng.standard_normal((2, 1))
    out = torch.full((2, 1, words, n), float("nan"), dtype=torch.complex64, device=cuda)
    dev = [torch.as_tensor(v, device=cuda) for v in (sos, delays, s.astype(np.complex64))]
    _lib.check(_lib.load().hpx_ideal_csi(_lib.ptr(dev[0]), paths, terms, _lib.ptr(dev[1]), cp + 1, _lib.ptr(dev[2]), 2, 1,
                                         words, n, cp, 0, _lib.ptr(out), _lib.stream_handle()))
    m = np.arange(words)[:, None] * (n + cp) + cp + np.arange(n)
    h = np.stack([(sos[p, :, 2, None, None] * np.exp(1j * (sos[p, :, 0, None, None] * m + sos[p, :, 1, None, None]))).sum(0)
                  for p in range(paths)]).mean(axis=2)  # (paths, words)
    bins = (np.arange(n) - n // 2) % n
    c = np.einsum("pw,pk->wk", h, np.exp(-2j * np.pi * np.outer(delays, bins) / n))
    # float32 sums of at most 74 paths and one product
    assert rel_err(out.cpu().numpy(), s[:, :, None, None] * c) < 1e-5


# the window of x in LDS and out of it (8 antennas of more than 64 KB; 2000 samples of delay), samples before the
# frame and after it, Taylor blocks and (a high rate) direct taps
@pytest.mark.parametrize("ntx,m,maxd,rate", [(1, 1, 0, 1e-5), (4, 300, 37, 1e-5), (8, 700, 800, 1e-5), (2, 5000, 2000, 1e-5),
                                             (3, 513, 20, 0.2)])
def test_tdl_propagate(cuda, ntx, m, maxd, rate):
    from hermespy_amd import _lib

    rng = np.random.default_rng(m)
    paths, terms, nrx = 6, 9, 2
    sos = _terms(rng, paths, terms)
    sos[..., 0] *= rate / 2e-4
    delays = rng.integers(0, maxd + 1, paths).astype(np.int32)
    delays[-1] = maxd
    x = (rng.standard_normal((ntx, m)) + 1j * rng.standard_normal((ntx, m))).astype(np.complex64)
    s = (rng.standard_normal((nrx, ntx)) + 1j * rng.standard_normal((nrx, ntx))).astype(np.complex64)
    y = torch.full((nrx, m + maxd), float("nan"), dtype=torch.complex64, device=cuda)
    dx, dsos, dd, ds = (torch.as_tensor(v, device=cuda) for v in (x, sos, delays, s))
    _lib.check(_lib.load().hpx_tdl_propagate(_lib.ptr(dx), ntx, m, m, _lib.ptr(dsos), paths, terms, rate, _lib.ptr(dd), maxd,
                                             _lib.ptr(ds), nrx, _lib.ptr(y), m + maxd, _lib.stream_handle()))
    want = np.zeros((nrx, m + maxd), complex)
    for p in range(paths):
        h = (sos[p, :, 2, None] * np.exp(1j * (sos[p, :, 0, None] * np.arange(m) + sos[p, :, 1, None]))).sum(0)
        want[:, delays[p]:delays[p] + m] += s.astype(complex) @ (h * x)
    assert rel_err(y.cpu().numpy(), want) < 1e-5
