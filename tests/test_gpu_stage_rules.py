"""Stage kernels on both sides of the rules that choose their workgroups by size, against float64."""

import numpy as np
import pytest
import torch

from conftest import rel_err

pytestmark = pytest.mark.gpu


def _terms(rng, paths, terms):
    return np.stack([rng.uniform(-2e-4, 2e-4, (paths, terms)), rng.uniform(-np.pi, np.pi, (paths, terms)),
                     rng.uniform(0.1, 1.0, (paths, terms)) / np.sqrt(paths * terms)], axis=-1)


# 1024 workgroups in all: words in as many shares as their subcarriers make, in fewer, and whole; terms side by side and in turn
@pytest.mark.parametrize("paths,terms,n,words", [(5, 21, 1024, 200), (5, 21, 4096, 300), (80, 21, 2048, 400), (80, 21, 512, 1030)])
def test_ideal_csi_of_many_words(cuda, paths, terms, n, words):
    from hermespy_amd import _lib

    rng = np.random.default_rng(words)
    cp = n // 4
    sos, delays = _terms(rng, paths, terms), rng.integers(0, cp + 1, paths).astype(np.int32)
    out = torch.full((words, n), float("nan"), dtype=torch.complex64, device=cuda)
    dev = [torch.as_tensor(v, device=cuda) for v in (sos, delays, np.ones(1, np.complex64))]
    _lib.check(_lib.load().hpx_ideal_csi(_lib.ptr(dev[0]), paths, terms, _lib.ptr(dev[1]), cp + 1, _lib.ptr(dev[2]), 1, 1,
                                         words, n, cp, 0, _lib.ptr(out), _lib.stream_handle()))
    assert bool(torch.isfinite(torch.view_as_real(out)).all())
    some = np.array([0, 1, words // 2, words - 1])
    m = some[:, None] * (n + cp) + cp + np.arange(n)
    h = np.stack([(sos[p, :, 2, None, None] * np.exp(1j * (sos[p, :, 0, None, None] * m + sos[p, :, 1, None, None]))).sum(0)
                  for p in range(paths)]).mean(axis=2)
    bins = (np.arange(n) - n // 2) % n
    c = np.einsum("pw,pk->wk", h, np.exp(-2j * np.pi * np.outer(delays, bins) / n))
    # float32 sums of at most 80 paths
    assert rel_err(out[torch.as_tensor(some, device=cuda)].cpu().numpy(), c) < 1e-5


# the window of x in LDS: few workgroups and many paths, some, and 4096 (little reuse; a large window of many paths);
# through memory beside each; samples before the frame and after it, Taylor blocks and (a high rate) direct taps
@pytest.mark.parametrize("ntx,paths,m,maxd,rate", [(8, 6, 700, 30, 1e-5), (8, 6, 700, 600, 1e-5), (2, 16, 513, 37, 0.2),
                                                   (4, 3, 1 << 18, 0, 1e-5), (1, 12, 1 << 18, 500, 1e-5),
                                                   (1, 2, 1 << 20, 90, 1e-5), (1, 2, 1 << 20, 300, 1e-5),
                                                   (8, 8, 1 << 20, 64, 1e-5), (5, 9, 1 << 20, 300, 1e-5)])
def test_tdl_window(cuda, ntx, paths, m, maxd, rate):
    from hermespy_amd import _lib

    rng = np.random.default_rng(m + paths)
    terms, nrx = 9, 2
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
    want = torch.zeros((nrx, m + maxd), dtype=torch.complex128, device=cuda)
    n = torch.arange(m, device=cuda, dtype=torch.float64)
    for p in range(paths):
        h = torch.zeros(m, dtype=torch.complex128, device=cuda)
        for rate_k, phase, amp in sos[p]:
            h += amp * torch.exp(1j * (rate_k * n + phase))
        want[:, delays[p]:delays[p] + m] += ds.to(torch.complex128) @ (h * dx.to(torch.complex128))
    assert rel_err(y.cpu().numpy(), want.cpu().numpy()) < 1e-5
