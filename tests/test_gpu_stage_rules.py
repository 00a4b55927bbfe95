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
