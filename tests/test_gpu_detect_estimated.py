"""Detection on estimated channels over its shares of a drop, frames with and without references, rows shorter
and longer than the workgroup, and bits in LDS and drawn per element."""

import numpy as np
import pytest
import torch

from conftest import rel_err
from oracle import mapping, philox

pytestmark = pytest.mark.gpu

SEED = 20261202


# (drops, Nrx, Ntx, words, N, order, references): one share of a word each, shares of several words, one share a
# drop (513 drops); rows of 16, 300 and 512 subcarriers; 128 KB of bits a word (drawn per element)
@pytest.mark.parametrize("drops,nr,nt,words,n,order,refs", [
    (1, 2, 2, 14, 512, 16, True), (2, 4, 4, 37, 16, 256, False), (200, 1, 1, 7, 64, 4, True), (513, 2, 1, 3, 64, 64, True),
    (3, 8, 8, 2, 300, 64, True), (1, 4, 4, 2, 32768, 256, False), (2, 3, 2, 5, 300, 16, False)])
def test_detect_estimated(cuda, drops, nr, nt, words, n, order, refs):
    from hermespy_amd import _lib

    rng = np.random.default_rng(drops + n)
    bps = int(np.log2(order))
    mask = rng.random((words, n)) < (0.8 if refs else 1.1)
    num_data = int(mask.sum())
    elements = np.where(mask, np.cumsum(mask, axis=1) - 1, -1).astype(np.int32)
    word_data = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int32)

    def normal(*shape):
        return ((rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / np.sqrt(2)).astype(np.complex64)

    h = normal(nt, drops, nr, words * n) + np.eye(nr, nt, dtype=np.complex64).T[:, None, :, None] * 3
    y = normal(drops, nr, words * n) * 2
    noise = rng.uniform(0.05, 0.2, drops)
    dev = [torch.as_tensor(v, device=cuda) for v in (y, h, noise, elements, word_data)]
    err = torch.full((drops,), -7, dtype=torch.int32, device=cuda)
    eq = torch.full((drops, nt, num_data), float("nan"), dtype=torch.complex64, device=cuda)
    _lib.check(_lib.load().hpx_detect_estimated(
        _lib.ptr(dev[0]), _lib.ptr(dev[1]), drops, nr, nt, words, n, _lib.ptr(dev[3]) if refs else None,
        _lib.ptr(dev[4]) if refs else None, num_data, order, _lib.HPX_DETECT_MMSE, _lib.ptr(dev[2]), SEED, 40, _lib.ptr(err),
        _lib.ptr(eq), _lib.stream_handle()))
    got, err = eq.cpu().numpy(), err.cpu().numpy()
    hd = h.astype(complex)[..., mask.reshape(-1)].transpose(1, 3, 2, 0)  # (drops, K, Nrx, Ntx)
    yd = y.astype(complex)[..., mask.reshape(-1)].transpose(0, 2, 1)[..., None]
    hh = hd.conj().swapaxes(-1, -2)
    want = np.linalg.solve(hh @ hd + noise[:, None, None, None] * np.eye(nt), hh @ yd)[..., 0].transpose(0, 2, 1)
    # float32 normal equations with one refinement step, condition numbers of a few hundred
    assert rel_err(got, want) < 1e-5
    for d in range(min(drops, 5)):
        tx = np.stack([philox.stream_bits(SEED, 40 + d, t, num_data * bps) for t in range(nt)])
        rx = np.stack([mapping.detect_bits(got[d, t].astype(complex), order).astype(np.uint8) for t in range(nt)])
        assert int(err[d]) == int(np.sum(tx != rx))
