"""The LMMSE interpolation kernel at the edges of its tiles, against a complex128 product of the same operands."""

import ctypes

import numpy as np
import pytest
import torch

from conftest import rel_err

pytestmark = pytest.mark.gpu

# (streams, rows, pilots, elements, rows per set): tiles of 64 rows x 128 elements and chunks of 32 pilots, one
# less, one more and far less; odd pilot counts (no 16-byte rows); empty sets; more sets than a launch takes
SHAPES = [(1, 1, 1, 1, [1]), (2, 70, 128, 300, [64, 0, 6]), (1, 200, 31, 127, [65, 63, 1]), (2, 129, 33, 129, [129]),
          (1, 40, 32, 128, [0, 40]), (3, 66, 64, 257, [3] * 20), (1, 64, 130, 640, [64])]


@pytest.mark.parametrize("tx,rows,pilots,elements,counts", SHAPES)
def test_lmmse_sets_match_complex128(cuda, tx, rows, pilots, elements, counts):
    from hermespy_amd import _lib

    lib, st = _lib.load(), _lib.stream_handle()
    g = torch.Generator(device=cuda).manual_seed(rows + pilots)
    c64 = lambda *s: torch.view_as_complex(torch.randn(*s, 2, generator=g, device=cuda))
    ls, filt = c64(tx, rows, pilots), c64(len(counts), tx, elements, pilots)
    order = torch.randperm(rows, generator=g, device=cuda).to(torch.int32)
    lists = [r.contiguous() for r in torch.split(order, counts + [rows - sum(counts)])][: len(counts)]
    est = torch.full((tx, rows, elements), complex(7.0, 7.0), dtype=torch.complex64, device=cuda)
    ptrs = (ctypes.c_void_p * len(counts))(*[r.data_ptr() if r.numel() else None for r in lists])
    num = (ctypes.c_int32 * len(counts))(*counts)
    _lib.check(lib.hpx_lmmse_apply_sets(_lib.ptr(ls), tx, rows, pilots, _lib.ptr(filt), elements, len(counts),
                                        ctypes.addressof(ptrs), ctypes.addressof(num), _lib.ptr(est), st))
    one = torch.full_like(est, complex(7.0, 7.0))
    for i, r in enumerate(lists):
        _lib.check(lib.hpx_lmmse_apply(_lib.ptr(ls), tx, rows, pilots, _lib.ptr(filt[i]), elements, _lib.ptr(r),
                                       r.numel(), _lib.ptr(one), st))
    assert torch.equal(torch.view_as_real(est), torch.view_as_real(one))
    want = torch.full((tx, rows, elements), complex(7.0, 7.0), dtype=torch.complex128)
    lsd, fd = ls.cpu().to(torch.complex128), filt.cpu().to(torch.complex128)
    for i, r in enumerate(lists):
        idx = r.cpu().long()
        for t in range(tx):
            want[t, idx] = lsd[t, idx] @ fd[i, t].T
    # float32 sums of up to 130 products of unit scale: 1e-5 of the norm with room; untouched rows exactly
    assert rel_err(est.cpu().numpy(), want.numpy()) < 1e-5


def test_own_row_lists_may_share_rows(cuda):
    """Row lists that are not ``rows_by_set``'s may name a row twice: the last set's filter wins."""

    from hermespy_amd.configs import mimo2x2_512_pilots
    from hermespy_amd.lmmse import LMMSEChannelEstimation

    cfg = mimo2x2_512_pilots()
    lm = LMMSEChannelEstimation(cfg, snr_db=(0.0, 20.0))
    ls = torch.view_as_complex(torch.randn(cfg.num_tx, 3, cfg.num_rx, lm.num_pilots, 2, device=cuda))
    every = torch.arange(6, dtype=torch.int32, device=cuda)
    got = lm.apply(ls, np.zeros(3, dtype=int), rows_by_set=[every, every[2:4].contiguous()])
    first, second = lm.apply(ls, np.zeros(3, dtype=int)), lm.apply(ls, np.ones(3, dtype=int))
    assert torch.equal(got[:, [0, 2]], first[:, [0, 2]]) and torch.equal(got[:, 1], second[:, 1])
