"""The float64 drop path at the edges of its tables, rounds and transforms, against the float64 oracle."""

import dataclasses

import numpy as np
import pytest
import torch

from conftest import oracle_link, rel_err
from oracle import drop as odrop

pytestmark = pytest.mark.gpu

# (N, words, prefix ratio, paths, sinusoids, Doppler Hz, order, DC): one short word (the sinusoids' tables fit
# one at a time), every transform length, no prefix (delays reach into the previous word), a prefix as
# long as the word, frames of one sample run more and less than a round of 2048 samples, more
# sinusoids than one table group, a Doppler beyond the float32 path's range
SHAPES = [(32, 1, 0.0, 1, 20, 50.0, 4, True), (32, 2, 0.25, 4, 7, 50.0, 16, False), (64, 14, 0.25, 5, 20, 50.0, 4, True),
          (64, 32, 0.0, 6, 20, 50.0, 4, True), (64, 33, 0.0, 6, 20, 50.0, 64, True), (128, 3, 1.0, 9, 50, 200.0, 16, True),
          (128, 13, 0.25, 7, 60, 50.0, 4, False), (256, 14, 1 / 16, 12, 20, 20.0, 256, True),
          (64, 14, 0.25, 5, 20, 20000.0, 4, True)]


@pytest.mark.parametrize("n,words,ratio,paths,sinusoids,doppler,order,dc", SHAPES)
def test_f64_shapes_match_oracle(cuda, n, words, ratio, paths, sinusoids, doppler, order, dc):
    from hermespy_amd.configs import siso_64
    from hermespy_amd.simulation import BatchedLink

    print("float64 shape", n, words, ratio, paths, sinusoids, doppler, flush=True)
    p = 10.0 ** (-0.2 * np.arange(paths))
    cfg = dataclasses.replace(siso_64(), num_subcarriers=n, words=words, prefix_ratio=ratio, delays=np.arange(paths) / 1e6,
                              power_profile=p / p.sum(), rice_factors=np.array([2.0] + [0.0] * (paths - 1)),
                              num_sinusoids=sinusoids, doppler=2 * np.pi * doppler, modulation_order=order,
                              dc_suppression=dc, detector="mmse")
    snrs = np.array([5.0, 15.0, 25.0])
    bl = BatchedLink(cfg)
    npw = torch.as_tensor(cfg.noise_power(snrs), dtype=torch.float64, device=cuda)
    err = torch.full((3,), -1, dtype=torch.int32, device=cuda)
    eq = torch.full((3, words * n), float("nan"), dtype=torch.complex128, device=cuda)
    bl.run_f64(7, 100, npw, err, eq)
    err, eq = err.cpu().numpy(), eq.cpu().numpy()
    link = oracle_link(cfg)
    for i, snr in enumerate(snrs):
        ref = odrop.run_drop(link, 7, 100 + i, float(snr), faithful=False)
        # MMSE is well conditioned: a thousand roundings of 1e-16 stay far below 1e-11
        assert rel_err(eq[i], ref.equalized[0]) < 1e-11
        assert int(err[i]) == ref.errors
