"""Words side by side in one workgroup and drops cut into segments of words: every output of a drop is the same
bit for bit whatever the launch holds beside it and whatever its workgroup, and agrees with the oracle."""

import dataclasses

import numpy as np
import pytest
import torch

from conftest import oracle_link, rel_err
from oracle import drop as odrop

pytestmark = pytest.mark.gpu

# (antennas, N, words, prefix ratio, paths, order): single words; frames that the batches of 7, 4 or 2 words and
# the segments do not divide; no or a short prefix, so that delays reach into the word before (and into
# the segment before); one word per batch with 8 antennas; 32 and 2048 subcarriers
SHAPES = [(1, 64, 1, 0.25, 5, 4), (1, 64, 15, 0.0, 9, 16), (2, 32, 13, 0.125, 4, 64), (2, 128, 5, 1 / 32, 23, 16),
          (4, 128, 14, 0.125, 7, 256), (4, 256, 9, 0.0, 12, 4), (8, 64, 6, 0.25, 3, 16), (8, 256, 3, 1 / 64, 20, 64),
          (2, 512, 14, 0.0, 23, 16), (4, 1024, 5, 1 / 64, 23, 16), (1, 2048, 2, 1 / 8, 8, 64)]


def _link(a, n, words, ratio, paths, order):
    from hermespy_amd.uneven import DropShape

    return dataclasses.replace(DropShape(a, n, paths, 2.0, min(300.0, 5.0 * n), order, 0.0).link(), words=words, prefix_ratio=ratio)


def _run(cfg, cuda, first, noise):
    from hermespy_amd.simulation import BatchedLink

    n = len(noise)
    out = {"equalized": (n, cfg.num_tx, cfg.num_data), "grid": (n, cfg.num_rx, cfg.words, cfg.num_subcarriers),
           "csi": (n, cfg.words, cfg.num_subcarriers), "spatial": (n, cfg.num_rx, cfg.num_tx)}
    out = {k: torch.full(s, complex(7.0, 7.0), dtype=torch.complex64, device=cuda) for k, s in out.items()}
    errors = torch.full((n,), -1, dtype=torch.int32, device=cuda)
    BatchedLink(cfg).run(99, first, torch.as_tensor(noise, dtype=torch.float64, device=cuda), errors, **out)
    return {"errors": errors, **{k: torch.view_as_real(v) for k, v in out.items()}}


@pytest.mark.parametrize("shape", SHAPES)
def test_drops_do_not_depend_on_their_launch(cuda, shape):
    cfg = _link(*shape)
    print("segments", shape, flush=True)
    count = 1100 if shape[1] <= 128 else 600  # beyond one round of the GPU for some of them: other segment counts
    noise = cfg.noise_power(np.linspace(0.0, 30.0, count))
    many = _run(cfg, cuda, 40, noise)
    for lo, hi in ((0, 1), (1, 4), (4, 60)):
        few = _run(cfg, cuda, 40 + lo, noise[lo:hi])
        for k, v in few.items():
            assert torch.equal(v, many[k][lo:hi]), (k, lo, hi)
    for size in (64, 128, 256, 512):
        pairs = cfg.num_subcarriers // (2 * size)
        if pairs > 4 or cfg.num_subcarriers > 16 * size:
            continue
        other = _run(dataclasses.replace(cfg, workgroup_size=size), cuda, 41, noise[1:9])
        for k, v in other.items():
            assert torch.equal(v, many[k][1:9]), (k, size)
    link = oracle_link(cfg)
    ref = odrop.run_drop(link, 99, 41, float(30.0 / (count - 1)), faithful=False)
    # float32 signals against float64: 1e-5 of the grid's norm, 1e-4 where MMSE divides by the channel
    grid = torch.view_as_complex(many["grid"][1]).cpu().numpy()
    assert rel_err(grid, ref.grid) < 1e-5
    assert rel_err(torch.view_as_complex(many["equalized"][1]).cpu().numpy(), ref.equalized) < 1e-4


def test_frames_and_uneven_classes_do_not_depend_on_their_launch(cuda):
    """Pilot frames (element maps and per-word data offsets) of 128 subcarriers, several words a batch; a
    heterogeneous batch of few drops (segments) against the single-link launches of the same drops."""

    from hermespy_amd.configs import comb_pilot_frame
    from hermespy_amd.uneven import DropShape, UnevenBatch

    mask, pilots = comb_pilot_frame(128, 7, (1, 4), 4, 2)
    mask[3] = 2  # a word of null elements: no data, no bits
    cfg = dataclasses.replace(_link(2, 128, 7, 1 / 32, 9, 16), frame_mask=mask, pilots=pilots)
    noise = cfg.noise_power(np.linspace(0.0, 30.0, 700))
    many, few = _run(cfg, cuda, 5, noise), _run(cfg, cuda, 5, noise[:3])
    wide = _run(dataclasses.replace(cfg, workgroup_size=512), cuda, 5, noise[:3])
    for k, v in few.items():
        assert torch.equal(v, many[k][:3]) and torch.equal(wide[k], v), k
    pop = [DropShape(a, n, 23, 2.0, 60.0, 16, 9.0) for a in (1, 2, 4, 8) for n in (128, 256, 512, 1024)]
    batch = UnevenBatch(pop, seed=99, first_drop=77)
    batch.errors.fill_(-1)
    batch.run()
    errors = batch.errors.cpu().numpy()
    for i, shape in enumerate(pop):
        link = shape.link()
        alone = _run(link, cuda, 77 + i, np.atleast_1d(link.noise_power(shape.snr_db)))
        assert int(alone["errors"][0]) == int(errors[i]), shape
