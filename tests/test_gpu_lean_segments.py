"""Drops beyond one CU's LDS cut into segments of words: the same decisions and symbols, bit for bit, as in one
piece."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 37, 129])
def test_segments_of_lean_drops_change_nothing(cuda, count):
    """`count` drops (seven segments, six, and more workgroups than the GPU holds at once or whole drops) against a
    batch of 257 of them, which runs in whole drops or other segments; replayed, since errors are added up."""

    from hermespy_amd.uneven import DropShape, UnevenBatch

    shapes = [DropShape(8, 2048, 5 + i % 19, 2.0, 100.0, 16, 10.0) for i in range(257)]
    whole = UnevenBatch(shapes, seed=3)
    whole.run()
    part = UnevenBatch(shapes[:count], seed=3, export_equalized=True)
    other = UnevenBatch(shapes[:count] + shapes[:257 - count], seed=3, export_equalized=True)
    other.run()
    part.capture()
    for _ in range(3):
        part.replay()
        torch.cuda.synchronize()
        assert torch.equal(part.errors, whole.errors[:count])
    for i in range(count):
        assert torch.equal(part.equalized[i], other.equalized[i])
