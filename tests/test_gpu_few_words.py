"""Heterogeneous classes whose drops have fewer word steps than the class has segments, beside drops that have more."""

import dataclasses

import pytest
import torch

from hermespy_amd.uneven import DropShape

pytestmark = pytest.mark.gpu


@dataclasses.dataclass
class Frame(DropShape):
    words: int = 14

    def link(self):
        return dataclasses.replace(super().link(), words=self.words)


# words side by side (128), one word a step, and drops beyond one CU's LDS (their tables filled by a launch before, or
# by the drop itself where it makes one segment)
@pytest.mark.parametrize("antennas,n", [(1, 128), (2, 512), (4, 1024), (8, 2048)])
def test_segments_of_few_words(cuda, antennas, n):
    """Seven drops (up to seven segments each) and 300 (whole) of the same frames: the same errors, drop by drop, replayed."""

    from hermespy_amd.uneven import UnevenBatch

    words = [1, 2, 3, 14, 5, 1, 9]
    shapes = [Frame(antennas, n, 5 + i % 7, 2.0, 100.0, 16, 9.0, words[i % 7]) for i in range(300)]
    whole = UnevenBatch(shapes, seed=4)
    whole.run()
    few = UnevenBatch(shapes[:7], seed=4)
    few.capture()
    for _ in range(3):
        few.errors.fill_(-1)
        few.replay()
        torch.cuda.synchronize()
        assert torch.equal(few.errors, whole.errors[:7])
