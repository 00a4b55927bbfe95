"""The float64 drop path on frames around one sample per thread (256 samples), against the float64 oracle."""

import pytest

from test_gpu_f64_shapes import test_f64_shapes_match_oracle as check

pytestmark = pytest.mark.gpu


# (N, words, prefix ratio, paths, sinusoids): 40, 160, 256, 264 and 288 samples (one sample a thread up to 256, then eight);
# tables of all sinusoids at once, in groups beyond the room they get (80 sinusoids), and in the frame's own
@pytest.mark.parametrize("n,words,ratio,paths,sinusoids", [(32, 1, 0.25, 15, 20), (128, 1, 0.25, 4, 20), (64, 4, 0.0, 9, 80),
                                                           (32, 8, 1 / 32, 3, 20), (32, 9, 0.0, 5, 80), (32, 1, 0.0, 2, 1)])
def test_short_frames(cuda, n, words, ratio, paths, sinusoids):
    check(cuda, n, words, ratio, paths, sinusoids, 50.0, 16, True)
