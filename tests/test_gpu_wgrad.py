"""Weight and bias gradients of the circular convolutions on the matrix cores and on the VALU fallback, at
the edges of their tiles, against float64 sums of the same bfloat16 operands."""

import numpy as np
import pytest
import torch

from conftest import rel_err

pytestmark = pytest.mark.gpu

# (samples, cin, cout, taps, dilation): one sample, a whole and a part chunk of 32; strips of 1, 2 and 7
# channel tiles; the bias column alone in its tile (5 x 64 + 1 columns) and inside one (5 x 8 + 1);
# shifts that wrap; input widths that take the VALU form (12: no 16-byte rows, 72: too wide)
SHAPES = [(1, 8, 32, 1, 1), (31, 8, 64, 5, 1), (33, 64, 64, 5, 16), (32, 64, 224, 5, 4), (65, 8, 224, 17, 1),
          (40, 16, 96, 3, 63), (7, 24, 128, 7, 9), (5, 56, 448, 5, 1), (9, 12, 64, 5, 2), (3, 72, 32, 3, 5),
          (4, 8, 40, 5, 1)]


@pytest.mark.parametrize("s,cin,cout,taps,dil", SHAPES)
@pytest.mark.parametrize("offset", [0, 1])
def test_wgrad_matches_float64(cuda, s, cin, cout, taps, dil, offset):
    """`offset` elements into a larger buffer: operands that are not 16-byte aligned take the VALU form."""

    from hermespy_amd import _lib

    lib, st = _lib.load(), _lib.stream_handle()
    g = torch.Generator(device=cuda).manual_seed(100 * s + cin + taps)

    def operand(channels):
        flat = torch.randn(s * 64 * channels + offset, generator=g, device=cuda).to(torch.bfloat16)
        return flat[offset:]

    x, dz = operand(cin), operand(cout)
    ws = torch.full((int(lib.hpx_conv1d_wgrad_workspace(s, cin, cout, taps)) // 4,), float("nan"), device=cuda)
    gw = torch.full((cout, taps, cin), float("nan"), device=cuda)
    gb = torch.full((cout,), float("nan"), device=cuda)
    _lib.check(lib.hpx_conv1d_wgrad(_lib.ptr(dz), _lib.ptr(x), s, cin, cout, taps, dil, _lib.ptr(ws), _lib.ptr(gw),
                                    _lib.ptr(gb), st))
    xd = x.double().cpu().reshape(s, 64, cin)
    zd = dz.double().cpu().reshape(s * 64, cout)
    for k in range(taps):
        want = zd.T @ torch.roll(xd, -(k - taps // 2) * dil, dims=1).reshape(s * 64, cin)
        # float32 accumulation of up to 64 s terms of unit scale: far below 1e-5 of the sum's norm
        assert rel_err(gw[:, k].cpu().numpy(), want.numpy()) < 1e-5
    assert np.abs(gb.cpu().numpy() - zd.sum(dim=0).numpy()).max() < 1e-5 * 64 * s
