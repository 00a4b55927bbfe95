"""The fused passes over the learned estimator's network (inference, training forward, backward through the
data) against float64 convolutions of the same bfloat16 operands, at the edges of their sample groups and tiles."""

import ctypes

import numpy as np
import pytest
import torch

from conftest import rel_err

pytestmark = pytest.mark.gpu

DILATIONS = (1, 4, 16, 1)
# float32 sums round a bfloat16 activation to its other neighbour (2^-8 away) about once in 10^4, so outputs
# differ by ~ sqrt(1e-4) 2^-8 = 4e-5 of their norm; a wrong row, tap or channel is a difference of order one
TOL = 1e-3


def _net(g, cout):
    shapes = [(64, 5, 8), (64, 5, 64), (64, 5, 64), (cout, 5, 64), (cout, 17, 8)]
    w = [(torch.randn(s, generator=g, device="cuda") * (2.0 / (s[1] * s[2])) ** 0.5).to(torch.bfloat16) for s in shapes]
    b = [torch.randn(s[0], generator=g, device="cuda") * 0.1 for s in shapes]
    return w, b


def _conv(a, w, dil):
    w = w.double()
    return sum(torch.roll(a, -(k - w.shape[1] // 2) * dil, dims=1) @ w[:, k].T for k in range(w.shape[1]))


def _forward(x, w, b):
    pre, act, a = [], [], x.double()
    for i in range(3):
        pre.append(_conv(a, w[i], DILATIONS[i]) + b[i].double())
        a = torch.nn.functional.gelu(pre[-1], approximate="tanh").to(torch.bfloat16).double()
        act.append(a)
    return pre, act, _conv(a, w[3], 1) + b[3].double() + _conv(x.double(), w[4], 1) + b[4].double()


def _pointers(tensors):
    return (ctypes.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])


# (drops, Nrx, Ntx, words, N): groups of 2, 4 and 8 samples with ragged ends; 1, 3 and 7 channel tiles; one
# (no four-channel stores), three (odd) and eight subcarriers a position
@pytest.mark.parametrize("drops,nr,nt,words,n", [(1, 1, 1, 16, 64), (3, 1, 1, 16, 192), (5, 3, 1, 2, 512), (1, 2, 2, 14, 512),
                                                 (683, 3, 1, 16, 64), (513, 2, 2, 2, 512), (1025, 2, 2, 14, 512),
                                                 (4099, 1, 1, 16, 192)])
@pytest.mark.parametrize("offset", [0, 1])
def test_estimate(cuda, drops, nr, nt, words, n, offset):
    """`offset` subcarriers into a larger buffer: an estimate that is not 16-byte aligned."""

    from hermespy_amd import _lib

    g = torch.Generator(device=cuda).manual_seed(drops + 10 * words + n)
    blk = n // 64
    cout = 2 * words * blk
    w, b = _net(g, cout)
    grid = torch.view_as_complex(torch.randn(drops, nr, words * n, 2, generator=g, device=cuda))
    pidx = torch.stack([torch.randperm(words * n, generator=g, device=cuda)[:128] for _ in range(nt)]).to(torch.int32)
    pval = torch.polar(torch.ones(nt, 128, device=cuda), torch.randn(nt, 128, generator=g, device=cuda))
    noise = torch.rand(drops, generator=g, device=cuda, dtype=torch.float64) + 0.01
    flat = torch.full((nt * drops * nr * words * n + offset,), float("nan"), dtype=torch.complex64, device=cuda)
    wp, bp = _pointers(w), _pointers(b)
    _lib.check(_lib.load().hpx_learned_estimate(
        _lib.ptr(grid), drops, nr, nt, words, n, _lib.ptr(pidx), _lib.ptr(pval), 128, _lib.ptr(noise),
        ctypes.addressof(wp), ctypes.addressof(bp), cout, _lib.ptr(flat[offset:]), _lib.stream_handle()))
    x = torch.zeros((nt, drops, nr, 64, 8), dtype=torch.float32, device=cuda)
    for t in range(nt):
        ls = (grid[:, :, pidx[t].long()] / pval[t]).reshape(drops, nr, 2, 64)
        for v in range(2):
            x[t, ..., 2 * v], x[t, ..., 2 * v + 1] = ls[:, :, v].real, ls[:, :, v].imag
        x[t, ..., 4] = 1.0 if t else -1.0
        x[t, ..., 5] = (-torch.log10(noise) / 3.0).float()[:, None, None]
    out = _forward(x.reshape(-1, 64, 8).to(torch.bfloat16), w, b)[2].reshape(-1, 64, words, blk, 2).permute(0, 2, 1, 3, 4)
    want = torch.view_as_complex(out.contiguous()).reshape(-1)
    assert rel_err(flat[offset:].cpu().numpy(), want.cpu().numpy()) < TOL


# two and four samples a workgroup, ragged
@pytest.mark.parametrize("s,cout", [(1, 32), (3, 96), (2047, 64), (2049, 224), (4099, 32)])
def test_training_forward(cuda, s, cout):
    from hermespy_amd import _lib

    g = torch.Generator(device=cuda).manual_seed(s)
    w, b = _net(g, cout)
    x = torch.randn(s, 64, 8, generator=g, device=cuda).to(torch.bfloat16)
    pre = [torch.full((s, 64, 64), float("nan"), device=cuda) for _ in range(3)]
    act = [torch.full((s, 64, 64), float("nan"), dtype=torch.bfloat16, device=cuda) for _ in range(3)]
    out = torch.full((s, 64, cout), float("nan"), device=cuda)
    wp, bp, pp, ap = _pointers(w), _pointers(b), _pointers(pre), _pointers(act)
    _lib.check(_lib.load().hpx_net_forward(_lib.ptr(x), s, wp, bp, cout, pp, ap, _lib.ptr(out), _lib.stream_handle()))
    want_pre, want_act, want = _forward(x, w, b)
    for i in range(3):
        assert rel_err(pre[i].cpu().numpy(), want_pre[i].cpu().numpy()) < TOL
        assert rel_err(act[i].double().cpu().numpy(), want_act[i].cpu().numpy()) < TOL
    assert rel_err(out.cpu().numpy(), want.cpu().numpy()) < TOL


@pytest.mark.parametrize("s", [1, 3, 2047, 2049])
def test_backward_through_the_data(cuda, s):
    from hermespy_amd import _lib

    g = torch.Generator(device=cuda).manual_seed(s + 1)
    w, _ = _net(g, 224)
    dz_out = torch.randn(s, 64, 224, generator=g, device=cuda).to(torch.bfloat16)
    pre = [torch.randn(s, 64, 64, generator=g, device=cuda) for _ in range(3)]
    dz = [torch.full((s, 64, 64), float("nan"), dtype=torch.bfloat16, device=cuda) for _ in range(3)]
    wt = [w[i].flip(1).permute(2, 1, 0).contiguous() for i in (1, 2, 3)]
    wp, pp, dp = _pointers(wt), _pointers(pre), _pointers(dz)
    _lib.check(_lib.load().hpx_net_backward(_lib.ptr(dz_out), s, 224, wp, pp, dp, _lib.stream_handle()))
    d = dz_out.double()
    for i in (2, 1, 0):
        p = pre[i].double().requires_grad_()
        torch.nn.functional.gelu(p, approximate="tanh").sum().backward()
        d = (_conv(d, wt[i], DILATIONS[i + 1]) * p.grad).to(torch.bfloat16).double()
        assert rel_err(dz[i].double().cpu().numpy(), d.cpu().numpy()) < TOL
    with pytest.raises(ValueError, match="not instantiated"):
        _lib.check(_lib.load().hpx_net_backward(_lib.ptr(dz_out), s, 192, wp, pp, dp, _lib.stream_handle()))


# one and three subcarriers a position, odd word counts, an output row shorter and longer than the workgroup
@pytest.mark.parametrize("drops,nr,nt,words,n", [(1, 1, 1, 1, 64), (5, 2, 2, 3, 192), (7, 1, 2, 14, 512)])
def test_loss_gradient(cuda, drops, nr, nt, words, n):
    """The gradient in float32 against float64, and in bfloat16 as the rounded float32 one."""

    from hermespy_amd import _lib

    g = torch.Generator(device=cuda).manual_seed(n)
    blk = n // 64
    out = torch.randn(nt * drops * nr, 64, words, blk, 2, generator=g, device=cuda)
    csi = torch.view_as_complex(torch.randn(drops, words, n, 2, generator=g, device=cuda))
    spatial = torch.view_as_complex(torch.randn(drops, nr, nt, 2, generator=g, device=cuda))
    group = (torch.arange(drops, device=cuda) % 2).to(torch.int32)
    lib, st = _lib.load(), _lib.stream_handle()
    got = {}
    for dtype, fn in ((torch.float32, lib.hpx_nmse_grad), (torch.bfloat16, lib.hpx_nmse_grad_bf16)):
        work = torch.zeros(6, dtype=torch.float64, device=cuda)
        loss = torch.zeros(1, dtype=torch.float64, device=cuda)
        grad = torch.full(out.shape, float("nan"), dtype=dtype, device=cuda)
        _lib.check(fn(_lib.ptr(out), _lib.ptr(csi), _lib.ptr(spatial), drops, nr, nt, words, n, _lib.ptr(group), 2,
                      _lib.ptr(work), _lib.ptr(grad), _lib.ptr(loss), st))
        got[dtype] = grad
    o = out.double().requires_grad_()
    h = spatial.permute(2, 0, 1)[..., None].to(torch.complex128) * csi.reshape(1, drops, 1, -1)
    est = torch.view_as_complex(o.permute(0, 2, 1, 3, 4).contiguous()).reshape(h.shape)
    err, power = (est - h).abs().square().sum(dim=(0, 2, 3)), h.abs().square().sum(dim=(0, 2, 3))
    used = [k for k in range(2) if (group == k).any()]
    want = sum(10 * torch.log10(err[group == k].sum() / power[group == k].sum()) for k in used) / len(used)
    want.backward()
    assert abs(float(loss) - float(want)) < 1e-5
    assert rel_err(got[torch.float32].cpu().numpy(), o.grad.cpu().numpy()) < 1e-5
    assert torch.equal(got[torch.bfloat16], got[torch.float32].to(torch.bfloat16))


def test_adam_of_several_tensors(cuda):
    """One launch over ragged tensors equals a launch per tensor and the separate weight copies, bit for bit."""

    from hermespy_amd import _lib

    lib, st = _lib.load(), _lib.stream_handle()
    g = torch.Generator(device=cuda).manual_seed(3)
    shapes = [(64, 5, 8), (1, 1, 1), (33, 3, 5), (257,), (0,), (256,)]
    state = [[torch.randn(s, generator=g, device=cuda) for _ in range(3)] + [torch.rand(s, generator=g, device=cuda)]
             for s in shapes]
    copies = [(torch.zeros(s, dtype=torch.bfloat16, device=cuda),
               torch.zeros(s[::-1], dtype=torch.bfloat16, device=cuda)) if len(s) == 3 else None for s in shapes]
    one = [[t.clone() for t in row] for row in state]
    entries = []
    for s, (p, gr, m1, m2), c in zip(shapes, one, copies):
        w, wt, taps, cin = (c[0].data_ptr(), c[1].data_ptr(), s[1], s[2]) if c else (None, None, 0, 0)
        entries.append(_lib.HpxAdamTensor(p.data_ptr(), gr.data_ptr(), m1.data_ptr(), m2.data_ptr(), w, wt, p.numel(), taps, cin))
    _lib.check(lib.hpx_adam_steps((_lib.HpxAdamTensor * len(entries))(*entries), len(entries), 1e-3, 0.9, 0.999, 1e-8, 7, st))
    for s, (p, gr, m1, m2), got, c in zip(shapes, state, one, copies):
        _lib.check(lib.hpx_adam_step(_lib.ptr(p), _lib.ptr(gr), _lib.ptr(m1), _lib.ptr(m2), p.numel(), 1e-3, 0.9, 0.999,
                                     1e-8, 7, st))
        assert all(torch.equal(a, b) for a, b in zip((p, m1, m2), (got[0], got[2], got[3])))
        if c:
            w, wt = torch.empty_like(c[0]), torch.empty_like(c[1])
            _lib.check(lib.hpx_conv1d_weight_copies(_lib.ptr(p), s[0], s[2], s[1], _lib.ptr(w), _lib.ptr(wt), st))
            assert torch.equal(w, c[0]) and torch.equal(wt, c[1])
