"""The training step's fused kernels against the layer-by-layer entry points, bit for bit: the same bfloat16
roundings and the same order of every float32 sum."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# (samples, cin, cout, taps, dilation): one sample, whole and part chunks of 32 and more than 32 chunks; channel
# groups of 32, 64 and 224; (tap, ci) columns that leave the bias a tile of its own (5 x 64) and that do not
SHAPES = [(1, 8, 32, 1, 1), (33, 8, 64, 5, 1), (70, 64, 64, 5, 16), (32, 64, 224, 5, 4), (1100, 8, 224, 17, 1),
          (40, 16, 96, 3, 63), (7, 24, 128, 7, 9), (5, 56, 448, 5, 1)]


def _wgrad(lib, st, dz, x, s, cin, cout, taps, dil):
    ws = torch.full((int(lib.hpx_conv1d_wgrad_workspace(s, cin, cout, taps)) // 4,), float("nan"), device="cuda")
    gw = torch.full((cout, taps, cin), float("nan"), device="cuda")
    gb = torch.full((cout,), float("nan"), device="cuda")
    from hermespy_amd import _lib

    _lib.check(lib.hpx_conv1d_wgrad(dz.data_ptr(), x.data_ptr(), s, cin, cout, taps, dil, ws.data_ptr(), gw.data_ptr(),
                                    gb.data_ptr(), st))
    return gw, gb


# 2^-70: products of the two operands are subnormal float32 values
@pytest.mark.parametrize("scale", [1.0, 2.0**-70])
@pytest.mark.parametrize("s,cin,cout,taps,dil", SHAPES)
def test_weight_gradients(cuda, s, cin, cout, taps, dil, scale):
    """Matrix cores against the VALU form (operands off 16-byte alignment take it), and the sum over chunks of 32
    samples in their order."""

    from hermespy_amd import _lib

    lib, st = _lib.load(), _lib.stream_handle()
    g = torch.Generator(device=cuda).manual_seed(s + cin)
    x, dz = ((torch.randn(s * 64 * c, generator=g, device=cuda) * scale).to(torch.bfloat16) for c in (cin, cout))
    gw, gb = _wgrad(lib, st, dz, x, s, cin, cout, taps, dil)
    shifted = [torch.cat([t.new_zeros(1), t])[1:] for t in (dz, x)]
    assert all(t.data_ptr() % 16 == 2 for t in shifted)
    vw, vb = _wgrad(lib, st, *shifted, s, cin, cout, taps, dil)
    assert torch.equal(gw, vw) and torch.equal(gb, vb)
    sw, sb = torch.zeros_like(gw), torch.zeros_like(gb)
    for s0 in range(0, s, 32):
        n = min(32, s - s0)
        pw, pb = _wgrad(lib, st, dz[s0 * 64 * cout:], x[s0 * 64 * cin:], n, cin, cout, taps, dil)
        sw += pw
        sb += pb
    assert torch.equal(gw, sw) and torch.equal(gb, sb)


def _by_layers(tr, ls):
    """A step's activations, output, gradients of every pre-activation, weight gradients and loss through the entry
    points of single layers, from the trainer's simulated drops."""

    from hermespy_amd import _lib
    from hermespy_amd.learned import CIN, DILATIONS, POSITIONS, SKIP_TAPS, TAPS, skip_shape

    lib, st = _lib.load(), _lib.stream_handle()
    net, c = tr.net, tr.cfg
    x = net.net_input(ls, tr.noise_power)
    out, cache = net.forward(x, keep=True)
    s, n = x.shape[0], len(net.shapes)
    work, loss, grad = torch.zeros_like(tr.work), torch.zeros_like(tr.loss), torch.empty_like(out)
    group = ((tr.first + torch.arange(tr.drops)) % tr.num_groups).to(torch.int32).cuda()
    _lib.check(lib.hpx_nmse_grad(out.data_ptr(), tr.csi.data_ptr(), tr.spatial.data_ptr(), tr.drops, c.num_rx, c.num_tx,
                                 c.words, c.num_subcarriers, group.data_ptr(), tr.num_groups, work.data_ptr(),
                                 grad.data_ptr(), loss.data_ptr(), st))
    dz, gw, gb = [None] * n, [None] * (n + 1), [None] * (n + 1)
    for i in range(n - 1, -1, -1):
        cin, cout, act = net.shapes[i]
        a_in, pre = cache[i]
        dz[i] = torch.empty((s, POSITIONS, cout), dtype=torch.bfloat16, device="cuda")
        if act:
            _lib.check(lib.hpx_gelu_backward(grad.data_ptr(), pre.data_ptr(), grad.numel(), dz[i].data_ptr(), st))
        else:
            _lib.check(lib.hpx_to_bf16(grad.data_ptr(), grad.numel(), dz[i].data_ptr(), st))
        gw[i], gb[i] = _wgrad(lib, st, dz[i], a_in, s, cin, cout, TAPS, DILATIONS[i])
        if i > 0:
            grad = torch.empty((s, POSITIONS, cin), device="cuda")
            _lib.check(lib.hpx_conv1d_forward(dz[i].data_ptr(), s, cout, TAPS, DILATIONS[i], net.wt16[i].data_ptr(), None,
                                              cin, 0, grad.data_ptr(), None, st))
    gw[n], gb[n] = _wgrad(lib, st, dz[-1], x, s, CIN, skip_shape(c)[1], SKIP_TAPS, 1)
    return cache, out, gw, gb, loss


def _config(words, n):
    """The 2x2 comb-pilot link with frames of words * n elements (2 words n / 64 output channels)."""

    import dataclasses

    from hermespy_amd.configs import comb_pilot_frame, mimo2x2_512_pilots

    base = mimo2x2_512_pilots()
    mask, pilots = comb_pilot_frame(n, words, (0, words - 1), n // 128, 2)
    return dataclasses.replace(base, num_subcarriers=n, words=words, frame_mask=mask, pilots=pilots,
                               bandwidth=base.bandwidth * n / 512)


# one and two tiles of positions per wavefront (fewer than 2048 samples and more)
@pytest.mark.parametrize("drops", [33, 520])
# 224 and 64 output channels
@pytest.mark.parametrize("words,n", [(14, 512), (4, 512), (16, 128)])
def test_training_step(cuda, drops, words, n):
    """Two Adam steps: activations, gradients and parameters are those of the layer-by-layer step; the loss, a float64
    sum of per-sample terms in the order their atomics arrive, is within 4096 roundings of it."""

    from hermespy_amd import _lib
    from hermespy_amd.learned import ConvNetEstimator, Trainer

    lib, st = _lib.load(), _lib.stream_handle()
    tr = Trainer(ConvNetEstimator(_config(words, n)), drops, seed=5)
    for k in range(2):
        tr.first = (1 << 20) + k * drops
        params = [p.clone() for p in tr.net.w + tr.net.b]
        moments = [m.clone() for m in tr.m1 + tr.m2]
        ls = tr.simulate(tr.first)
        cache, out, gw, gb, loss = _by_layers(tr, ls)
        x = tr.net.net_input(ls, tr.noise_power)
        got, pre, act = tr._forward(x)
        assert torch.equal(got, out)
        for i in range(3):
            assert torch.equal(pre[i], cache[i][1]) and torch.equal(act[i], cache[i + 1][0])
        step = tr.step(tr.first)
        assert abs(float(step) - float(loss)) <= 4096 * 2.3e-16 * abs(float(loss))
        assert all(torch.equal(a, b) for a, b in zip(tr.gw + tr.gb, gw + gb))
        for p, gr, m1, m2, new in zip(params, gw + gb, moments[:len(params)], moments[len(params):], tr.net.w + tr.net.b):
            _lib.check(lib.hpx_adam_step(p.data_ptr(), gr.data_ptr(), m1.data_ptr(), m2.data_ptr(), p.numel(), tr.lr,
                                         *tr.betas, tr.eps, tr.step_count, st))
            assert torch.equal(p, new)
        for w, w16 in zip(tr.net.w, tr.net.w16):
            assert torch.equal(w.to(torch.bfloat16), w16)


# one and two tiles of positions per wavefront
@pytest.mark.parametrize("s", [5, 2050])
def test_weights_of_any_alignment(cuda, s):
    """Inference and training forward read weights and biases one element off their 16-byte boundary: the same bits."""

    from hermespy_amd import _lib

    lib, st = _lib.load(), _lib.stream_handle()
    g = torch.Generator(device=cuda).manual_seed(s)
    shapes = [(64, 5, 8), (64, 5, 64), (64, 5, 64), (64, 5, 64), (64, 17, 8)]
    w = [(torch.randn(sh, generator=g, device=cuda) * 0.1).to(torch.bfloat16) for sh in shapes]
    b = [torch.randn(64, generator=g, device=cuda) for _ in shapes]
    x = torch.randn(s, 64, 8, generator=g, device=cuda).to(torch.bfloat16)
    grid = torch.view_as_complex(torch.randn(s, 4, 512, 2, generator=g, device=cuda))
    pidx = torch.arange(0, 256, 2, dtype=torch.int32, device=cuda)
    pval = torch.ones(128, dtype=torch.complex64, device=cuda)
    noise = torch.ones(s, dtype=torch.float64, device=cuda)

    def pointers(tensors):
        return (ctypes.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])

    def passes(weights, biases):
        wp, bp = pointers(weights), pointers(biases)
        est = torch.full((s, 4, 512), complex("nan"), dtype=torch.complex64, device=cuda)
        _lib.check(lib.hpx_learned_estimate(grid.data_ptr(), s, 1, 1, 4, 512, pidx.data_ptr(), pval.data_ptr(), 128,
                                            noise.data_ptr(), ctypes.addressof(wp), ctypes.addressof(bp), 64,
                                            est.data_ptr(), st))
        pre = [torch.empty((s, 64, 64), device=cuda) for _ in range(3)]
        act = [torch.empty((s, 64, 64), dtype=torch.bfloat16, device=cuda) for _ in range(3)]
        out = torch.empty((s, 64, 64), device=cuda)
        pp, ap = pointers(pre), pointers(act)
        _lib.check(lib.hpx_net_forward(x.data_ptr(), s, wp, bp, 64, pp, ap, out.data_ptr(), st))
        return [est, out, *pre, *act]

    shifted = [torch.cat([t.new_zeros(1), t.reshape(-1)])[1:] for t in w + b]
    assert all(t.data_ptr() % 16 == t.element_size() for t in shifted)
    for got, want in zip(passes(shifted[:5], shifted[5:]), passes(w, b)):
        assert torch.equal(got, want)


# one workgroup per sample, and samples in shares (a pair or none for the last threads)
@pytest.mark.parametrize("drops,words,n", [(1, 14, 4096), (3, 3, 192), (1100, 1, 64)])
def test_loss_gradient_of_any_alignment(cuda, drops, words, n):
    """Outputs and gradients one element off the boundary of a pair: the bits of aligned ones, float32 and bfloat16,
    which for one group are scale (out - H)."""

    from hermespy_amd import _lib

    lib, st = _lib.load(), _lib.stream_handle()
    g = torch.Generator(device=cuda).manual_seed(n)
    blk = n // 64
    out = torch.randn(drops, 64, words, blk, 2, generator=g, device=cuda)
    csi = torch.view_as_complex(torch.randn(drops, words, n, 2, generator=g, device=cuda))
    spatial = torch.ones(drops, 1, 1, dtype=torch.complex64, device=cuda)

    def gradient(fn, dtype, offset):
        flat = torch.full((out.numel() + offset,), float("nan"), dtype=dtype, device=cuda)
        src = torch.cat([out.new_zeros(offset), out.reshape(-1)])
        work = torch.zeros(3, dtype=torch.float64, device=cuda)
        loss = torch.zeros(1, dtype=torch.float64, device=cuda)
        _lib.check(fn(src[offset:].data_ptr(), csi.data_ptr(), spatial.data_ptr(), drops, 1, 1, words, n, None, 1,
                      work.data_ptr(), flat[offset:].data_ptr(), loss.data_ptr(), st))
        return flat[offset:], work

    got, work = gradient(lib.hpx_nmse_grad, torch.float32, 1)
    h = torch.view_as_real(csi).reshape(drops, words, 64, blk, 2).permute(0, 2, 1, 3, 4)
    assert torch.equal(got, (work[2].float() * (out - h)).reshape(-1))
    assert torch.equal(gradient(lib.hpx_nmse_grad_bf16, torch.bfloat16, 1)[0], got.to(torch.bfloat16))
    assert torch.equal(gradient(lib.hpx_nmse_grad, torch.float32, 0)[0], got)
