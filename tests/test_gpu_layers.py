"""The host-side layer engines on the GPU: autograd Functions, side effects, the reference's
golden vectors through the HIP path, analogues of the reference's own tests for this path
(test_slayer002/003/009/010/011, test_slayerLoihi001/002) and size-independent properties at
the benchmark's full tensor sizes.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import slayerpytorch_amd as snn
from oracle import oracle as O
from slayerpytorch_amd import slayerCuda, slayerLoihiCuda
from slayerpytorch_amd.slayer import alphaKernel

from _util import golden, raster_from_aer, raster_from_events, rel_err

pytestmark = pytest.mark.gpu

DEV = "cuda"
REL_TOL = 1e-5


def neuron(**kw):
    d = {"theta": 10.0, "tauSr": 10.0, "tauRef": 1.0, "scaleRef": 2.0, "tauRho": 1.0, "scaleRho": 1.0}
    d.update(kw)
    return d


def loihi_neuron(**kw):
    d = {"type": "LOIHI", "vThMant": 80, "vDecay": 128, "iDecay": 1024, "refDelay": 1, "wgtExp": 0,
         "tauRho": 1, "scaleRho": 1}
    d.update(kw)
    return d


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def host(t):
    return t.detach().cpu().numpy()


# ------------------------------------------------------------------------------------------ psp
@pytest.mark.parametrize("recursion", [True, False])
def test_psp_forward_backward_matches_oracle(recursion, monkeypatch):
    import slayerpytorch_amd.slayer as slayer_module
    monkeypatch.setattr(slayer_module, "PSP_RECURSION", recursion)
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 300}).to(DEV)
    rng = np.random.default_rng(0)
    x = (rng.random((3, 4, 5, 5, 300)) < 0.05).astype(np.float32)
    g = rng.standard_normal(x.shape).astype(np.float32)
    xt = dev(x).requires_grad_(True)
    y = layer.psp(xt)
    y.backward(dev(g))
    srm = host(layer.srmKernel)
    if recursion:
        # the alpha kernel as a recursion over time: the sum over the taps to rounding
        assert layer._srmKernelIsAlpha() == (10.0, 1.0)
        assert rel_err(host(y), O.conv(x, srm, 1.0)) <= REL_TOL
    else:
        assert layer._srmKernelIsAlpha() is None
        assert np.array_equal(host(y), O.conv(x, srm, 1.0))
    # (the correlation of these rows runs on the matrix cores: another summation order than the chain)
    assert rel_err(host(xt.grad), O.corr(g, srm, 1.0)) <= REL_TOL
    assert layer.srmKernel.grad is None


def test_psp_takes_the_sums_for_a_kernel_that_is_not_the_layers_alpha_kernel():
    # an edited or replaced srmKernel is filtered as it is (the recursion only stands in for the kernel that
    # calculateSrmKernel built): the chain's bits on spike trains
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 300}).to(DEV)
    rng = np.random.default_rng(1)
    x = (rng.random((2, 3, 1, 1, 300)) < 0.05).astype(np.float32)
    assert layer._srmKernelIsAlpha() is not None
    layer.srmKernel[3] *= 1.5                      # in place: the tensor's version changes
    assert layer._srmKernelIsAlpha() is None
    assert np.array_equal(host(layer.psp(dev(x))), O.conv(x, host(layer.srmKernel), 1.0))
    layer.srmKernel = torch.ones(40, device=DEV)   # replaced
    assert layer._srmKernelIsAlpha() is None
    assert np.array_equal(host(layer.psp(dev(x))), O.conv(x, np.ones(40, np.float32), 1.0))


def test_psp_equals_padded_conv3d_layer():
    # reference test_slayer011: psp == pspLayer (left-padded conv3d with the flipped kernel), ||d|| / numel < 1e-6
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 300}).to(DEV)
    x = (torch.rand((2, 2, 34, 34, 300), device=DEV) < 0.02).float()
    k = layer.srmKernel
    padded = F.pad(x.reshape(2, 1, 1, -1, 300), (k.numel() - 1, 0))
    want = F.conv3d(padded, torch.flip(k, [0]).reshape(1, 1, 1, 1, -1)).reshape(x.shape) * 1.0
    got = layer.psp(x)
    assert (torch.norm(got - want) / got.numel()).item() < 1e-6


def test_psp_accepts_non_contiguous_input_and_tensor_Ts():
    layer = snn.layer(neuron(), {"Ts": 0.5, "tSample": 100}).to(DEV)
    x = torch.randn((2, 3, 4, 100, 5), device=DEV).permute(0, 1, 2, 4, 3)       # time last, not contiguous
    assert not x.is_contiguous()
    want = O.conv(host(x.contiguous()), host(layer.srmKernel), 0.5)
    assert rel_err(host(layer.psp(x)), want) <= REL_TOL      # (the layer filters its alpha kernel as a recursion)
    # the extension accepts a 0-dim tensor wherever the reference passed one for Ts
    got = slayerCuda.conv(x.contiguous(), layer.srmKernel, torch.tensor(0.5, device=DEV))
    assert np.array_equal(host(got), want)


# ------------------------------------------------------------------------------------------ spike
def test_spike_forward_side_effect_and_backward():
    nd = neuron(tauRho=0.7, scaleRho=1.3)
    layer = snn.layer(nd, {"Ts": 1.0, "tSample": 300}).to(DEV)
    rng = np.random.default_rng(1)
    u = (rng.standard_normal((2, 8, 6, 6, 300)) * 5).astype(np.float32)
    g = rng.standard_normal(u.shape).astype(np.float32)
    ref = host(layer.refKernel)
    want_s, want_u = O.get_spikes(u, ref, 10.0, 1.0)

    ut = dev(u)
    src = ut.clone().requires_grad_(True)
    pre = src * 1.0                                   # contiguous non-leaf: spike() updates it in place
    s = layer.spike(pre)
    assert np.array_equal(host(s), want_s)
    assert np.array_equal(host(pre), want_u), "membrane potential must reflect the refractory response"
    s.backward(dev(g))
    # the gradient uses the post-refractory potential that was saved
    want_g = O.spike_bwd(g, want_u, 10.0, 0.7 * 10.0, 1.3)
    np.testing.assert_allclose(host(src.grad), want_g, rtol=REL_TOL, atol=1e-30)


def test_spike_non_contiguous_input_is_left_untouched():
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 64}).to(DEV)
    rng = np.random.default_rng(2)
    u = (rng.standard_normal((2, 3, 4, 64, 5)) * 6).astype(np.float32)
    ut = dev(u).permute(0, 1, 2, 4, 3)
    before = host(ut).copy()
    s = layer.spike(ut)
    want_s, _ = O.get_spikes(before, host(layer.refKernel), 10.0, 1.0)
    assert np.array_equal(host(s), want_s)
    assert np.array_equal(host(ut), before)          # the kernel worked on a contiguous copy


@pytest.mark.parametrize("T", [300, 350])
def test_pspSpike_layer_call_matches_spike_of_psp(T, monkeypatch):
    # the MLP ordering spike(psp(fc(x))) of the reference's example as one forward and one backward kernel
    from slayerpytorch_amd import slayer as slayer_module
    monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", False)      # the two Functions as they are
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": T}).to(DEV)
    rng = np.random.default_rng(T)
    shape = (2, 24, 1, 1, T)
    a = (rng.standard_normal(shape) * 3).astype(np.float32)
    g = rng.standard_normal(shape).astype(np.float32)
    x1 = dev(a).requires_grad_(True)
    s1 = layer.pspSpike(x1)
    s1.backward(dev(g))
    x2 = dev(a).requires_grad_(True)
    s2 = layer.spike(layer.psp(x2))
    s2.backward(dev(g))
    assert torch.equal(s1, s2) and float(s1.detach().sum()) > 0
    if T % 4 == 0:  # the separate correlation of such rows runs on the matrix cores, the fused backward as a chain
        assert rel_err(host(x1.grad), host(x2.grad)) <= REL_TOL
    else:
        assert torch.equal(x1.grad, x2.grad)


@pytest.mark.parametrize("T", [300, 350, 600])
@pytest.mark.parametrize("use", ["psp", "both", "spikes"])
def test_spikePsp_layer_call_matches_psp_of_spike(T, use, monkeypatch):
    # the CNN ordering psp(spike(u)) of the reference's example: same spikes and PSP signal as the two calls, and one
    # backward kernel for whichever of the two results were used (T = 600: rows beyond the recursion take the sums over the taps)
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": T}).to(DEV)
    rng = np.random.default_rng(T)
    shape = (2, 24, 1, 1, T)
    u = (rng.standard_normal(shape) * 6 + 3).astype(np.float32)
    ga, gs = dev(rng.standard_normal(shape).astype(np.float32)), dev(rng.standard_normal(shape).astype(np.float32))

    def loss(s, a):
        return ((a * ga).sum() if use != "spikes" else 0) + ((s * gs).sum() if use != "psp" else 0)

    u1 = dev(u).requires_grad_(True)
    w1 = u1 * 1.0                       # (the spike function updates its input in place)
    s1, a1 = layer.spikePsp(w1)
    loss(s1, a1).backward()
    from slayerpytorch_amd import slayer as slayer_module
    monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", False)      # the two Functions as they are
    u2 = dev(u).requires_grad_(True)
    w2 = u2 * 1.0
    s2 = layer.spike(w2)
    a2 = layer.psp(s2)
    loss(s2, a2).backward()
    assert torch.equal(s1, s2) and torch.equal(a1, a2) and torch.equal(w1, w2) and float(s1.detach().sum()) > 0
    if use == "spikes" or T % 4 != 0 or T > 512:
        # (rows of whole vectors beyond the recursion: the separate correlation runs on the matrix cores)
        assert torch.equal(u1.grad, u2.grad) or (T > 512 and rel_err(host(u1.grad), host(u2.grad)) <= REL_TOL)
    else:
        assert torch.equal(u1.grad, u2.grad)
    assert float(u1.grad.abs().sum()) > 0


def test_psp_of_fresh_spikes_sends_its_gradient_past_the_spike_function(monkeypatch):
    """Reference-style code, spike(conv(psp(spike(conv(psp(x)))))): psp() recognises a tensor that spike() has just
    returned and runs correlation + surrogate gradient as one kernel; same values and the same gradients as with the two
    Functions apart - bit for bit while the spikes have no other user, to rounding when they have."""
    from slayerpytorch_amd import slayer as slayer_module
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 300}).to(DEV)
    torch.manual_seed(5)
    conv1, conv2 = layer.conv(2, 6, 3, padding=1, weightScale=60).to(DEV), layer.conv(6, 4, 3, padding=1, weightScale=60).to(DEV)
    rng = np.random.default_rng(31)
    x = dev((rng.random((2, 2, 8, 8, 300)) < 0.05).astype(np.float32))
    g = dev(rng.standard_normal((2, 4, 8, 8, 300)).astype(np.float32))
    gs = dev(rng.standard_normal((2, 6, 8, 8, 300)).astype(np.float32))

    def run(pair, extra, touch=None):
        monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", pair)
        for m in (conv1, conv2):
            m.weight.grad = None
        s1 = layer.spike(conv1(layer.psp(x)))
        if touch == "inplace":
            s1 = s1.mul_(1.0)                        # no longer what the spike function returned
        elif touch == "detach":
            s1 = s1.detach()
        a2 = layer.psp(s1)
        s2 = layer.spike(conv2(a2))
        out = (layer.psp(s2) * g).sum()
        if extra:
            out = out + (s1 * gs).sum()              # the hidden spikes have a second user
        out.backward()
        return s2.detach().clone(), conv1.weight.grad.clone() if conv1.weight.grad is not None else None, conv2.weight.grad.clone()

    apart = run(False, False)
    paired = run(True, False)
    assert float(apart[0].sum()) > 0 and float(apart[1].abs().sum()) > 0
    assert all(torch.equal(a, b) for a, b in zip(apart, paired))
    apart2, paired2 = run(False, True), run(True, True)
    assert torch.equal(apart2[0], paired2[0]) and torch.equal(apart2[2], paired2[2])
    assert rel_err(host(paired2[1]), host(apart2[1])) <= REL_TOL and not torch.equal(apart2[1], apart[1])
    # spikes that were modified, or detached, are not paired
    assert all(torch.equal(a, b) for a, b in zip(run(False, False, "inplace"), run(True, False, "inplace")))
    detached = run(True, False, "detach")
    assert detached[1] is None and torch.equal(detached[2], apart[2])
    # the pairing really happened: the node behind the PSP signal
    monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", True)
    s1 = layer.spike(conv1(layer.psp(x)))
    assert type(layer.psp(s1).grad_fn).__name__ == "_pspOfSpikeFunctionBackward"
    assert type(layer.psp(s1 * 1.0).grad_fn).__name__ == "_pspFunctionBackward"
    with torch.no_grad():
        assert layer.psp(s1).grad_fn is None


def test_spike_of_a_fresh_psp_signal_sends_its_gradient_past_the_filter(monkeypatch):
    """Reference-style MLP code, spike(psp(fc(spike(psp(fc(x)))))): spike() recognises a signal that psp() has just
    returned and runs surrogate gradient + correlation as one kernel; same spikes, and the same gradients bit for bit
    as with the two Functions apart; a signal that was touched in between is not paired."""
    from slayerpytorch_amd import slayer as slayer_module
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 300}).to(DEV)
    torch.manual_seed(6)
    fc1, fc2 = layer.dense(40, 30, weightScale=80).to(DEV), layer.dense(30, 7, weightScale=80).to(DEV)
    rng = np.random.default_rng(32)
    x = dev((rng.random((3, 40, 1, 1, 300)) < 0.05).astype(np.float32))
    g = dev(rng.standard_normal((3, 7, 1, 1, 300)).astype(np.float32))

    def run(pair, touch=False):
        monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", pair)
        for m in (fc1, fc2):
            m.weight.grad = None
        a1 = layer.psp(fc1(x))
        if touch:
            a1 = a1 * 1.0
        s1 = layer.spike(a1)
        s2 = layer.spike(layer.psp(fc2(s1)))
        (layer.psp(s2) * g).sum().backward()
        return s2.detach().clone(), fc1.weight.grad.clone(), fc2.weight.grad.clone(), type(s1.grad_fn).__name__

    apart, paired, touched = run(False), run(True), run(True, True)
    assert float(apart[0].sum()) > 0 and float(apart[1].abs().sum()) > 0
    assert apart[3] == "_spikeFunctionBackward" and paired[3] == "_spikeOfPspFunctionBackward" and touched[3] == "_spikeFunctionBackward"
    for other in (paired, touched):
        assert all(torch.equal(a, b) for a, b in zip(apart[:3], other[:3]))


@pytest.mark.parametrize("C,H,W,T,window", [(3, 8, 8, 300, 2), (4, 7, 9, 173, 2), (2, 5, 6, 173, 2), (4, 9, 7, 520, 3),
                                            (1, 10, 7, 520, 3), (2, 8, 7, 40, 3),
                                            (2, 6, 8, 9, (2, 4)), (4, 5, 5, 3, 2), (1, 2, 2, 20, 2)])
def test_pool_of_fresh_psp_sends_its_gradient_past_filter_and_spike_function(C, H, W, T, window, monkeypatch):
    """pool(psp(spike(u))): the pooling layer correlates its gradient while it is still pooled and sends it to u in one
    kernel.  Same values as with the Functions apart and as torch's own pooling of the extended tensor; the gradient to
    rounding (weight and filter change places: two roundings per term, REL_TOL).  A psp tensor that is still held gets its
    own gradient."""
    from slayerpytorch_amd import slayer as slayer_module
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": max(T, 100)}).to(DEV)
    pool = layer.pool(window).to(DEV)
    with torch.no_grad():
        pool.weight.mul_(torch.rand(pool.weight.shape, device=DEV) + 0.5)     # a weight per position of the window
    torch.manual_seed(7)
    u0 = torch.randn((4, C, H, W, T), device=DEV) * 6 + 5
    KH, KW = pool.kernel_size[0], pool.kernel_size[1]
    g = torch.randn((4, C, (H + H % KH) // KH, (W + W % KW) // KW, T), device=DEV)

    def run(pair, hold):
        monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", pair)
        u = u0.clone().requires_grad_(True)
        a = layer.psp(layer.spike(u * 1.0))
        values = a.detach()
        y = pool(a)
        name = type(y.grad_fn).__name__
        wanted = [u, a] if hold else [u]
        del a
        return y.detach(), values, name, torch.autograd.grad(y, wanted, g)

    y0, a0, _, (ref,) = run(False, False)
    y1, _, name, (got,) = run(True, False)
    assert torch.equal(y0, y1) and float(ref.abs().sum()) > 0
    if C > 1 and (H + H % KH) % KH != 0:             # windows run from one channel into the next
        assert name == "ViewBackward0"
    elif y1.numel() % 4 == 0 if T <= 512 else T % 4 == 0:
        assert name == "_poolOfPspFunctionBackward"
    assert rel_err(host(got), host(ref)) <= REL_TOL
    (ref_u, ref_a), (got_u, got_a) = run(False, True)[3], run(True, True)[3]
    assert torch.equal(ref_u, got_u) and torch.equal(ref_a, got_a)
    padded = F.pad(a0.double().cpu(), (0, 0, 0, W % KW, 0, H % KH))
    want = F.conv3d(padded.reshape(4, 1, -1, *padded.shape[3:]), pool.weight.detach().double().cpu(), None, (KH, KW, 1))
    assert rel_err(host(y1), want.reshape(y1.shape).numpy()) <= REL_TOL


@pytest.mark.parametrize("window", [2, 3, 4, 5, (3, 2), (2, 5)])
@pytest.mark.parametrize("C", [1, 2, 3, 4])
def test_pool_layer_is_the_convolution_of_the_channels_below_one_another(window, C):
    """The pooling layer is one convolution of the extended tensor viewed as (N, 1, C H, W, T), whatever the height: windows
    run from one channel into the next where they do not divide the extended height, shapes whose result is no whole number of
    channels are refused, images smaller than the window have no pixel, if they are not refused, and a weight that requires a
    gradient changes nothing."""
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 100}).to(DEV)
    pool = layer.pool(window).to(DEV)
    KH, KW = pool.kernel_size[0], pool.kernel_size[1]
    with torch.no_grad():
        pool.weight.mul_(torch.rand(pool.weight.shape, device=DEV) + 0.5)
    rng = np.random.default_rng(17 * C + KH + KW)
    refused = taken = 0
    for H in range(1, 14):
        for W, T in ((1, 8), (7, 5), (10, 3)):
            x0 = dev(rng.standard_normal((2, C, H, W, T)).astype(np.float32))

            def expression(x, w):
                y = F.pad(x, (0, 0, 0, W % KW, 0, H % KH))
                y = F.conv3d(y.reshape(2, 1, -1, *y.shape[3:]), w, None, (KH, KW, 1))
                return y.reshape(2, C, -1, *y.shape[3:])

            xd, wd = x0.double().cpu().requires_grad_(True), pool.weight.detach().double().cpu()
            try:
                want = expression(xd, wd)
            except RuntimeError:
                want = None
            for learnable in (False, True):
                pool.weight.requires_grad_(learnable)
                x = x0.clone().requires_grad_(True)
                if want is None:
                    small = C * (H + H % KH) < KH or W + W % KW < KW
                    try:
                        got = pool(x)
                    except RuntimeError:
                        got = None
                    assert got is None or (small and got.numel() == 0), (H, W, T)
                    refused += 1
                    continue
                got = pool(x)
                assert got.shape == want.shape, (H, W, T)
                g = dev(rng.standard_normal(tuple(got.shape)).astype(np.float32))
                (wantG,) = torch.autograd.grad(want, xd, g.double().cpu(), retain_graph=True)
                (gotG,) = torch.autograd.grad(got, x, g)
                assert rel_err(host(got), want.detach().numpy()) <= 1e-6 and rel_err(host(gotG), wantG.numpy()) <= 1e-6, (H, W, T)
                taken += 1
    assert taken > 0 and (refused > 0) == (window != 2)


@pytest.mark.parametrize("learnable", [True, False])
def test_delay_of_fresh_spikes_sends_its_gradient_past_the_spike_function(learnable, monkeypatch):
    """Reference-style delay(spike(u)) / delayShift(spike(u), d): the delay recognises a tensor that spike() has just
    returned and runs the gradient's shift and the surrogate gradient as one kernel; same values, same gradients for
    the membrane potential and the delays, bit for bit."""
    from slayerpytorch_amd import slayer as slayer_module
    params = {"type": "SRMALPHA", "theta": 10, "tauSr": 2.0, "tauRef": 1.0, "scaleRef": 2, "tauRho": 1, "scaleRho": 1}
    layer = snn.layer(params, {"Ts": 1.0, "tSample": 120}).cuda()
    torch.manual_seed(4)
    u0 = (torch.randn((3, 6, 2, 2, 120)) * 6 + 4).cuda()
    g = torch.randn_like(u0)
    dl = layer.delay((6, 2, 2)).cuda()
    with torch.no_grad():
        dl.delay.mul_(9.0)

    def run(pair):
        monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", pair)
        dl.delay.grad = None
        u = u0.clone().requires_grad_(True)
        s = layer.spike(u * 1.0)
        out = dl(s) if learnable else layer.delayShift(s, 3.0)
        out.backward(g)
        return out.detach().clone(), u.grad.clone(), (dl.delay.grad.clone() if learnable else None), type(out.grad_fn).__name__

    apart, paired = run(False), run(True)
    assert paired[3] == "_delayOfSpikeFunctionBackward" and apart[3] != paired[3]
    assert torch.equal(apart[0], paired[0]) and torch.equal(apart[1], paired[1]) and float(apart[1].abs().sum()) > 0
    if learnable:
        assert torch.equal(apart[2], paired[2]) and float(apart[2].abs().sum()) > 0


def test_get_spikes_requires_five_dimensions():
    f = torch.ones(3, device=DEV)
    with pytest.raises(IndexError):
        slayerCuda.getSpikes(torch.zeros((4, 10), device=DEV), f, 1.0, 1.0)
    with pytest.raises(RuntimeError):
        slayerCuda.getSpikes(torch.zeros((1, 2, 3, 10), device=DEV), f, 1.0, 1.0)
    with pytest.raises(RuntimeError, match="contiguous"):
        slayerCuda.conv(torch.zeros((4, 10, 3), device=DEV).permute(0, 2, 1), f, 1.0)
    with pytest.raises(RuntimeError, match="Float"):
        slayerCuda.conv(torch.zeros((4, 10), device=DEV, dtype=torch.float64), f, 1.0)
    with pytest.raises(RuntimeError, match="shift and number of neurons must be same"):
        slayerCuda.shift(torch.zeros((2, 3, 1, 1, 10), device=DEV), torch.zeros(5, device=DEV), 1.0)


# ------------------------------------------------------------------------------------------ delay
def check_shift(x, y, k):
    if k > 0:
        return torch.equal(x[:-k], y[k:]) and not y[:k].any()
    if k == 0:
        return torch.equal(x, y)
    return torch.equal(x[-k:], y[:k]) and not y[k:].any()


def test_shift_per_neuron_like_reference_test009():
    Ts = 0.1
    layer = snn.layer(neuron(), {"Ts": Ts, "tSample": 50}).to(DEV)
    N, C, H, W, D = 5, 10, 20, 30, 500
    delay = layer.delay((C, H, W)).to(DEV)
    x = torch.randn((N, C, H, W, D), device=DEV)
    delay.delay.data = torch.rand(delay.delay.shape, device=DEV) * 2 - 1
    y = slayerCuda.shift(x, delay.delay.data, Ts)
    d = host(delay.delay.data)
    xs, ys = x.cpu(), y.cpu()
    rng = np.random.default_rng(0)
    for _ in range(400):                              # a random sample of neurons; all rows are checked below
        n, c, h, w = rng.integers(N), rng.integers(C), rng.integers(H), rng.integers(W)
        k = int(np.float32(d[c, h, w]) / np.float32(Ts))
        assert check_shift(xs[n, c, h, w], ys[n, c, h, w], k)
    assert np.array_equal(host(y), O.shift(host(x), d, Ts))
    y4 = layer.delayShift(x, 4)
    assert torch.equal(y4[..., 4:], x[..., :-4]) and not y4[..., :4].any()


def test_delay_shift_backward_shifts_the_other_way():
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 100}).to(DEV)
    x = torch.randn((2, 3, 4, 4, 100), device=DEV, requires_grad=True)
    g = torch.randn_like(x)
    for delay in (3, 3.0, torch.tensor(3.0), torch.tensor([3.0], device=DEV)):
        x.grad = None
        layer.delayShift(x, delay).backward(g)
        assert np.array_equal(host(x.grad), O.shift(host(g), -3, 1.0))
    d = torch.rand((3, 4, 4), device=DEV) * 20 - 5
    x.grad = None
    layer.delayShift(x, d).backward(g)
    assert np.array_equal(host(x.grad), O.shift(host(g), -host(d), 1.0))


def test_delay_layer_gradients_like_reference_test010():
    """Autograd delay gradient == -sum(e * d(psp)/dt) * Ts, in both operator orders."""
    Ts, Ns, N, Nin, Nout = 0.1, 500, 5, 25, 1
    nd = neuron(tauSr=1.0)
    layer = snn.layer(nd, {"Ts": Ts, "tSample": 50}).to(DEV)
    torch.manual_seed(0)
    fc1 = layer.dense(Nin, Nout).to(DEV)
    delay = layer.delay((Nin, 1, 1)).to(DEV)
    spikeIn = ((torch.rand((N, Nin, 1, 1, Ns), device=DEV) > 0.8).float() / Ts)
    spikeDes = ((torch.rand((N, Nout, 1, 1, Ns), device=DEV) > 0.8).float() / Ts)

    def loss_of(spikeOut):
        err = layer.psp(spikeOut - spikeDes)
        return 0.5 * torch.sum(err ** 2) * Ts

    grads = []

    class Probe(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.view_as(x)

        @staticmethod
        def backward(ctx, g):
            grads.append(g)
            return g

    pspDelayed = delay(layer.psp(spikeIn))
    uOut = fc1(Probe.apply(pspDelayed))
    loss_of(layer.spike(uOut)).backward()
    errorRec = grads[0]
    diffFilter = torch.tensor([1, -1], dtype=torch.float, device=DEV) / Ts
    dpsp_dt = slayerCuda.conv(pspDelayed.detach().contiguous(), diffFilter, 1)
    manual = -torch.sum(errorRec * dpsp_dt, [0, -1], keepdim=True).reshape((Nin, 1, 1)) * Ts
    assert torch.norm(manual - delay.delay.grad).item() < 1e-4
    assert torch.norm(manual).item() > 1e-3

    # delay before psp gives the same gradient (both are time-invariant linear maps)
    delay.delay.grad = None
    loss_of(layer.spike(fc1(layer.psp(delay(spikeIn))))).backward()
    assert torch.norm(manual - delay.delay.grad).item() < 1e-4


def test_delay_layer_per_channel_broadcast_and_oracle_gradient():
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 64}).to(DEV)
    delay = layer.delay(3).to(DEV)                       # one delay per channel, input has H, W > 1
    delay.delay.data = torch.tensor([0.0, 2.0, 5.0], device=DEV).reshape(3, 1, 1)
    x = torch.randn((2, 3, 4, 5, 64), device=DEV, requires_grad=True)
    g = torch.randn_like(x)
    y = delay(x)
    y.backward(g)
    lut = np.repeat(np.array([0.0, 2.0, 5.0], np.float32), 20).reshape(3, 4, 5)
    assert np.array_equal(host(y), O.shift(host(x), lut, 1.0))
    assert np.array_equal(host(x.grad), O.shift(host(g), -lut, 1.0))
    per_neuron = O.delay_grad(host(y), host(g), 1.0)    # (3, 4, 5): summed over the repeat by autograd
    assert rel_err(host(delay.delay.grad).reshape(3), per_neuron.reshape(3, -1).sum(1)) < 1e-4


# ------------------------------------------------------------------------------------------ golden chains
def test_golden_250_25_1_spike_chain_like_reference_test002():
    snn_d = golden("snn_250_25_1.npz")
    Ts, Ns = 0.1, 500
    nd = neuron(tauSr=1.0)
    layer = snn.layer(nd, {"Ts": Ts, "tSample": 50}, fullRefKernel=True).to(DEV)
    assert layer.srmKernel.numel() == 77 and layer.refKernel.numel() == 160
    fc1, fc2 = layer.dense(250, 25).to(DEV), layer.dense(25, 1).to(DEV)
    fc1.weight.data = dev(snn_d["w1learned"]).reshape(25, 250, 1, 1, 1)
    fc2.weight.data = dev(snn_d["w2learned"]).reshape(1, 25, 1, 1, 1)
    x = dev(raster_from_aer(snn_d["spikeIn"], 250, Ns, Ts, 1 / Ts)).reshape(1, 250, 1, 1, Ns)
    uHid = fc1(layer.psp(x))
    pre = host(uHid).copy()
    sHid = layer.spike(uHid)
    want = raster_from_aer(snn_d["spikeHid"], 25, Ns, Ts, 1 / Ts)
    assert np.array_equal(host(sHid).reshape(25, Ns), want)
    sOut = layer.spike(layer.psp(fc2(sHid)))
    assert np.array_equal(np.nonzero(host(sOut).reshape(-1))[0], np.array([203, 355, 447]))
    # spike function triples recorded for hidden neuron 0: u before, u after, spikes
    d = snn_d["spikeFuncHid"][:-1]
    assert np.abs(pre.reshape(25, Ns)[0] - d[:, 0]).max() < 2e-3
    assert np.abs(host(uHid).reshape(25, Ns)[0] - d[:, 1]).max() < 2e-3
    assert np.array_equal(host(sHid).reshape(25, Ns)[0], d[:, 2])


def test_golden_gradients_like_reference_test003():
    snn_d = golden("snn_250_25_1.npz")
    Ts, Ns = 0.1, 500
    nd = neuron(tauSr=1.0, tauRho=0.1)
    layer = snn.layer(nd, {"Ts": Ts, "tSample": 50}, fullRefKernel=True).to(DEV)
    fc1, fc2 = layer.dense(250, 25).to(DEV), layer.dense(25, 1).to(DEV)
    fc1.weight = torch.nn.Parameter(dev(snn_d["w1Initial"]).reshape(25, 250, 1, 1, 1))
    fc2.weight = torch.nn.Parameter(dev(snn_d["w2Initial"]).reshape(1, 25, 1, 1, 1))
    x = dev(raster_from_aer(snn_d["spikeIn"], 250, Ns, Ts, 1 / Ts)).reshape(1, 250, 1, 1, Ns)
    des = dev(raster_from_aer(snn_d["spikeOut"], 1, Ns, Ts, 1 / Ts)).reshape(1, 1, 1, 1, Ns)
    s1 = layer.spike(layer.psp(fc1(x)))
    s2 = layer.spike(layer.psp(fc2(s1)))
    error = snn.loss({"neuron": nd, "simulation": {"Ts": Ts, "tSample": 50}, "training": {"error": {"type": "SpikeTime"}}}).to(DEV)
    loss = error.spikeTime(s2, des)
    assert float(loss.detach()) == pytest.approx(float((0.5 * torch.sum(layer.psp(s2 - des) ** 2) * Ts).detach()), rel=1e-6)
    loss.backward()
    g2 = host(fc2.weight.grad).reshape(1, 25)
    g1 = host(fc1.weight.grad).reshape(25, 250)
    assert np.linalg.norm(snn_d["gradW2Initial"] - g2) / g2.size < 1e-4
    assert np.linalg.norm(snn_d["gradW1Initial"] - g1) / g1.size < 1e-4


def test_golden_output_layer_and_gradients_torch_validate():
    """The legacy traces of the 250-25-1 network at Ts = 0.1 through the layer engine and autograd: hidden and
    output spikes (266 and 11), the output neuron's potential, the error signal of the spike-time loss and both
    weight gradients (Wgrad1, Wgrad2: a second joint pin of psp, spike, the surrogate gradient and corr next to
    the gradW*Initial files).  The files carry 5 digits."""
    tv = golden("torch_validate.npz")
    Ts, Ns = 0.1, 501
    nd = neuron(tauSr=1.0, tauRho=0.43429)                         # pdf tau = tauRho * theta = 4.3429
    layer = snn.layer(nd, {"Ts": Ts, "tSample": 50}, fullRefKernel=True).to(DEV)
    fc1, fc2 = layer.dense(250, 25).to(DEV), layer.dense(25, 1).to(DEV)
    fc1.weight = torch.nn.Parameter(dev(tv["W12"]).reshape(25, 250, 1, 1, 1))
    fc2.weight = torch.nn.Parameter(dev(tv["W23"]).reshape(1, 25, 1, 1, 1))
    s1 = dev(raster_from_events(tv["s1_shape"], tv["s1_events"], tv["s1_values"])).reshape(1, 250, 1, 1, Ns)
    a1 = layer.psp(s1)
    assert np.abs(host(a1).reshape(250, Ns) - tv["a1"]).max() < 1e-4
    u2 = fc1(a1)
    s2 = layer.spike(u2)
    assert np.array_equal(host(s2).reshape(25, Ns), tv["s2"]) and float((s2 > 0).sum()) == 266
    u3 = fc2(layer.psp(s2))
    s3 = layer.spike(u3)
    assert np.array_equal(host(s3).reshape(1, Ns), tv["s3"]) and float((s3 > 0).sum()) == 11
    assert np.abs(host(u3).reshape(1, Ns) - tv["u3"]).max() < 2e-2   # (the potential after the refractory response)
    des = dev(tv["des_s"]).reshape(1, 1, 1, 1, Ns)
    e3 = layer.psp(s3 - des)
    assert np.abs(host(e3).reshape(1, Ns) - tv["e3"]).max() < 2e-4
    error = snn.loss({"neuron": nd, "simulation": {"Ts": Ts, "tSample": 50}, "training": {"error": {"type": "SpikeTime"}}}).to(DEV)
    error.spikeTime(s3, des).backward()
    assert rel_err(host(fc2.weight.grad).reshape(1, 25), tv["Wgrad2"]) < 2e-3
    assert rel_err(host(fc1.weight.grad).reshape(25, 250), tv["Wgrad1"]) < 2e-3


def test_numSpikes_loss_matches_host_side_formulation():
    # the reference computes the target region, the desired counts and the count error with numpy on
    # the host (src/spikeLoss.py:84-104); the same numbers, and the gradient, from device tensors
    Ts, T = 1.0, 300
    nd = neuron()
    desc = {"neuron": nd, "simulation": {"Ts": Ts, "tSample": T},
            "training": {"error": {"type": "NumSpikes", "tgtSpikeRegion": {"start": 50, "stop": 250},
                                   "tgtSpikeCount": {True: 60, False: 10}}}}
    error = snn.loss(desc).to(DEV)
    rng = np.random.default_rng(4)
    out = ((rng.random((3, 10, 1, 1, T)) < 0.1) / Ts).astype(np.float32)
    cls = np.zeros((3, 10, 1, 1, 1), np.float32)
    cls[np.arange(3), rng.integers(0, 10, 3)] = 1
    x = dev(out).requires_grad_(True)
    loss = error.numSpikes(x, dev(cls))
    loss.backward()
    # host-side formulation with the oracle's PSP filter
    srm = host(error.slayer.srmKernel)
    region = np.zeros(out.shape)
    region[..., 50:250] = 1
    actual = out[..., 50:250].sum(4, keepdims=True) * Ts
    desired = np.where(cls == True, 60, 10)      # noqa: E712
    count_error = (actual - desired) / 200
    e = O.conv((out - (region * out).astype(np.float32)), srm, Ts) + (count_error * region).astype(np.float32)
    assert float(loss.detach()) == pytest.approx(0.5 * float((e.astype(np.float64) ** 2).sum()) * Ts, rel=1e-5)
    want_grad = O.corr((e * np.float32(Ts)).astype(np.float32), srm, Ts)
    assert rel_err(host(x.grad), want_grad) < REL_TOL


# ------------------------------------------------------------------------------------------ Loihi
def test_loihi_chip_recordings_like_reference_loihi_test001():
    snn_d, chip = golden("snn_250_25_1.npz"), golden("loihi_chip.npz")
    Ts, Ns = 0.1, 500
    layer = snn.loihi(loihi_neuron(), {"Ts": Ts, "tSample": 50}).to(DEV)
    fc1, fc2 = layer.dense(250, 25).to(DEV), layer.dense(25, 1).to(DEV)
    W1 = np.round(snn_d["w1learned"].astype(np.float64) * 4 / 2) * 2
    W2 = np.round(snn_d["w2learned"].astype(np.float64) * 4 / 2) * 2
    fc1.weight.data = dev(W1.astype(np.float32)).reshape(25, 250, 1, 1, 1)
    fc2.weight.data = dev(W2.astype(np.float32)).reshape(1, 25, 1, 1, 1)
    x = dev(raster_from_aer(snn_d["spikeIn"], 250, Ns, Ts, 1 / Ts, offset=49)).reshape(1, 250, 1, 1, Ns)
    sH, vH, _ = layer.spikeLoihiFull(fc1(x))
    sH = layer.delayShift(sH, 1)
    sO, vO, _ = layer.spikeLoihiFull(fc2(sH))
    sO = layer.delayShift(sO, 1)
    want = raster_from_aer(chip["hiddenSpikes"], 25, Ns, Ts, 1 / Ts, time_first=False)
    assert torch.norm(sH.reshape(25, Ns).cpu() - torch.from_numpy(want)).item() < 1e-3
    assert np.array_equal(np.nonzero(host(sO).reshape(-1))[0], np.array([57, 60]))
    assert torch.norm(vH[0, 24, 0, 0, :-1].cpu() - torch.from_numpy(chip["hiddenVoltage24"]).float()).item() < 1e-3
    assert torch.norm(vO[..., :-1].cpu().reshape(-1) - torch.from_numpy(chip["outputVoltage"]).float()).item() < 1e-3


@pytest.mark.parametrize("refDelay", [2, 9, 17])
def test_loihi_random_network_like_reference_loihi_test002(refDelay):
    rng = np.random.default_rng(refDelay)
    numSrc, numDst, T = 128, 64, 200
    layer = snn.loihi(loihi_neuron(refDelay=refDelay, scaleRho=768), {"Ts": 1, "tSample": T}).to(DEV)
    weight = np.round((rng.random((numDst, numSrc)) - 0.5) * 10) * 2
    w = weight.dot(rng.random((numSrc, T)) > 0.8).astype(np.float32)
    spike, voltage, current = layer.spikeLoihiFull(dev(w))                  # 2-D input, as in the reference test
    want = O.loihi_get_spikes(w, 0, 80 * 64, 1024, 128, refDelay)
    assert np.array_equal(host(spike), want[0]) and np.array_equal(host(voltage), want[1])
    assert np.array_equal(host(current), want[2])


def test_loihi_autograd_backward():
    Ts = 1.0
    nd = loihi_neuron(scaleRho=2.0)
    layer = snn.loihi(nd, {"Ts": Ts, "tSample": 300}).to(DEV)
    rng = np.random.default_rng(3)
    w = (2 * rng.integers(-64, 64, size=(2, 6, 5, 5, 300)) * (rng.random((2, 6, 5, 5, 300)) < 0.3)).astype(np.float32)
    g = rng.standard_normal(w.shape).astype(np.float32)
    wt = dev(w).requires_grad_(True)
    s = layer.spikeLoihi(wt)
    s.backward(dev(g))
    ws, wv, _ = O.loihi_get_spikes(w, 0, 5120, 1024, 128, 1)
    assert np.array_equal(host(s), ws) and ws.sum() > 0
    psp = host(layer.srmKernel)
    want = O.corr(O.spike_bwd(g, wv, 5120.0, 5120.0, nd["scaleRho"]), psp, Ts)
    assert rel_err(host(wt.grad), want) < REL_TOL
    assert len(psp) == 110 and nd["scaleRho"] == pytest.approx(2.0 / 195.0)


@pytest.mark.parametrize("Ts,delay", [(1.0, 1), (1.0, 40), (0.5, 1.0), (1.0, 0)])
def test_loihi_spike_with_fused_delay_matches_spike_then_delayShift(Ts, delay):
    # the Loihi network blocks of the reference do delayShift(spikeLoihi(x), 1); the layer offers it as one call
    nd = loihi_neuron(scaleRho=2.0)
    layer = snn.loihi(nd, {"Ts": Ts, "tSample": 300}).to(DEV)
    rng = np.random.default_rng(11)
    shape = (2, 6, 5, 5, 300)
    w = ((2 * rng.integers(-64, 64, size=shape) * (rng.random(shape) < 0.3)) / Ts).astype(np.float32)
    g = rng.standard_normal(shape).astype(np.float32)
    a = dev(w).requires_grad_(True)
    fused = layer.spikeLoihi(a, delay)
    fused.backward(dev(g))
    b = dev(w).requires_grad_(True)
    two = layer.delayShift(layer.spikeLoihi(b), delay)
    two.backward(dev(g))
    assert torch.equal(fused, two) and float(fused.detach().sum()) > 0
    assert torch.equal(a.grad, b.grad)
    # without a gradient to compute the layer asks the kernel for the spikes only
    with torch.no_grad():
        assert torch.equal(layer.spikeLoihi(dev(w), delay), two)


@pytest.mark.parametrize("delay,delayTs", [(0.3, 0.1), (0.7, 0.1), (2.9999999, 1.0), (5.0, 2.5), (-0.3, 0.1), (4.0, 0.1)])
def test_loihi_fused_delay_uses_the_shift_kernels_quotient(delay, delayTs):
    # delay / delayTs in fp32, truncated toward zero, like the shift kernel: 0.3 / 0.1 is 3 steps there (2 in double
    # precision); negative and long delays, a delay per neuron and tensors take the separate shift
    layer = snn.loihi(loihi_neuron(scaleRho=2.0), {"Ts": 1.0, "tSample": 120}).to(DEV)
    rng = np.random.default_rng(13)
    shape = (2, 3, 2, 2, 120)
    w = (2 * rng.integers(-64, 64, size=shape) * (rng.random(shape) < 0.3)).astype(np.float32)
    with torch.no_grad():
        plain = layer.spikeLoihi(dev(w))
        want = layer.delayShift(plain, delay, delayTs)
        assert torch.equal(layer.spikeLoihi(dev(w), delay, delayTs), want)
        assert torch.equal(want, dev(O.shift(host(plain), delay, delayTs)))
    assert float(plain.sum()) > 0


@pytest.mark.parametrize("C,H,W,T,window,delay", [(3, 8, 8, 310, 2, 1), (2, 7, 9, 173, 2, 1), (1, 5, 6, 64, (2, 3), 0), (4, 3, 2, 33, 2, 5),
                                                  (2, 9, 7, 40, 3, 2), (1, 10, 7, 40, 3, 2), (2, 8, 7, 40, 3, 2),
                                                  (2, 4, 4, 300, 2, 1), (2, 4, 4, 12, 2, 1)])
def test_loihi_neuron_takes_the_gradient_of_a_pooling_layer_as_it_is(C, H, W, T, window, delay, monkeypatch):
    """pool(spikeLoihi(x)): the neuron's backward kernel spreads the pooled gradient over the windows on the way in.  The same
    bits as through the pooling layer's own gradient where the kernel sums over rows as they come; also with a second user of
    the spikes, a backward pass that is run twice, one that runs on another stream, spikes that are still held, and an infinity."""
    from slayerpytorch_amd import slayer as slayer_module
    layer = snn.loihi(loihi_neuron(), {"Ts": 1, "tSample": T}).to(DEV)
    pool = layer.pool(window).to(DEV)
    with torch.no_grad():
        pool.weight.mul_(torch.arange(1, 1 + pool.weight.numel(), device=DEV).reshape(pool.weight.shape) / 2.0)
    rng = np.random.default_rng(C + H + W + T)
    x0 = dev((2 * rng.integers(-128, 128, (2, C, H, W, T)) * (rng.random((2, C, H, W, T)) < 0.3)).astype(np.float32))
    KH, KW = pool.kernel_size[0], pool.kernel_size[1]
    g = dev(rng.standard_normal((2, C, (H + H % KH) // KH, (W + W % KW) // KW, T)).astype(np.float32))
    more = dev(rng.standard_normal(x0.shape).astype(np.float32))

    def run(pair, how, g=g):
        monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", pair)
        x = x0.clone().requires_grad_(True)
        s = layer.spikeLoihi(x * 1.0, delay=delay)
        y = pool(s)
        name = type(y.grad_fn).__name__
        wanted = [x, s] if how == "held" else [x]
        out = (y * g).sum() + ((s * more).sum() if how == "both" else 0.0)
        del s
        if how == "twice":
            torch.autograd.grad(out, wanted, retain_graph=True)
        return name, y.detach(), torch.autograd.grad(out, wanted)

    for how in ("once", "both", "twice", "held"):
        (_, y0, ref), (name, y1, got) = run(False, how), run(True, how)
        assert name == ("ViewBackward0" if C > 1 and (H + H % KH) % KH != 0 else "_poolOfSpikesFunctionBackward") and torch.equal(y0, y1)
        assert len(ref) == len(got) and all(torch.equal(a, b) for a, b in zip(ref, got)), how
    bad = g.clone()
    bad[1, C - 1, 0, 0, T // 2] = float("inf")
    ref, got = run(False, "once", bad)[2][0], run(True, "once", bad)[2][0]
    assert torch.equal(torch.isfinite(ref), torch.isfinite(got)) and rel_err(host(got.nan_to_num(0, 0, 0)), host(ref.nan_to_num(0, 0, 0))) <= REL_TOL
    monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", True)
    x = x0.clone().requires_grad_(True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    s = layer.spikeLoihi(x * 1.0, delay=delay)
    with torch.cuda.stream(side):
        side.wait_stream(torch.cuda.default_stream())
        y = pool(s)
        del s
        gs = g * 1.0
    torch.cuda.current_stream().wait_stream(side)
    (got,) = torch.autograd.grad(y, x, gs)
    assert torch.equal(got, run(False, "once")[2][0])


def test_loihi_delay_per_neuron_or_tensor_takes_the_separate_shift():
    layer = snn.loihi(loihi_neuron(scaleRho=2.0), {"Ts": 1.0, "tSample": 120}).to(DEV)
    rng = np.random.default_rng(14)
    shape = (2, 3, 2, 2, 120)
    w = (2 * rng.integers(-64, 64, size=shape) * (rng.random(shape) < 0.3)).astype(np.float32)
    table = dev((rng.random((3, 2, 2)) * 6).astype(np.float32))
    with torch.no_grad():
        plain = layer.spikeLoihi(dev(w))
        assert torch.equal(layer.spikeLoihi(dev(w), table), layer.delayShift(plain, table))
        one = torch.tensor([2.0], device=DEV)
        assert torch.equal(layer.spikeLoihi(dev(w), one), layer.delayShift(plain, one))


def test_loihi_Ts_scaling_of_input_and_output():
    layer = snn.loihi(loihi_neuron(), {"Ts": 0.1, "tSample": 20}).to(DEV)
    rng = np.random.default_rng(4)
    w = (20 * rng.integers(-30, 60, size=(1, 9, 1, 1, 200))).astype(np.float32)      # spikes of amplitude 1/Ts times weights
    s, v, u = layer.spikeLoihiFull(dev(w))
    ws, wv, wu = O.loihi_get_spikes((w * np.float32(0.1)).astype(np.float32), 0, 5120, 1024, 128, 1)
    assert np.array_equal(host(s), ws / np.float32(0.1)) and np.array_equal(host(v), wv)
    with pytest.raises(ValueError):
        slayerLoihiCuda.getSpikes(dev(w), 0, 5120, 1024, 128, 0)


# ------------------------------------------------------------------------------------------ full sizes
FULL = (12, 16, 34, 34, 300)          # largest activation tensor of the NMNIST-CNN-shaped config


def test_full_size_spike_sampled_rows_and_checksum():
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 300}).to(DEV)
    g = torch.Generator(device="cpu").manual_seed(0)
    u = torch.randn(FULL, generator=g) * 5.0
    ud = u.to(DEV)
    s = slayerCuda.getSpikes(ud, layer.refKernel, 10.0, 1.0)
    rows = np.random.default_rng(0).choice(12 * 16 * 34 * 34, 4096, replace=False)
    un = u.reshape(-1, 300).numpy()[rows].reshape(1, 4096, 1, 1, 300)
    want_s, want_u = O.get_spikes(un, host(layer.refKernel), 10.0, 1.0)
    idx = torch.from_numpy(rows).to(DEV)
    assert np.array_equal(host(s.reshape(-1, 300)[idx]), want_s.reshape(4096, 300))
    assert np.array_equal(host(ud.reshape(-1, 300)[idx]), want_u.reshape(4096, 300))
    # size-independent properties: spikes are 0 or 1/Ts and sit on supra-threshold samples (nu[0] = 0);
    # the refractory update is linear in the spikes: u_after = u_before + conv(spikes, nu) up to rounding
    assert torch.all((s == 0) | (s == 1.0))
    assert torch.all(ud[s > 0] >= 10.0)
    assert 0.005 < (s > 0).float().mean().item() < 0.05
    rebuilt = u.to(DEV) + slayerCuda.conv(s, layer.refKernel, 1.0)
    assert (rebuilt - ud).abs().max().item() < 1e-4


def test_full_size_psp_linearity_adjoint_and_sampled_rows():
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 300}).to(DEV)
    k = layer.srmKernel
    g = torch.Generator(device="cpu").manual_seed(1)
    x = (torch.rand(FULL, generator=g) < 0.02).float().to(DEV)
    y = torch.randn(FULL, generator=g).to(DEV)
    cx = slayerCuda.conv(x, k, 1.0)
    cy = slayerCuda.corr(y, k, 1.0)
    lhs = (cx.double() * y.double()).sum().item()
    rhs = (x.double() * cy.double()).sum().item()
    assert abs(lhs - rhs) <= 1e-6 * abs(lhs)                                   # <conv x, y> = <x, corr y>
    both = slayerCuda.conv(2.0 * x + y, k, 1.0)
    assert rel_err(host(both[0, 0]), host(2.0 * cx[0, 0] + slayerCuda.conv(y, k, 1.0)[0, 0])) < REL_TOL
    rows = np.random.default_rng(1).choice(12 * 16 * 34 * 34, 2048, replace=False)
    idx = torch.from_numpy(rows).to(DEV)
    assert np.array_equal(host(cx.reshape(-1, 300)[idx]), O.conv(host(x.reshape(-1, 300)[idx]), host(k), 1.0))
    assert rel_err(host(cy.reshape(-1, 300)[idx]), O.corr(host(y.reshape(-1, 300)[idx]), host(k), 1.0)) <= REL_TOL


def test_full_size_shift_roundtrip():
    g = torch.Generator(device="cpu").manual_seed(2)
    x = torch.randn(FULL, generator=g).to(DEV)
    y = slayerCuda.shift(x, 1.0, 1.0)
    assert torch.equal(y[..., 1:], x[..., :-1]) and not y[..., 0].any()
    back = slayerCuda.shift(y, 1.0, 1.0, sign=-1.0)
    assert torch.equal(back[..., :-1], x[..., :-1]) and not back[..., -1].any()


def test_full_size_loihi_sampled_rows():
    shape = (8, 16, 32, 32, 300)      # largest tensor of the Loihi DVS-gesture-shaped config
    g = torch.Generator(device="cpu").manual_seed(3)
    w = (2 * torch.randint(-128, 128, shape, generator=g) * (torch.rand(shape, generator=g) < 0.05)).float()
    s, v, u = slayerLoihiCuda.getSpikes(w.to(DEV), 0, 5120, 1024, 128, 1)
    rows = np.random.default_rng(3).choice(8 * 16 * 32 * 32, 4096, replace=False)
    want = O.loihi_get_spikes(w.reshape(-1, 300).numpy()[rows], 0, 5120, 1024, 128, 1)
    idx = torch.from_numpy(rows).to(DEV)
    for got, exp in zip((s, v, u), want):
        assert np.array_equal(host(got.reshape(-1, 300)[idx]), exp)
    assert want[0].sum() > 0
    # invariants of the neuron: first sample is zero, spikes are 0/1, reported voltage at a spike is vDecay
    assert not s[..., 0].any() and not v[..., 0].any() and not u[..., 0].any()
    assert torch.all((s == 0) | (s == 1)) and torch.all(v[s > 0] == 128)


def test_delay_stress_config_shapes():
    # long-sequence delay config: (64, 256, 1, 1, 2000) with delays U[0, 62], tauSr = 1 (8 taps)
    layer = snn.layer(neuron(tauSr=1.0), {"Ts": 1.0, "tSample": 2000}).to(DEV)
    assert layer.srmKernel.numel() == 8
    g = torch.Generator(device="cpu").manual_seed(4)
    x = (torch.rand((64, 256, 1, 1, 2000), generator=g) < 0.005).float().to(DEV).requires_grad_(True)
    delay = layer.delay(256).to(DEV)
    delay.delay.data = (torch.rand((256, 1, 1), generator=g) * 62).to(DEV)
    y = delay(layer.psp(x))
    grad = torch.randn(y.shape, generator=g).to(DEV)
    y.backward(grad)
    a = O.conv(host(x), host(layer.srmKernel), 1.0)
    want_y = O.shift(a, host(delay.delay.data), 1.0)
    assert np.array_equal(host(y), want_y)
    assert rel_err(host(delay.delay.grad), O.delay_grad(want_y, host(grad), 1.0)) < REL_TOL
    want_gx = O.corr(O.shift(host(grad), -host(delay.delay.data), 1.0), host(layer.srmKernel), 1.0)
    assert np.array_equal(host(x.grad), want_gx)


def test_loihi_cnn_inference_is_bit_exact():
    """A small Loihi network in the ordering of the reference's gesture example
    (exampleLoihi/03_IBMGesture/ibmGestureTrain.py:55-79): pool, conv, pool, dense with weights on Loihi's even
    integer grid, every layer followed by a shift of one step.  Sums of small integers are exact in fp32, so the
    whole pipeline must reproduce the oracle chain (synapse -> integer neuron -> shift) bit for bit."""
    from oracle import oracle as O
    desc = {"type": "LOIHI", "vThMant": 80, "vDecay": 128, "iDecay": 1024, "refDelay": 1, "wgtExp": 0,
            "tauRho": 1, "scaleRho": 1}
    layer = snn.loihi(desc, {"Ts": 1, "tSample": 64}).cuda()
    torch.manual_seed(3)
    pool1, conv1, pool2 = layer.pool(2), layer.conv(2, 8, 3, padding=1, weightScale=30), layer.pool(2)
    fc = layer.dense(4 * 4 * 8, 5, weightScale=60)
    mods = [m.cuda() for m in (pool1, conv1, pool2, fc)]
    rng = np.random.default_rng(12)
    x = (rng.random((2, 2, 16, 16, 64)) < 0.05).astype(np.float32)

    s = torch.from_numpy(x).cuda()
    ref = x
    with torch.no_grad():
        for k, m in enumerate(mods):
            w = (m.weight if m.preHookFx is None else m.preHookFx(m.weight)).detach().cpu().numpy()[..., 0]
            if k == 3:
                s = s.reshape(2, -1, 1, 1, 64)
                ref = ref.reshape(2, -1, 1, 1, 64)
                z = np.einsum("ok,nkt->not", w.reshape(5, -1).astype(np.float64), ref.reshape(2, -1, 64)).reshape(2, 5, 1, 1, 64)
            elif k == 1:
                z = O.synapse_conv(ref, w, 1, 1)
            else:
                N, C, H, W, T = ref.shape
                z = O.synapse_conv(ref.reshape(N, 1, C * H, W, T), w, 2).reshape(N, C, H // 2, W // 2, T)
            assert np.array_equal(z, np.round(z))                      # integer weighted spikes
            spikes = O.loihi_get_spikes(z.astype(np.float32), 0, desc["theta"], 1024, 128, 1)[0]
            ref = O.shift(spikes, 1.0, 1.0)
            s = layer.spikeLoihi(m(s), delay=1)
            assert np.array_equal(s.cpu().numpy(), ref), "layer %d" % k
    assert ref.sum() > 0


@pytest.mark.parametrize("learnable", [True, False])
def test_spike_delayed_layer_matches_spike_then_delay(learnable):
    """spikeLayer.spikeDelayed against delay(spike(u)) / delayShift(spike(u), d): same spikes, same
    gradient with respect to the membrane potential and, for a delay layer, the delays."""
    params = {"type": "SRMALPHA", "theta": 10, "tauSr": 2.0, "tauRef": 1.0, "scaleRef": 2, "tauRho": 1, "scaleRho": 1}
    layer = snn.layer(params, {"Ts": 1.0, "tSample": 120}).cuda()
    torch.manual_seed(4)
    u0 = (torch.randn((3, 6, 2, 2, 120)) * 6 + 4).cuda()
    g = torch.randn_like(u0)
    if learnable:
        dl = layer.delay((6, 2, 2)).cuda()
        with torch.no_grad():
            dl.delay.mul_(9.0)
        dl2 = layer.delay((6, 2, 2)).cuda()
        with torch.no_grad():
            dl2.delay.copy_(dl.delay)
    ua = u0.clone().requires_grad_(True)
    ub = u0.clone().requires_grad_(True)
    # the spike function updates its input in place: give each path its own copy inside the graph
    if learnable:
        sa = dl(layer.spike(ua * 1.0))
        sb = layer.spikeDelayed(ub * 1.0, dl2)
    else:
        sa = layer.delayShift(layer.spike(ua * 1.0), 4.0, 1.0)
        sb = layer.spikeDelayed(ub * 1.0, 4.0, 1.0)
    assert torch.equal(sa, sb) and float(sa.sum()) > 0
    sa.backward(g)
    sb.backward(g)
    assert torch.equal(ua.grad, ub.grad)
    if learnable:
        assert torch.equal(dl.delay.grad, dl2.delay.grad) and float(dl.delay.grad.abs().sum()) > 0


@pytest.mark.parametrize("Ts,T,shape", [(1.0, 300, (4, 10, 1, 1)), (0.5, 128, (2, 3, 2, 2)), (1.0, 20000, (1, 2, 1, 1))])
def test_spike_time_loss_kernel_matches_tensor_expression(Ts, T, shape):
    """The fused loss (error signal + squared sum in two launches) against the reference's expression
    1/2 * sum(psp(out - desired)^2) * Ts evaluated with torch ops on the same psp kernel: the loss to
    rounding of the sum, the gradient bit for bit (the error signal is the same arithmetic).  T = 20000
    does not fit the fused kernel and takes the tensor expression."""
    params = {"type": "SRMALPHA", "theta": 10, "tauSr": 5.0, "tauRef": 1.0, "scaleRef": 2, "tauRho": 1, "scaleRho": 1}
    sim = {"Ts": Ts, "tSample": int(T * Ts)}
    error = snn.loss({"neuron": params, "simulation": sim, "training": {"error": {"type": "SpikeTime"}}}).cuda()
    torch.manual_seed(5)
    out = ((torch.rand(shape + (T,)) < 0.05).float() / Ts).cuda().requires_grad_(True)
    des = ((torch.rand(shape + (T,)) < 0.05).float() / Ts).cuda()
    loss = error.spikeTime(out, des)
    loss.backward()
    out2 = out.detach().clone().requires_grad_(True)
    e = error.slayer.psp(out2 - des)
    ref = 1 / 2 * torch.sum(e ** 2) * Ts
    ref.backward()
    assert abs(float(loss) - float(ref)) <= 1e-5 * abs(float(ref)) and float(ref) > 0
    Fl = error.slayer.srmKernel.numel()
    if 34 <= Fl <= 129 and T % 4 == 0 and T <= 60000 // 4:
        # the tensor expression's psp of this dense difference runs on the matrix cores, the fused kernel filters
        # with the chain: equal to rounding
        assert rel_err(out.grad.cpu().numpy(), out2.grad.cpu().numpy()) <= 1e-5
    else:
        assert torch.equal(out.grad, out2.grad)
    # against the oracle's psp
    eo = O.conv((out.detach() - des).cpu().numpy(), error.slayer.srmKernel.cpu().numpy(), Ts)
    assert abs(float(loss) - 0.5 * float((eo.astype(np.float64) ** 2).sum()) * Ts) <= 1e-5 * abs(float(ref))


@pytest.mark.parametrize("Ts,T,region,shape", [(1.0, 300, (0, 150), (4, 10, 1, 1)), (0.5, 129, (10, 1000), (2, 3, 1, 2)),
                                               (1.0, 65, (-20, -3), (1, 1, 1, 1)), (1.0, 4, (3, 1), (3, 2, 1, 1))])
def test_count_loss_kernel_matches_the_tensor_expressions(Ts, T, region, shape, monkeypatch):
    """The spike-count loss in two launches against the tensor expressions that stand for rows that do not fit it: loss and
    gradient to rounding (1e-5), for regions inside, across the end, counted from the end and empty, and classes given as
    truth values or numbers."""
    from slayerpytorch_amd import spikeLoss as module
    params = neuron(tauSr=5.0)
    error = snn.loss({"neuron": params, "simulation": {"Ts": Ts, "tSample": int(T * Ts) + 50}, "training": {"error": {
        "type": "NumSpikes", "tgtSpikeRegion": {"start": region[0] * Ts, "stop": region[1] * Ts},
        "tgtSpikeCount": {True: 20, False: 3}}}}).to(DEV)
    torch.manual_seed(3)
    out = ((torch.rand(shape + (T,)) < 0.2).float() / Ts).to(DEV)
    cls = (torch.rand(shape + (1,)) < 0.5).to(DEV)

    def run(wanted, scale=1):
        x = out.clone().requires_grad_(True)
        loss = error.numSpikes(x, wanted, scale)
        loss.backward()
        return type(loss.grad_fn).__name__, float(loss.detach()), host(x.grad)

    got = run(cls)
    assert got[0] == "_countLossFunctionBackward"
    assert all(a == b for a, b in zip(got[:2], run(cls.float())[:2]))
    scaled = run(cls, 2.5)
    monkeypatch.setattr(module, "_fits", lambda *a: False)
    for mine, scale in ((got, 1), (scaled, 2.5)):
        want = run(cls, scale)
        assert want[0] != mine[0] and abs(mine[1] - want[1]) <= 1e-5 * abs(want[1]) and want[1] > 0
        assert rel_err(mine[2], want[2]) <= REL_TOL


@pytest.mark.parametrize("scale", [100.0, 0.5])
def test_cpu_plumbing_configuration(scale):
    """The reference's CPU-runnable case: Bernoulli(0.02) spikes (4, 2, 34, 34, 300), dense 2312 -> 512 as a
    conv3d with N(0,1) * scale weights - scale 100 as that configuration is stated (every neuron with a positive
    drive then fires at each step), and 0.5, where the layer fires a few per cent of the time and the potentials
    cross the threshold slowly - a pspLayer-style conv3d PSP (left-padded, flipped SRM kernel, tauSr = 10) on the
    CPU with torch, threshold / refractory spikes by the oracle - against dense -> psp -> spike of this package on
    the GPU.  The membrane potentials agree to fp32 rounding; spikes may flip only where the potential sits
    within that rounding of the threshold."""
    params = {"type": "SRMALPHA", "theta": 10, "tauSr": 10.0, "tauRef": 1.0, "scaleRef": 2, "tauRho": 1, "scaleRho": 1}
    layer = snn.layer(params, {"Ts": 1.0, "tSample": 300})
    torch.manual_seed(0)
    x = (torch.rand((4, 2, 34, 34, 300)) < 0.02).float()
    fc = layer.dense((34, 34, 2), 512)
    with torch.no_grad():
        fc.weight.copy_(torch.randn(fc.weight.shape) * scale)
    srm = layer.srmKernel.clone()
    # CPU: conv3d dense, then the PSP as a conv3d over time with the flipped kernel (src/slayer.py:760-791)
    with torch.no_grad():
        z = F.conv3d(x, fc.weight)
        pad = F.pad(z, (srm.numel() - 1, 0)).reshape(4 * 512, 1, 1, 1, -1)
        a_cpu = F.conv3d(pad, srm.flip(0).reshape(1, 1, 1, 1, -1)).reshape(z.shape)
    s_cpu, u_cpu = O.get_spikes(a_cpu.numpy(), layer.refKernel.numpy(), params["theta"], 1.0)
    # GPU
    layer = layer.cuda()
    fc = fc.cuda()
    with torch.no_grad():
        a_gpu = layer.psp(fc(x.cuda()))
        assert rel_err(a_gpu.cpu().numpy(), a_cpu.numpy()) <= 1e-5
        s_gpu = layer.spike(a_gpu)
    flips = float((s_gpu.cpu().numpy() != s_cpu).mean())
    assert 0.005 < float(s_cpu.mean()) < (0.5 if scale < 1 else 0.9)
    assert flips <= 1e-4, "spike flip rate %g" % flips


def _pairs():
    """name -> (the tensor in between, the result) of x: calls whose backward passes run as one."""
    srm = snn.layer(neuron(), {"Ts": 1.0, "tSample": 300}).to(DEV)
    chip = snn.loihi(loihi_neuron(), {"Ts": 1, "tSample": 300}).to(DEV)
    pool, chipPool = srm.pool(2).to(DEV), chip.pool(2).to(DEV)

    def pool_psp(x):
        a = srm.psp(srm.spike(x))
        return a, pool(a)

    def pool_spikes(x):
        s = chip.spikeLoihi(x)
        return s, chipPool(s)

    def pool_psp_spike(x):
        s = srm.spike(x)
        return s, pool(srm.psp(s))

    def spike_psp(x):
        a = srm.psp(x)
        return a, srm.spike(a)

    def psp_spike(x):
        s = srm.spike(x)
        return s, srm.psp(s)

    def delay_spike(x):
        s = srm.spike(x)
        return s, delay(s)

    def shift_spike(x):
        s = srm.spike(x)
        return s, srm.delayShift(s, 3.0)

    delay = srm.delay((3, 4, 6)).to(DEV)
    return {"pool of psp": pool_psp, "pool of psp of spikes": pool_psp_spike, "pool of Loihi spikes": pool_spikes,
            "spike of psp": spike_psp, "psp of spikes": psp_spike, "delay of spikes": delay_spike, "shift of spikes": shift_spike}


# ways of asking for the gradient of a tensor after its last use: (what `ask` returns is held, the tensor is let go)
def _tensor_hook(t, seen):
    t.register_hook(lambda g: (seen.append(g.clone()), g * 2)[1])


def _node_prehook(t, seen):
    t.grad_fn.register_prehook(lambda gs: (seen.append(gs[0].clone()), (gs[0] * 2,))[1])


def _node_hook(t, seen):
    t.grad_fn.register_hook(lambda gradIn, gradOut: seen.append(gradOut[0].clone()))


def _retained(t, seen):
    t.retain_grad()
    return t


@pytest.mark.parametrize("ask", [_tensor_hook, _node_prehook, _node_hook, _retained, "edge", "again"])
@pytest.mark.parametrize("pair", ["pool of psp", "pool of psp of spikes", "pool of Loihi spikes", "spike of psp", "psp of spikes",
                                  "delay of spikes", "shift of spikes"])
def test_a_gradient_that_is_asked_for_after_the_call_is_there(pair, ask, monkeypatch):
    """A hook on the tensor between two paired calls, or on its node, registered after the second call on a tensor that is then
    let go, sees and changes the gradient as with the Functions apart; so does autograd.grad for the tensor's edge."""
    from slayerpytorch_amd import slayer as slayer_module
    rng = np.random.default_rng(5)
    x0 = dev((rng.integers(-3, 9, (2, 3, 4, 6, 300)) * 12).astype(np.float32))
    calls = _pairs()[pair]

    def run(paired):
        monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", paired)
        x = x0.clone().requires_grad_(True)
        seen = []
        between, y = calls(x * 1.0)
        g = torch.linspace(-1.0, 2.0, y.numel(), device=DEV).reshape(y.shape)
        if ask == "edge":
            edge = torch.autograd.graph.get_gradient_edge(between)
            del between
            return list(torch.autograd.grad(y, [x, edge], g))
        if ask == "again":                           # watched in one pass, and not in the next
            handle = between.register_hook(lambda g: (seen.append(g.clone()), g * 2)[1])
            del between
            first = torch.autograd.grad(y, x, g, retain_graph=True)
            handle.remove()
            return [*first, *torch.autograd.grad(y, x, g), *seen]
        held = ask(between, seen)
        del between
        (grad,) = torch.autograd.grad(y, x, g) if held is None else (y.backward(g), x.grad)[1:]
        return [grad, *seen, *(() if held is None else (held.grad,))]

    want, got = run(False), run(True)
    assert len(want) == len(got) >= 2 and all(float(w.abs().sum()) > 0 for w in want)
    for a, b in zip(got, want):
        assert a.shape == b.shape and rel_err(host(a), host(b)) <= REL_TOL


@pytest.mark.parametrize("pair", ["pool of psp", "spike of psp"])
@pytest.mark.parametrize("paired", [True, False])
def test_a_filter_that_was_changed_in_place_between_the_calls_is_noticed(pair, paired, monkeypatch):
    """The gradient belongs to the filter that the signal was made with: a filter that was changed in place since is an error
    of the backward pass, as for any saved tensor, and not the filter of a paired kernel."""
    from slayerpytorch_amd import slayer as slayer_module
    monkeypatch.setattr(slayer_module, "PAIR_SPIKE_PSP", paired)
    layer = snn.layer(neuron(), {"Ts": 1.0, "tSample": 300}).to(DEV)
    pool = layer.pool(2).to(DEV)
    x = torch.randn((2, 3, 4, 6, 300), device=DEV).mul_(9).requires_grad_(True)
    a = layer.psp(layer.spike(x * 1.0)) if pair == "pool of psp" else layer.psp(x * 1.0)
    layer.srmKernel.mul_(2.0)
    y = pool(a) if pair == "pool of psp" else layer.spike(a)
    del a
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


@pytest.mark.parametrize("pair", ["pool of psp", "pool of Loihi spikes", "psp of spikes"])
def test_a_signal_whose_users_send_no_gradient_sends_zeros(pair):
    """A Function that answers None for the signal between the two calls, or for the result: zeros at the input, and what comes
    by the other way where there is one."""
    class Nothing(torch.autograd.Function):
        @staticmethod
        def forward(ctx, a):
            return a.clone()

        @staticmethod
        def backward(ctx, g):
            return None

    x = dev(np.random.default_rng(6).integers(-20, 90, (2, 3, 4, 6, 300)).astype(np.float32)).requires_grad_(True)
    between, y = _pairs()[pair](x * 1.0)
    if pair != "psp of spikes":                      # (the spike function by itself passes on that there is none)
        (grad,) = torch.autograd.grad(Nothing.apply(between).sum(), x, retain_graph=True)
        assert grad.shape == x.shape and not grad.any()
    (grad,) = torch.autograd.grad(Nothing.apply(y).sum(), x, retain_graph=True)
    assert not grad.any()
    both = Nothing.apply(between).sum() + y.sum()
    (want,) = torch.autograd.grad(y.sum(), x, retain_graph=True)
    (grad,) = torch.autograd.grad(both, x, retain_graph=True)
    assert want.any() and torch.equal(grad, want)
    del between
    (again,) = torch.autograd.grad(both, x)
    assert float((again - want).norm()) <= 1e-5 * float(want.norm())


@pytest.mark.parametrize("pair", ["pool of Loihi spikes", "delay of spikes", "shift of spikes"])
def test_paired_calls_in_a_compiled_model(pair):
    """torch.compile around calls whose backward passes run as one: the values of the calls as they are, a second time as well.
    (Not of ``psp``, whose look at its filter torch.compile does not take.)"""
    call = _pairs()[pair]

    class Model(torch.nn.Module):
        def forward(self, x):
            return call(x * 1.0)[1]

    x = dev((np.random.default_rng(8).integers(-3, 9, (2, 3, 4, 6, 300)) * 12).astype(np.float32)).requires_grad_(True)
    want = Model()(x)
    g = torch.linspace(-1.0, 2.0, want.numel(), device=DEV).reshape(want.shape)
    (wantGrad,) = torch.autograd.grad(want, x, g)
    torch._dynamo.reset()
    compiled = torch.compile(Model(), backend="eager")
    for _ in range(2):
        got = compiled(x)
        (grad,) = torch.autograd.grad(got, x, g)
        assert torch.equal(got, want) and rel_err(host(grad), host(wantGrad)) <= REL_TOL
