"""Host-side checks that need no GPU: the C-ABI library loads and exports every symbol the
header declares, and the Python modules reject bad arguments before anything is launched, with
the error behaviour of the reference bindings (src/cuda/slayerKernels.cu:7-10, 35, 102;
src/cuda/slayerLoihiKernels.cu:12-19)."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

from slayerpytorch_amd import _lib, slayerCuda, slayerLoihiCuda
import slayerpytorch_amd as snn

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "slayer_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(slayer_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = declared_symbols()
    assert len(names) >= 13 and "slayer_conv_f32" in names and "slayer_loihi_get_spikes_f32" in names
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for name in names:
        assert hasattr(lib, name), "libslayer_hip.so does not export %s" % name
    assert sorted(_lib.SIGNATURES) == names, "python binding table and header disagree"


def test_abi_version_and_status_strings():
    lib = _lib.load()
    assert lib.slayer_hip_abi_version() == _lib.ABI_VERSION == 1
    assert lib.slayer_status_string(0) == b"ok"
    assert lib.slayer_status_string(1) == b"invalid argument"
    assert lib.slayer_status_string(77) == b"unknown status"
    with pytest.raises(_lib.SlayerHipError, match="invalid argument"):
        _lib.check(1, "slayer_conv_f32")


def test_argument_validation_in_the_c_abi_without_launch():
    lib = _lib.load()
    # empty tensors are a successful no-op, whatever the pointers
    assert lib.slayer_conv_f32(None, None, None, 0, 10, 3, 1.0, None) == 0
    assert lib.slayer_get_spikes_f32(None, None, None, 5, 0, 3, 1.0, 1.0, None) == 0
    # null pointers with work to do, negative sizes, refDelay 0, bad sign
    assert lib.slayer_conv_f32(None, None, None, 4, 10, 3, 1.0, None) == 1
    assert lib.slayer_corr_f32(None, None, None, -1, 10, 3, 1.0, None) == 1
    assert lib.slayer_shift_f32(None, None, 1.0, 4, 10, 1.0, None) == 1
    assert lib.slayer_shift_lut_f32(None, None, None, 3, 2, 4, 10, 1.0, 1.0, None) == 1     # lutSize != nPerBatch
    assert lib.slayer_shift_lut_f32(None, None, None, 4, 0, 4, 10, 1.0, 0.5, None) == 1     # sign must be +-1
    assert lib.slayer_loihi_get_spikes_f32(None, None, None, None, 0, 0, 0, 64, 0, 0, 0, None) == 1   # refDelay 0
    assert lib.slayer_loihi_get_spikes_f32(None, None, None, None, 0, 0, 26, 64, 0, 0, 1, None) == 1  # 1 << 32
    assert lib.slayer_spike_bwd_f32(None, None, None, 1.0, 0.0, 1.0, 4, None) == 1
    assert lib.slayer_delay_grad_workspace_bytes(64, 256, 2000) == 64 * 256 * 4
    assert lib.slayer_delay_grad_workspace_bytes(0, 256, 2000) == 0


def test_cpu_tensors_are_rejected_like_the_reference():
    x = torch.zeros(1, 2, 1, 1, 10)
    f = torch.ones(3)
    for call in (lambda: slayerCuda.conv(x, f, 1.0), lambda: slayerCuda.corr(x, f, 1.0),
                 lambda: slayerCuda.shift(x, f, 1.0), lambda: slayerCuda.shift(x, 1.0),
                 lambda: slayerCuda.getSpikes(x, f, 1.0, 1.0),
                 lambda: slayerLoihiCuda.getSpikes(x, 0, 64, 0, 0, 1),
                 lambda: slayerLoihiCuda.getSpikesDelayed(x, 0, 64, 0, 0, 1, 1, voltage=False),
                 lambda: slayerCuda.pspSpike(x, f, f, 1.0, 1.0),
                 lambda: slayerCuda.spikeBackward(x, x, 1.0, 1.0, 1.0),
                 lambda: slayerCuda.spikeBackwardCorr(x, x, f, 1.0, 1.0, 1.0, 1.0),
                 lambda: slayerCuda.delayGrad(x, x, 1.0)):
        with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
            call()


def test_non_tensor_and_bad_scalar_arguments():
    f = torch.ones(3)
    with pytest.raises(TypeError):
        slayerCuda.conv([1.0, 2.0], f, 1.0)
    with pytest.raises(TypeError):
        slayerLoihiCuda.getSpikes(None, 0, 64, 0, 0, 1)


def test_loihi_integer_arguments_follow_unsigned_conversion():
    from slayerpytorch_amd.slayerLoihiCuda import _unsigned
    assert _unsigned(5, "x") == 5 and _unsigned(torch.tensor(7), "x") == 7
    import numpy as np
    assert _unsigned(np.int64(3), "x") == 3
    for bad in (-1, 1.5, "3", 1 << 32, torch.tensor(1.0)):
        with pytest.raises(TypeError):
            _unsigned(bad, "x")


def test_scalar_conversion_accepts_numbers_and_one_element_tensors():
    from slayerpytorch_amd.slayerCuda import _scalar
    import numpy as np
    assert _scalar(2, "Ts") == 2.0 and _scalar(torch.tensor(0.5), "Ts") == 0.5
    assert _scalar(np.float32(0.25), "Ts") == 0.25
    with pytest.raises(TypeError):
        _scalar(torch.ones(2), "Ts")
    with pytest.raises(TypeError):
        _scalar("1.0", "Ts")


def test_layer_objects_build_without_gpu():
    neuron = {"theta": 10, "tauSr": 10.0, "tauRef": 1.0, "scaleRef": 2, "tauRho": 1, "scaleRho": 1}
    layer = snn.layer(neuron, {"Ts": 1.0, "tSample": 300})
    assert layer.srmKernel.numel() == 77 and layer.refKernel.numel() == 11
    assert set(layer.state_dict()) == {"srmKernel", "refKernel"}        # buffers travel with the state dict
    assert layer.refKernel[1].item() == pytest.approx(-20.0)
    delay = layer.delay((4, 3, 2))
    assert delay.delay.shape == (4, 3, 2) and delay.delay.requires_grad
    assert layer.delay(5).delay.shape == (5, 1, 1)
    fc = layer.dense(12, 7)
    assert fc.weight.shape == (7, 12, 1, 1, 1)
    assert layer.dense((3, 4, 2), 5).weight.shape == (5, 2, 4, 3, 1)
    ld = {"type": "LOIHI", "vThMant": 80, "vDecay": 128, "iDecay": 1024, "refDelay": 1, "wgtExp": 0,
          "tauRho": 1, "scaleRho": 1}
    loihi = snn.loihi(ld, {"Ts": 1, "tSample": 300})
    assert ld["theta"] == 5120 and loihi.maxPspKernel == 195.0 and ld["scaleRho"] == pytest.approx(1 / 195.0)
    w = loihi.dense(8, 4)
    q = w.preHookFx(w.weight)
    assert torch.all(q == torch.round(q / 2) * 2)                        # weights quantised in steps of 2


def test_dense_layer_as_matrix_product_equals_the_3d_convolution():
    # the reference's dense layer is a conv3d whose kernel spans the whole (H, W) extent; the same
    # numbers from one matrix product per batch item (time stays innermost)
    import torch.nn.functional as F
    neuron = {"theta": 10, "tauSr": 1.0, "tauRef": 1.0, "scaleRef": 2, "tauRho": 1, "scaleRho": 1}
    layer = snn.layer(neuron, {"Ts": 1.0, "tSample": 50})
    torch.manual_seed(0)
    for inF, shape in (((3, 4, 2), (2, 2, 4, 3, 17)), (12, (3, 12, 1, 1, 9)), ((5, 2), (1, 1, 2, 5, 4))):
        fc = layer.dense(inF, 6)
        x = torch.randn(shape, requires_grad=True)
        y = fc(x)
        ref = F.conv3d(x, fc.weight)
        assert y.shape == ref.shape == (shape[0], 6, 1, 1, shape[-1])
        assert torch.allclose(y, ref, rtol=1e-5, atol=1e-5)
        gy = torch.randn_like(y)
        gx, gw = torch.autograd.grad(y, (x, fc.weight), gy, retain_graph=True)
        rx, rw = torch.autograd.grad(ref, (x, fc.weight), gy)
        assert torch.allclose(gx, rx, rtol=1e-5, atol=1e-5) and torch.allclose(gw, rw, rtol=1e-4, atol=1e-4)


def test_loss_module_builds_without_gpu_and_checks_its_type():
    neuron = {"theta": 10, "tauSr": 1.0, "tauRef": 1.0, "scaleRef": 2, "tauRho": 1, "scaleRho": 1}
    desc = {"neuron": neuron, "simulation": {"Ts": 1.0, "tSample": 100},
            "training": {"error": {"type": "NumSpikes", "tgtSpikeRegion": {"start": 0, "stop": 100},
                                   "tgtSpikeCount": {True: 20, False: 5}}}}
    error = snn.loss(desc)
    assert error.slayer.srmKernel.numel() == 8
    with pytest.raises(AssertionError, match="SpikeTime"):
        error.spikeTime(torch.zeros(1, 1, 1, 1, 100), torch.zeros(1, 1, 1, 1, 100))


def test_dropin_modules_re_export_the_extension_api():
    import importlib
    import sys
    sys.path.insert(0, os.path.join(ROOT, "slayerpytorch_amd", "dropin"))
    try:
        sc = importlib.import_module("slayerCuda")
        slc = importlib.import_module("slayerLoihiCuda")
    finally:
        sys.path.pop(0)
        sys.modules.pop("slayerCuda", None)
        sys.modules.pop("slayerLoihiCuda", None)
    for name in ("getSpikes", "conv", "corr", "shift"):
        assert getattr(sc, name) is getattr(slayerCuda, name)
    assert slc.getSpikes is slayerLoihiCuda.getSpikes


def test_bench_refuses_more_than_one_gpu():
    import subprocess
    import sys
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode != 0 and "one GPU" in (r.stderr + r.stdout)


def test_synapse_and_event_wrappers_need_the_gpu():
    """No CPU path: the synapse ops and the event binning reject CPU tensors before any launch."""
    import slayerpytorch_amd as snn
    from slayerpytorch_amd import synapse
    x, w = torch.zeros((1, 2, 5, 5, 4)), torch.zeros((3, 2, 3, 3))
    with pytest.raises(RuntimeError):
        slayerCuda.getSpikesDelayed(torch.zeros((1, 2, 1, 1, 8)), torch.zeros(3), 10.0, 1.0, 2.0)
    with pytest.raises(RuntimeError):
        slayerCuda.spikeBackwardDelayed(torch.zeros((1, 2, 1, 1, 8)), torch.zeros((1, 2, 1, 1, 8)), 10.0, 10.0, 1.0, 2.0)
    with pytest.raises(RuntimeError):
        synapse.conv(x, w)
    with pytest.raises(RuntimeError):
        synapse.convGradInput(torch.zeros((1, 3, 3, 3, 4)), w, x.shape)
    with pytest.raises(RuntimeError):
        synapse.convGradWeight(torch.zeros((1, 3, 3, 3, 4)), x, w.shape)
    layer = snn.layer({"theta": 10, "tauSr": 1.0, "tauRef": 1.0, "scaleRef": 2, "tauRho": 1, "scaleRho": 1},
                      {"Ts": 1.0, "tSample": 10})
    for mod in (layer.conv(2, 3, 3), layer.pool(2), layer.convTranspose(2, 3, 3), layer.unpool(2)):
        with pytest.raises(RuntimeError):
            mod(torch.zeros((1, 2, 6, 6, 4)))
    assert layer.conv(2, 3, (3, 2), stride=(2, 1), padding=1).weight.shape == (3, 2, 3, 2, 1)
    assert float(layer.pool(2).weight.flatten()[0]) == pytest.approx(11.0)
    with pytest.raises(RuntimeError):
        snn.io.event([1], [1], [0], [1.0]).toSpikeTensor(torch.zeros((1, 4, 4, 8)))


def test_event_class_decodes_like_the_oracle():
    """Host-side members of an event read from file bytes (x, y, p shifted to start at 0, t in ms)."""
    import os
    import slayerpytorch_amd as snn
    from oracle import oracle as O
    g = np.load(os.path.join(os.path.dirname(__file__), "golden", "spike_events.npz"))
    for key, fmt in (("nmnist_bs2", 2), ("ntidigits_bs1", 1), ("sample_bs3", 3)):
        ev = snn.io.event._fromBytes(g[key], fmt)
        x, y, p, t = O.decode_events(g[key], fmt)
        assert np.array_equal(ev.x, x) and np.array_equal(ev.p, p - p.min()) and np.array_equal(ev.t, t / 1000)
        assert ev.dim == (1 if fmt == 1 else 2)
        if fmt != 1:
            assert np.array_equal(ev.y, y)


def test_dropout_and_replicate_in_time():
    """Dropout zeroes whole time rows (src/slayer.py:748-759); replicateInTime repeats along T."""
    layer = snn.layer({"theta": 10, "tauSr": 1.0, "tauRef": 1.0, "scaleRef": 2, "tauRho": 1, "scaleRho": 1},
                      {"Ts": 1.0, "tSample": 10})
    torch.manual_seed(0)
    y = layer.dropout(0.5)(torch.ones(4, 3, 5, 5, 10))
    sums = y.sum(-1).flatten()
    assert set(sums.tolist()) == {0.0, 20.0}
    x = torch.rand(2, 3, 4, 4)
    r = layer.replicateInTime(x)
    assert r.shape == (2, 3, 4, 4, 10) and torch.equal(r[..., 7], x)


def test_synapse_geometries_beyond_the_kernels_fall_back_to_torch():
    """The synapse kernels index a filter window of less than 16 MiB and batch items below 2 GiB; the decision is
    made on the host from the sizes alone, and the differentiable ops then call torch's conv3d /
    conv_transpose3d like the reference's layers do (here on CPU tensors: the fallback never reaches the
    library).  Geometries within the limits keep the kernels - and reject CPU tensors."""
    import torch.nn.functional as F
    from slayerpytorch_amd import synapse
    assert synapse.supported((12, 2, 34, 34, 300), (16, 2, 5, 5), 1, 2)
    assert not synapse.supported((1, 2, 346, 260, 5000), (8, 2, 5, 5), 1, 2)          # 5 rows of 346 x 5000 samples
    assert not synapse.supported((1, 16, 128, 128, 8192), (16, 16, 3, 3), 1, 1)       # 4 GiB per batch item
    # a small tensor whose dilated, padded window is 24.6 MB
    geo = dict(stride=1, padding=(1000, 0), dilation=(1000, 1), groups=1)
    x = torch.randn((1, 1, 4, 64, 32), requires_grad=True)
    w = torch.randn((2, 1, 2, 3, 1), requires_grad=True)
    assert not synapse.supported(x.shape, w.shape, **geo)
    y = synapse.synapseConv(x, w, **geo)
    want = F.conv3d(x, w, None, (1, 1, 1), (1000, 0, 0), (1000, 1, 1), 1)
    assert torch.equal(y, want) and y.shape == (1, 2, 1004, 62, 32)
    y.sum().backward()
    assert x.grad is not None and w.grad is not None and float(w.grad.abs().sum()) > 0
    # the transposed op of the same geometry
    z = torch.randn((1, 2, 1004, 62, 32))
    t = synapse.synapseConvTranspose(z, w.detach(), **geo)
    assert torch.equal(t, F.conv_transpose3d(z, w.detach(), None, (1, 1, 1), (1000, 0, 0), 0, 1, (1000, 1, 1)))
    assert t.shape == x.shape
    with pytest.raises(RuntimeError, match="CUDA"):
        synapse.synapseConv(torch.zeros((1, 2, 5, 5, 4)), torch.zeros((3, 2, 3, 3)), 1, 1)


def test_plans_are_kept_for_whole_numbers_only():
    """A layer's plan is kept by its sizes: what was refused before an equal one was kept is refused after, a list, an array or
    a changed tensor is worked out anew, and a geometry beyond the limits raises every time."""
    from slayerpytorch_amd import synapse
    a, w = (1, 2, 9, 9, 8), (4, 2, 3, 3)
    for _ in range(2):
        assert synapse.outShape(a, w, 2, 1) == synapse.outShape(list(a), list(w), [2, 2], (1, 1)) == (1, 4, 5, 5, 8)
        assert synapse.outShape(torch.Size(a), w + (1,), (2, 2), 1) == (1, 4, 5, 5, 8)
        with pytest.raises(TypeError):
            synapse.outShape(a, w, 2.0, 1)
        with pytest.raises(RuntimeError):
            synapse.outShape(a, (4, 3, 3, 3))
        with pytest.raises(RuntimeError):
            synapse.outShape((1, 64, 4096, 4096, 4), (6, 64, 3, 3))
    stride = torch.tensor(1)
    assert synapse.outShape(a, w, (stride, 1)) == (1, 4, 7, 7, 8)
    stride.fill_(2)
    assert synapse.outShape(a, w, (stride, 1)) == (1, 4, 4, 7, 8)


def test_an_unknown_name_of_the_native_calls_is_an_attribute_error():
    assert hasattr(_lib._Host(), "conv2d") and not hasattr(_lib._Host(), "conv4d")
    assert getattr(_lib.host, "conv4d", None) is None
    with pytest.raises(AttributeError, match="conv4d"):
        _lib.host.conv4d


def test_pool_layer_extends_odd_extents_by_zeros():
    """The pooled tensor and its gradient for odd heights and widths, against the extension that the layer stands for."""
    from slayerpytorch_amd import slayer, synapse
    layer = slayer._poolLayer(1.0, 2)
    seen = []
    keep, synapse.synapseConv = synapse.synapseConv, lambda x, *rest: seen.append(x) or x
    try:
        for H, W in [(5, 4), (4, 5), (5, 7), (4, 6)]:
            x = torch.randn(2, 3, H, W, 6, requires_grad=True)
            layer(x)
            got = seen.pop().reshape(2, 3, H + H % 2, W + W % 2, 6)
            assert torch.equal(got[:, :, :H, :W], x) and not got[:, :, H:].any() and not got[:, :, :, W:].any()
            g = torch.randn_like(got)
            got.backward(g)
            assert torch.equal(x.grad, g[:, :, :H, :W])
    finally:
        synapse.synapseConv = keep


def test_whole_row_spike_kernel_stays_within_its_rows(tmp_path):
    """Every block of LDS that the whole-row spike kernel touches lies within its row's pitch, for every row length, number
    of taps and number of rows that it serves: from spike to spike (block b and the `rounds` from there on, and a finished
    row's visits to its padding) and sample by sample (spike_walk_block)."""
    import subprocess
    source = tmp_path / "walk.cpp"
    source.write_text("""
#include "spike_rows.h"
#include <cstdio>
#include <initializer_list>
using namespace slayer;
int main()
{
    long shapes = 0, beyond = 0;
    for (int rows : {1, 1500, 3000, 5000, 1000000})
        for (int T = 1; T <= 4100; ++T)
            for (int taps = 0; taps <= 4096; taps += taps < 140 ? 1 : 97) {
                const SpikeRowsLayout l = spike_rows_layout(T, taps, rows, 256);
                if (!l.served) continue;
                ++shapes;
                const int pitch = l.pitch / l.parts;
                bool good = l.pitch % l.parts == 0 && l.pitch % 4 == 0 && l.blocks * l.parts >= T && l.blocks + l.rounds <= pitch &&
                            (l.rounds - 1) * l.parts >= taps - 1 && l.ldsBytes <= 64 * 1024;
                const SpikeWalk walk = spike_walk(l.parts, l.rounds);
                const int blocks = (T + walk.lanes - 1) / walk.lanes, end = l.pitch / walk.lanes, step = 32 / walk.lanes;
                good = good && l.pitch % walk.lanes == 0;
                for (int b0 = 0; walk.exists && b0 < blocks; b0 += step)
                    for (int m = 0; m < step + walk.rounds - 1; ++m) {
                        const int b = spike_walk_block(b0, m, walk.rounds, end);
                        // within the row; a block that is not the one asked for is padding, and so is the one taken for it
                        good = good && b >= 0 && b < end && (b == b0 + m || (b >= blocks && b0 + m >= blocks));
                    }
                if (!good) {
                    if (++beyond < 5) std::printf("rows %d T %d taps %d: %d lanes, %d blocks, pitch %d\\n", rows, T, taps, l.parts, l.blocks, pitch);
                }
            }
    std::printf("%ld shapes, %ld beyond\\n", shapes, beyond);
    return beyond != 0 || shapes < 100000;
}
""")
    program = str(tmp_path / "walk")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "slayerpytorch_amd", "csrc"), str(source), "-o", program],
                   check=True, timeout=120)
    r = subprocess.run([program], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout


def test_whole_rows_or_pieces_where_each_was_measured_faster(tmp_path):
    """Rows by length that took longer whole than in pieces, and the other way round (256 compute units, 11 taps)."""
    import subprocess
    pieces = [(640, 16000), (640, 40000), (700, 12000), (700, 16000), (760, 11000), (760, 16000), (800, 12000), (1000, 10000),
              (1000, 40000), (1200, 8000), (1500, 8000), (4036, 8000), (8000, 3)]
    whole = [(300, 200000), (600, 16000), (600, 40000), (640, 8000), (640, 12000), (640, 20000), (700, 11000), (700, 24000),
             (760, 10000), (800, 8000), (1000, 8000), (1200, 6000), (1500, 4000), (3000, 1000)]
    source = tmp_path / "rule.cpp"
    source.write_text("""
#include "spike_rows.h"
#include <cstdio>
int main()
{
    long T, rows;
    while (std::scanf("%ld %ld", &T, &rows) == 2)
        std::printf("%d\\n", slayer::spike_rows_better_in_pieces(slayer::spike_rows_layout(T, 11, rows, 256), T, rows, 256) ? 1 : 0);
}
""")
    program = str(tmp_path / "rule")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "slayerpytorch_amd", "csrc"), str(source), "-o", program],
                   check=True, timeout=120)
    r = subprocess.run([program], input="".join("%d %d\n" % s for s in pieces + whole), capture_output=True, text=True, timeout=60)
    assert r.stdout.split() == ["1"] * len(pieces) + ["0"] * len(whole)


def test_pooling_kernels_take_windows_that_lie_in_one_channel():
    """poolSupported and the entry points agree: sizes where the pooling layer, a convolution of the channels below one another,
    has no window in two channels and at least one window (EINVAL for the null pointers), and no others (EUNSUPPORTED)."""
    from slayerpytorch_amd import _lib, synapse
    lib = _lib.load()
    for KH in range(1, 6):
        for KW in (1, 2, 3):
            for C in range(1, 5):
                for H in range(1, 14):
                    for W in (1, 4, 7):
                        rows = C * (H + H % KH)
                        channels = [{row // (H + H % KH) for row in range(y, y + KH)} for y in range(0, rows - KH + 1, KH)]
                        takes = H + H % KH >= KH and W + W % KW >= KW and all(len(c) == 1 for c in channels) \
                            and len(channels) == C * ((H + H % KH) // KH)
                        sizes = (2, C, H, W, 8)
                        assert synapse.poolSupported(sizes, (1, 1, KH, KW)) == takes, (sizes, KH, KW)
                        assert lib.slayer_pool_f32(None, None, None, *sizes, KH, KW, None) == (1 if takes else 2)
                        assert lib.slayer_pool_grad_input_f32(None, None, None, None, 0.0, 1.0, 0.0, *sizes, KH, KW, None) == (1 if takes else 2)


@pytest.mark.parametrize("how", ["nobody", "tensor hook", "node prehook", "node hook", "retain_grad", "asked for", "edge", "several"])
def test_a_gradient_that_someone_watches_is_known_in_the_backward_pass(how):
    """host.watched(ctx) for a Function that may send its gradient past its first argument: every way of looking at that
    argument's gradient, registered after the call and with the tensor let go."""
    answers, seen = [], []

    class First(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            ctx.set_materialize_grads(False)
            return x * 2

        @staticmethod
        def backward(ctx, g):
            return None if g is None else g * 2

    class Second(torch.autograd.Function):
        @staticmethod
        def forward(ctx, a, x):
            return a * 3

        @staticmethod
        def backward(ctx, g):
            answers.append(_lib.host.watched(ctx))
            return (g * 3, None) if answers[-1] else (None, g * 6)

    x = torch.ones(3, requires_grad=True)
    a = First.apply(x)
    y = Second.apply(a, x).sum()
    wanted = [x]
    if how == "tensor hook":
        a.register_hook(lambda g: (seen.append(g), g * 2)[1])
    elif how == "node prehook":
        a.grad_fn.register_prehook(lambda gs: (seen.append(gs[0]), (gs[0] * 2,))[1])
    elif how == "node hook":
        a.grad_fn.register_hook(lambda gi, go: (seen.append(go[0]), (gi[0] * 2,))[1])
    elif how == "retain_grad":
        a.retain_grad()
    elif how == "several":
        torch.autograd.graph.register_multi_grad_hook([a], lambda gs: seen.append(gs[0]))
    elif how in ("asked for", "edge"):
        wanted = [x, a] if how == "asked for" else [x, torch.autograd.graph.get_gradient_edge(a)]
    if how != "retain_grad":
        del a
    got = torch.autograd.grad(y, wanted)
    assert answers == [how != "nobody"]
    assert torch.equal(got[0], torch.full((3,), 12.0 if how in ("tensor hook", "node prehook", "node hook") else 6.0))
    assert all(torch.equal(g, torch.full((3,), 3.0)) for g in (*seen, *got[1:]))
    assert len(seen) == (how in ("tensor hook", "node prehook", "node hook", "several"))


@pytest.mark.parametrize("traceable", [True, False])
def test_a_function_of_this_package_can_be_compiled(traceable):
    """torch.compile takes a model that calls one of the package's Functions: into its graph where it can follow the Function,
    around it where it cannot (the kernels are called through ctypes and an extension module)."""
    from slayerpytorch_amd._function import Function
    _lib.host.unwrapped(torch.ones(1))               # the extension module is there, as in a model that has run before

    class Scaled(Function):
        @staticmethod
        def forward(ctx, x, k):
            ctx.k = k
            return x * k if traceable else torch.from_numpy(x.detach().numpy() * (k if _lib.host.unwrapped(x) else 0.0))

        @staticmethod
        def backward(ctx, g):
            return g * ctx.k, None

    class Model(torch.nn.Module):
        def forward(self, x):
            return Scaled.apply(x + 1, 3.0) * 2

    torch._dynamo.reset()
    model = torch.compile(Model(), backend="eager", fullgraph=traceable)
    x = torch.ones(3, requires_grad=True)
    y = model(x)
    (grad,) = torch.autograd.grad(y.sum(), x)
    assert torch.equal(y, torch.full((3,), 12.0)) and torch.equal(grad, torch.full((3,), 6.0))
