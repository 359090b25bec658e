"""Cases by which the speed of this framework is measured: whole passes of the networks that its benchmark, tests and
configurations use, through the public entry points (``snn.layer``, ``snn.loihi``, ``snn.loss``, ``snn.io``).

``listed()`` the cases, ``draw(rng)`` one more of the same ranges, ``prepare(case, seed)`` inputs and weights on the
GPU, ``run(state)`` one pass and its outputs, ``work(case)`` bytes and operations that the pass cannot do without,
``tolerance(case)`` how far two correct implementations of the same precision differ.
"""
import math

import numpy as np
import torch

import slayerpytorch_amd as snn


def listed():
    return [
        # the 250-25-1 network of the tests' fixture, one sample, Ts = 0.1: the smallest training step there is,
        # all launches and host work
        dict(name="small_train", kind="mlp", order="psp_first", batch=1, channels=250, height=1, width=1, hidden=25,
             outputs=1, steps=500, Ts=0.1, tauSr=1.0, rate=0.01, train=True, loss="SpikeTime"),
        # one sample through the NMNIST MLP: serving latency
        dict(name="mlp_single", kind="mlp", order="fc_first", batch=1, channels=2, height=34, width=34, hidden=512,
             outputs=10, steps=350, Ts=1.0, tauSr=10.0, rate=0.015, train=False, loss="SpikeTime"),
        # the NMNIST MLP's training step at its batch size: ordinary, many short kernels, sparse dense-layer input
        dict(name="mlp_train", kind="mlp", order="fc_first", batch=12, channels=2, height=34, width=34, hidden=512,
             outputs=10, steps=350, Ts=1.0, tauSr=10.0, rate=0.015, train=True, loss="SpikeTime"),
        # the NMNIST CNN's training step at its batch size: the framework's main workload
        dict(name="cnn_train", kind="cnn", batch=12, height=34, width=34, steps=300, rate=0.02, train=True,
             loss="SpikeTime"),
        # the same network on a large batch: every tensor beyond the caches
        dict(name="cnn_train_large", kind="cnn", batch=64, height=34, width=34, steps=300, rate=0.02, train=True,
             loss="NumSpikes"),
        # the same network forward only: evaluation
        dict(name="cnn_infer", kind="cnn", batch=32, height=34, width=34, steps=300, rate=0.02, train=False,
             loss="SpikeTime"),
        # odd extents everywhere: an image whose halves are odd, an odd number of time steps, few samples
        dict(name="cnn_train_ragged", kind="cnn", batch=5, height=29, width=37, steps=173, rate=0.03, train=True,
             loss="NumSpikes"),
        # long sequences through two dense layers with a learnable delay per neuron
        dict(name="delay_train", kind="delay", batch=64, inputs=200, hidden=256, steps=2000, rate=0.005),
        # the gesture network on the Loihi neuron, quantised weights: evaluation at the benchmark's length
        dict(name="gesture_infer", kind="gesture", batch=8, size=128, steps=300, rate=0.01, train=False),
        # and its training step at the length and batch size of the gesture recordings
        dict(name="gesture_train", kind="gesture", batch=4, size=128, steps=1450, rate=0.01, train=True),
        # the temporal kernels alone, forward and backward, on the largest activation tensor of the CNN
        dict(name="temporal", kind="temporal", batch=12, channels=16, height=34, width=34, steps=300, delay=1),
        # a batch of event files to a spike tensor: what a data loader does before each of the steps above
        dict(name="events", kind="events", batch=12, count=5000, height=34, width=34, steps=300, binning="OR"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over lo..hi by its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "cnn", "cnn", "cnn", "delay", "gesture", "temporal", "events"])
    train = rng.random() < 0.7
    loss = rng.choice(["SpikeTime", "NumSpikes"])
    if kind == "mlp":
        small = rng.random() < 0.4
        return dict(kind="mlp", order=rng.choice(["psp_first", "fc_first"]), batch=_log(rng, 1, 32),
                    channels=rng.randint(20, 400) if small else 2, height=1 if small else rng.randint(20, 40),
                    width=1 if small else rng.randint(20, 40), hidden=_log(rng, 20, 512), outputs=rng.randint(1, 20),
                    steps=_log(rng, 100, 500), Ts=1.0, tauSr=10.0, rate=round(rng.uniform(0.01, 0.03), 4), train=train,
                    loss=loss)
    if kind == "cnn":
        height, width, steps = rng.randint(20, 40), rng.randint(20, 40), _log(rng, 100, 400)
        most = 64 * 34 * 34 * 300 // (height * width * steps)
        return dict(kind="cnn", batch=_log(rng, 1, min(48, most)), height=height, width=width, steps=steps,
                    rate=round(rng.uniform(0.01, 0.04), 4), train=train, loss=loss)
    if kind == "delay":
        return dict(kind="delay", batch=_log(rng, 1, 64), inputs=_log(rng, 30, 256), hidden=_log(rng, 30, 256),
                    steps=_log(rng, 200, 2000), rate=round(rng.uniform(0.003, 0.02), 4))
    if kind == "gesture":
        size, steps = 16 * rng.randint(2, 8), _log(rng, 100, 1450)
        return dict(kind="gesture", batch=_log(rng, 1, min(8, 4 * 1450 // steps)), size=size, steps=steps,
                    rate=round(rng.uniform(0.005, 0.02), 4), train=train)
    if kind == "temporal":
        channels, height, width, steps = _log(rng, 1, 64), rng.randint(1, 36), rng.randint(1, 36), _log(rng, 60, 2000)
        most = max(1, 12 * 16 * 34 * 34 * 300 // (channels * height * width * steps))
        return dict(kind="temporal", batch=_log(rng, 1, min(64, most)), channels=channels, height=height, width=width,
                    steps=steps, delay=rng.randint(0, 20))
    size, steps = rng.randint(20, 128), _log(rng, 60, 1450)
    most = max(1, 64 * 2 * 34 * 34 * 300 // (2 * size * size * steps))
    return dict(kind="events", batch=_log(rng, 1, min(64, most)), count=_log(rng, 300, 20000), height=size, width=size,
                steps=steps, binning=rng.choice(["OR", "SUM"]))


_REGION = 0.5      # part of the time axis in which the spike-count loss counts


def _srm(case, tauSr=10.0, Ts=1.0):
    """Neuron and simulation of the SRM networks (theta 10, tauRef 1), and the loss' descriptor."""
    neuron = {"type": "SRMALPHA", "theta": 10.0, "tauSr": tauSr, "tauRef": 1.0, "scaleRef": 2.0,
              "tauRho": 0.1 if Ts < 1 else 1.0, "scaleRho": 1.0}
    sim = {"Ts": Ts, "tSample": case["steps"] * Ts}
    error = {"type": case.get("loss", "SpikeTime"), "tgtSpikeCount": {True: 20, False: 3},
             "tgtSpikeRegion": {"start": 0, "stop": int(case["steps"] * Ts * _REGION)}}
    return neuron, sim, {"neuron": neuron, "simulation": sim, "training": {"error": error}}


def _spikes(gen, shape, rate, Ts=1.0):
    return (torch.rand(shape, generator=gen, device="cuda") < rate).float().div_(Ts)


def _target(case, gen, outputs, net, Ts=1.0):
    """What the loss compares with: a target train, or a one-hot class."""
    if case["loss"] == "SpikeTime":
        return _spikes(gen, (case["batch"], outputs, 1, 1, case["steps"]), 0.01, Ts)
    wanted = torch.randint(0, outputs, (case["batch"],), generator=gen, device="cuda")
    return torch.nn.functional.one_hot(wanted, outputs).bool().reshape(case["batch"], outputs, 1, 1, 1)


# Weight scales at which the layers of these networks fire as trained ones do, a few per cent of the time (measured;
# pooled layers fire more, their weights are constants).
_MLP_SCALE = {"psp_first": (1.0, 16.0), "fc_first": (1.0, 9.0)}
_CNN_SCALE = (1.0, 1.5, 2.2, 8.0)
_DELAY_SCALE = (110.0, 60.0)


def _first_scale(rate):
    """Weight scale of a first layer: independent input spikes at this rate through a filter of time constant 10 have a
    mean square of 18.5 rate + (27.2 rate)^2."""
    return 21.0 / math.sqrt(18.5 * rate + (27.2 * rate) ** 2)


def prepare(case, seed):
    torch.manual_seed(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case, "kind": case["kind"]}
    if case["kind"] == "mlp":
        neuron, sim, net = _srm(case, case["tauSr"], case["Ts"])
        layer = snn.layer(neuron, sim).cuda()
        shape = (case["batch"], case["channels"], case["height"], case["width"], case["steps"])
        flat = case["height"] == case["width"] == 1
        scale = _MLP_SCALE[case["order"]]
        fc1 = layer.dense(case["channels"] if flat else (case["width"], case["height"], case["channels"]), case["hidden"],
                          weightScale=scale[0] * _first_scale(case["rate"])).cuda()
        fc2 = layer.dense(case["hidden"], case["outputs"], weightScale=scale[1]).cuda()
        state.update(layer=layer, synapses=[fc1, fc2], input=_spikes(gen, shape, case["rate"], case["Ts"]),
                     target=_target(case, gen, case["outputs"], net, case["Ts"]), error=snn.loss(net).cuda())
    elif case["kind"] == "cnn":
        neuron, sim, net = _srm(case)
        layer = snn.layer(neuron, sim).cuda()
        shape = (case["batch"], 2, case["height"], case["width"], case["steps"])
        _, (h, w) = _cnn_extents(case)
        synapses = [layer.conv(2, 16, 5, padding=1, weightScale=_CNN_SCALE[0] * _first_scale(case["rate"])), layer.pool(2),
                    layer.conv(16, 32, 3, padding=1, weightScale=_CNN_SCALE[1]), layer.pool(2),
                    layer.conv(32, 64, 3, padding=1, weightScale=_CNN_SCALE[2]),
                    layer.dense((w, h, 64), 10, weightScale=_CNN_SCALE[3])]
        state.update(layer=layer, synapses=[s.cuda() for s in synapses], input=_spikes(gen, shape, case["rate"]),
                     target=_target(case, gen, 10, net), error=snn.loss(net).cuda())
    elif case["kind"] == "delay":
        neuron, sim, net = _srm(case, tauSr=1.0)
        layer = snn.layer(neuron, sim).cuda()
        shape = (case["batch"], case["inputs"], 1, 1, case["steps"])
        fc1 = layer.dense(case["inputs"], case["hidden"], weightScale=_DELAY_SCALE[0]).cuda()
        fc2 = layer.dense(case["hidden"], case["inputs"], weightScale=_DELAY_SCALE[1]).cuda()
        d1, d2 = layer.delay(case["hidden"]).cuda(), layer.delay(case["inputs"]).cuda()
        with torch.no_grad():
            d1.delay.mul_(62.0)
            d2.delay.mul_(62.0)
        state.update(layer=layer, synapses=[fc1, fc2], delays=[d1, d2], input=_spikes(gen, shape, case["rate"]),
                     target=_spikes(gen, shape, 0.01), error=snn.loss(net).cuda())
    elif case["kind"] == "gesture":
        neuron = {"type": "LOIHI", "vThMant": 80, "vDecay": 128, "iDecay": 1024, "refDelay": 1, "wgtExp": 0, "tauRho": 1,
                  "scaleRho": 1}
        sim = {"Ts": 1, "tSample": case["steps"]}
        layer = snn.loihi(neuron, sim).cuda()
        synapses = [layer.pool(4), layer.conv(2, 16, 5, padding=2, weightScale=10), layer.pool(2),
                    layer.conv(16, 32, 3, padding=1, weightScale=50), layer.pool(2),
                    layer.dense((case["size"] // 16) ** 2 * 32, 512), layer.dense(512, 11)]
        net = {"neuron": dict(neuron), "simulation": sim, "training": {"error": {"type": "SpikeTime"}}}
        state.update(layer=layer, synapses=[s.cuda() for s in synapses],
                     input=_spikes(gen, (case["batch"], 2, case["size"], case["size"], case["steps"]), case["rate"]),
                     target=_spikes(gen, (case["batch"], 11, 1, 1, case["steps"]), 0.02),
                     error=snn.loss(net, snn.loihi).cuda())
    elif case["kind"] == "temporal":
        neuron, sim, _ = _srm(case)
        shape = (case["batch"], case["channels"], case["height"], case["width"], case["steps"])
        # weighted input spikes, smooth potentials above the threshold for runs of samples
        x = _spikes(gen, shape, 0.05).mul_(torch.randn(shape, generator=gen, device="cuda").mul_(9.0))
        state.update(layer=snn.layer(neuron, sim).cuda(), input=x.requires_grad_(True),
                     grad=torch.randn(shape, generator=gen, device="cuda"))
    else:
        rng = np.random.default_rng(seed)
        files = []
        for _ in range(case["batch"]):
            n = case["count"]
            x, y, p = rng.integers(0, case["width"], n), rng.integers(0, case["height"], n), rng.integers(0, 2, n)
            # a few events lie beyond the tensor's last time step, as in recordings that were cut
            t = np.sort(rng.integers(0, min(1050 * case["steps"], 1 << 23), n))
            packed = np.zeros((n, 5), dtype=np.uint8)
            packed[:, 0], packed[:, 1], packed[:, 2] = x, y, ((t >> 16) & 0x7F) | (p << 7)
            packed[:, 3], packed[:, 4] = (t >> 8) & 0xFF, t & 0xFF
            files.append(packed.reshape(-1))
        # (what io.read2Dspikes makes of a file's bytes; files come from the page cache in earnest, not from disk)
        state.update(events=[snn.io.event._fromBytes(f, 2) for f in files])
    return state


def _forward(state):
    layer, s = state["layer"], state["input"]
    if state["kind"] == "mlp":
        for fc in state["synapses"]:
            s = layer.spike(layer.psp(fc(s))) if state["case"]["order"] == "fc_first" else layer.spike(fc(layer.psp(s)))
    elif state["kind"] == "cnn":
        for synapse in state["synapses"]:
            s = layer.spike(synapse(layer.psp(s)))
    elif state["kind"] == "delay":
        for fc, delay in zip(state["synapses"], state["delays"]):
            s = delay(layer.spike(layer.psp(fc(s))))
    else:
        for k, synapse in enumerate(state["synapses"]):
            if k == 5:
                s = s.reshape(s.shape[0], -1, 1, 1, s.shape[-1])
            s = layer.spikeLoihi(synapse(s), delay=1)
    return s


def run(state):
    case, kind = state["case"], state["kind"]
    if kind == "events":
        empty = torch.zeros((case["batch"], 2, case["height"], case["width"], case["steps"]), device="cuda")
        return snn.io.toSpikeTensorBatch(state["events"], empty, 1.0, binningMode=case["binning"])
    if kind == "temporal":
        layer, x = state["layer"], state["input"]
        out = layer.delayShift(layer.spike(layer.psp(x)), case["delay"])
        (grad,) = torch.autograd.grad(out, x, state["grad"])
        return {"raster": out.detach() > 0, "grad": grad}
    if kind != "delay" and not case["train"]:
        with torch.no_grad():
            return _forward(state) > 0      # the raster of the output layer
    weights = [s.weight for s in state["synapses"] if s.weight.requires_grad] + [d.delay for d in state.get("delays", [])]
    for w in weights:
        w.grad = None
    out = _forward(state)
    if case.get("loss") == "NumSpikes":
        loss = state["error"].numSpikes(out, state["target"])
    else:
        loss = state["error"].spikeTime(out, state["target"])
    loss.backward()
    return [loss.detach()] + [w.grad for w in weights]


def _cnn_extents(case):
    """Extents of the layers' outputs: conv 5x5 padded by 1, pool, conv 3x3 padded by 1, pool (odd extents are
    extended by one row)."""
    h, w = case["height"] - 2, case["width"] - 2
    half = lambda v: (v + v % 2) // 2
    h2, w2 = half(h), half(w)
    h4, w4 = half(h2), half(w2)
    return [(2 * case["height"] * case["width"], 16 * h * w, 50), (16 * h * w, 16 * h2 * w2, 0),
            (16 * h2 * w2, 32 * h2 * w2, 144), (32 * h2 * w2, 32 * h4 * w4, 0), (32 * h4 * w4, 64 * h4 * w4, 288),
            (64 * h4 * w4, 10, 64 * h4 * w4)], (h4, w4)


def work(case):
    """Each call of the pass is taken to read its input tensors once and to write its output tensors once (a user's
    program holds every one of them); operations are the synapses' multiply-adds, three times as many with
    gradients.  Samples are counted per time step."""
    steps = case["batch"] * case["steps"]
    if case["kind"] == "events":
        return {"bytes": 5.0 * case["batch"] * case["count"] + 8.0 * steps * case["height"] * case["width"], "flops": 0}
    if case["kind"] == "temporal":
        # psp 2, spike 3 (the potential is updated in place), shift 2; backward: shift 2, surrogate gradient and
        # correlation 3
        n = float(steps * case["channels"] * case["height"] * case["width"])
        return {"bytes": 4 * 12 * n, "flops": 0}
    if case["kind"] == "mlp":
        first = case["channels"] * case["height"] * case["width"]
        layers = [(first, case["hidden"], first), (case["hidden"], case["outputs"], case["hidden"])]
    elif case["kind"] == "cnn":
        layers = _cnn_extents(case)[0]
    elif case["kind"] == "delay":
        layers = [(case["inputs"], case["hidden"], case["inputs"]), (case["hidden"], case["inputs"], case["hidden"])]
    else:
        q = (case["size"] // 4) ** 2
        layers = [(32 * q, 2 * q, 0), (2 * q, 16 * q, 50), (16 * q, 4 * q, 0), (4 * q, 8 * q, 144), (8 * q, 2 * q, 0),
                  (2 * q, 512, 2 * q), (512, 11, 512)]
    train = case.get("train", True)
    moved, products = 0.0, 0.0
    for k, (n_in, n_out, taps) in enumerate(layers):
        fed = (2 * n_in if case["kind"] == "cnn" or case.get("order") == "psp_first" else 0) \
            + (2 * n_out if case["kind"] == "delay" or case.get("order") == "fc_first" else 0)
        neuron = {"gesture": 2 + train, "delay": 3 + 2}.get(case["kind"], 3)
        moved += fed + n_in + n_out + neuron * n_out
        products += 2.0 * n_out * taps
        if train:
            # the neuron's gradient with the filter's correlation, the synapse's two gradients (none for the
            # network's input), the delays' gradient
            moved += 3 * n_out + (n_in + n_out if taps else 0) + (n_in + n_out if k else 0)
            moved += 2 * n_out if case["kind"] == "delay" else 0
            products += 2.0 * n_out * taps * (2 if k else 1)
    return {"bytes": 4.0 * steps * moved, "flops": steps * products}


def tolerance(case):
    """Whole numbers where the path is in whole numbers (Loihi neuron forward, events).  Elsewhere the potentials are
    32-bit sums whose rounding moves a few spikes in a million across the threshold, and every such spike moves the
    gradients behind it, the more the smaller the batch (measured: filters as sums over their taps and library
    products against the recursion and the framework's products; about four times the largest difference seen)."""
    if case["kind"] == "events" or (case["kind"] == "gesture" and not case["train"]):
        return "exact"
    if case["kind"] == "gesture":
        return {"rel": 1e-5}
    if case["kind"] == "temporal":
        return {"rel": 1e-3, "max": 0.99, "differ": 1e-6}
    if case["kind"] == "delay":
        return {"rel": 1e-3, "max": 0.2}
    if case["kind"] == "mlp":
        return {"rel": 3e-3, "max": 0.2, "differ": 2e-3}
    return {"rel": 8e-3 if case["batch"] * case["steps"] >= 2000 else 3e-2, "max": 0.6, "differ": 6e-3}
