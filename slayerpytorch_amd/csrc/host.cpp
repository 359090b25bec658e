// The calls that a layer makes on every pass, from Python to the C ABI in one step each: what slayerCuda.py,
// slayerLoihiCuda.py and synapse.py do around an entry point - looking at the tensors, allocating the result and
// workspaces, finding the stream - costs 4 to 6 us per call in Python and ctypes, as much as the launch itself and more
// than the kernels of a small network take.
//
// Every function takes the positional arguments of its namesake there and answers None for anything but the plain case
// (exact torch.Tensor objects, contiguous fp32 on one GPU, Python numbers, sizes that the entry point takes): the caller
// then goes through its own checks, which raise what they always raised, and its general path.  Nothing has been launched
// where None is returned: a launch that reports an error - it may be one that another HIP call left, the kernel running all
// the same - raises here.  No state is kept.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/function_hook.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/autograd/python_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <string>

#include "../../include/slayer_hip.h"

namespace {

// A tensor whose memory may be handed to a kernel as it is.
bool plain(const at::Tensor &t)
{
    using c10::DispatchKey;
    return t.defined() && t.is_cuda() && t.scalar_type() == at::kFloat && t.layout() == at::kStrided && t.has_storage() &&
           t.is_contiguous() && !t.is_neg() && !t.is_quantized() && !t.is_nested() &&
           !t.key_set().has_any(c10::DispatchKeySet({DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                                     DispatchKey::Functionalize}));
}

// The arguments of a call; ok goes false with the first one that is not plain.
struct Args {
    const char *name;    // of the function
    PyObject *const *a;
    Py_ssize_t n;
    bool ok;
    c10::Device device;

    Args(const char *function, PyObject *const *args, Py_ssize_t count, Py_ssize_t expected)
        : name(function), a(args), n(count), ok(count == expected), device(c10::DeviceType::CUDA, -1) {}

    const at::Tensor *tensor(Py_ssize_t i)
    {
        if (!ok || !THPVariable_CheckExact(a[i])) return fail();
        const at::Tensor &t = THPVariable_Unpack(a[i]);
        if (!plain(t) || (device.index() >= 0 && t.device() != device)) return fail();
        device = t.device();
        return &t;
    }
    const at::Tensor *tensorOrNone(Py_ssize_t i) { return ok && a[i] == Py_None ? nullptr : tensor(i); }
    double number(Py_ssize_t i)
    {
        if (ok && PyFloat_CheckExact(a[i])) return PyFloat_AS_DOUBLE(a[i]);
        if (ok && PyLong_CheckExact(a[i])) {
            const double v = PyLong_AsDouble(a[i]);
            if (v == -1.0 && PyErr_Occurred()) PyErr_Clear();
            else return v;
        }
        ok = false;
        return 0.0;
    }
    int64_t integer(Py_ssize_t i)
    {
        if (ok && (PyLong_CheckExact(a[i]) || PyBool_Check(a[i]))) {
            int overflow = 0;
            const long long v = PyLong_AsLongLongAndOverflow(a[i], &overflow);
            if (!overflow && !(v == -1 && PyErr_Occurred())) return v;
            PyErr_Clear();
        }
        ok = false;
        return 0;
    }
    bool truth(Py_ssize_t i)
    {
        if (ok && PyBool_Check(a[i])) return a[i] == Py_True;
        ok = false;
        return false;
    }
    // a whole number within [lo, hi]
    int64_t within(Py_ssize_t i, int64_t lo, int64_t hi)
    {
        const int64_t v = integer(i);
        if (v < lo || v > hi) ok = false;
        return v;
    }
    // (h, w) from an int or a tuple of two ints
    void pair(Py_ssize_t i, int32_t &h, int32_t &w)
    {
        if (!ok) return;
        if (PyLong_CheckExact(a[i])) {
            h = w = narrow(a[i]);
        } else if (PyTuple_CheckExact(a[i]) && PyTuple_GET_SIZE(a[i]) == 2) {
            h = narrow(PyTuple_GET_ITEM(a[i], 0));
            w = narrow(PyTuple_GET_ITEM(a[i], 1));
        } else {
            ok = false;
        }
    }

  private:
    const at::Tensor *fail()
    {
        ok = false;
        return nullptr;
    }
    int32_t narrow(PyObject *o)
    {
        if (!PyLong_CheckExact(o)) { ok = false; return 0; }
        int overflow = 0;
        const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
        if (overflow || v < 0 || v > (1 << 24)) { ok = false; return 0; }
        return static_cast<int32_t>(v);
    }
};

template <typename T = float> T *ptr(const at::Tensor &t) { return t.numel() ? static_cast<T *>(t.data_ptr()) : nullptr; }
template <typename T = float> T *ptr(const at::Tensor *t) { return t ? ptr<T>(*t) : nullptr; }

void rows(const at::Tensor &x, int64_t &n, int64_t &T)
{
    T = x.dim() ? x.size(-1) : 1;
    n = T ? x.numel() / T : 0;
}

at::Tensor floats(at::IntArrayRef shape, const c10::Device &device)
{
    return at::empty(shape, at::TensorOptions().dtype(at::kFloat).device(device));
}

// The package's error for a launch that reported one, as _lib.check raises it.
[[noreturn]] void raise_launch_error(const char *name)
{
    const std::string text = std::string(name) + " failed: " + slayer_status_string(SLAYER_ELAUNCH) + " (" + slayer_last_hip_error() + ")";
    THPObjectPtr module(PyImport_ImportModule("slayerpytorch_amd._lib"));
    THPObjectPtr error(module ? PyObject_GetAttrString(module.get(), "SlayerHipError") : nullptr);
    if (error) PyErr_SetString(error.get(), text.c_str());
    throw python_error();
}

// Runs the entry point on the tensors' device and PyTorch's current stream there, without the interpreter's lock (as a
// ctypes call does).  True: launched.  False: refused, nothing was launched.
template <typename Call> bool launch(const Args &a, Call call)
{
    const c10::DeviceGuard guard(a.device);
    void *stream = c10::hip::getCurrentHIPStream(a.device.index()).stream();
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = call(stream);
    Py_END_ALLOW_THREADS
    if (status == SLAYER_ELAUNCH) raise_launch_error(a.name);
    return status == SLAYER_OK;
}

PyObject *none() { Py_RETURN_NONE; }
PyObject *wrapped(bool launched, const at::Tensor &t) { return launched ? THPVariable_Wrap(t) : none(); }

#define SLAYER_HOST(NAME) PyObject *NAME(PyObject *, PyObject *const *args, Py_ssize_t nargs)
#define SLAYER_ARGS(COUNT) Args a(__func__, args, nargs, COUNT)
#define SLAYER_PLAIN \
    if (!a.ok) return none()

bool same(const at::Tensor *x, const at::Tensor *y) { return x && y && x->sizes() == y->sizes(); }

// ---- the temporal kernels ------------------------------------------------------------------------------
SLAYER_HOST(getSpikes)   // (d_u, d_nu, theta, Ts)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(4);
    const at::Tensor *u = a.tensor(0), *nu = a.tensor(1);
    const float theta = a.number(2), Ts = a.number(3);
    SLAYER_PLAIN;
    if (u->dim() != 5) return none();
    const at::Tensor s = at::empty_like(*u);
    int64_t n, T;
    rows(*u, n, T);
    const int64_t taps = nu->dim() ? nu->size(-1) : 1;
    return wrapped(launch(a, [&](void *st) { return slayer_get_spikes_f32(ptr(s), ptr(u), ptr(nu), n, T, taps, theta, Ts, st); }), s);
    END_HANDLE_TH_ERRORS
}

template <int (*ENTRY)(float *, const float *, const float *, int64_t, int64_t, int64_t, float, void *)>
SLAYER_HOST(fir)         // (input, filter, Ts)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(3);
    const at::Tensor *x = a.tensor(0), *f = a.tensor(1);
    const float Ts = a.number(2);
    SLAYER_PLAIN;
    const at::Tensor y = at::empty_like(*x);
    int64_t n, T;
    rows(*x, n, T);
    return wrapped(launch(a, [&](void *st) { return ENTRY(ptr(y), ptr(x), ptr(f), n, T, f->numel(), Ts, st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(pspAlpha)    // (input, filter, tau, mult, Ts, causal)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(6);
    const at::Tensor *x = a.tensor(0), *f = a.tensor(1);
    const float tau = a.number(2), mult = a.number(3), Ts = a.number(4);
    const bool causal = a.truth(5);
    SLAYER_PLAIN;
    if (f->numel() < 1) return none();
    const at::Tensor y = at::empty_like(*x);
    int64_t n, T;
    rows(*x, n, T);
    return wrapped(launch(a, [&](void *st) {
        return slayer_psp_alpha_f32(ptr(y), ptr(x), ptr(f), n, T, f->numel(), tau, mult, Ts, causal ? 1 : 0, st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(spikeBackward)   // (gradOutput, membranePotential, theta, tau, scale)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(5);
    const at::Tensor *g = a.tensor(0), *u = a.tensor(1);
    const float theta = a.number(2), tau = a.number(3), scale = a.number(4);
    SLAYER_PLAIN;
    if (!same(g, u)) return none();
    const at::Tensor y = at::empty_like(*g);
    return wrapped(launch(a, [&](void *st) { return slayer_spike_bwd_f32(ptr(y), ptr(g), ptr(u), theta, tau, scale, g->numel(), st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(spikeBackwardPspAlpha)   // (gradOutput, membranePotential, filter, tauSr, mult, theta, tau, scale, Ts)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(9);
    const at::Tensor *g = a.tensor(0), *u = a.tensor(1), *f = a.tensor(2);
    float v[6];
    for (int i = 0; i < 6; ++i) v[i] = a.number(3 + i);
    SLAYER_PLAIN;
    if (!same(g, u) || f->numel() < 1) return none();
    const at::Tensor y = at::empty_like(*g);
    int64_t n, T;
    rows(*g, n, T);
    return wrapped(launch(a, [&](void *st) {
        return slayer_spike_bwd_psp_alpha_f32(ptr(y), ptr(g), ptr(u), ptr(f), n, T, f->numel(), v[0], v[1], v[2], v[3], v[4], v[5], st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(pspSpikeBackwardAlpha)   // (gradPsp, gradSpike or None, membranePotential, filter, tauSr, mult, theta, tau, scale, Ts)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(10);
    const at::Tensor *g = a.tensor(0), *more = a.tensorOrNone(1), *u = a.tensor(2), *f = a.tensor(3);
    float v[6];
    for (int i = 0; i < 6; ++i) v[i] = a.number(4 + i);
    SLAYER_PLAIN;
    if (!same(g, u) || (more && !same(g, more)) || f->numel() < 1) return none();
    const at::Tensor y = at::empty_like(*g);
    int64_t n, T;
    rows(*g, n, T);
    return wrapped(launch(a, [&](void *st) {
        return slayer_psp_spike_bwd_alpha_f32(ptr(y), ptr(g), ptr(more), ptr(u), ptr(f), n, T, f->numel(), v[0], v[1], v[2], v[3], v[4], v[5], st); }), y);
    END_HANDLE_TH_ERRORS
}

// A delay as a number or as a table with one entry per neuron of a batch item (or one entry).
struct Delay {
    const at::Tensor *table = nullptr;
    double value = 0.0;
    Delay(Args &a, Py_ssize_t i)
    {
        if (!a.ok) return;
        if (THPVariable_Check(a.a[i])) table = a.tensor(i);
        else value = a.number(i);
    }
    bool fits(const at::Tensor &x, int64_t n) const
    {
        return !table || table->numel() == 1 || (x.dim() > 0 && x.size(0) > 0 && table->numel() == n / x.size(0));
    }
};

SLAYER_HOST(shift)       // (input, number or table, Ts, sign)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(4);
    const at::Tensor *x = a.tensor(0);
    const Delay delay(a, 1);
    const float Ts = a.number(2);
    const double sign = a.number(3);
    SLAYER_PLAIN;
    int64_t n, T;
    rows(*x, n, T);
    if (!delay.fits(*x, n)) return none();
    const at::Tensor y = at::empty_like(*x);
    if (!delay.table)
        return wrapped(launch(a, [&](void *st) {
            return slayer_shift_f32(ptr(y), ptr(x), static_cast<float>(delay.value * sign), n, T, Ts, st); }), y);
    const bool one = delay.table->numel() == 1;
    const int64_t nBatch = one ? 1 : x->size(0), perBatch = one ? n : n / nBatch;
    return wrapped(launch(a, [&](void *st) {
        return slayer_shift_lut_f32(ptr(y), ptr(x), ptr(delay.table), delay.table->numel(), nBatch, perBatch, T, Ts, static_cast<float>(sign), st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(spikeBackwardDelayed)   // (gradOutput, membranePotential, theta, tau, scale, delay, delayTs)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(7);
    const at::Tensor *g = a.tensor(0), *u = a.tensor(1);
    const float theta = a.number(2), tau = a.number(3), scale = a.number(4);
    const Delay delay(a, 5);
    const float delayTs = a.number(6);
    SLAYER_PLAIN;
    int64_t n, T;
    rows(*g, n, T);
    if (!same(g, u) || !delay.fits(*g, n)) return none();
    const at::Tensor y = at::empty_like(*g);
    return wrapped(launch(a, [&](void *st) {
        return slayer_spike_bwd_delayed_f32(ptr(y), ptr(g), ptr(u), ptr(delay.table), delay.table ? delay.table->numel() : 0,
                                            static_cast<float>(delay.value),
                                            delayTs, n, T, theta, tau, scale, st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(delayGrad)   // (output, gradOutput, Ts)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(3);
    const at::Tensor *y = a.tensor(0), *g = a.tensor(1);
    const float Ts = a.number(2);
    SLAYER_PLAIN;
    if (!same(y, g) || y->dim() < 2) return none();
    const int64_t T = y->size(-1), nBatch = y->size(0);
    const at::IntArrayRef shape = y->sizes().slice(1, y->dim() - 2);
    int64_t perBatch = 1;
    for (int64_t d : shape) perBatch *= d;
    const at::Tensor out = floats(shape, a.device);
    const int64_t bytes = slayer_delay_grad_workspace_bytes(nBatch, perBatch, T);
    const at::Tensor work = floats({(bytes < 4 ? 4 : bytes) / 4}, a.device);
    return wrapped(launch(a, [&](void *st) {
        return slayer_delay_grad_f32(ptr(out), ptr(y), ptr(g), work.data_ptr<float>(), nBatch, perBatch, T, Ts, st); }), out);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(spikeBackwardDelayedCorr)   // (gradOutput, membranePotential, filter, delaySteps, theta, tau, scale, Ts)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(8);
    const at::Tensor *g = a.tensor(0), *u = a.tensor(1), *f = a.tensor(2);
    const int64_t steps = a.integer(3);
    const float theta = a.number(4), tau = a.number(5), scale = a.number(6), Ts = a.number(7);
    SLAYER_PLAIN;
    if (!same(g, u)) return none();
    const at::Tensor y = at::empty_like(*g);
    int64_t n, T;
    rows(*g, n, T);
    return wrapped(launch(a, [&](void *st) {
        return slayer_spike_bwd_delayed_corr_f32(ptr(y), ptr(g), ptr(u), ptr(f), n, T, f->numel(), steps, theta, tau, scale, Ts, st); }), y);
    END_HANDLE_TH_ERRORS
}

// ---- the Loihi neuron ----------------------------------------------------------------------------------
SLAYER_HOST(loihiSpikesDelayed)   // (weightedSpikes, wgtExp, theta, iDecay, vDecay, refDelay, delaySteps, voltage): [spike, voltage or None]
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(8);
    const at::Tensor *x = a.tensor(0);
    const int64_t wgtExp = a.within(1, 0, 25), theta = a.within(2, 0, 0x7fffffff), iDecay = a.within(3, 0, 0xffffffffLL),
                  vDecay = a.within(4, 0, 0xffffffffLL), refDelay = a.within(5, 1, 0xffffffffLL), delay = a.within(6, 0, 31);
    const bool voltage = a.truth(7);
    SLAYER_PLAIN;
    const at::Tensor s = at::empty_like(*x);
    at::Tensor v;
    if (voltage) v = at::empty_like(*x);
    int64_t n, T;
    rows(*x, n, T);
    const bool launched = launch(a, [&](void *st) {
        return slayer_loihi_get_spikes_delayed_f32(ptr(s), voltage ? ptr(v) : nullptr, nullptr, ptr(x), n, T, static_cast<uint32_t>(wgtExp),
                                                   static_cast<int32_t>(theta), static_cast<uint32_t>(iDecay), static_cast<uint32_t>(vDecay),
                                                   static_cast<uint32_t>(refDelay), static_cast<int32_t>(delay), st); });
    if (!launched) return none();
    PyObject *list = PyList_New(3);
    if (!list) return nullptr;
    PyList_SET_ITEM(list, 0, THPVariable_Wrap(s));
    PyList_SET_ITEM(list, 1, voltage ? THPVariable_Wrap(v) : none());
    PyList_SET_ITEM(list, 2, none());
    return list;
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(quantize)    // (weights, step)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(2);
    const at::Tensor *w = a.tensor(0);
    const double step = a.number(1);
    SLAYER_PLAIN;
    if (step == 0.0 || step != step) return none();
    const at::Tensor y = at::empty_like(*w);
    return wrapped(launch(a, [&](void *st) { return slayer_quantize_f32(ptr(y), ptr(w), w->numel(), step, st); }), y);
    END_HANDLE_TH_ERRORS
}

// ---- losses --------------------------------------------------------------------------------------------
PyObject *lossAndError(bool launched, const at::Tensor &loss, const at::Tensor &error)
{
    if (!launched) return none();
    PyObject *both = PyTuple_New(2);
    if (!both) return nullptr;
    PyTuple_SET_ITEM(both, 0, THPVariable_Wrap(loss));
    PyTuple_SET_ITEM(both, 1, THPVariable_Wrap(error));
    return both;
}

SLAYER_HOST(spikeLoss)   // (spikeOut, spikeDesired, srmKernel, Ts, addend or None)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(5);
    const at::Tensor *out = a.tensor(0), *desired = a.tensor(1), *srm = a.tensor(2);
    const float Ts = a.number(3);
    const at::Tensor *addend = a.tensorOrNone(4);
    SLAYER_PLAIN;
    if (!same(out, desired) || (addend && !same(out, addend))) return none();
    int64_t n, T;
    rows(*out, n, T);
    const at::Tensor loss = floats({}, a.device), error = at::empty_like(*out), work = floats({n > 0 ? n : 1}, a.device);
    return lossAndError(launch(a, [&](void *st) {
        return slayer_spike_loss_f32(loss.data_ptr<float>(), ptr(error), ptr(out), ptr(desired), ptr(addend), ptr(srm), work.data_ptr<float>(),
                                     n, T, srm->numel(), Ts, st); }), loss, error);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(spikeLossGrad)   // (error, gradLoss, srmKernel, Ts)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(4);
    const at::Tensor *error = a.tensor(0), *g = a.tensor(1), *srm = a.tensor(2);
    const float Ts = a.number(3);
    SLAYER_PLAIN;
    if (g->numel() != 1) return none();
    int64_t n, T;
    rows(*error, n, T);
    const at::Tensor y = at::empty_like(*error);
    return wrapped(launch(a, [&](void *st) {
        return slayer_spike_loss_grad_f32(ptr(y), ptr(error), ptr(g), ptr(srm), n, T, srm->numel(), Ts, st); }), y);
    END_HANDLE_TH_ERRORS
}

// ---- synapses ------------------------------------------------------------------------------------------
// Geometry of a synapse on an input of the given sizes; false where the kernels do not take it or it is no geometry at all.
bool geometry(Args &a, at::IntArrayRef in, at::IntArrayRef w, Py_ssize_t first, slayer_synapse_geom &g, int32_t &OH, int32_t &OW)
{
    if (in.size() != 5 || (w.size() != 4 && !(w.size() == 5 && w[4] == 1))) return false;
    for (int64_t v : in)
        if (v < 0 || v > INT32_MAX) return false;
    for (int64_t v : w)
        if (v < 0 || v > INT32_MAX) return false;
    g.N = in[0]; g.C = in[1]; g.H = in[2]; g.W = in[3]; g.T = in[4];
    g.O = w[0]; g.KH = w[2]; g.KW = w[3];
    a.pair(first, g.strideH, g.strideW);
    a.pair(first + 1, g.padH, g.padW);
    a.pair(first + 2, g.dilH, g.dilW);
    const int64_t groups = a.within(first + 3, 1, INT32_MAX);
    if (!a.ok || g.C % groups || g.O % groups || w[1] * groups != g.C) return false;
    g.groups = static_cast<int32_t>(groups);
    return slayer_synapse_out_shape(&g, &OH, &OW) == SLAYER_OK;
}

SLAYER_HOST(conv2d)      // (input, weight, stride, padding, dilation, groups)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(6);
    const at::Tensor *x = a.tensor(0), *w = a.tensor(1);
    SLAYER_PLAIN;
    slayer_synapse_geom g;
    int32_t OH, OW;
    if (!geometry(a, x->sizes(), w->sizes(), 2, g, OH, OW)) return none();
    const at::Tensor y = floats({g.N, g.O, OH, OW, g.T}, a.device);
    return wrapped(launch(a, [&](void *st) { return slayer_synapse_conv_f32(ptr(y), ptr(x), ptr(w), &g, st); }), y);
    END_HANDLE_TH_ERRORS
}

bool output_of(const at::Tensor &t, const slayer_synapse_geom &g, int32_t OH, int32_t OW)
{
    return t.sizes() == at::IntArrayRef({g.N, g.O, OH, OW, g.T});
}

SLAYER_HOST(conv2dGradInput)   // (gradOutput, weight, input, stride, padding, dilation, groups): the input's sizes are what is needed
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(7);
    const at::Tensor *go = a.tensor(0), *w = a.tensor(1), *x = a.tensor(2);
    SLAYER_PLAIN;
    slayer_synapse_geom g;
    int32_t OH, OW;
    if (!geometry(a, x->sizes(), w->sizes(), 3, g, OH, OW) || !output_of(*go, g, OH, OW)) return none();
    const at::Tensor y = floats(x->sizes(), a.device);
    return wrapped(launch(a, [&](void *st) { return slayer_synapse_conv_grad_input_f32(ptr(y), ptr(go), ptr(w), &g, st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(conv2dGradWeight)  // (gradOutput, input, weight, stride, padding, dilation, groups): the weight's sizes are what is needed
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(7);
    const at::Tensor *go = a.tensor(0), *x = a.tensor(1), *w = a.tensor(2);
    SLAYER_PLAIN;
    slayer_synapse_geom g;
    int32_t OH, OW;
    if (!geometry(a, x->sizes(), w->sizes(), 3, g, OH, OW) || !output_of(*go, g, OH, OW)) return none();
    const at::Tensor y = floats(w->sizes(), a.device);
    const int64_t bytes = slayer_synapse_conv_grad_weight_workspace_bytes(&g);
    const at::Tensor work = floats({(bytes + 3) / 4}, a.device);
    return wrapped(launch(a, [&](void *st) { return slayer_synapse_conv_grad_weight_f32(ptr(y), ptr(go), ptr(x), ptr(work), &g, st); }), y);
    END_HANDLE_TH_ERRORS
}

bool window(const at::Tensor &w) { return (w.dim() == 4 || w.dim() == 5) && w.size(2) > 0 && w.size(3) > 0 && w.numel() == w.size(2) * w.size(3); }

SLAYER_HOST(pool)        // (input, weight)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(2);
    const at::Tensor *x = a.tensor(0), *w = a.tensor(1);
    SLAYER_PLAIN;
    if (x->dim() != 5 || !window(*w)) return none();
    const int64_t H = x->size(2), W = x->size(3), KH = w->size(2), KW = w->size(3);
    const at::Tensor y = floats({x->size(0), x->size(1), (H + H % KH) / KH, (W + W % KW) / KW, x->size(4)}, a.device);
    return wrapped(launch(a, [&](void *st) {
        return slayer_pool_f32(ptr(y), ptr(x), ptr(w), x->size(0), x->size(1), H, W, x->size(4), KH, KW, st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(poolSpikeBackward)   // (gradOutput, weight, membranePotential, theta, tau, scale)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(6);
    const at::Tensor *g = a.tensor(0), *w = a.tensor(1), *u = a.tensor(2);
    const float theta = a.number(3), tau = a.number(4), scale = a.number(5);
    SLAYER_PLAIN;
    if (u->dim() != 5 || !window(*w)) return none();
    const int64_t H = u->size(2), W = u->size(3), KH = w->size(2), KW = w->size(3);
    if (g->sizes() != at::IntArrayRef({u->size(0), u->size(1), (H + H % KH) / KH, (W + W % KW) / KW, u->size(4)})) return none();
    const at::Tensor y = at::empty_like(*u);
    return wrapped(launch(a, [&](void *st) {
        return slayer_pool_grad_input_f32(ptr(y), ptr(g), ptr(w), ptr(u), theta, tau, scale, u->size(0), u->size(1), H, W, u->size(4), KH, KW, st); }), y);
    END_HANDLE_TH_ERRORS
}

// The dense layer: x (N, K, T) or the output gradient (N, O, T), weight (O, K).
SLAYER_HOST(denseEvents)   // (input, weight)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(2);
    const at::Tensor *x = a.tensor(0), *w = a.tensor(1);
    SLAYER_PLAIN;
    if (x->dim() != 3 || w->dim() != 2 || w->size(1) != x->size(1)) return none();
    const int64_t N = x->size(0), K = x->size(1), T = x->size(2), O = w->size(0);
    const at::Tensor y = floats({N, O, T}, a.device), work = floats({(slayer_dense_events_workspace_bytes(N, K, O, T) + 3) / 4}, a.device);
    return wrapped(launch(a, [&](void *st) { return slayer_dense_events_f32(ptr(y), ptr(x), ptr(w), ptr(work), N, K, O, T, st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(denseEventsGradWeight)   // (gradOutput, input)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(2);
    const at::Tensor *g = a.tensor(0), *x = a.tensor(1);
    SLAYER_PLAIN;
    if (x->dim() != 3 || g->dim() != 3 || g->size(0) != x->size(0) || g->size(2) != x->size(2)) return none();
    const int64_t N = x->size(0), K = x->size(1), T = x->size(2), O = g->size(1);
    const at::Tensor y = floats({O, K}, a.device),
                     work = floats({(slayer_dense_events_grad_weight_workspace_bytes(N, K, O, T) + 3) / 4}, a.device);
    return wrapped(launch(a, [&](void *st) { return slayer_dense_events_grad_weight_f32(ptr(y), ptr(g), ptr(x), ptr(work), N, K, O, T, st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(denseThin)   // (input, weight)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(2);
    const at::Tensor *x = a.tensor(0), *w = a.tensor(1);
    SLAYER_PLAIN;
    if (x->dim() != 3 || w->dim() != 2 || w->size(1) != x->size(1)) return none();
    const int64_t N = x->size(0), K = x->size(1), T = x->size(2), O = w->size(0);
    const int64_t bytes = slayer_dense_thin_workspace_bytes(N, K, O, T, 0);
    const at::Tensor y = floats({N, O, T}, a.device);
    at::Tensor work;
    if (bytes) work = floats({bytes / 4}, a.device);
    return wrapped(launch(a, [&](void *st) {
        return slayer_dense_thin_f32(ptr(y), ptr(w), ptr(x), bytes ? ptr(work) : nullptr, N, K, O, T, st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(denseThinGradInput)   // (gradOutput, weight)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(2);
    const at::Tensor *g = a.tensor(0), *w = a.tensor(1);
    SLAYER_PLAIN;
    if (g->dim() != 3 || w->dim() != 2 || w->size(0) != g->size(1)) return none();
    const int64_t N = g->size(0), K = w->size(1), T = g->size(2), O = g->size(1);
    const at::Tensor y = floats({N, K, T}, a.device);
    return wrapped(launch(a, [&](void *st) { return slayer_dense_thin_grad_input_f32(ptr(y), ptr(w), ptr(g), N, K, O, T, st); }), y);
    END_HANDLE_TH_ERRORS
}

SLAYER_HOST(denseThinGradWeight)   // (gradOutput, input)
{
    HANDLE_TH_ERRORS
    SLAYER_ARGS(2);
    const at::Tensor *g = a.tensor(0), *x = a.tensor(1);
    SLAYER_PLAIN;
    if (x->dim() != 3 || g->dim() != 3 || g->size(0) != x->size(0) || g->size(2) != x->size(2)) return none();
    const int64_t N = x->size(0), K = x->size(1), T = x->size(2), O = g->size(1);
    const int64_t bytes = slayer_dense_thin_workspace_bytes(N, K, O, T, 1);
    const at::Tensor y = floats({O, K}, a.device);
    at::Tensor work;
    if (bytes) work = floats({bytes / 4}, a.device);
    return wrapped(launch(a, [&](void *st) {
        return slayer_dense_thin_grad_weight_f32(ptr(y), ptr(g), ptr(x), bytes ? ptr(work) : nullptr, N, K, O, T, st); }), y);
    END_HANDLE_TH_ERRORS
}

// (arguments...): whether every tensor among them is an exact torch.Tensor with memory of its own, which no functorch
// transform, dead or alive, has wrapped
SLAYER_HOST(unwrapped)
{
    using c10::DispatchKey;
    static const c10::DispatchKeySet wrappers({DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                               DispatchKey::Functionalize});
    for (Py_ssize_t i = 0; i < nargs; ++i) {
        if (THPVariable_CheckExact(args[i])) {
            const at::Tensor &t = THPVariable_Unpack(args[i]);
            if (!t.defined() || !t.has_storage() || t.key_set().has_any(wrappers)) Py_RETURN_FALSE;
        } else if (THPVariable_Check(args[i])) {
            Py_RETURN_FALSE;
        }
    }
    Py_RETURN_TRUE;
}

// (ctx, nodes = 1): whether someone looks at the gradient of this Function's first tensor argument in the backward pass that is
// running - a hook on the tensor or on the node behind it, retain_grad, or the pass was asked for it - so that the gradient
// may not go past that node; with more `nodes`, at that of the node's first argument as well, and so on.  True where there is
// no such pass.
SLAYER_HOST(watched)
{
    using namespace torch::autograd;
    HANDLE_TH_ERRORS
    const long nodes = nargs == 2 ? PyLong_AsLong(args[1]) : 1;
    if (nargs < 1 || nargs > 2 || nodes < 1 || !THPFunction_Check(args[0])) {
        PyErr_Clear();
        Py_RETURN_TRUE;
    }
    const std::shared_ptr<PyNode> own = reinterpret_cast<THPFunction *>(args[0])->cdata.lock();
    const auto *info = get_current_graph_task_exec_info();
    if (!own || !info) Py_RETURN_TRUE;
    Node *node = own.get();
    for (long i = 0; i < nodes; ++i) {
        node = node->num_outputs() ? node->next_edge(0).function.get() : nullptr;
        if (!node) Py_RETURN_FALSE;
        const auto asked = info->find(node);
        if (!node->pre_hooks().empty() || !node->tensor_pre_hooks().empty() || !node->retains_grad_hooks().empty() || !node->post_hooks().empty() ||
            (asked != info->end() && asked->second.captures_ && !asked->second.captures_->empty()))
            Py_RETURN_TRUE;
    }
    Py_RETURN_FALSE;
    END_HANDLE_TH_ERRORS
}

#define SLAYER_METHOD(NAME, FN) {NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(FN)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    SLAYER_METHOD("getSpikes", getSpikes),
    SLAYER_METHOD("conv", (fir<slayer_conv_f32>)),
    SLAYER_METHOD("corr", (fir<slayer_corr_f32>)),
    SLAYER_METHOD("pspAlpha", pspAlpha),
    SLAYER_METHOD("spikeBackward", spikeBackward),
    SLAYER_METHOD("spikeBackwardPspAlpha", spikeBackwardPspAlpha),
    SLAYER_METHOD("pspSpikeBackwardAlpha", pspSpikeBackwardAlpha),
    SLAYER_METHOD("shift", shift),
    SLAYER_METHOD("spikeBackwardDelayed", spikeBackwardDelayed),
    SLAYER_METHOD("delayGrad", delayGrad),
    SLAYER_METHOD("spikeBackwardDelayedCorr", spikeBackwardDelayedCorr),
    SLAYER_METHOD("loihiSpikesDelayed", loihiSpikesDelayed),
    SLAYER_METHOD("quantize", quantize),
    SLAYER_METHOD("spikeLoss", spikeLoss),
    SLAYER_METHOD("spikeLossGrad", spikeLossGrad),
    SLAYER_METHOD("conv2d", conv2d),
    SLAYER_METHOD("conv2dGradInput", conv2dGradInput),
    SLAYER_METHOD("conv2dGradWeight", conv2dGradWeight),
    SLAYER_METHOD("pool", pool),
    SLAYER_METHOD("poolSpikeBackward", poolSpikeBackward),
    SLAYER_METHOD("denseEvents", denseEvents),
    SLAYER_METHOD("denseEventsGradWeight", denseEventsGradWeight),
    SLAYER_METHOD("denseThin", denseThin),
    SLAYER_METHOD("denseThinGradInput", denseThinGradInput),
    SLAYER_METHOD("denseThinGradWeight", denseThinGradWeight),
    SLAYER_METHOD("unwrapped", unwrapped),
    SLAYER_METHOD("watched", watched),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_slayer_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__slayer_host() { return PyModule_Create(&module); }
