"""The convolutions and transforms that programs have this library do, as
timing cases: small cubes, where launches and latency count, the sizes of the
benchmark (64^3, 128^3, 256^3, 512^3), batches with a shared filter and with
one filter per cube, mixed batches, the plain 3D transform in both directions,
the split-FP16 form, the filter set-up, and the drop-in call on host buffers.

A case is a dict:
  kind   "conv"    cubes on the device, filter spectra made beforehand
         "fft"     plain 3D transform of cubes on the device
         "setup"   spectra of new filters, then the convolution with them
         "mixed"   a prepared batch of several edges, replayed
         "dropin"  fpgaf_conv3D on host buffers (filter transform included)
  n      cube edge; count: cubes (mixed: n32 .. n256 instances of each edge)
  own    one filter per cube (else all cubes share one)
  split  split-FP16 matrix-core form; inverse: direction of "fft"
  log    log-uniform magnitudes in [1e-3, 1e3) with uniform phase, else
         uniform [-1, 1) real and imaginary parts
"""
import math
import random

import numpy as np
import torch

import convfpga_amd as C
from convfpga_amd import api

EDGES = (8, 16, 32, 64, 128, 256, 512)
MIXED_EDGES = (32, 64, 128, 256)
# plans that the persistent batch runs, by edge (the graph batch runs any)
PERSISTENT_PLANS = {32: api.CF_PLAN_PLANE3, 64: api.CF_PLAN_PLANE3,
                    128: api.CF_PLAN_SPLIT3_G24M2H, 256: api.CF_PLAN_SPLIT3_G24M2H}


def _conv(name, n, count=1, own=False, split=False, log=False):
    return {"name": name, "kind": "conv", "n": n, "count": count, "own": own, "split": split, "log": log}


def listed():
    return [
        # the smallest cubes: one call's latency, as in a loop over small volumes
        _conv("conv_16", 16),
        # one cube at the command line's default edge
        _conv("conv_64", 64),
        # many small signals against one kernel (a batch of measurements)
        _conv("conv_64x64_shared", 64, count=64),
        # single cubes of the medium size
        _conv("conv_128", 128),
        # the headline workload: one large cube, spectrum precomputed
        _conv("conv_256", 256),
        # the largest edge, larger than every cache
        _conv("conv_512", 512),
        # the matrix-core form on a batch with wide-ranging magnitudes, own filters
        _conv("split_256x4_log", 256, count=4, own=True, split=True, log=True),
        # a replayed batch of uneven sizes, every instance with its own filter
        {"name": "mixed_29", "kind": "mixed", "n32": 16, "n64": 8, "n128": 4, "n256": 1, "persistent": False},
        # forward transforms of an odd number of cubes
        {"name": "fft_128x3", "kind": "fft", "n": 128, "count": 3, "inverse": False, "log": False},
        # one large inverse transform
        {"name": "ifft_256", "kind": "fft", "n": 256, "count": 1, "inverse": True, "log": False},
        # a new filter for every convolution (matched filtering with changing templates)
        {"name": "setup_conv_256", "kind": "setup", "n": 256, "count": 1, "log": False},
        # the reference's own call: host buffers in and out, filter transform included
        {"name": "dropin_64", "kind": "dropin", "n": 64, "log": False},
    ]


def _log_int(rng, most):
    """1 .. most, spread over the logarithm."""
    return min(most, int(math.exp(rng.uniform(0.0, math.log(most + 1.0)))))


def draw(rng):
    kind = rng.choices(("conv", "split", "mixed", "fft", "setup", "dropin"), (6, 1, 2, 3, 2, 1))[0]
    log = rng.random() < 0.3
    if kind == "split":
        return {"kind": "conv", "n": 256, "count": rng.randint(1, 5), "own": rng.random() < 0.5, "split": True, "log": log}
    if kind == "mixed":
        persistent = rng.random() < 0.3
        return {"kind": "mixed", "n32": rng.randint(0, 24), "n64": rng.randint(1, 12), "n128": rng.randint(0, 5),
                "n256": rng.randint(0, 2), "persistent": persistent}
    if kind == "dropin":
        return {"kind": "dropin", "n": rng.choice(EDGES[:5]), "log": log}
    if kind == "setup":
        n = rng.choice(EDGES[:6])
        return {"kind": "setup", "n": n, "count": _log_int(rng, max(1, min(64, 2 * 256 ** 3 // n ** 3))), "log": log}
    n = rng.choice(EDGES)
    count = _log_int(rng, max(1, min(512, 5 * 256 ** 3 // n ** 3)))
    if kind == "fft":
        return {"kind": "fft", "n": n, "count": count, "inverse": rng.random() < 0.5, "log": log}
    return {"kind": "conv", "n": n, "count": count, "own": rng.random() < 0.5, "split": False, "log": log}


# ---- inputs ------------------------------------------------------------------
def _complex_values(shape, seed, log, device):
    """complex64 values of `shape` from `seed`: uniform parts, or log-uniform magnitudes and uniform phase."""
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    u = torch.rand(tuple(shape) + (2,), generator=g, device=device, dtype=torch.float32)
    if not log:
        return torch.view_as_complex(u * 2.0 - 1.0)
    return torch.polar(torch.pow(10.0, 6.0 * u[..., 0] - 3.0), 2.0 * math.pi * u[..., 1])


def _signals(case, seed, device):
    n = case["n"]
    return _complex_values((case.get("count", 1), n, n, n), 4 * seed, case["log"], device)


def _filters(case, seed, device):
    n = case["n"]
    many = case["count"] if case["kind"] == "setup" or case.get("own") else 1
    return _complex_values((many, n, n, n), 4 * seed + 1, case["log"], device)


def _mixed_groups(case):
    return [(n, case["n%d" % n]) for n in MIXED_EDGES if case["n%d" % n] > 0]


def _mixed_inputs(n, count, seed, device):
    return (_complex_values((count, n, n, n), 4 * seed + 1024 * n, False, device),
            _complex_values((count, n, n, n), 4 * seed + 1024 * n + 1, False, device))


_ready = False


def _library():
    """The library, initialised once per process as a program does at its start."""
    global _ready
    if not _ready:
        rc = C.fpga_initialize()
        if rc != 0:
            raise RuntimeError("fpga_initialize -> %d" % rc)
        _ready = True


# ---- a pass ------------------------------------------------------------------
def prepare(case, seed):
    _library()
    kind = case["kind"]
    if kind == "dropin":
        sig, filt = (f(case, seed, "cpu").numpy().reshape(-1).copy() for f in (_signals, _filters))
        return {"case": case, "sig": sig, "filt": filt, "out": np.zeros_like(sig)}
    if kind == "mixed":
        specs, instances = [], []
        for n, count in _mixed_groups(case):
            sig, filt = _mixed_inputs(n, count, seed, "cuda")
            out = torch.empty_like(sig)
            if case["persistent"]:
                api.set_plan(n, PERSISTENT_PLANS[n])
            spec = C.Spectrum(n, filt, count)
            if case["persistent"]:
                api.set_plan(n, api.CF_PLAN_AUTO)
            specs.append(spec)
            instances += [(sig[k], out[k], spec.view(k)) for k in range(count)]
        outs = [out for _, out, _ in instances]
        if case["persistent"]:  # one launch takes them in any order; the graph runs neighbours of one edge together
            random.Random(seed).shuffle(instances)
        batch = api.Batch(instances, mode=api.CF_BATCH_PERSISTENT if case["persistent"] else api.CF_BATCH_GRAPH)
        return {"case": case, "batch": batch, "specs": specs, "outs": outs}
    sig = _signals(case, seed, "cuda")
    state = {"case": case, "sig": sig, "out": torch.empty_like(sig)}
    if kind == "setup":
        state["filt"] = _filters(case, seed, "cuda")
    elif kind == "conv":
        filt = _filters(case, seed, "cuda")
        state["spec"] = C.Spectrum(case["n"], filt, filt.shape[0])
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "conv":
        C.conv3d_device(state["spec"], state["sig"], state["out"], case["count"],
                        precision=api.CF_PREC_SPLIT_FP16 if case["split"] else api.CF_PREC_FP32)
        return state["out"]
    if kind == "fft":
        C.fft3d_device(case["n"], state["sig"], state["out"], case["count"], case["inverse"])
        return state["out"]
    if kind == "setup":
        spec = C.Spectrum(case["n"], state["filt"], case["count"])
        C.conv3d_device(spec, state["sig"], state["out"], case["count"])
        spec.close()
        return state["out"]
    if kind == "mixed":
        state["batch"].launch()
        return state["outs"]
    t = C.fpgaf_conv3D(case["n"], state["sig"], state["filt"], state["out"])
    if not t.valid:
        raise RuntimeError("fpgaf_conv3D: " + api.last_error())
    return state["out"]


# ---- what a pass cannot do without --------------------------------------------
def work(case):
    def fft_flops(n):
        return 15.0 * n ** 3 * math.log2(n)  # 5 P log2 P for P = n^3 points

    kind = case["kind"]
    if kind == "mixed":
        parts = [(n, count, 2) for n, count in _mixed_groups(case)]
    else:
        n, count = case["n"], case.get("count", 1)
        if kind == "fft":
            return {"bytes": 16.0 * n ** 3 * count, "flops": fft_flops(n) * count}
        if kind == "conv" and not case["own"]:
            return {"bytes": 8.0 * n ** 3 * (2 * count + 1), "flops": count * (2 * fft_flops(n) + 6.0 * n ** 3)}
        parts = [(n, count, 2 if kind == "conv" else 3)]
    # signal, own filter (or its spectrum) and output of every cube
    return {"bytes": sum(24.0 * n ** 3 * count for n, count, _ in parts),
            "flops": sum(count * (ffts * fft_flops(n) + 6.0 * n ** 3) for n, count, ffts in parts)}


# ---- the values in 64 bits ------------------------------------------------------
def _convolve(sig, filt, scale=1.0):
    """Circular convolution of each cube with its (or the shared) filter, in complex128."""
    out = torch.empty(sig.shape, dtype=torch.complex128, device=sig.device)
    h = None
    for k in range(sig.shape[0]):
        if h is None or filt.shape[0] > 1:
            h = torch.fft.fftn(filt[k].to(torch.complex128))
        out[k] = torch.fft.ifftn(torch.fft.fftn(sig[k].to(torch.complex128)) * h)
    return out if scale == 1.0 else out * scale


def exact(case, seed):
    kind = case["kind"]
    if kind == "mixed":
        return [x for n, count in _mixed_groups(case)
                for x in _convolve(*_mixed_inputs(n, count, seed, "cuda")).unbind(0)]
    if kind == "fft":
        sig, n = _signals(case, seed, "cuda"), case["n"]
        out = torch.empty(sig.shape, dtype=torch.complex128, device=sig.device)
        for k in range(sig.shape[0]):
            x = sig[k].to(torch.complex128)
            out[k] = torch.fft.ifftn(x) * float(n ** 3) if case["inverse"] else torch.fft.fftn(x)
        return out
    if kind == "dropin":
        return _convolve(_signals(case, seed, "cpu"), _filters(case, seed, "cpu"), float(case["n"] ** 3)).reshape(-1).numpy()
    return _convolve(_signals(case, seed, "cuda"), _filters(case, seed, "cuda"))
