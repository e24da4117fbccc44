"""Performance cases of batched prediction.

What a user of this package has it do, by entry point:

  mlp       RuntimePredictor.predict_batch: run-time predictions of one
            operation kind for a batch of feature rows, from one row to the
            million rows of the benchmark.
  scale     wave_scale: kernel records in GPU memory scaled from one device to
            one or several others, from the kernels of one trace to 64 million.
  trace     Trace.to_device: one training-iteration trace predicted for one
            other device, kernels and MLP operations together.
  sweep     TracePlan.prepare(...).launch(): one trace predicted for many
            devices (prepared once per set of devices, launched per question).
  deferred  the reference's own loop, a strategy call per kernel object and the
            times read afterwards, through the deferred strategy.

Inference only: the path has no backward pass.  Features and times are float64,
launch fields int32, network weights and predictions float32.
"""
import math

import numpy as np
import torch

from habitat_amd import Device, synthetic
from habitat_amd.analysis.mlp.mlp import RuntimePredictor
from habitat_amd.analysis.predictor import Predictor
from habitat_amd.analysis.wave_scaling.batch import KernelRecords, WaveScaleOutput, wave_scale
from habitat_amd.analysis.wave_scaling.deferred import deferred_unified_wave_scaling
from habitat_amd.analysis.wave_scaling.metadata import NullMetadataManager

HIDDEN_LAYERS, WIDTH = 8, 1024   # the reference's network shape
KINDS = ("conv2d", "linear", "bmm", "lstm")
INPUTS = {kind: len(names) + 4 for kind, names in synthetic.MLP_FEATURES.items()}
TRACE_DESTINATIONS = ("P100", "P4000", "RTX2070", "RTX2080Ti", "T4", "MI355X")
SCALE_DESTINATIONS = ("MI355X", "P4000", "RTX2070", "RTX2080Ti", "T4", "P100", "GTX1080Ti", "P4")

# A ResNet-50-shaped trace: distinct MLP rows (23 convolutions, 1 linear) and
# kernel records.
TRACE_CONV_ROWS, TRACE_LINEAR_ROWS, TRACE_RECORDS = 23, 1, 908


def listed():
    return [
        # one operation asked for on one device (an interactive question)
        {"name": "mlp_1_row", "path": "mlp", "kind": "lstm", "rows": 1},
        # the operations of one trace of a recurrent or attention model
        {"name": "mlp_54_rows", "path": "mlp", "kind": "bmm", "rows": 54},
        # a few traces, or one trace for a handful of devices
        {"name": "mlp_700_rows", "path": "mlp", "kind": "linear", "rows": 700},
        # one trace's distinct convolutions for 256 devices and the origin
        {"name": "mlp_5911_rows", "path": "mlp", "kind": "conv2d", "rows": 5911},
        # the benchmark's batch: a database of operations evaluated at once
        {"name": "mlp_1M_rows", "path": "mlp", "kind": "conv2d", "rows": 1_000_000},
        # the kernels of one trace, all outputs, buffers made by the call
        {"name": "scale_900", "path": "scale", "records": 900, "dests": 1, "options": True,
         "waves": True, "own_out": False},
        # the benchmark's headline: a million records, one destination
        {"name": "scale_1M", "path": "scale", "records": 1_000_000, "dests": 1, "options": False,
         "waves": False, "own_out": True},
        # a million records to every other device of the table at once, with the
        # register table's column and records without metrics among them
        {"name": "scale_1M_to_7", "path": "scale", "records": 1_000_003, "dests": 7,
         "options": True, "waves": False, "own_out": True},
        # a record database beyond every cache
        {"name": "scale_64M", "path": "scale", "records": 64_000_000, "dests": 1,
         "options": False, "waves": False, "own_out": True},
        # a training iteration predicted for one device, from Python objects to times
        {"name": "trace_to_device", "path": "trace", "batch": 32, "dest": "T4"},
        # the same for a sweep of 256 device designs
        {"name": "sweep_256_devices", "path": "sweep", "batch": 32, "devices": 256},
        # the reference's loop over a trace's kernel objects
        {"name": "deferred_900_kernels", "path": "deferred", "kernels": 908, "dest": "P100"},
    ]


def _log_int(rng, low, high):
    """Log-uniform over [low, high]."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    path = rng.choice(["mlp", "mlp", "mlp", "scale", "scale", "trace", "sweep", "deferred"])
    if path == "mlp":
        return {"path": "mlp", "kind": rng.choice(KINDS), "rows": _log_int(rng, 1, 1_000_000)}
    if path == "scale":
        dests = rng.choice([1, 1, 2, 3, 5, 7])
        return {"path": "scale", "records": _log_int(rng, 1, 64_000_000 // dests), "dests": dests,
                "options": rng.random() < 0.5, "waves": rng.random() < 0.3,
                "own_out": rng.random() < 0.5}
    if path == "trace":
        return {"path": "trace", "batch": rng.randint(1, 256), "dest": rng.choice(TRACE_DESTINATIONS)}
    if path == "sweep":
        return {"path": "sweep", "batch": rng.randint(1, 256), "devices": _log_int(rng, 2, 1024)}
    return {"path": "deferred", "kernels": _log_int(rng, 1, 20_000),
            "dest": rng.choice(TRACE_DESTINATIONS)}


# ---------------------------------------------------------------- inputs
def _predictor_of(kind, seed):
    """A network with weights as trained ones are: activations that keep their
    size from layer to layer and predictions of a few milliseconds, with its
    weights uploaded."""
    torch.manual_seed(seed)
    rp = RuntimePredictor(kind, HIDDEN_LAYERS, WIDTH)
    with torch.no_grad():
        for name, p in rp.model.named_parameters():
            if name.startswith(("fc1", "mlp")) and name.endswith("weight"):
                p.mul_(math.sqrt(6.0))
        rp.model.fc2.bias.fill_(4.0)
    _, mu, sigma = synthetic.mlp_features(kind, 2048, seed=seed)
    rp.set_normalization(mu, sigma)
    rp.predict_batch(mu[None, :])
    return rp


def _records(n, options, seed):
    """Kernel records as a profiler leaves them, all of which can have run on a
    V100: launch sizes, times and DRAM traffic over several decades."""
    g = torch.Generator("cuda").manual_seed(seed)

    def uniform(low, high):
        return torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (high - low) + low

    def integer(low, high):
        return torch.randint(low, high + 1, (n,), generator=g, device="cuda", dtype=torch.int32)

    block = 64 << integer(0, 4)
    limit = torch.clamp(65536 // block, max=255)
    smem = integer(0, 48 * 1024)
    cols = {
        "num_blocks": torch.floor(2.0 ** uniform(0, 20)).to(torch.int32),
        "block_size": block,
        "dynamic_smem": smem - smem // 2,
        "static_smem": smem // 2,
        "regs_per_thread": torch.minimum(integer(16, 255), limit.to(torch.int32)),
        "run_time_ns": torch.floor(10.0 ** uniform(3, 7)),
        "flop_sp_efficiency": 10.0 ** uniform(-2, 2),
        "dram_read_bytes": torch.floor(10.0 ** uniform(3, 10)),
        "dram_write_bytes": torch.floor(10.0 ** uniform(3, 10)),
    }
    dest_regs = has_metrics = None
    if options:
        # every second kernel is in the register table, 30 % carry metrics
        dest_regs = torch.where(integer(0, 1) == 1, torch.minimum(integer(16, 255), limit),
                                torch.full_like(block, -1)).to(torch.int32)
        has_metrics = (uniform(0, 1) < 0.3).to(torch.uint8)
    return KernelRecords(cols, dest_regs, has_metrics)


def _trace_predictor(seed):
    return Predictor(mlp_predictors={kind: _predictor_of(kind, seed)
                                     for kind in ("conv2d", "linear")})


def _kernels(count, seed):
    """`count` measured kernel objects of one or more traces."""
    kernels, part = [], 0
    while len(kernels) < count:
        trace = synthetic.resnet50_trace(Device.V100, batch=32, seed=seed * 64 + part)
        for op in trace.operations:
            for rt in (op.forward, op.backward):
                if rt is not None:
                    kernels.extend(rt.kernels)
        part += 1
    return kernels[:count]


def prepare(case, seed):
    path = case["path"]
    if path == "mlp":
        rp = _predictor_of(case["kind"], seed)
        x, _, _ = synthetic.mlp_features(case["kind"], case["rows"], seed=seed + 1)
        return {"path": path, "predictor": rp, "rows": torch.from_numpy(x).cuda()}
    if path == "scale":
        n, dests = case["records"], case["dests"]
        out = None
        if case["own_out"]:
            out = WaveScaleOutput(n, dests, torch.device("cuda", torch.cuda.current_device()),
                                  waves=case["waves"], status=True)
        first = 0 if dests == 1 else 1   # several: the other devices of the table
        return {"path": path, "records": _records(n, case["options"], seed), "out": out,
                "dests": [getattr(Device, d) for d in SCALE_DESTINATIONS[first:first + dests]],
                "waves": case["waves"]}
    if path == "trace":
        return {"path": path, "predictor": _trace_predictor(seed),
                "trace": synthetic.resnet50_trace(Device.V100, batch=case["batch"], seed=seed),
                "dest": getattr(Device, case["dest"])}
    if path == "sweep":
        trace = synthetic.resnet50_trace(Device.V100, batch=case["batch"], seed=seed)
        devices, feats = synthetic.device_sweep(case["devices"], seed=seed)
        features = {d.name: list(f) for d, f in zip(devices, feats)}
        features[Device.V100.name] = [16, 900, 80, 14.028]
        plan = _trace_predictor(seed).plan_trace(trace)
        return {"path": path, "sweep": plan.prepare(devices, features)}
    return {"path": path, "kernels": _kernels(case["kernels"], seed),
            "dest": getattr(Device, case["dest"]), "registers": NullMetadataManager()}


# ---------------------------------------------------------------- one pass
def run(state):
    path = state["path"]
    if path == "mlp":
        return state["predictor"].predict_batch(state["rows"])
    if path == "scale":
        out = wave_scale(state["records"], Device.V100, state["dests"], out=state["out"],
                         waves=state["waves"])
        return {"time_ns": out.time_ns, "occ_origin": out.occ_origin, "occ_dest": out.occ_dest,
                "wave_origin": out.wave_origin, "wave_dest": out.wave_dest, "status": out.status}
    if path == "trace":
        predicted = state["trace"].to_device(state["dest"], state["predictor"])
        return {"total_ms": predicted.run_time_ms,
                "operations_ms": np.array([op.run_time_ms for op in predicted.operations])}
    if path == "sweep":
        res = state["sweep"].launch()
        return {"total_ms": res.total_ms, "pass_kernel_ns": res.pass_kernel_ns,
                "special_ms": res.special_ms, "bad_records": res.bad_records,
                "clamped_ops": res.clamped_ops}
    predicted = [deferred_unified_wave_scaling(k, Device.V100, state["dest"], state["registers"])
                 for k in state["kernels"]]
    return np.array([k.run_time_ns for k in predicted], np.float64)


# ------------------------------------------------- what a pass cannot do without
def _mlp_work(kind, rows):
    f = INPUTS[kind]
    weights = 4 * ((f + 1) * WIDTH + HIDDEN_LAYERS * (WIDTH + 1) * WIDTH + WIDTH + 1)
    flops = 2.0 * rows * (f * WIDTH + HIDDEN_LAYERS * WIDTH * WIDTH + WIDTH)
    return weights + rows * (8 * f + 4), flops


def work(case):
    path = case["path"]
    if path == "mlp":
        moved, flops = _mlp_work(case["kind"], case["rows"])
        return {"bytes": moved, "flops": flops}
    if path == "scale":
        per = 52 + (5 if case["options"] else 0) + 4 + (4 if case["waves"] else 0)
        per += case["dests"] * (13 + (4 if case["waves"] else 0))
        return {"bytes": case["records"] * per}
    if path in ("trace", "sweep"):
        devices = 2 if path == "trace" else case["devices"] + 1   # the origin's rows too
        conv, conv_flops = _mlp_work("conv2d", TRACE_CONV_ROWS * devices)
        linear, linear_flops = _mlp_work("linear", TRACE_LINEAR_ROWS * devices)
        # records in; per destination the passes' sums (two per operation) and the operations' times
        moved = conv + linear + TRACE_RECORDS * 57 + (devices - 1) * 8 * (250 + 54)
        return {"bytes": moved, "flops": conv_flops + linear_flops}
    return {"bytes": case["kernels"] * (64 + 9)}


def tolerance(case):
    """About four times the differences seen from an evaluation in 64 bits;
    integers and statuses are equal.  Float32 networks of ten layers: 2e-7 over
    a batch, 8e-7 at the worst row (torch's own float32 forward: 1e-7 and 4e-7).
    A trace or sweep divides two predictions: 4e-7 and 1.3e-6.  Scaled times,
    float64 through one power: 9e-15."""
    if case["path"] == "mlp":
        return {"rel": 8e-7, "max": 4e-6}
    if case["path"] in ("trace", "sweep"):
        return {"rel": 1.6e-6, "max": 6e-6}
    return {"rel": 4e-14, "max": 4e-14}
