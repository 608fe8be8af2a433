"""The work this framework is timed on: dedispersion of one beam or many, in
one step or two, over bytes, packed and float samples, resident on the device
or streamed from the host, the peak search that follows it, and the cost model
of the learned tuner.  Sizes run from the smallest call (128 channels, 128 DMs,
4096 samples) to batches of beams that fill the device.

``listed`` gives the cases, ``draw`` another one of the same ranges,
``prepare`` what a program holds before the call, ``run`` one pass through the
public entry points, ``work`` the bytes and additions a pass cannot do without
and ``exact`` the results in 64 bits, in plain torch and numpy.
"""
from __future__ import annotations

import ctypes
import math
import random

import numpy as np
import torch

from dedispersion_amd import DDError, Observation, Plan, detect_peaks, detect_peaks_batch
from dedispersion_amd._lib import check, load
from dedispersion_amd.beams import BeamSet
from dedispersion_amd.learned import FEATURES, Network
from dedispersion_amd.streaming import StreamEngine
from dedispersion_amd.workloads import (ARTS_BANDWIDTH, ARTS_CHANNELS, ARTS_MIN_FREQ, PADDING, SAMPLING_TIME,
                                        Workload)

ARTS_SPAN = ARTS_CHANNELS * ARTS_BANDWIDTH  # 300 MHz
WIDTHS = 7  # boxcars 1 .. 64
HIDDEN, LAYERS = 64, 3  # the tuner's network


def listed():
    return [
        # One beam of a small survey: the shortest call, latency and launches.
        single("small_single", 128, 128, 4096, span=100.0, min_freq=1400.0, dm_step=0.5, zapped=2),
        # One ARTS beam, every DM in one step: the heaviest single launch.
        single("arts_single", ARTS_CHANNELS, 2048, 24576),
        # Two beams seen as three synthesized ones, nothing a multiple of a tile, DMs from 40 up.
        single("ragged_single", 1000, 301, 5003, beams=2, sbeams=3, first_dm=40.0, dm_step=0.3, zapped=37),
        # 2-bit samples as many recorders store them.
        single("packed_single", ARTS_CHANNELS, 1024, 12288, bits=2),
        # Samples that were normalised to floats beforehand.
        single("float_single", 768, 512, 12288, bits=32),
        # A small two-step plan: launches and short rows.
        two_step("small_two_step", 256, 16, 8, 16, 5000),
        # The ARTS beam in two steps, 64 x 32 DMs.
        two_step("arts_two_step", ARTS_CHANNELS, 32, 64, 32, 24576),
        # Many uneven beams replayed as one graph: the production batch.
        {"name": "beam_batch", "kind": "batch", "beams": 16, "layout": 4, "chunks": 0},
        # 1.024 s chunks of four beams arriving together at the streaming engine, from pinned host memory.
        {"name": "stream_chunks", "kind": "stream", "beams": 4, "channels": ARTS_CHANNELS, "subbands": 32, "coarse": 64,
         "fine": 32, "samples": 12500},
        # The search over the rows of a batch of beams.
        {"name": "peak_batch", "kind": "peaks", "sets": 12, "layout": 4},
        # Training the tuner's cost model on four swept layouts: loss and gradients.
        {"name": "tuner_gradient", "kind": "gradient", "rows": 2880},
        # Ranking the 720 configurations of one layout.
        {"name": "tuner_predict", "kind": "predict", "rows": 720},
    ]


def single(name, channels, dms, samples, bits=8, beams=1, sbeams=1, min_freq=ARTS_MIN_FREQ, span=ARTS_SPAN, first_dm=0.0,
           dm_step=0.2, zapped=None):
    return {"name": name, "kind": "single", "channels": channels, "dms": dms, "samples": samples, "bits": bits,
            "beams": beams, "sbeams": sbeams, "min_freq": min_freq, "span": span, "first_dm": first_dm,
            "dm_step": dm_step, "zapped": channels // 20 if zapped is None else zapped}


def two_step(name, channels, subbands, coarse, fine, samples, bits=8):
    return {"name": name, "kind": "two_step", "channels": channels, "subbands": subbands, "coarse": coarse, "fine": fine,
            "samples": samples, "bits": bits}


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["single", "single", "single", "packed", "float", "two_step", "two_step", "batch", "stream",
                       "peaks", "tuner"])
    if kind in ("single", "packed", "float"):
        bits = {"single": 8, "packed": rng.choice([1, 2, 4]), "float": 32}[kind]
        while True:
            c = single(None, log(64, 1536), log(32, 2048), log(1024, 24576), bits=bits, beams=rng.choice([1, 1, 2]),
                       min_freq=rng.choice([1250.0, 1400.0]), span=rng.uniform(100.0, 300.0),
                       first_dm=rng.choice([0.0, 0.0, rng.uniform(1.0, 60.0)]), dm_step=rng.uniform(0.1, 0.5))
            c["sbeams"] = c["beams"] + rng.choice([0, 0, 1])
            del c["name"]
            # float rows are added four bytes at a time, in order: a quarter of the byte cases' range
            if c["channels"] * c["dms"] * c["samples"] * c["sbeams"] <= (1.9e10 if bits == 32 else 7.7e10):
                return c
    if kind == "two_step":
        subbands = rng.choice([8, 16, 32])
        c = two_step(None, subbands * rng.randint(8, 48), subbands, log(4, 64), rng.choice([8, 16, 24, 32]),
                     log(1024, 24576), bits=rng.choice([8, 8, 32, 4]))
        del c["name"]
        return c
    if kind == "batch":
        return {"kind": "batch", "beams": rng.randint(2, 16), "layout": rng.randint(5, 10 ** 6), "chunks": rng.choice([0, 0, 2])}
    if kind == "stream":
        subbands = rng.choice([16, 32])
        return {"kind": "stream", "beams": rng.randint(1, 4), "channels": subbands * rng.randint(16, 48),
                "subbands": subbands, "coarse": log(8, 64), "fine": rng.choice([16, 32]), "samples": log(4000, 12500)}
    if kind == "peaks":
        return {"kind": "peaks", "sets": log(1, 12), "layout": rng.randint(5, 10 ** 6)}
    return {"kind": rng.choice(["gradient", "predict"]), "rows": log(64, 2880)}


# ---- what the cases are made of ----

def f32(v):
    return np.float32(v)


def observation(case):
    """The Observation of a single or two-step case; streams and batches are
    two-step beams of the ARTS band."""
    if case["kind"] == "single":
        return Observation(
            nr_channels=case["channels"], min_freq=case["min_freq"], channel_bandwidth=case["span"] / case["channels"],
            sampling_time=SAMPLING_TIME, nr_samples_per_batch=case["samples"], nr_dms=case["dms"],
            first_dm=case["first_dm"], dm_step=case["dm_step"], nr_beams=case["beams"],
            nr_synthesized_beams=case["sbeams"])
    return Observation(
        nr_channels=case["channels"], min_freq=ARTS_MIN_FREQ, channel_bandwidth=ARTS_SPAN / case["channels"],
        sampling_time=SAMPLING_TIME, nr_samples_per_batch=case["samples"], nr_dms=case["fine"], first_dm=0.0,
        dm_step=0.2, nr_subbands=case["subbands"], nr_dms_subbanding=case["coarse"], first_dm_subbanding=0.0,
        dm_step_subbanding=f32(0.2).item() * case["fine"])


def delays(rows, first, step, o):
    """Samples of delay per unit DM of every row, in float32 as the shift
    tables are defined."""
    freq = f32(first) + np.arange(rows, dtype=np.float32) * f32(step)
    top = f32(first) + f32(rows - 1) * f32(step)
    one = f32(1.0)
    d = f32(4148.808) * (one / (freq * freq) - one / (top * top))
    d = d * f32(o.nr_samples_per_batch) / (f32(o.nr_samples_per_batch) * f32(o.sampling_time))
    d[-1] = 0.0
    return d


def tables(o):
    """Delays of the channels, of the channels relative to their subband's top
    one, and of the subbands."""
    ch = delays(o.nr_channels, o.min_freq, o.channel_bandwidth, o)
    per = o.nr_channels // o.nr_subbands
    sub = delays(o.nr_subbands, f32(o.min_freq) + f32(per - 1) * f32(o.channel_bandwidth),
                 f32(per) * f32(o.channel_bandwidth), o)
    return ch, ch - np.repeat(ch[per - 1::per], per), sub


def shifts(table, first, step, dms):
    """Whole-sample shifts [row][DM]."""
    dm = f32(first) + np.arange(dms, dtype=np.float32) * f32(step)
    return (dm[None, :] * table[:, None]).astype(np.uint32).astype(np.int64)


def dispersed(samples, delay, first, step, dms):
    last = f32(first) + f32(dms - 1) * f32(step)
    return int(math.ceil(f32(samples) + f32(delay) * last))


def lengths(o):
    """Input samples per row, and step one's output samples per row."""
    ch, _, sub = tables(o)
    if not o.nr_dms_subbanding:
        return dispersed(o.nr_samples_per_batch, ch[0], o.first_dm, o.dm_step, o.nr_dms), 0
    s1 = dispersed(o.nr_samples_per_batch, sub[0], o.first_dm, o.dm_step, o.nr_dms)
    return dispersed(s1, ch[0], o.first_dm_subbanding, o.dm_step_subbanding, o.nr_dms_subbanding), s1


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed & (2 ** 62 - 1))


def noise(o, bits, seed, samples):
    """One input, [beams][channels][samples]: noise with pulses for 8 bits,
    uniform fields for packed samples, normalised noise for floats."""
    g = generator(seed)
    shape = (o.nr_beams, o.nr_channels, samples)
    if bits < 8:
        return torch.randint(0, 1 << bits, shape, generator=g, device="cuda", dtype=torch.uint8)
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    r = random.Random(seed)
    table = torch.from_numpy(tables(o)[0]).cuda()
    last = max(o.nr_dms_subbanding, 1) * o.nr_dms - 1
    for _ in range(4):  # dispersed boxcars, 2.5 sigma in every channel
        dm = o.first_dm + o.dm_step * r.randint(0, last)
        t0, width = r.randrange(max(1, o.nr_samples_per_batch - 16)), r.randint(1, 16)
        at = t0 + (table * dm).long()[:, None] + torch.arange(width, device="cuda")[None, :]
        b = r.randrange(o.nr_beams)
        x[b].scatter_add_(1, at.clamp(max=samples - 1), torch.full(at.shape, 2.5, device="cuda"))
    return x if bits == 32 else (x * 16 + 128).round_().clamp_(0, 255).to(torch.uint8)


def rows_of(values, bits, pitch):
    """The samples in the device layout: rows of `pitch` elements, packed
    least significant field first."""
    b, c, s = values.shape
    if bits < 8:
        per = 8 // bits
        n = -(-s // per)
        wide = torch.zeros(b, c, n * per, dtype=torch.uint8, device="cuda")
        wide[:, :, :s] = values
        wide = wide.view(b, c, n, per)
        values = wide[..., 0].clone()
        for k in range(1, per):
            values |= wide[..., k] << (k * bits)
    out = torch.zeros(b, c, pitch, dtype=values.dtype, device="cuda")
    out[:, :, :values.shape[2]] = values
    return out


def zapped_of(channels, count, seed):
    flags = [0] * channels
    for c in random.Random(seed + 1).sample(range(channels), count):
        flags[c] = 1
    return flags


def beams_of(case, seed):
    """Sizes and seeds of a batch's beams: DM counts and samples uneven, as in
    workloads.batched_beams."""
    r = random.Random(case["layout"])
    out = []
    for b in range(case["beams"]):
        coarse, samples = r.choice([16, 32, 64, 128]), r.choice([8192, 16384, 24576, 32768])
        out.append(({"kind": "two_step", "channels": ARTS_CHANNELS, "subbands": 32, "coarse": coarse, "fine": 32,
                     "samples": samples}, seed * 1000 + b))
    return out


def sets_of(case):
    r = random.Random(case["layout"])
    return [(r.choice([128, 512, 1024, 2048, 4096]), r.choice([4096, 8192, 12500, 16384, 24576, 32768]))
            for _ in range(case["sets"])]


def peak_rows(rows, samples, seed):
    """Rows as dedispersion leaves them: sums of about 1459 channels of bytes,
    some with a boxcar."""
    g = generator(seed)
    x = torch.randn(rows, samples, generator=g, device="cuda").mul_(611.0).add_(186752.0)
    r = random.Random(seed)
    for _ in range(max(1, rows // 16)):
        w, t = r.randint(1, 64), r.randrange(samples - 64)
        x[r.randrange(rows), t:t + w] += r.uniform(500.0, 4000.0)
    return x.round_().clamp_(min=0.0)


class Wrapped:
    """A device buffer of the streaming engine, for torch."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 2}


def stream():
    return torch.cuda.current_stream().cuda_stream


# ---- the passes ----

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("single", "two_step"):
        o = observation(case)
        bits = case["bits"]
        plan = Plan(o, PADDING, input_bits=bits)
        plan.set_zapped_channels(zapped_of(o.nr_channels, zapped_count(case), seed))
        z = plan.sizes
        n, s1 = lengths(o)
        two = kind == "two_step"
        if n != (z.nr_dispersed_samples_subbanding if two else z.nr_dispersed_samples):
            raise DDError("the plan's sizes differ from the definition's")
        d_in = rows_of(noise(o, bits, seed, n), bits, z.sub_in_pitch if two else z.in_pitch)
        state = {"kind": kind, "plan": plan, "in": d_in, "bits": bits, "s1": s1}
        if two:
            state["mid"] = torch.zeros(o.nr_beams, o.nr_dms_subbanding, o.nr_subbands, z.sub_out_pitch, device="cuda")
            state["out"] = torch.zeros(o.nr_synthesized_beams, o.nr_dms_subbanding * o.nr_dms, z.out_pitch, device="cuda")
        else:
            state["out"] = torch.zeros(o.nr_synthesized_beams, o.nr_dms, z.out_pitch, device="cuda")
        return state
    if kind == "batch":
        works = []
        for c, s in beams_of(case, seed):
            o = observation(c)
            flags = zapped_of(o.nr_channels, zapped_count(c), s)
            works.append(Workload(f"beam-{s}", o, zapped=[k for k, f in enumerate(flags) if f], noise="uniform", seed=s))
        beams = BeamSet(torch, works, pulses=False, chunks=case["chunks"])
        for (c, s), plan, d_in in zip(beams_of(case, seed), beams.plans, beams.inputs):
            o = plan.obs
            d_in.copy_(rows_of(noise(o, 8, s, lengths(o)[0]), 8, plan.sizes.sub_in_pitch).view(-1))
        return {"kind": kind, "beams": beams}
    if kind == "stream":
        o = observation(case)
        plan = Plan(o, PADDING)
        plan.set_zapped_channels(zapped_of(o.nr_channels, zapped_count(case), seed))
        z = plan.sizes
        nb = case["beams"]
        chunks = []
        for b in range(nb):
            host = torch.empty(o.nr_channels, case["samples"], dtype=torch.uint8, pin_memory=True)
            host.copy_(noise(o, 8, seed * 64 + b, case["samples"])[0])
            chunks.append(host)
        budget = nb * (z.sub_input_elements + 4 * (z.intermediate_elements + z.sub_output_elements)) + (1 << 30)
        state = {"kind": kind, "plan": plan, "chunks": chunks, "engine": StreamEngine(plan, nb, budget, max_slots=nb)}
        run(state)  # the beams are under way: their history is not empty
        return state
    if kind == "peaks":
        sets = [(peak_rows(r, s, seed * 64 + k), torch.zeros(r, 5, dtype=torch.int32, device="cuda"))
                for k, (r, s) in enumerate(sets_of(case))]
        return {"kind": kind, "sets": sets}
    net = Network(HIDDEN, LAYERS, seed)
    x, t = features(case, seed)
    return {"kind": kind, "net": net, "rows": case["rows"], "x": x, "t": t, "loss": torch.zeros(1, device="cuda"),
            "grad": torch.zeros(net.n_params, device="cuda"), "y": torch.zeros(case["rows"], device="cuda")}


def zapped_count(case):
    return case.get("zapped", case["channels"] // 20)


def features(case, seed):
    g = generator(seed)
    x = torch.randn(case["rows"], len(FEATURES), generator=g, device="cuda")
    return x, torch.randn(case["rows"], generator=g, device="cuda")


def run(state):
    kind = state["kind"]
    if kind == "single":
        plan = state["plan"]
        call = plan.dedisperse_f32 if state["bits"] == 32 else plan.dedisperse
        call(state["in"].data_ptr(), state["out"].data_ptr(), stream=stream())
        return state["out"][:, :, :plan.sizes.nr_samples]
    if kind == "two_step":
        plan = state["plan"]
        one = plan.step_one_f32 if state["bits"] == 32 else plan.step_one
        one(state["in"].data_ptr(), state["mid"].data_ptr(), stream=stream())
        plan.step_two(state["mid"].data_ptr(), state["out"].data_ptr(), stream=stream())
        return [state["mid"][..., :state["s1"]], state["out"][:, :, :plan.sizes.nr_samples]]
    if kind == "batch":
        beams = state["beams"]
        beams.run()
        return [out.view(-1, p.sizes.out_pitch)[:, :p.sizes.nr_samples] for p, out in zip(beams.plans, beams.outs)]
    if kind == "stream":
        engine, plan = state["engine"], state["plan"]
        for b, chunk in enumerate(state["chunks"]):
            engine.submit(b, chunk.data_ptr(), chunk.stride(0), b)
        outs = {}
        while len(outs) < len(state["chunks"]):
            for e in engine.progress():
                outs[e["beam"]] = e["output"]
                engine.release(e["slot"])
        z = plan.sizes
        shape = (plan.obs.nr_dms_subbanding * plan.obs.nr_dms, z.out_pitch)
        rows = [torch.as_tensor(Wrapped(outs[b], shape), device="cuda")[:, :z.nr_samples] for b in sorted(outs)]
        for r in rows:
            r.engine = engine  # the buffers are the engine's: it lives as long as they do
        return rows
    if kind == "peaks":
        sets = state["sets"]
        if len(sets) == 1:
            rows, peaks = sets[0]
            detect_peaks(rows.data_ptr(), rows.shape[0], rows.shape[1], rows.stride(0), WIDTHS, peaks.data_ptr(), stream())
        else:
            detect_peaks_batch([(rows.data_ptr(), rows.shape[0], rows.shape[1], rows.stride(0), peaks.data_ptr())
                                for rows, peaks in sets], WIDTHS, stream())
        return [[p.view(torch.float32)[:, :3], p[:, 3:]] for _, p in sets]
    net = state["net"]
    if kind == "gradient":
        check(load().dd_mlp_loss_grad(net.handle, state["x"].data_ptr(), state["t"].data_ptr(), state["rows"],
                                      ctypes.c_void_p(state["loss"].data_ptr()), ctypes.c_void_p(state["grad"].data_ptr()),
                                      stream() or None))
        return [state["loss"], state["grad"]]
    net.forward(state["x"], state["rows"], state["y"], stream())
    return state["y"]


# ---- what a pass cannot do without ----

def work(case):
    kind = case["kind"]
    if kind == "single":
        n, _ = lengths(observation(case))
        live = case["channels"] - zapped_count(case)
        outputs = case["sbeams"] * case["dms"] * case["samples"]
        return {"bytes": case["beams"] * live * n * case["bits"] / 8 + 4 * outputs, "flops": live * outputs}
    if kind in ("two_step", "stream"):
        n, s1 = lengths(observation(case))
        live = case["channels"] - zapped_count(case)
        beams = case.get("beams", 1)
        outputs = case["coarse"] * case["fine"] * case["samples"]
        sums = case["coarse"] * s1
        moved = live * n * case.get("bits", 8) / 8 + 4 * outputs
        if kind == "two_step":
            moved += 2 * 4 * sums * case["subbands"]  # step one's output and step two's input
        return {"bytes": beams * moved, "flops": beams * (live * sums + case["subbands"] * outputs)}
    if kind == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for c, _ in beams_of(case, 0):
            w = work({**c, "kind": "stream"})
            total = {k: total[k] + w[k] for k in total}
        return total
    if kind == "peaks":
        sets = sets_of(case)
        samples = sum(r * s for r, s in sets)
        return {"bytes": 4 * samples + 20 * sum(r for r, _ in sets), "flops": 2 * WIDTHS * samples}
    n, params = len(FEATURES), network_shape()
    weights = sum(a * b + b for a, b in params)
    passes = 1 if kind == "predict" else 3
    moved = 4 * (case["rows"] * (n + 1) + weights * (1 if kind == "predict" else 2))
    return {"bytes": moved, "flops": 2.0 * passes * case["rows"] * weights}


def network_shape():
    return [(len(FEATURES) if k == 0 else HIDDEN, HIDDEN if k < LAYERS else 1) for k in range(LAYERS + 1)]


# ---- the results in 64 bits ----

def shifted_sums(rows, table, samples):
    """sum over r of rows[r][t + table[r][d]], [DMs][samples], in 64 bits."""
    table = torch.as_tensor(table, device="cuda")
    out = torch.zeros(table.shape[1], samples, dtype=torch.float64, device="cuda")
    at = torch.arange(samples, device="cuda")
    for r in range(len(rows)):
        x = rows[r].double().contiguous()
        out += x[table[r][:, None] + at[None, :]]
    return out


def exact_two_step(o, values, flags):
    """Step one's and step two's results of one beam's samples [channels][n]."""
    _, relative, sub = tables(o)
    _, s1 = lengths(o)
    per = o.nr_channels // o.nr_subbands
    t1 = shifts(relative, o.first_dm_subbanding, o.dm_step_subbanding, o.nr_dms_subbanding)
    mid = torch.zeros(o.nr_dms_subbanding, o.nr_subbands, s1, dtype=torch.float64, device="cuda")
    for sb in range(o.nr_subbands):
        live = [c for c in range(sb * per, (sb + 1) * per) if not flags[c]]
        mid[:, sb] = shifted_sums([values[c] for c in live], t1[live], s1)
    t2 = shifts(sub, o.first_dm, o.dm_step, o.nr_dms)
    out = torch.cat([shifted_sums(mid[c], t2, o.nr_samples_per_batch) for c in range(o.nr_dms_subbanding)])
    return mid, out


def exact(case, seed):
    kind = case["kind"]
    if kind == "single":
        o = observation(case)
        values = noise(o, case["bits"], seed, lengths(o)[0])
        flags = zapped_of(o.nr_channels, zapped_count(case), seed)
        live = [c for c in range(o.nr_channels) if not flags[c]]
        table = shifts(tables(o)[0], o.first_dm, o.dm_step, o.nr_dms)[live]
        per_beam = [shifted_sums([values[b][c] for c in live], table, o.nr_samples_per_batch) for b in range(o.nr_beams)]
        return torch.stack([per_beam[b % o.nr_beams] for b in range(o.nr_synthesized_beams)])
    if kind == "two_step":
        o = observation(case)
        values = noise(o, case["bits"], seed, lengths(o)[0])
        mid, out = exact_two_step(o, values[0], zapped_of(o.nr_channels, zapped_count(case), seed))
        return [mid[None], out[None]]
    if kind == "batch":
        outs = []
        for c, s in beams_of(case, seed):
            o = observation(c)
            flags = zapped_of(o.nr_channels, zapped_count(c), s)
            outs.append(exact_two_step(o, noise(o, 8, s, lengths(o)[0])[0], flags)[1].float())  # whole numbers
        return outs
    if kind == "stream":
        o = observation(case)
        flags = zapped_of(o.nr_channels, zapped_count(case), seed)
        n, _ = lengths(o)
        history = n - case["samples"]
        outs = []
        for b in range(case["beams"]):
            x = noise(o, 8, seed * 64 + b, case["samples"])[0]
            before = torch.zeros(o.nr_channels, history, dtype=torch.uint8, device="cuda")
            kept = min(history, case["samples"])  # one chunk came before this one
            before[:, history - kept:] = x[:, case["samples"] - kept:]
            outs.append(exact_two_step(o, torch.cat([before, x], 1), flags)[1].float())  # whole numbers
        return None if history > case["samples"] else outs
    if kind == "peaks":
        return [[exact_peaks(peak_rows(r, s, seed * 64 + k)), None] for k, (r, s) in enumerate(sets_of(case))]
    net = Network(HIDDEN, LAYERS, seed)  # its initial weights, and no more
    return exact_network(case, *(v.double().cpu().numpy() for v in features(case, seed)), net.get_params().astype(np.float64))


def exact_peaks(x):
    rows, s = x.shape
    x = x.double()
    mean = x.mean(1)
    sigma = (x.square().mean(1) - mean.square()).clamp(min=0).sqrt()
    total = torch.cat([torch.zeros(rows, 1, dtype=torch.float64, device="cuda"), x.cumsum(1)], 1)
    best = None
    for k in range(WIDTHS):
        w = 1 << k
        if w > s:
            break
        snr = ((total[:, w:] - total[:, :-w]).amax(1) - w * mean) / (sigma * math.sqrt(w))
        best = snr if best is None else torch.maximum(best, snr)
    return torch.stack([best, mean, sigma], 1)


def exact_network(case, x, t, flat):
    layers, at = [], 0
    for a, b in network_shape():
        layers.append((flat[at:at + a * b].reshape(a, b), flat[at + a * b:at + a * b + b]))
        at += a * b + b
    acts = [x]
    for k, (w, b) in enumerate(layers):
        y = acts[-1] @ w + b
        acts.append(np.maximum(y, 0.0) if k < LAYERS else y)
    if case["kind"] == "predict":
        return acts[-1][:, 0]
    d = acts[-1][:, 0] - t
    g, parts = (2.0 / len(t)) * d[:, None], []
    for k in range(LAYERS, -1, -1):
        parts[:0] = [(acts[k].T @ g).ravel(), g.sum(0)]
        if k:
            g = (g @ layers[k][0].T) * (acts[k] > 0)
    return [np.array([np.mean(d * d)]), np.concatenate(parts)]
