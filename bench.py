"""Benchmark: production ATA Mode-B block on one MI355X.

Workload (one step = one block): CI8 voltages A=28, F=192, T=8192, P=2 and
CF32 phasors for B=16 beams, resident in HBM -> beamform (FP32 precision) ->
channelize (FFT of length 4 along T, fftshift) -> polarize (XY -> LR), CF32
output [16, 768, 2048, 2], in one fused kernel.  The split-FP16 variant of the
same kernel is timed beside it.

value = beamformed Msamples/s = B*F*T*P / (time per block) / 1e6.

Successive steps read successive blocks out of NSETS resident voltage blocks
(3 x 176 MB of CI8, more than MI355X's 256 MB Infinity Cache in front of
HBM), as a stream of new blocks would; one block re-read every step would
be served largely from that cache, not from HBM.

The ``cpu_baseline`` leg times the vectorised numpy port of the same chain
on the host's cores and checks both GPU variants against the complex128
oracle on a few channels.

``unfused_f32`` times the same block as one plain FP32 kernel per reference
module (cast, beamformer, channelizer, polarizer); ``split_f16`` reports its
speedup over both that chain and the fused FP32 kernel.

Extra legs (not the headline value; ``--no-extra`` skips them):
``batched`` -- 32 uneven blocks in one persistent launch, autotuned;
``mode_a`` -- split-FP16 beamform -> FFT-8192 -> Stokes I on A28 F192 T16384 B8;
``calibration`` -- fused Stokes-I loss/gradient and Adam steps on A42 F384 T2048 B4;
``kernels`` -- achieved HBM rate of the bandwidth-bound kernels (polarizer,
detector, cast, gather, permutation, channelizer) on the block's beams;
``ingest`` -- GUPPI RAW blocks read into pinned memory, copied to HBM and
beamformed, per stage and end to end;
``reference_benchmarks`` -- every module at the arguments of the reference's
own benchmark suite (benchmarks/modules);
``mode_b_bundle``, ``mode_h_bundle`` -- the reference's Mode-B and Mode-H
bundle benchmark configurations through a Runner with host buffers, per
block.
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)
# The modules' INFO lines go to stdout; the bench's stdout is one JSON line.
os.environ.setdefault("BLADE_QUIET", "1")

METRIC = "beamformed Msamples/s + % HBM/MFMA roofline; split-FP16 vs FP32 @ ≤1e-5 err"
A, F, T, P, B, RATE = 28, 192, 8192, 2, 16, 4

WARMUP_S = 2.0
NSETS = 3          # voltage blocks cycled per step (3 x 176 MB > 256 MB last-level cache)
HBM_PEAK_GBS = 8000.0
MFMA16_PEAK_TFLOPS = 2500.0


def algorithmic_counts():
    """Bytes and flops of one block (unit: one beamformed complex sample)."""
    n_in = A * F * T * P                       # CI8 complex samples, 2 B each
    n_out = B * F * T * P                      # CF32 complex samples, 8 B each
    n_w = B * A * F * P                        # CF32 phasors
    bytes_ = 2 * n_in + 8 * n_out + 8 * n_w
    flops_bf = 8 * A * n_out                   # one complex MAC = 8 real flops
    flops_fft = 5 * 2 * n_out                  # 5 log2(C) per sample, C = 4
    flops_pol = 4 * n_out
    return bytes_, flops_bf + flops_fft + flops_pol, flops_bf


def gpu_leg(steps, warmup):
    import torch
    from blade_amd import ops

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(1)
    xs = [torch.clamp(torch.round(torch.randn((A, F, T, P, 2), device=dev, generator=g) * 16.0),
                      -127, 127).to(torch.int8) for _ in range(NSETS)]
    rng = np.random.default_rng(1)
    tau = rng.uniform(-50e-9, 50e-9, size=(B, A))
    freq = 1.0e9 + np.arange(F) * 0.5e6
    w_np = np.exp(-2j * np.pi * tau[:, :, None] * freq[None, None, :])
    w_np = np.repeat(w_np[:, :, :, None, None], P, axis=4).astype(np.complex64)
    w = torch.from_numpy(w_np).to(dev)
    outs = {p: [torch.empty((B, F * RATE, T // RATE, P), dtype=torch.complex64, device=dev)
                for _ in range(NSETS)] for p in ("f32", "f16x2")}
    stream = torch.cuda.current_stream(dev)
    cursor = [0]

    def step(prec):
        i = cursor[0] % NSETS
        cursor[0] += 1
        ops.beamform_chain(xs[i], w, False, False, RATE, True, prec, out=outs[prec][i], stream=stream)

    results = {}
    for prec in ("f32", "f16x2"):
        # W warm-up steps, continued until the GPU has been busy for at least
        # WARMUP_S seconds: the clocks ramp up over the first ~1 s of load.
        t_w = time.perf_counter()
        n = 0
        while n < warmup or time.perf_counter() - t_w < WARMUP_S:
            step(prec)
            n += 1
            if n % 64 == 0:
                torch.cuda.synchronize()
        torch.cuda.synchronize()
        # Per-launch HIP events on the launching stream (kernel duration) ...
        ev = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
              for _ in range(steps)]
        t_wall0 = time.perf_counter()
        for s, e in ev:
            s.record(stream)
            step(prec)
            e.record(stream)
        torch.cuda.synchronize()
        t_wall = time.perf_counter() - t_wall0
        per = [s.elapsed_time(e) for s, e in ev]
        # ... and the whole timed region back to back (step time).
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for _ in range(steps):
            step(prec)
        e1.record(stream)
        torch.cuda.synchronize()
        region_ms = e0.elapsed_time(e1)
        results[prec] = dict(kernel_ms=float(np.mean(per)), kernel_ms_median=float(np.median(per)),
                             step_ms=region_ms / steps, wall_ms=t_wall * 1e3 / steps)
    # split-FP16 vs FP32 on the full block (device-side norm).
    d = outs["f16x2"][0] - outs["f32"][0]
    rel = float(torch.linalg.vector_norm(d) / torch.linalg.vector_norm(outs["f32"][0]))
    return results, rel, (xs[0], w, {p: o[0] for p, o in outs.items()})


def cpu_leg(x, w, outs, budget_s=12.0):
    """Time the numpy port on the host and check the GPU against the oracle.

    The port runs on N threads (the host's cores, at most 16), each on its
    own two channels of the block, with BLAS held to one thread per call:
    numpy releases the interpreter lock inside these array operations, so
    the threads run in parallel and `cores` is the number of threads used.
    """
    from concurrent.futures import ThreadPoolExecutor

    import threadpoolctl

    import oracle as O

    nthr = max(1, min(16, len(os.sched_getaffinity(0))))
    per = 2                                     # channels per thread
    fs = min(F, nthr * per)
    nthr = fs // per
    x_np = x[:, :fs].cpu().numpy()
    w_np = w[:, :, :fs].cpu().numpy()
    parts = [(x_np[:, k * per:(k + 1) * per], w_np[:, :, k * per:(k + 1) * per]) for k in range(nthr)]

    def run_part(pw):
        O.beamform_chain_c64(pw[0], pw[1], RATE, True)

    times = []
    with threadpoolctl.threadpool_limits(limits=1), ThreadPoolExecutor(nthr) as ex:
        list(ex.map(run_part, parts))                   # warm-up
        t0 = time.perf_counter()
        while (time.perf_counter() - t0 < budget_s) or len(times) < 3:
            t1 = time.perf_counter()
            list(ex.map(run_part, parts))
            times.append(time.perf_counter() - t1)
            if len(times) >= 400:
                break
    t_med = float(np.median(times))
    value = B * fs * T * P / t_med / 1e6
    # One thread on a slice of the same block (a shorter run: median of >= 3).
    fs1 = 4
    x1, w1 = x_np[:, :fs1], w_np[:, :, :fs1]
    with threadpoolctl.threadpool_limits(limits=1):
        O.beamform_chain_c64(x1, w1, RATE, True)
        t1s = []
        t0 = time.perf_counter()
        while (time.perf_counter() - t0 < budget_s / 2) or len(t1s) < 3:
            t1 = time.perf_counter()
            O.beamform_chain_c64(x1, w1, RATE, True)
            t1s.append(time.perf_counter() - t1)
            if len(t1s) >= 30:
                break
    value_1t = B * fs1 * T * P / float(np.median(t1s)) / 1e6
    # parity on 2 channels against the complex128 oracle
    fc = 2
    ref = O.polarizer(O.channelizer(O.beamformer_ata(x[:, :fc].cpu().numpy(), w[:, :, :fc].cpu().numpy()), RATE))
    errs = {}
    for prec, o in outs.items():
        got = o[:, :fc * RATE].cpu().numpy()
        errs[prec] = O.norm_rel_err(got, ref)
    return {
        "value": round(value, 2), "unit": "Msamples/s", "cores": int(nthr), "kind": "port",
        "sample": f"vectorised numpy complex64 beamform->FFT4->polarize on F={fs} of the "
                  f"A{A} F{F} T{T} B{B} block, {nthr} threads with {per} channels each "
                  f"(BLAS 1 thread per call), median of {len(times)} runs ({sum(times):.1f} s); "
                  f"scaled per beamformed sample",
        "cpu_model": _cpu_model(),
        "single_thread": {"value": round(value_1t, 2), "unit": "Msamples/s", "cores": 1,
                          "sample": f"F={fs1}, median of {len(t1s)} runs ({sum(t1s):.1f} s)"},
        "host": {"os_cpu_count": os.cpu_count(), "affinity_cores": len(os.sched_getaffinity(0))},
    }, errs


def _events_ms(fn, iters):
    import torch
    s = torch.cuda.current_stream()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(s)
    for _ in range(iters):
        fn()
    e1.record(s)
    e1.synchronize()
    return e0.elapsed_time(e1) / iters


def _ci8(shape, gen):
    import torch
    v = torch.randn(tuple(shape) + (2,), device="cuda", generator=gen) * 16.0
    return torch.clamp(torch.round(v), -127, 127).to(torch.int8)


def unfused_leg(iters=20):
    """The same Mode-B block through one plain FP32 kernel per reference
    module, in the reference's order (Cast CI8 -> CF32, Beamformer, Channelizer
    at rate 4, Polarizer in place), with this library's kernels and the
    voltage blocks cycled as in the main leg.  Device time per block."""
    import torch
    from blade_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(5)
    xs = [_ci8((A, F, T, P), gen) for _ in range(NSETS)]
    w = torch.randn((B, A, F, 1, P), dtype=torch.complex64, device="cuda", generator=gen)
    xf = torch.empty((A, F, T, P), dtype=torch.complex64, device="cuda")
    y = torch.empty((B, F, T, P), dtype=torch.complex64, device="cuda")
    ch = torch.empty((B, F * RATE, T // RATE, P), dtype=torch.complex64, device="cuda")
    k = [0]

    def chain():
        x = xs[k[0] % NSETS]
        k[0] += 1
        ops.cast(x, "cf32", out=xf, in_type="ci8")
        ops.beamformer(xf, w, False, False, "f32", out=y)
        ops.channelizer(y, RATE, out=ch)
        ops.polarizer(ch, out=ch)

    _events_ms(chain, 3)
    ms = _events_ms(chain, iters)
    return {"workload": "Mode-B block as four FP32 kernels: cast CI8->CF32, beamform (CF32 in), "
                        "channelize rate 4, polarize in place",
            "ms_per_block": round(ms, 4)}


def batched_leg(iters=20):
    """32 uneven blocks (A in {14,20,27,28}, F in {64..1024}, T in {1024..8192},
    B in 4..64, drawn from seed 2026) in one persistent launch, autotuned."""
    import torch
    from blade_amd import autotune, ops
    rng = np.random.default_rng(2026)
    shapes = [(int(rng.choice([14, 20, 27, 28])), int(rng.choice([64, 128, 256, 1024])),
               int(rng.choice([1024, 2048, 4096, 8192])), int(rng.integers(4, 65))) for _ in range(32)]
    gen = torch.Generator(device="cuda").manual_seed(3)
    blocks = []
    for (a, f, t, b) in shapes:
        x = _ci8((a, f, t, 2), gen)
        ph = torch.polar(torch.ones((b, a, f, 1, 2), device="cuda"),
                         torch.rand((b, a, f, 1, 2), device="cuda", generator=gen) * 6.283185307179586)
        blocks.append((x, ph.to(torch.complex64), torch.empty((b, f, t, 2), dtype=torch.complex64, device="cuda")))
    n_out = sum(b * f * t * 2 for (a, f, t, b) in shapes)
    bytes_ = sum(2 * a * f * t * 2 + 8 * b * f * t * 2 + 8 * b * a * f * 2 for (a, f, t, b) in shapes)
    flops = sum(8 * a * b * f * t * 2 for (a, f, t, b) in shapes)
    out = {"workload": "32 blocks, seed 2026", "blocks": len(shapes), "beamformed_samples": n_out,
           "alg_bytes": bytes_, "alg_flops": flops}
    for prec in ("f32", "f16x2"):
        tuning, _ = autotune.tune_batched(blocks, prec, iters=3, warmup=2)
        bb = ops.BatchedBeamformer(blocks, prec, tuning)
        _events_ms(bb, 5)
        ms = _events_ms(bb, iters)
        out[prec] = {"ms_per_batch": round(ms, 4), "msamples_per_s": round(n_out / ms / 1e3, 1),
                     "hbm_gbs": round(bytes_ / ms / 1e6, 1), "tflops": round(flops / ms / 1e9, 2),
                     "tuning": tuning}
    return out


def mode_a_leg(iters=20):
    """Mixed-precision Mode A block: CI8 A28 F192 T16384, split-FP16 beamform of
    B8 -> FFT-8192 -> Stokes I over 4 spectra (2 blocks), F32 filterbank."""
    import torch
    from blade_amd import ops
    A_, F_, T_, B_, C, N = 28, 192, 16384, 8, 8192, 4
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = _ci8((A_, F_, T_, 2), gen)
    rng = np.random.default_rng(2)
    tau = torch.from_numpy(rng.uniform(-200e-9, 200e-9, size=(B_, A_))).cuda()
    cal = torch.ones((A_, F_, 1, 2), dtype=torch.complex128, device="cuda")
    w = ops.phasor_ata(tau, cal, 9.904e9, 0.5e6, 0.0, 0, out_type="cf32")
    y = torch.empty((B_, F_, T_, 2), dtype=torch.complex64, device="cuda")
    out = torch.empty((B_, F_ * C, 1, 1), dtype=torch.float32, device="cuda")
    state = {"k": 0}

    def block():
        ops.beamformer(x, w, False, False, "f16x2", out=y)
        ops.channelizer_detector(y, C, N, 1, out=out, accumulate=state["k"] % 2 == 1)
        state["k"] += 1

    _events_ms(block, 10)
    ms = _events_ms(block, iters)
    t_bf = _events_ms(lambda: ops.beamformer(x, w, False, False, "f16x2", out=y), iters)
    t_cd = _events_ms(lambda: ops.channelizer_detector(y, C, N, 1, out=out, accumulate=True), iters)
    return {"workload": "CI8 A28 F192 T16384 -> split-FP16 beamform B8 -> FFT-8192 -> Stokes I (4 spectra, 2 blocks)",
            "ms_per_block": round(ms, 4), "beamform_ms": round(t_bf, 4), "channelize_detect_ms": round(t_cd, 4),
            "msamples_per_s": round(B_ * F_ * T_ * 2 / ms / 1e3, 1),
            "realtime_factor": round((T_ / 0.5e6) / (ms * 1e-3), 1)}


def gradient_leg(iters=20):
    """The fused Stokes-I loss + phasor gradient alone on A42 F384 T2048 B4
    (the calibration leg's inner kernel), for kernel traces and counters."""
    import torch
    from blade_amd import ops
    A_, F_, T_, B_ = 42, 384, 2048, 4
    gen = torch.Generator(device="cuda").manual_seed(6)
    x = _ci8((A_, F_, T_, 2), gen)
    w = torch.polar(torch.ones((B_, A_, F_, 1, 2), device="cuda"),
                    torch.rand((B_, A_, F_, 1, 2), device="cuda", generator=gen) * 6.283185307179586).to(torch.complex64)
    lam = [1.0, 0.0, 0.0, 0.0]
    out = {"workload": "A42 F384 T2048 P2 B4, loss = -Stokes I of beam 0", "calls_per_precision": 5 + iters}
    for prec in ("f32", "f16x2"):
        _events_ms(lambda: ops.stokes_i_loss_and_grad(x, w, lam, precision=prec), 5)
        g_ms = _events_ms(lambda: ops.stokes_i_loss_and_grad(x, w, lam, precision=prec), iters)
        out["grad_ms" if prec == "f32" else "grad_ms_f16x2"] = round(g_ms, 4)
    return out


def calibration_leg(steps=200):
    """Gain calibration on A42 F384 T2048 B4: fused Stokes-I loss + gradient
    (beams recomputed, never stored) and full Adam steps on unit-modulus gains."""
    import torch
    from blade_amd import ops
    from blade_amd.calibration import calibrate
    A_, F_, T_, B_ = 42, 384, 2048, 4
    gen = torch.Generator(device="cuda").manual_seed(6)
    x = _ci8((A_, F_, T_, 2), gen)
    w = torch.polar(torch.ones((B_, A_, F_, 1, 2), device="cuda"),
                    torch.rand((B_, A_, F_, 1, 2), device="cuda", generator=gen) * 6.283185307179586).to(torch.complex64)
    lam = [1.0, 0.0, 0.0, 0.0]
    _events_ms(lambda: ops.stokes_i_loss_and_grad(x, w, lam), 5)
    g_ms = _events_ms(lambda: ops.stokes_i_loss_and_grad(x, w, lam), 20)
    freqs = 1.0e9 + torch.arange(F_, dtype=torch.float64, device="cuda") * 0.5e6

    def timed(n, precision, delays=False):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        extra = dict(fit_delays=True, freqs_hz=freqs, delay_lr=1e-10) if delays else {}
        out = calibrate(x, w, steps=n, lr=0.05, precision=precision, **extra)
        torch.cuda.synchronize()
        return time.perf_counter() - t0, out

    res = {}
    for key, prec, delays in (("f32", "f32", False), ("f16x2", "f16x2", False), ("delays", "f32", True)):
        timed(10, prec, delays)                 # first capture, library set-up
        t_short, _ = timed(20, prec, delays)
        t_full, (_, _, losses) = timed(steps, prec, delays)
        # The per-call set-up (reference loss, 3 eager steps, graph capture)
        # is the same for both runs; the difference is what each further
        # step costs.
        res[key] = ((t_full - t_short) * 1e3 / (steps - 20), t_full, losses)
    step_ms, t_full, losses = res["f32"]
    bytes_ = A_ * F_ * T_ * 2 * 2
    return {"workload": "A42 F384 T2048 P2 B4, loss = -Stokes I of beam 0", "grad_ms": round(g_ms, 4),
            "grad_input_gbs": round(bytes_ / g_ms / 1e6, 1), "adam_step_ms": round(step_ms, 3),
            "adam_step_ms_f16x2": round(res["f16x2"][0], 3),
            "adam_step_ms_gains_and_delays": round(res["delays"][0], 3),
            "loss_last_f16x2": round(res["f16x2"][2][-1], 4),
            "calibrate_total_ms": round(t_full * 1e3, 1), "adam_steps": steps,
            "loss_first_last": [round(losses[0], 4), round(losses[-1], 4)]}


def kernels_leg(iters=20):
    """Achieved HBM rate of the bandwidth-bound kernels of the path at the
    production block's sizes (algorithmic bytes = bytes read + written once)."""
    import torch
    from blade_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(7)
    beams = torch.randn((16, 192, 8192, 2), dtype=torch.complex64, device="cuda", generator=gen)
    nb = beams.numel() * 8
    x8s = [_ci8((28, 192, 8192, 2), gen) for _ in range(2)]   # 2 x 176 MB > last-level cache
    k8 = [0]

    def next_x8():
        k8[0] += 1
        return x8s[k8[0] % 2]
    out = {}

    def rate(name, fn, nbytes):
        _events_ms(fn, 3)
        ms = _events_ms(fn, iters)
        out[name] = {"us": round(ms * 1e3, 1), "gbs": round(nbytes / ms / 1e6, 1),
                     "hbm_frac": round(nbytes / ms / 1e6 / HBM_PEAK_GBS, 3)}

    pol = torch.empty_like(beams)
    rate("polarizer_cf32", lambda: ops.polarizer(beams, out=pol), 2 * nb)
    det = torch.empty((16, 192, 8192 // 4, 1), dtype=torch.float32, device="cuda")
    rate("detector_stokes_i_int4", lambda: ops.detector(beams, 4, 1, out=det), nb + det.numel() * 4)
    cf = torch.empty((28, 192, 8192, 2), dtype=torch.complex64, device="cuda")
    rate("cast_ci8_cf32", lambda: ops.cast(next_x8(), "cf32", out=cf, in_type="ci8"),
         x8s[0].numel() + cf.numel() * 8)
    g = torch.empty((16, 192, 8192 * 2, 2), dtype=torch.complex64, device="cuda")
    rate("gather_x2_time", lambda: ops.gather(beams, g, 2, 2, 0), 2 * nb)
    rate("permutation_aftp_atpf", lambda: ops.permutation(beams, (0, 2, 3, 1)), 2 * nb)
    ch = torch.empty_like(beams)
    for C in (4, 64, 1024, 8192):
        rate(f"channelizer_c{C}", lambda C=C: ops.channelizer(beams, C, out=ch), 2 * nb)
    cd = torch.empty((16, 192 * 8192, 1, 1), dtype=torch.float32, device="cuda")
    rate("channelizer_detector_c8192", lambda: ops.channelizer_detector(beams, 8192, 1, 1, out=cd),
         nb + cd.numel() * 4)
    return out


def reference_benchmarks_leg(iters=20):
    """Each module at the arguments of the reference's own benchmark suite
    (benchmarks/modules/*/generic.hh, beamformer/ata.hh): the same shapes,
    one process() per iteration on resident buffers, as the reference times
    them.  Inputs under 256 MB stay in the Infinity Cache across iterations,
    as they stay in a GPU's L2 in the reference's runs.  Algorithmic bytes =
    read + written once."""
    import torch
    from blade_amd import ops
    gen = torch.Generator(device="cuda").manual_seed(11)
    out = {}

    def cf32(*shape):
        return torch.randn(shape, dtype=torch.complex64, device="cuda", generator=gen)

    def rate(name, fn, nbytes):
        _events_ms(fn, 3)
        ms = _events_ms(fn, iters)
        out[name] = {"us": round(ms * 1e3, 1), "gbs": round(nbytes / ms / 1e6, 1)}

    for b_, a_ in ((1, 20), (2, 20), (8, 20), (1, 42)):      # beamformer/ata.hh:15-18
        x = cf32(a_, 192, 8192, 2)
        w = cf32(b_, a_, 192, 1, 2)
        y = torch.empty((b_, 192, 8192, 2), dtype=torch.complex64, device="cuda")
        rate(f"beamformer_cf32_B{b_}_A{a_}", lambda: ops.beamformer(x, w, False, False, "f32", out=y),
             x.numel() * 8 + w.numel() * 8 + y.numel() * 8)
        del x, w, y
    for a_ in (2, 16, 64):                                       # cast/generic.hh:15-49
        n = a_ * 192 * 8192 * 2
        x = cf32(a_, 192, 8192, 2)
        y = torch.empty_like(x)
        rate(f"cast_cf32_cf32_A{a_}", lambda: ops.cast(x, "cf32", out=y), 16 * n)
        del x
        x8 = _ci8((a_, 192, 8192, 2), gen)
        rate(f"cast_ci8_cf32_A{a_}", lambda: ops.cast(x8, "cf32", out=y, in_type="ci8"), 10 * n)
        del y
        h = ops.cast(x8, "cf16", in_type="ci8")
        rate(f"cast_ci8_cf16_A{a_}", lambda: ops.cast(x8, "cf16", out=h, in_type="ci8"), 6 * n)
        del x8, h
    x = cf32(16, 192, 8192, 2)                                   # channelizer/generic.hh:15
    y = torch.empty_like(x)
    rate("channelizer_A16_C8192", lambda: ops.channelizer(x, 8192, out=y), 2 * x.numel() * 8)
    del y
    for a_, i_, p_ in ((2, 8, 4), (16, 8, 4), (2, 32, 4), (16, 32, 4), (2, 64, 4), (16, 64, 4),
                       (2, 64, 1), (16, 64, 1)):                 # detector/generic.hh:15-37
        xa = x[:a_]
        d = torch.empty((a_, 192, 8192 // i_, p_), dtype=torch.float32, device="cuda")
        rate(f"detector_A{a_}_I{i_}_P{p_}", lambda: ops.detector(xa, i_, p_, out=d),
             xa.numel() * 8 + d.numel() * 4)
    del x
    x = cf32(20, 192, 8192, 2)                                   # duplicate/generic.hh:13-25
    y = torch.empty_like(x)
    rate("duplicate_cf32", lambda: ops.gather(x, y, 0, 1, 0), 2 * x.numel() * 8)
    xr = torch.view_as_real(x)[..., 0].contiguous()
    yr = torch.empty_like(xr)
    rate("duplicate_f32", lambda: ops.gather(xr, yr, 0, 1, 0), 2 * xr.numel() * 4)
    del x, y, xr, yr
    for f_, t_ in ((192, 8192), (131072, 1)):                    # gather/generic.hh:15-30
        x = cf32(5, f_, t_, 2)
        y = torch.empty((5, f_, t_ * 64, 2), dtype=torch.complex64, device="cuda")
        rate(f"gather_cf32_x64_F{f_}_T{t_}", lambda: ops.gather(x, y, 2, 64, 3), 2 * x.numel() * 8)
        xh = torch.randn((5, f_, t_, 2), device="cuda", generator=gen).to(torch.float16)
        yh = torch.empty((5, f_, t_ * 64, 2), dtype=torch.float16, device="cuda")
        rate(f"gather_f16_x64_F{f_}_T{t_}", lambda: ops.gather(xh, yh, 2, 64, 3, type_name="f16"),
             2 * xh.numel() * 2)
        del x, y, xh, yh
    x = cf32(2, 192, 8192, 2)                                    # permutation/generic.hh:13-15
    for idx in ((0, 1, 2, 3), (0, 2, 1, 3), (0, 2, 3, 1)):
        rate("permutation_" + "".join("AFTP"[i] for i in idx), lambda: ops.permutation(x, idx),
             2 * x.numel() * 8)
    for a_ in (2, 16):                                           # polarizer/generic.hh:15-30
        xa = cf32(a_, 192, 8192, 2)
        ya = torch.empty_like(xa)
        rate(f"polarizer_cf32_A{a_}", lambda: ops.polarizer(xa, out=ya), 2 * xa.numel() * 8)
        xh = ops.cast(xa, "cf16")
        yh = torch.empty_like(xh)
        rate(f"polarizer_cf16_A{a_}", lambda: ops.polarizer(xh, out=yh), 2 * xa.numel() * 4)
        del xa, ya, xh, yh
    return out


# ITRF positions (m) of the 20 ATA antennas of the reference's Mode-B
# benchmark (benchmarks/bundles/ata/mode-b/mode_b.hh:70-89).
ATA20 = [(-2524041.5388905862, -4123587.965024342, 4147646.4222955606),
         (-2524068.187873109, -4123558.735413135, 4147656.21282186),
         (-2524087.2078100787, -4123532.397416349, 4147670.9866770394),
         (-2524103.384010733, -4123511.111598937, 4147682.4133068994),
         (-2524056.730228759, -4123515.287949227, 4147706.4850287656),
         (-2523986.279601761, -4123497.427940991, 4147766.732988923),
         (-2523970.301363642, -4123515.238502669, 4147758.790023165),
         (-2523983.5419911123, -4123528.1422073604, 4147737.872218138),
         (-2523941.5221860334, -4123568.125040547, 4147723.8292249846),
         (-2524074.096220788, -4123468.5182652213, 4147742.0422435375),
         (-2524058.6409591637, -4123466.5112451194, 4147753.4513993543),
         (-2524026.989692545, -4123480.9405167866, 4147758.2356800516),
         (-2524048.5254066754, -4123468.3463909747, 4147757.835369889),
         (-2524000.5641107005, -4123498.2984570004, 4147756.815976133),
         (-2523945.086670364, -4123480.3638816103, 4147808.127865142),
         (-2523950.6822576034, -4123444.7023326857, 4147839.7474427638),
         (-2523880.869769226, -4123514.3375464156, 4147813.413426994),
         (-2523930.3747946257, -4123454.3080821196, 4147842.6449955846),
         (-2523898.1150373477, -4123456.314794732, 4147860.3045849088),
         (-2523824.598229116, -4123527.93080514, 4147833.98936114)]


def _mode_b_reference_config(bl, out_shape, beams, detector):
    """The ModeB configuration of the reference's bundle benchmarks
    (benchmarks/bundles/ata/mode-b/mode_b.hh:55-115, mode-bh/mode_bh.hh:146-196):
    20 ATA antennas, unit calibrations, 6500.125 MHz, `beams` beams (the
    first off the boresight) and the incoherent beam."""
    import math
    in_shape = (20, 192, 8192, 2)
    cal = bl.array_tensor((20, 192, 1, 2), dtype=bl.cf64, device=bl.cpu)
    np.copyto(cal.as_numpy(), np.ones((20, 192, 1, 2), dtype=np.complex128))
    return {
        "input_shape": in_shape, "output_shape": out_shape,
        "pre_beamformer_channelizer_rate": 1,
        "phasor_observation_frequency_hz": 6500.125e6, "phasor_channel_bandwidth_hz": 0.5e6,
        "phasor_total_bandwidth_hz": 1.024e9, "phasor_frequency_start_index": 352,
        "phasor_reference_antenna_index": 0,
        "phasor_array_reference_position": bl.lla(lon=math.radians(-121.470733),
                                                  lat=math.radians(40.815987), alt=1020.86),
        "phasor_boresight_coordinate": bl.ra_dec(ra=0.64169, dec=1.079896295),
        "phasor_antenna_positions": [bl.xyz(*q) for q in ATA20],
        "phasor_antenna_calibrations": cal,
        "phasor_beam_coordinates": [bl.ra_dec(ra=0.63722, dec=1.07552424)] +
                                   [bl.ra_dec(ra=0.64169, dec=1.079896295)] * (beams - 1),
        "beamformer_incoherent_beam": True,
        "detector_enable": detector, "detector_integration_size": 1,
        "detector_number_of_output_polarizations": 1,
    }, cal


def _drive_async(bl, p, n_outputs, ins, outs):
    """The reference benchmarks' run loop (benchmarks/bundles/ata/mode-b/
    mode_b.hh:127-154): enqueue with the two host buffers in turn, dequeue,
    until `n_outputs` outputs came back.  Returns the wall time in seconds."""
    state = {"in": 0, "out": 0, "done": 0}

    def input_callback():
        p.transfer_in(*ins[state["in"] % 2])
        state["in"] += 1
        return bl.result.success

    def output_callback():
        p.transfer_out(*outs[state["out"] % 2])
        state["out"] += 1
        return bl.result.success

    def callback(input_id, output_id, did_output):
        if did_output:
            state["done"] += 1
        return bl.result.success

    t0 = time.perf_counter()
    while state["done"] < n_outputs:
        p.enqueue(input_callback, output_callback, state["in"], state["out"])
        p.dequeue(callback)
    dt = time.perf_counter() - t0
    # Untimed: collect the block still in flight, so that the next run starts
    # from an idle runner and none is left queued when the runner goes away.
    deadline = time.perf_counter() + 60
    while p.dequeue(callback) != bl.result.runner_queue_empty:
        if time.perf_counter() > deadline:
            raise RuntimeError("runner did not drain within 60 s")
    return dt


def _mode_b_pipeline(bl, config, in_shape, out_shape):
    @bl.runner
    class ModeB:
        def __init__(self):
            self.input.dut = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
            self.input.date = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
            self.input.buffer = bl.array_tensor(in_shape, dtype=bl.ci8)
            self.output.buffer = bl.array_tensor(out_shape, dtype=bl.f32)
            self.module.mode_b = bl.module(bl.modeb, config,
                                           (self.input.dut, self.input.date, self.input.buffer),
                                           it=bl.ci8, ot=bl.f32, telescope=bl.ata)

        def transfer_in(self, dut, date, buffer):
            self.copy(self.input.dut, dut)
            self.copy(self.input.date, date)
            self.copy(self.input.buffer, buffer)

        def transfer_out(self, buffer):
            self.copy(self.output.buffer, self.module.mode_b.get_output())
            self.copy(buffer, self.output.buffer)

    return ModeB()


def _host_inputs(bl, in_shape, seed, count=2):
    ins = []
    rng = np.random.default_rng(seed)
    for k in range(count):
        dut = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
        date = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
        buf = bl.array_tensor(in_shape, dtype=bl.ci8, device=bl.cpu)
        np.copyto(buf.as_numpy(), np.clip(np.round(rng.normal(size=in_shape + (2,)) * 16), -127, 127)
                  .astype(np.int8))
        dut.as_numpy()[0] = 0.0
        date.as_numpy()[0] = (1649366473.0 + k * 0.016384) / 86400 + 2440587.5
        ins.append((dut, date, buf))
    return ins


def mode_b_bundle_async_leg(blocks=24):
    """The reference's Mode-B bundle benchmark as it runs there
    (benchmarks/bundles/ata/mode-b/mode_b.hh:55-154): CI8 [20,192,8192,2] ->
    8 beams + incoherent -> Stokes I -> F32 [9,192,8192,1] through the
    Runner's enqueue/dequeue on two streams with two host buffers each way,
    so block N+1's copy in overlaps block N's compute and copy out.  Wall
    time per block over `blocks` blocks after two."""
    import blade_amd as bl
    in_shape, out_shape = (20, 192, 8192, 2), (9, 192, 8192, 1)
    config, _cal = _mode_b_reference_config(bl, out_shape, 8, True)
    p = _mode_b_pipeline(bl, config, in_shape, out_shape)
    ins = _host_inputs(bl, in_shape, 3)
    outs = [(bl.array_tensor(out_shape, dtype=bl.f32, device=bl.cpu),) for _ in range(2)]
    _drive_async(bl, p, 2, ins, outs)
    dt = _drive_async(bl, p, blocks, ins, outs)
    ms = dt * 1e3 / blocks
    return {"workload": "reference Mode-B benchmark through enqueue/dequeue: CI8 [20,192,8192,2] -> "
                        "8 beams + incoherent, Stokes I -> F32 [9,192,8192,1], two host buffers each way",
            "ms_per_block": round(ms, 3), "realtime_factor": round(16.384 / ms, 2),
            "blocks": blocks, "finite": bool(np.isfinite(outs[0][0].as_numpy()).all())}


def mode_bh_bundle_leg(outputs=3):
    """The reference's Mode-BH bundle benchmark (benchmarks/bundles/ata/
    mode-bh/mode_bh.hh:41-196): CI8 [20,192,8192,2] -> Mode B (2 beams +
    incoherent, CF32 beams) -> Gather x8 along time -> Mode H at rate 65536
    (Stokes I) -> F32 [3,12582912,1,1], through enqueue/dequeue with two host
    buffers each way; eight Mode-B blocks per output.  Wall time per output
    over `outputs` outputs after one."""
    import blade_amd as bl
    in_shape = (20, 192, 8192, 2)
    g_in, g_out = (3, 192, 8192, 2), (3, 192, 65536, 2)
    out_shape = (3, 192 * 65536, 1, 1)
    config_b, _cal = _mode_b_reference_config(bl, g_in, 2, False)
    config_h = {"input_shape": g_out, "output_shape": out_shape, "polarizer_convert_to_circular": False,
                "detector_integration_size": 1, "detector_number_of_output_polarizations": 1}

    @bl.runner
    class ModeBH:
        def __init__(self):
            self.input.dut = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
            self.input.date = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
            self.input.buffer = bl.array_tensor(in_shape, dtype=bl.ci8)
            self.output.buffer = bl.array_tensor(out_shape, dtype=bl.f32)
            inp = (self.input.dut, self.input.date, self.input.buffer)
            self.module.mode_b = bl.module(bl.modeb, config_b, inp, it=bl.ci8, ot=bl.cf32, telescope=bl.ata)
            self.module.gather = bl.module(bl.gather, {"axis": 2, "multiplier": 8},
                                           self.module.mode_b.get_output(), ot=bl.cf32)
            self.module.mode_h = bl.module(bl.modeh, config_h, self.module.gather.get_output(),
                                           ot=bl.f32)

        def transfer_in(self, dut, date, buffer):
            self.copy(self.input.dut, dut)
            self.copy(self.input.date, date)
            self.copy(self.input.buffer, buffer)

        def transfer_out(self, buffer):
            self.copy(self.output.buffer, self.module.mode_h.get_output())
            self.copy(buffer, self.output.buffer)

    p = ModeBH()
    ins = _host_inputs(bl, in_shape, 4)
    outs = [(bl.array_tensor(out_shape, dtype=bl.f32, device=bl.cpu),) for _ in range(2)]
    _drive_async(bl, p, 1, ins, outs)
    dt = _drive_async(bl, p, outputs, ins, outs)
    ms = dt * 1e3 / outputs
    return {"workload": "reference Mode-BH benchmark through enqueue/dequeue: CI8 [20,192,8192,2] -> "
                        "2 beams + incoherent -> gather x8 -> FFT 65536 -> Stokes I -> F32 "
                        "[3,12582912,1,1]; 8 input blocks (131 ms of sky) per output",
            "ms_per_output": round(ms, 3), "realtime_factor": round(8 * 16.384 / ms, 2),
            "outputs": outputs, "finite": bool(np.isfinite(outs[0][0].as_numpy()).all())}


def mode_b_bundle_leg(blocks=10):
    """The reference's Mode-B bundle benchmark configuration
    (benchmarks/bundles/ata/mode-b/mode_b.hh:55-115): CI8 [20,192,8192,2] ->
    delays and phasors for 8 beams + incoherent beam -> beamform -> Stokes I
    -> F32 [9,192,8192,1], through a Runner with host buffers (copy in, the
    bundle, copy out, synchronously per block).  Wall time per block."""
    import blade_amd as bl
    in_shape, out_shape = (20, 192, 8192, 2), (9, 192, 8192, 1)
    config, _cal = _mode_b_reference_config(bl, out_shape, 8, True)

    @bl.runner
    class ModeB:
        def __init__(self):
            self.input.dut = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
            self.input.date = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
            self.input.buffer = bl.array_tensor(in_shape, dtype=bl.ci8)
            self.output.buffer = bl.array_tensor(out_shape, dtype=bl.f32)
            self.module.mode_b = bl.module(bl.modeb, config,
                                           (self.input.dut, self.input.date, self.input.buffer),
                                           it=bl.ci8, ot=bl.f32, telescope=bl.ata)

        def transfer_in(self, dut, date, buffer):
            self.copy(self.input.dut, dut)
            self.copy(self.input.date, date)
            self.copy(self.input.buffer, buffer)

        def transfer_out(self, buffer):
            self.copy(self.output.buffer, self.module.mode_b.get_output())
            self.copy(buffer, self.output.buffer)

    dut = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
    date = bl.tensor(1, dtype=bl.f64, device=bl.cpu)
    host_in = bl.array_tensor(in_shape, dtype=bl.ci8, device=bl.cpu)
    host_out = bl.array_tensor(out_shape, dtype=bl.f32, device=bl.cpu)
    rng = np.random.default_rng(3)
    np.copyto(host_in.as_numpy(), np.clip(np.round(rng.normal(size=in_shape + (2,)) * 16), -127, 127)
              .astype(np.int8))
    dut.as_numpy()[0] = 0.0
    p = ModeB()
    times = []
    for k in range(blocks + 2):
        date.as_numpy()[0] = (1649366473.0 + k * 0.016384) / 86400 + 2440587.5
        t0 = time.perf_counter()
        p(dut, date, host_in, host_out)
        times.append(time.perf_counter() - t0)
    ms = float(np.median(times[2:])) * 1e3
    return {"workload": "reference Mode-B benchmark: CI8 [20,192,8192,2] -> 8 beams + incoherent, "
                        "Stokes I -> F32 [9,192,8192,1], host buffers in and out",
            "ms_per_block": round(ms, 3), "realtime_factor": round(16.384 / ms, 2),
            "finite": bool(np.isfinite(host_out.as_numpy()).all())}


def mode_h_bundle_leg(blocks=10):
    """The reference's Mode-H bundle benchmark configuration
    (benchmarks/bundles/generic/mode-h/mode_h.hh:47-55): CF32 [8,192,8192,2]
    -> channelizer at rate 8192 -> XY -> LR -> Stokes I -> F32
    [8,1572864,1,1], through a Runner with host buffers, one synchronous call
    per block (wall time), and the fused device kernel alone (HIP events)."""
    import torch
    import blade_amd as bl
    from blade_amd import ops
    in_shape, out_shape = (8, 192, 8192, 2), (8, 192 * 8192, 1, 1)
    config = {"input_shape": in_shape, "output_shape": out_shape,
              "polarizer_convert_to_circular": True,
              "detector_integration_size": 1, "detector_number_of_output_polarizations": 1}

    @bl.runner
    class ModeH:
        def __init__(self):
            self.input.buffer = bl.array_tensor(in_shape, dtype=bl.cf32)
            self.output.buffer = bl.array_tensor(out_shape, dtype=bl.f32)
            self.module.mode_h = bl.module(bl.modeh, config, self.input.buffer, it=bl.cf32, ot=bl.f32)

        def transfer_in(self, buffer):
            self.copy(self.input.buffer, buffer)

        def transfer_out(self, buffer):
            self.copy(self.output.buffer, self.module.mode_h.get_output())
            self.copy(buffer, self.output.buffer)

    host_in = bl.array_tensor(in_shape, dtype=bl.cf32, device=bl.cpu)
    host_out = bl.array_tensor(out_shape, dtype=bl.f32, device=bl.cpu)
    rng = np.random.default_rng(8)
    np.copyto(host_in.as_numpy(), (rng.random(in_shape) + 1j * rng.random(in_shape)).astype(np.complex64))
    p = ModeH()
    times = []
    for _ in range(blocks + 2):
        t0 = time.perf_counter()
        p(host_in, host_out)
        times.append(time.perf_counter() - t0)
    ms = float(np.median(times[2:])) * 1e3
    x = torch.randn(in_shape, dtype=torch.complex64, device="cuda")
    d = torch.empty((8, 192 * 8192, 1, 1), dtype=torch.float32, device="cuda")
    fn = lambda: ops.channelizer_detector(x, 8192, 1, 1, out=d)
    _events_ms(fn, 3)
    dev_ms = _events_ms(fn, 20)
    return {"workload": "reference Mode-H benchmark: CF32 [8,192,8192,2] -> FFT 8192 -> XY->LR -> "
                        "Stokes I -> F32 [8,1572864,1,1], host buffers in and out",
            "ms_per_block": round(ms, 3), "realtime_factor": round(16.384 / ms, 2),
            "fused_kernel_us": round(dev_ms * 1e3, 1),
            "finite": bool(np.isfinite(host_out.as_numpy()).all())}


def ingest_leg(nblocks=6):
    """Ingest of GUPPI RAW blocks of the Mode-B shape (A28 F192 T8192, CI8,
    176 MB per block) from a file in the page cache: the reader fills its
    pinned step buffer (file -> host), the block goes to HBM on a copy
    stream (host -> device), and the fused FP32 chain runs on the compute
    stream while the reader fills the next block."""
    import shutil
    import tempfile
    import torch
    import blade_amd as bl
    from blade_amd import ops
    tmp = tempfile.mkdtemp(prefix="blade_ingest_")
    try:
        path = os.path.join(tmp, "ingest.0000.raw")
        rng = np.random.default_rng(11)
        blk = np.clip(np.round(rng.normal(0, 16, size=(A, F, T, P, 2))), -127, 127).astype(np.int8)
        cards = [("BLOCSIZE", blk.nbytes), ("OBSNCHAN", A * F), ("NANTS", A), ("NPOL", 4), ("NBITS", 8),
                 ("DIRECTIO", 1), ("CHAN_BW", 0.5), ("OBSFREQ", 6500.125), ("SCHAN", 352),
                 ("SYNCTIME", 1649366400), ("PIPERBLK", 16), ("PKTIDX", 0)]
        head = b"".join(f"{k:<8.8}= {str(v):<70.70}".encode() for k, v in cards) + f"{'END':<80}".encode()
        head += b" " * (-len(head) % 512)
        with open(path, "wb") as fh:
            for _ in range(nblocks):
                fh.write(head)
                blk.tofile(fh)
        del blk
        cfg = {"filepath": path, "step_number_of_time_samples": 0,
               "step_number_of_frequency_channels": 0, "step_number_of_aspects": 0}
        gen = torch.Generator(device="cuda").manual_seed(3)
        w = torch.randn((B, A, F, 1, P), dtype=torch.complex64, device="cuda", generator=gen)
        y = torch.empty((B, F * RATE, T // RATE, P), dtype=torch.complex64, device="cuda")
        copy_s = torch.cuda.Stream()
        comp = torch.cuda.current_stream()
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(4)]

        def run():
            r = bl.module(bl.guppi_reader, cfg, (), ot=bl.ci8)
            host = torch.from_numpy(r.get_step_output_buffer().as_numpy())
            dev = [torch.empty(host.shape, dtype=torch.int8, device="cuda") for _ in range(2)]
            t_read, t_h2d, t_iter = [], [], []
            torch.cuda.synchronize()
            for s in range(nblocks):
                a = time.perf_counter()
                assert r.process(s) == bl.result.success
                t_read.append(time.perf_counter() - a)
                d = dev[s % 2]
                with torch.cuda.stream(copy_s):
                    ev[0].record(copy_s)
                    d.copy_(host, non_blocking=True)
                    ev[1].record(copy_s)
                comp.wait_event(ev[1])
                ops.beamform_chain(d, w, False, False, RATE, True, "f32", out=y)
                ev[1].synchronize()      # the step buffer is refilled next: its copy must be done
                t_h2d.append(ev[0].elapsed_time(ev[1]) * 1e-3)
                t_iter.append(time.perf_counter() - a)
            torch.cuda.synchronize()
            return host, dev, t_read, t_h2d, t_iter

        run()                            # first-use costs (allocations, twiddles, page cache)
        host, dev, t_read, t_h2d, t_iter = run()
        nbytes = host.numel()
        # The first block of a reader also pays the first touch of its fresh
        # pinned step buffer; the steady state is the mean over the rest.
        first_ms = t_read[0] * 1e3
        t_read, t_h2d, t_iter = t_read[1:], t_h2d[1:], t_iter[1:]
        ev[2].record(comp)
        ops.beamform_chain(dev[0], w, False, False, RATE, True, "f32", out=y)
        ev[3].record(comp)
        ev[3].synchronize()
        t_comp = ev[2].elapsed_time(ev[3]) * 1e-3
        rd, hd = float(np.mean(t_read)), float(np.mean(t_h2d))
        per_block = float(np.mean(t_iter))
        return {"workload": f"{nblocks} GUPPI RAW blocks CI8 [28,192,8192,2] (176.2 MB each), page cache -> "
                            "pinned step buffer -> HBM -> fused FP32 Mode-B chain",
                "read_ms": round(rd * 1e3, 2), "read_gbs": round(nbytes / rd / 1e9, 2),
                "h2d_ms": round(hd * 1e3, 2), "h2d_gbs": round(nbytes / hd / 1e9, 2),
                "compute_ms": round(t_comp * 1e3, 3),
                "ms_per_block": round(per_block * 1e3, 2),
                "realtime_factor": round((T / 0.5e6) / per_block, 2),
                "host_pinned": bool(host.is_pinned()),
                "first_read_ms": round(first_ms, 2),
                "note": "one step buffer: the next read waits for the copy; compute overlaps the next read"}
    finally:
        shutil.rmtree(tmp, ignore_errors=True)


def _extra(fn):
    try:
        return fn()
    except Exception as e:  # an extra leg never hides the headline line
        return {"error": f"{type(e).__name__}: {e}"}


def _async_blit_child():
    """The asynchronous Mode-B leg in a child process started with
    HSA_ENABLE_SDMA=0: host<->device copies then run as kernels on the
    Runner's streams, so one block's input copy overlaps the other's output
    copy.  HIP reads the variable at start-up, hence the separate process."""
    import subprocess
    env = dict(os.environ, HSA_ENABLE_SDMA="0")
    r = subprocess.run([sys.executable, os.path.abspath(__file__), "--leg", "mode_b_bundle_async"],
                       env=env, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=600)
    if r.returncode != 0:
        return {"error": f"child exited {r.returncode}: {r.stderr.strip()[-300:]}"}
    res = json.loads(r.stdout.strip().splitlines()[-1])["mode_b_bundle_async"]
    return {"env": "HSA_ENABLE_SDMA=0", "ms_per_block": res.get("ms_per_block"),
            "realtime_factor": res.get("realtime_factor"), "finite": res.get("finite")}


def _cpu_model():
    try:
        with open("/proc/cpuinfo") as fh:
            for line in fh:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-extra", action="store_true",
                    help="skip the batched, Mode-A and calibration legs")
    ap.add_argument("--kernel-only", choices=["f32", "f16x2"],
                    help="profiling mode: launch only this variant of the fused kernel, then a "
                         "plain 1 GiB device copy (blade_gather) that calibrates HBM counters")
    ap.add_argument("--leg", choices=["batched", "mode_a", "calibration", "kernels", "ingest",
                                      "reference_benchmarks", "mode_b_bundle", "mode_h_bundle",
                                      "mode_b_bundle_async", "mode_bh_bundle", "unfused_f32", "gradient"],
                    help="profiling mode: run only this extra leg and print its JSON")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (asked for --gpus {args.gpus}); the path shards by "
              "coarse channel with no exchange, so N GPUs would each run this block on F/N channels.",
              file=sys.stderr)
        sys.exit(2)
    if args.kernel_only:
        kernel_only(args.kernel_only, args.steps, args.warmup)
        return
    if args.leg:
        legs = {"batched": batched_leg, "mode_a": mode_a_leg, "calibration": calibration_leg,
                "kernels": kernels_leg, "ingest": ingest_leg,
                "reference_benchmarks": reference_benchmarks_leg, "mode_b_bundle": mode_b_bundle_leg,
                "mode_h_bundle": mode_h_bundle_leg, "mode_b_bundle_async": mode_b_bundle_async_leg,
                "mode_bh_bundle": mode_bh_bundle_leg, "unfused_f32": unfused_leg,
                "gradient": gradient_leg}
        print(json.dumps({args.leg: legs[args.leg]()}))
        return

    res, rel_f16_vs_f32, bufs = gpu_leg(args.steps, args.warmup)
    bytes_, flops, flops_bf = algorithmic_counts()
    f32 = res["f32"]
    t_k = f32["kernel_ms"] * 1e-3
    achieved_tflops = flops / t_k / 1e12
    achieved_gbs = bytes_ / t_k / 1e9
    t_step = f32["step_ms"] * 1e-3
    value = B * F * T * P / t_step / 1e6
    # The fraction reported is the larger of the HBM fraction (algorithmic
    # bytes) and the matrix-core fraction: the kernel multiplies each FP32
    # phasor as three exact BF16 parts, so the matrix cores execute three
    # times the contraction's flops, against the dense BF16 peak.
    hbm_frac = achieved_gbs / HBM_PEAK_GBS
    executed_tflops = 3 * flops_bf / t_k / 1e12
    mfma_frac = executed_tflops / MFMA16_PEAK_TFLOPS
    if mfma_frac >= hbm_frac:
        roof = {"bound": "mfma", "achieved": round(executed_tflops, 2), "peak": MFMA16_PEAK_TFLOPS,
                "unit": "TFLOP/s", "frac": round(mfma_frac, 4)}
    else:
        roof = {"bound": "hbm", "achieved": round(achieved_gbs, 1), "peak": HBM_PEAK_GBS,
                "unit": "GB/s", "frac": round(hbm_frac, 4)}
    roof["mfma_frac"] = round(mfma_frac, 4)
    roof["traffic"] = _traffic()
    roof["kernel"] = "beamform_kernel<4,2,true,2,2,true,12> (NT=4, MW=2, CI8, FP32 phasors as three exact BF16 parts on BF16 MFMA with FP32 accumulation, Mode-B epilogue: FFT-4 + polarize; phasors packed into LDS by each workgroup)"
    roof["kernel_ms"] = round(f32["kernel_ms"], 5)
    roof["hbm_gbs"] = round(achieved_gbs, 1)
    roof["hbm_frac"] = round(achieved_gbs / HBM_PEAK_GBS, 4)
    roof["alg_bytes"] = bytes_
    roof["alg_flops"] = flops
    roof["alg_tflops"] = round(achieved_tflops, 2)

    h = res["f16x2"]
    t_h = h["kernel_ms"] * 1e-3
    split = {
        "value": round(B * F * T * P / (h["step_ms"] * 1e-3) / 1e6, 2),
        "kernel_ms": round(h["kernel_ms"], 5),
        "hbm_gbs": round(bytes_ / t_h / 1e9, 1),
        "hbm_frac": round(bytes_ / t_h / 1e9 / HBM_PEAK_GBS, 4),
        "speedup_vs_f32": round(f32["kernel_ms"] / h["kernel_ms"], 3),
        "rel_err_vs_f32": rel_f16_vs_f32,
    }
    unfused = unfused_leg()
    split["speedup_vs_unfused_f32"] = round(unfused["ms_per_block"] / h["kernel_ms"], 3)
    line = {
        "metric": METRIC, "value": round(value, 2), "unit": "Msamples/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(f32["step_ms"], 5),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": "ATA Mode-B block: CI8 A28 F192 T8192 P2 -> beamform B16 (FP32) "
                               "-> FFT4 channelize -> polarize XY->LR, CF32 [16,768,2048,2]",
                   "A": A, "F": F, "T": T, "P": P, "B": B, "rate": RATE,
                   "input": "CI8 N(0,16^2) rounded+clipped", "parallelism": "single GPU"},
        "roofline": roof,
        "split_f16": split,
        "unfused_f32": unfused,
        "realtime_factor": round((T / 0.5e6) / t_step, 1),
    }
    if not args.no_extra:
        line["batched"] = _extra(batched_leg)
        line["mode_a"] = _extra(mode_a_leg)
        line["calibration"] = _extra(calibration_leg)
        line["kernels"] = _extra(kernels_leg)
        line["ingest"] = _extra(ingest_leg)
        line["reference_benchmarks"] = _extra(reference_benchmarks_leg)
        line["mode_b_bundle"] = _extra(mode_b_bundle_leg)
        line["mode_h_bundle"] = _extra(mode_h_bundle_leg)
        line["mode_b_bundle_async"] = _extra(mode_b_bundle_async_leg)
        line["mode_b_bundle_async"]["blit_copies"] = _extra(_async_blit_child)
        line["mode_bh_bundle"] = _extra(mode_bh_bundle_leg)
    if not args.no_cpu:
        x, w, outs = bufs
        cpu, errs = cpu_leg(x, w, outs)
        line["cpu_baseline"] = cpu
        line["err_vs_fp64_oracle"] = {k: float(v) for k, v in errs.items()}
    else:
        line["cpu_baseline"] = None
    print(json.dumps(line))


def kernel_only(prec, steps, warmup):
    import torch
    from blade_amd import ops

    dev = torch.device("cuda:0")
    xs = [torch.randint(-127, 128, (A, F, T, P, 2), dtype=torch.int8, device=dev) for _ in range(NSETS)]
    w = torch.randn((B, A, F, 1, P), dtype=torch.complex64, device=dev)
    outs = [torch.empty((B, F * RATE, T // RATE, P), dtype=torch.complex64, device=dev)
            for _ in range(NSETS)]
    for i in range(warmup + steps):
        ops.beamform_chain(xs[i % NSETS], w, False, False, RATE, True, prec, out=outs[i % NSETS])
    # Calibration copy: exactly 1 GiB read + 1 GiB written.
    src = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
    dst = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
    src.fill_(1)
    for _ in range(3):
        ops.gather(src, dst, 0, 1, 0, type_name="i8")
    torch.cuda.synchronize()
    print(f"kernel-only {prec}: {warmup + steps} launches + 3 x 1 GiB copies done", flush=True)


def _traffic():
    """HBM bytes per launch of the fused kernel, from the committed rocprofv3
    FETCH_SIZE/WRITE_SIZE summary (None if it has not been recorded)."""
    p = os.path.join(ROOT, "profiles", "traffic_beamform_chain_f32.json")
    try:
        with open(p) as fh:
            return json.load(fh).get("hbm_bytes_per_launch")
    except (OSError, ValueError):
        return None


if __name__ == "__main__":
    main()
