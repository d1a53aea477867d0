"""The workloads whose speed is measured: what one pass is, on which inputs.

``listed()`` are the standing cases, ``draw(rng)`` makes further ones of the
same ranges, ``prepare(case, seed)`` holds what a program has in hand before
the call (device buffers, as the Pipeline modules keep them), ``run(state)``
is one pass through the public entry points, ``exact(case, seed)`` the same
outputs from plain torch in 64 bits, and ``work(case)`` the bytes and
operations a pass cannot do without.

Kinds of pass:

* ``chain``    beamform -> channelize (rate 1, 2 or 4) -> [polarize] of one block
* ``mode_a``   two blocks: beamform, fine channelizer and Stokes I over both
* ``spectra``  channelizer at any rate
* ``mode_h``   channelizer -> [polarizer] -> detector
* ``gradient`` Stokes-I loss of weighted beams and its phasor gradient (forward + backward)
* ``adjoint``  beamforming under autograd: beams forward, phasor gradient backward
* ``batch``    beamformer blocks of different shapes in one launch

Voltages are CI8 Gaussian noise of sigma 16, phasors
``exp(-j 2 pi f tau)`` with delays within +-100 ns times per-antenna
calibrations of about unit amplitude, beams (inputs of the channelizer) CF32
Gaussian noise: what the telescope path meets.
"""

from __future__ import annotations

import math

import torch

from blade_amd import calibration, ops

# ----------------------------------------------------------------- the cases


def listed():
    return [
        # A short real-time block of plain beams with the incoherent beam: the
        # smallest call of the path, where latency counts.
        dict(name="plain-small", kind="chain", dtype="ci8", precision="f32", A=20, F=192, T=512, B=8,
             incoherent=True, rate=1, polarize=False),
        # The production Mode-B block (16 beams, FFT-4, XY -> LR) in FP32 ...
        dict(name="mode-b", kind="chain", dtype="ci8", precision="f32", A=28, F=192, T=8192, B=16,
             incoherent=False, rate=4, polarize=True),
        # ... and with split-FP16 phasors.
        dict(name="mode-b-f16x2", kind="chain", dtype="ci8", precision="f16x2", A=28, F=192, T=8192, B=16,
             incoherent=False, rate=4, polarize=True),
        # A block no tile size divides: odd antennas, channels and beams, a
        # capture of 3000 samples, incoherent beam, FFT-2.
        dict(name="ragged", kind="chain", dtype="ci8", precision="f32", A=27, F=117, T=3000, B=11,
             incoherent=True, rate=2, polarize=False),
        # The beamformer module on CF32 voltages (the reference's own
        # beamformer benchmark: 20 antennas, 8 beams).
        dict(name="beamformer-cf32", kind="chain", dtype="cf32", precision="f32", A=20, F=192, T=8192, B=8,
             incoherent=False, rate=1, polarize=False),
        # Mode A: 8 split-FP16 beams of two blocks into a fine filterbank of
        # 8192 channels, Stokes I over the 4 spectra.
        dict(name="mode-a", kind="mode_a", precision="f16x2", A=28, F=192, T=16384, B=8, C=8192),
        # Mode H with full Stokes: a medium-resolution filterbank, short
        # integrations, circular polarizations.
        dict(name="mode-h", kind="mode_h", A=8, F=192, T=8192, C=512, N=8, pols=4, polarize=True),
        # The fine channelizer of the reference's Mode-BH benchmark: 3 beams
        # of 8 gathered blocks at rate 65536.
        dict(name="spectra-65536", kind="spectra", A=3, F=192, T=65536, C=65536),
        # A rate that is no power of two (0.5 MHz channels to 0.5 kHz).
        dict(name="spectra-1000", kind="spectra", A=8, F=96, T=12000, C=1000),
        # One loss + gradient evaluation of the gain calibration.
        dict(name="gradient", kind="gradient", precision="f32", A=42, F=384, T=2048, B=4),
        # Beamforming inside a differentiable program, forward and backward.
        dict(name="adjoint", kind="adjoint", A=42, F=384, T=2048, B=4),
        # Uneven blocks (several observations' sub-bands) in one launch.
        dict(name="batch", kind="batch", precision="f32",
             blocks="28x128x4096x16 14x256x2048x40 20x64x8192x8 27x256x1024x4 "
                    "28x64x4096x64 20x128x2048x24 14x1024x1024x12 27x64x2048x33"),
    ]


# A drawn case stays below this many bytes of inputs and outputs.
_DRAW_BYTES = 600_000_000


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth_rate(rng, lo, hi):
    """An even rate in [lo, hi] made of 2, 3, 5 and 7, powers of two half of the time."""
    if rng.random() < 0.5:
        return 2 ** rng.randint(math.ceil(math.log2(lo)), math.floor(math.log2(hi)))
    while True:
        c = 2
        target = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        while c < target:
            c *= rng.choice((2, 2, 2, 3, 5, 7))
        if lo <= c <= hi:
            return c


def _fit(case):
    """Fewer channels until the case fits the byte bound."""
    while work(case)["bytes"] > _DRAW_BYTES and case["F"] > 1:
        case["F"] = max(1, case["F"] * 3 // 4)
    return case


def draw(rng):
    kind = rng.choice(("chain", "chain", "chain", "mode_a", "mode_h", "mode_h", "spectra", "spectra",
                       "gradient", "adjoint", "batch"))
    A = _log_int(rng, 6, 64)
    F = _log_int(rng, 16, 384)
    if kind == "chain":
        rate = rng.choice((1, 1, 2, 4))
        T = _log_int(rng, 256, 16384)
        T = max(rate, T // 64 * 64) if rng.random() < 0.5 else T
        if rate > 1:
            T = T // 4 * 4
        dtype = rng.choice(("ci8", "ci8", "ci8", "cf32"))
        precision = "f32" if dtype == "cf32" else rng.choice(("f32", "f32", "f16x2"))
        return _fit(dict(kind=kind, dtype=dtype, precision=precision, A=A, F=F, T=T, B=_log_int(rng, 1, 40),
                         incoherent=rng.random() < 0.4, rate=rate, polarize=rate > 1 and rng.random() < 0.6))
    if kind == "mode_a":
        C = _smooth_rate(rng, 128, 8192)
        return _fit(dict(kind=kind, precision=rng.choice(("f32", "f16x2")), A=A, F=F, T=C * rng.randint(1, 4),
                         B=_log_int(rng, 1, 16), C=C))
    if kind == "mode_h":
        C = _smooth_rate(rng, 32, 8192)
        N = _log_int(rng, 1, 16)
        S = N * max(1, _log_int(rng, 8, 16384) // (C * N))
        return _fit(dict(kind=kind, A=rng.randint(1, 16), F=F, T=C * S, C=C, N=N, pols=rng.choice((1, 4)),
                         polarize=rng.random() < 0.5))
    if kind == "spectra":
        C = _smooth_rate(rng, 16, 65536)
        S = max(1, _log_int(rng, 16, 32768) // C)
        return _fit(dict(kind=kind, A=rng.randint(1, 16), F=F, T=C * S, C=C))
    if kind == "batch":
        shapes = []
        for _ in range(rng.randint(3, 10)):
            shapes.append((rng.choice((14, 20, 27, 28)), rng.choice((64, 128, 256)), 64 * _log_int(rng, 8, 64),
                           _log_int(rng, 4, 64)))
        case = dict(kind=kind, precision=rng.choice(("f32", "f16x2")), blocks="")
        while True:
            case["blocks"] = " ".join("x".join(map(str, s)) for s in shapes)
            if work(case)["bytes"] <= _DRAW_BYTES or len(shapes) == 1:
                return case
            shapes.pop()
    T = _log_int(rng, 256, 4096)
    T = T // 4 * 4 if rng.random() < 0.7 else T
    case = dict(kind=kind, A=A, F=F, T=T, B=_log_int(rng, 1, 16))
    if kind == "gradient":
        case["precision"] = rng.choice(("f32", "f32", "f16x2"))
    return _fit(case)


def _blocks(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["blocks"].split()]


# ---------------------------------------------------------------- the inputs


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _voltages(gen, A, F, T):
    x = torch.randn((A, F, T, 2, 2), device="cuda", generator=gen)
    return x.mul_(16.0).round_().clamp_(-127, 127).to(torch.int8)


def _phasors(gen, B, A, F):
    f = 1.0e9 + 0.5e6 * torch.arange(F, device="cuda", dtype=torch.float64)
    tau = (torch.rand((B, A, 1, 1, 1), device="cuda", generator=gen, dtype=torch.float64) - 0.5) * 200e-9
    phase = -2.0 * math.pi * f[None, None, :, None, None] * tau
    gain = 1.0 + 0.1 * torch.randn((1, A, F, 1, 2), device="cuda", generator=gen, dtype=torch.float64)
    return torch.polar(gain.expand(B, A, F, 1, 2).contiguous(),
                       phase.expand(B, A, F, 1, 2).contiguous()).to(torch.complex64)


def _cf32(gen, *shape, scale=1.0):
    return torch.randn(shape, device="cuda", dtype=torch.complex64, generator=gen) * scale


def _inputs(case, seed):
    """The input tensors of one pass, from the seed alone."""
    gen = _generator(seed)
    kind = case["kind"]
    if kind == "batch":
        return [(_voltages(gen, A, F, T), _phasors(gen, B, A, F)) for A, F, T, B in _blocks(case)]
    A, F, T = case["A"], case["F"], case["T"]
    if kind in ("spectra", "mode_h"):
        return {"x": _cf32(gen, A, F, T, 2, scale=64.0)}
    B = case["B"]
    if kind == "chain":
        x = _voltages(gen, A, F, T) if case["dtype"] == "ci8" else _cf32(gen, A, F, T, 2, scale=16.0)
        return {"x": x, "w": _phasors(gen, B, A, F)}
    if kind == "mode_a":
        return {"x": [_voltages(gen, A, F, T) for _ in range(2)], "w": _phasors(gen, B, A, F)}
    if kind == "gradient":
        # beam 0 calibrates on the source, the others weigh in less
        return {"x": _voltages(gen, A, F, T), "w": _phasors(gen, B, A, F),
                "lam": [1.0] + [0.25] * (B - 1)}
    return {"x": _voltages(gen, A, F, T), "w": _phasors(gen, B, A, F), "gy": _cf32(gen, B, F, T, 2)}


def _groups(case):
    S = case["T"] // case["C"]
    return S // case["N"] if case["N"] <= S else 1


def prepare(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    if kind == "batch":
        blocks = [(x, w, torch.empty((w.shape[0],) + tuple(x.shape[1:4]), dtype=torch.complex64, device="cuda"))
                  for x, w in inp]
        return {"case": case, "plan": ops.BatchedBeamformer(blocks, case["precision"])}
    state = dict(inp, case=case)
    F, T = case["F"], case["T"]
    if kind == "chain":
        nb, r = case["B"] + int(case["incoherent"]), case["rate"]
        state["out"] = torch.empty((nb, F * r, T // r, 2), dtype=torch.complex64, device="cuda")
    elif kind == "mode_a":
        state["beams"] = torch.empty((case["B"], F, T, 2), dtype=torch.complex64, device="cuda")
        state["out"] = torch.empty((case["B"], F * case["C"], 1, 1), dtype=torch.float32, device="cuda")
    elif kind == "mode_h":
        state["out"] = torch.empty((case["A"], F * case["C"], _groups(case), case["pols"]), dtype=torch.float32,
                                   device="cuda")
    elif kind == "spectra":
        state["out"] = torch.empty((case["A"], F * case["C"], T // case["C"], 2), dtype=torch.complex64,
                                   device="cuda")
    else:
        state["w"] = state["w"].requires_grad_(True)
    return state


# ---------------------------------------------------------------- one pass


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "chain":
        return ops.beamform_chain(state["x"], state["w"], case["incoherent"], False, case["rate"], case["polarize"],
                                  case["precision"], out=state["out"])
    if kind == "mode_a":
        n = 2 * (case["T"] // case["C"])           # the spectra of both blocks
        for k, x in enumerate(state["x"]):
            ops.beamformer(x, state["w"], precision=case["precision"], out=state["beams"])
            ops.channelizer_detector(state["beams"], case["C"], n, 1, out=state["out"], accumulate=k == 1)
        return state["out"]
    if kind == "mode_h":
        return ops.channelizer_detector(state["x"], case["C"], case["N"], case["pols"], out=state["out"],
                                        polarize=case["polarize"])
    if kind == "spectra":
        return ops.channelizer(state["x"], case["C"], out=state["out"])
    if kind == "gradient":
        loss = calibration.stokes_i_power(state["x"], state["w"], state["lam"], case["precision"])
        (grad,) = torch.autograd.grad(loss, state["w"])
        return loss.detach(), grad
    if kind == "adjoint":
        y = calibration.beamform(state["x"], state["w"])
        (grad,) = torch.autograd.grad(y, state["w"], state["gy"])
        return y.detach(), grad
    return state["plan"]()


# ---------------------------------------------------------- 64-bit reference


def _c128(x):
    """CI8 [..., 2] or CF32 as complex128."""
    return torch.view_as_complex(x.double()) if x.dtype == torch.int8 else x.to(torch.complex128)


def _channel_steps(F, per_channel):
    step = max(1, int(2 ** 25 // max(1, per_channel)))
    return [(f, min(F, f + step)) for f in range(0, F, step)]


def _beams64(x, w, incoherent=False):
    """sum_a x w of every beam, and the incoherent beam, [B', F, T, 2]."""
    B, A, F, _, P = w.shape
    T = x.shape[2]
    out = torch.empty((B + int(incoherent), F, T, P), dtype=torch.complex128, device="cuda")
    for f0, f1 in _channel_steps(F, (A + B) * T * P):
        v = _c128(x[:, f0:f1]).permute(1, 3, 0, 2).contiguous()                    # [f, P, A, T]
        ww = w[:, :, f0:f1, 0].to(torch.complex128).permute(2, 3, 0, 1).contiguous()   # [f, P, B, A]
        out[:B, f0:f1] = torch.matmul(ww, v).permute(2, 0, 3, 1)
        if incoherent:
            w2 = ww[:, :, 0].abs().square()
            out[B, f0:f1] = (v.abs().square() * w2[..., None]).sum(2).permute(0, 2, 1)
    return out


def _spectra64(x, C):
    """fftshift(FFT) of every C samples, [A, F, T, P] -> [A, F C, T/C, P]."""
    A, F, T, P = x.shape
    out = torch.empty((A, F, C, T // C, P), dtype=torch.complex128, device="cuda")
    for f0, f1 in _channel_steps(F, A * T * P):
        v = x[:, f0:f1].to(torch.complex128).reshape(A, f1 - f0, T // C, C, P)
        out[:, f0:f1] = torch.fft.fftshift(torch.fft.fft(v, dim=3), dim=3).permute(0, 1, 3, 2, 4)
    return out.reshape(A, F * C, T // C, P)


def _circular64(x):
    return torch.stack((x[..., 0] + 1j * x[..., 1], x[..., 0] - 1j * x[..., 1]), dim=-1)


def _detect64(x, n, pols):
    """Stokes I or [XX*, YY*, Re XY*, Im XY*] over n consecutive samples."""
    X, Y = x[..., 0], x[..., 1]
    if pols == 1:
        d = (X.abs().square() + Y.abs().square())[..., None]
    else:
        xy = X * Y.conj()
        d = torch.stack((X.abs().square(), Y.abs().square(), xy.real, xy.imag), dim=-1)
    a, f, t, q = d.shape
    return d.reshape(a, f, t // n, n, q).sum(3)


def exact(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    if kind == "batch":
        return [_beams64(x, w) for x, w in inp]
    if kind == "chain":
        y = _beams64(inp["x"], inp["w"], case["incoherent"])
        if case["rate"] > 1:
            y = _spectra64(y, case["rate"])
        return _circular64(y) if case["polarize"] else y
    if kind == "spectra":
        return _spectra64(inp["x"], case["C"])
    if kind == "mode_h":
        y = _spectra64(inp["x"], case["C"])
        return _detect64(_circular64(y) if case["polarize"] else y, case["N"], case["pols"])
    if kind == "mode_a":
        total = 0.0
        for x in inp["x"]:
            y = _spectra64(_beams64(x, inp["w"]), case["C"])
            total = total + _detect64(y, case["T"] // case["C"], 1)
        return total
    y = _beams64(inp["x"], inp["w"])
    if kind == "gradient":
        lam = torch.tensor(inp["lam"], dtype=torch.float64, device="cuda")
        loss = -(lam * y.abs().square().sum((1, 2, 3))).sum()
        gy = -2.0 * lam[:, None, None, None] * y          # PyTorch's gradient of y
        return loss, _adjoint64(inp["x"], gy)
    return y, _adjoint64(inp["x"], inp["gy"].to(torch.complex128))


def _adjoint64(x, gy):
    """sum_t gy conj(x), [B, A, F, 1, P]."""
    B, F, T, P = gy.shape
    A = x.shape[0]
    out = torch.empty((B, A, F, 1, P), dtype=torch.complex128, device="cuda")
    for f0, f1 in _channel_steps(F, (A + B) * T * P):
        v = _c128(x[:, f0:f1]).conj().resolve_conj().permute(1, 3, 2, 0).contiguous()   # [f, P, T, A]
        g = gy[:, f0:f1].permute(1, 3, 0, 2).contiguous()                               # [f, P, B, T]
        out[:, :, f0:f1, 0] = torch.matmul(g, v).permute(2, 3, 0, 1)
    return out


# ------------------------------------------------- what a pass cannot avoid


def _beam_work(A, F, T, B, in_bytes, incoherent=False):
    nb = B + int(incoherent)
    return {"bytes": in_bytes * A * F * T * 2 + 8 * B * A * F * 2 + 8 * nb * F * T * 2,
            "flops": 8 * A * B * F * T * 2 + (5 * A * F * T * 2 if incoherent else 0)}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        parts = [_beam_work(A, F, T, B, 2) for A, F, T, B in _blocks(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    A, F, T = case["A"], case["F"], case["T"]
    n = A * F * T * 2                               # complex samples of the input
    if kind == "chain":
        r = _beam_work(A, F, T, case["B"], 2 if case["dtype"] == "ci8" else 8, case["incoherent"])
        nb = case["B"] + int(case["incoherent"])
        per = (5 * math.log2(case["rate"])) + (4 if case["polarize"] else 0)
        return {"bytes": r["bytes"], "flops": r["flops"] + int(per * nb * F * T * 2)}
    if kind == "mode_a":
        B, C = case["B"], case["C"]
        ny = B * F * T * 2
        return {"bytes": 2 * 2 * n + 8 * B * A * F * 2 + 4 * B * F * C,
                "flops": 2 * int(8 * A * ny + 5 * math.log2(C) * ny + 4 * ny)}
    if kind == "mode_h":
        return {"bytes": 8 * n + 4 * A * F * case["C"] * _groups(case) * case["pols"],
                "flops": int((5 * math.log2(case["C"]) + (4 if case["pols"] == 1 else 8)) * n)}
    if kind == "spectra":
        return {"bytes": 16 * n, "flops": int(5 * math.log2(case["C"]) * n)}
    B = case["B"]
    nw, ny = B * A * F * 2, B * F * T * 2
    if kind == "gradient":                          # beams recomputed, never stored
        return {"bytes": 2 * n + 16 * nw, "flops": 16 * A * ny + 6 * ny}
    return {"bytes": 2 * 2 * n + 16 * nw + 16 * ny, "flops": 16 * A * ny}
