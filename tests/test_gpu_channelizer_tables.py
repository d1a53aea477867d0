"""First use of a channelizer rate: the twiddle tables are whole for every
stream, and built outside a capture.  Each case is the first of its rate in a
process of its own."""

import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parent.parent

PRELUDE = """
import math, sys
import torch
from blade_amd import ops
def block(C, P, S=3):
    gen = torch.Generator(device="cuda").manual_seed(C + P)
    x = torch.randn((2, 5, S * C, P), dtype=torch.complex64, device="cuda", generator=gen)
    v = x.to(torch.complex128).reshape(2, 5, S, C, P)
    ref = torch.fft.fftshift(torch.fft.fft(v, dim=3), dim=3).permute(0, 1, 3, 2, 4).reshape(2, 5 * C, S, P)
    return x, ref, [torch.zeros_like(ref, dtype=torch.complex64) for _ in range(2)]
def check(C, y, ref, what):
    err = float((y.to(ref.dtype) - ref).norm() / ref.norm())
    print(C, what, err, flush=True)
    assert err <= 2 * math.log2(C) * 2.0 ** -24, (C, what, err)
def power(ref):
    return (ref.abs() ** 2).sum(-1, keepdim=True)
"""

# (rate, polarizations): mixed radices, the tables of the run-time radices,
# both passes of the long rates, a rate that factors into no small radix
TWO_STREAMS = """
a, b = torch.cuda.Stream(), torch.cuda.Stream()
m = torch.randn(4096, 4096, device="cuda")
for C, P in ((1000, 2), (64, 2), (512, 2), (1000, 1), (16384, 2), (65536, 2), (20000, 2), (22, 2)):
    x, ref, (ya, yb) = block(C, P)
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        for _ in range(40):                      # about 40 ms of work ahead of the first use
            m = m @ m
            m = m / m.norm()
    ops.channelizer(x, C, out=ya, stream=a)
    ops.channelizer(x, C, out=yb, stream=b)
    b.synchronize()
    check(C, yb, ref, "second stream")
    a.synchronize()
    check(C, ya, ref, "first stream")
"""

# The first use is inside a capture that allows allocations; an eager call
# comes before the first replay.
IN_CAPTURE = """
for C, P in ((1000, 2), (512, 2), (1000, 1)):
    x, ref, (yg, ye) = block(C, P)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="relaxed"):
        ops.channelizer(x, C, out=yg)
    ops.channelizer(x, C, out=ye)
    torch.cuda.synchronize()
    check(C, ye, ref, "eager before the replay")
    for _ in range(3):
        yg.zero_()
        g.replay()
        torch.cuda.synchronize()
        check(C, yg, ref, "replay")
"""

# After a plan, the first call of a small rate may be captured (nothing is
# allocated): the detector, and in place (rate == number of samples).
PLANNED = """
from blade_amd import _lib
for C in (1, 2, 4, 6, 14, 16, 32):
    _lib.call("blade_channelizer_plan", C, None)
    x, ref, _ = block(C, 2)
    z, zref, _ = block(C, 2, S=1)
    y = torch.zeros((2, 5 * C, 3, 1), device="cuda")
    zin = z.clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.channelizer_detector(x, C, 1, 1, out=y)
        ops.channelizer(z, C, out=z)
    for _ in range(3):
        y.zero_()
        z.copy_(zin)
        g.replay()
        torch.cuda.synchronize()
        check(max(C, 2) ** 2, y, power(ref), "detector")
        check(max(C, 2), z.view(zref.shape), zref, "in place")
"""

# An eager call at one shape warms its rate for every other shape, number of
# polarizations and the detector, whichever kernels these take.
WARMED = """
def captured(run, y, ref, C, what):
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run()
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        check(C, y, ref, what)
for C, P, S in ((4096, 2, 1), (2048, 2, 3), (1000, 1, 3), (1024, 2, 2), (64, 1, 2), (16384, 2, 1)):
    x, ref, (y, _) = block(C, P, S)
    ops.channelizer(x, C, out=y)
    check(C, y, ref, "warm")
    for P, S in ((1, 3), (2, 8)) if C < 16384 else ((1, 3),):
        x, ref, (y, _) = block(C, P, S)
        captured(lambda: ops.channelizer(x, C, out=y), y, ref, C, f"P {P} S {S}")
    if C <= 8192:
        ab = ref[..., 0] * ref[..., 1].conj()
        four = torch.stack((ref[..., 0].abs() ** 2, ref[..., 1].abs() ** 2, ab.real, ab.imag), -1)
        d = torch.zeros(four.shape, device="cuda")
        captured(lambda: ops.channelizer_detector(x, C, 1, 4, out=d), d, four, C * C, "detector")
"""


@pytest.mark.parametrize("script", [TWO_STREAMS, IN_CAPTURE, PLANNED, WARMED],
                         ids=["two_streams", "in_capture", "planned", "warmed"])
def test_first_use(script):
    r = subprocess.run([sys.executable, "-u", "-c", PRELUDE + script], cwd=ROOT, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=110)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
