"""Channelizer kernels at the edges of their plans, against the FP64 DFT.

Bar: an FFT of C points rounds about 2 log2(C) times on the way of a value
(one butterfly level and one twiddle each), so the normwise relative error is
within 2 log2(C) * 2^-24 (random rounding leaves it well below).
"""

import math

import pytest
import torch

from blade_amd import ops

pytestmark = pytest.mark.gpu


def _spectra(x, C):
    A, F, T, P = x.shape
    v = x.to(torch.complex128).reshape(A, F, T // C, C, P)
    return torch.fft.fftshift(torch.fft.fft(v, dim=3), dim=3).permute(0, 1, 3, 2, 4).reshape(A, F * C, T // C, P)


def _rand(seed, *shape):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, dtype=torch.complex64, device="cuda", generator=gen)


def _err(y, ref):
    return float((y.to(ref.dtype) - ref).abs().square().sum().sqrt() / ref.abs().square().sum().sqrt())


def _bar(C):
    return 2 * math.log2(C) * 2.0 ** -24


@pytest.mark.parametrize("A,F,S,C", [(1, 1, 1, 16384), (1, 3, 1, 16384), (1, 5, 2, 16384), (2, 1, 3, 32768),
                                     (1, 1, 1, 65536), (1, 3, 2, 65536)])
def test_four_step(A, F, S, C):
    # odd spectrum counts leave a grid that is no multiple of 8 workgroups
    x = _rand(C + S, A, F, S * C, 2)
    assert _err(ops.channelizer(x, C), _spectra(x, C)) <= _bar(C)


@pytest.mark.parametrize("alias", ["none", "same", "shifted"])
def test_four_step_groups(alias):
    """802 spectra (one group of the 192 MiB scratch and a short one), two per
    channel: apart, in place, and with the output one channel behind the input
    in the same buffer."""
    C, S, F = 16384, 2, 401
    n = F * S * C * 2
    buf = _rand(9, n + S * C * 2)
    off = S * C * 2 if alias == "shifted" else 0
    x = buf[off:off + n].view(1, F, S * C, 2)
    ref = _spectra(x[:, [0, 1, 382, 383, 384, 385, 400]], C)
    out = torch.empty_like(buf[:n]) if alias == "none" else buf[:n]
    y = ops.channelizer(x, C, out=out.view(1, F * C, S, 2))
    y = y.view(F, C, S, 2)[[0, 1, 382, 383, 384, 385, 400]].reshape(1, 7 * C, S, 2)
    assert _err(y, ref) <= _bar(C)


MIXED = [18, 20, 24, 28, 30, 32, 36, 42, 50, 54, 60, 64, 70, 84, 90, 98, 126, 128, 150, 162, 196, 210, 250, 360, 486, 490,
         686, 1000, 1176, 1458, 2058, 2500, 3430, 4096, 4374, 4802, 5000, 6250, 7680, 8064, 8100]


@pytest.mark.parametrize("C", MIXED)
def test_mixed_radices(C):
    """Every radix in every position; spectra that fill no workgroup, one and
    several per channel, and in place."""
    for A, F, S in ((1, 3, 1), (2, 7, 5), (1, 5, 8)):
        x = _rand(C + S, A, F, S * C, 2)
        ref = _spectra(x, C)
        assert _err(ops.channelizer(x, C), ref) <= _bar(C)
        if S == 1:
            ops.channelizer(x, C, out=x)
            assert _err(x.view(ref.shape), ref) <= _bar(C)


def _detect(spec, n, pols):
    X, Y = spec[..., 0], spec[..., 1]
    if pols == 1:
        d = (X.abs().square() + Y.abs().square())[..., None]
    else:
        xy = X * Y.conj()
        d = torch.stack((X.abs().square(), Y.abs().square(), xy.real, xy.imag), dim=-1)
    a, f, t, q = d.shape
    return d.reshape(a, f, t // n, n, q).sum(3)


@pytest.mark.parametrize("C", [4, 6, 18, 32, 64, 128, 256, 512, 1024, 2048, 4096, 8192, 96, 490, 1000, 4802, 8100])
@pytest.mark.parametrize("A,F,S,N", [(1, 1, 1, 1), (1, 1, 6, 2), (1, 3, 7, 1), (2, 5, 9, 3), (1, 37, 4, 4), (1, 2, 40, 40)])
@pytest.mark.parametrize("pols", [1, 4])
def test_integrations_of_a_block(C, A, F, S, N, pols):
    """Every integration is an item of its own: counts that leave slots of the
    last workgroup idle, several integrations per channel, then the same block
    added again.  Sums of N powers round N more times."""
    x = _rand(C + S + N, A, F, S * C, 2)
    ref = _detect(_spectra(x, C), N, pols)
    bar = 2 * _bar(C) + (N + 4) * 2.0 ** -24
    y = ops.channelizer_detector(x, C, N, pols)
    assert y.shape == ref.shape and _err(y, ref) <= bar
    if N == S:                                  # stepped over two blocks
        ops.channelizer_detector(x, C, 2 * N, pols, out=y)
        ops.channelizer_detector(x, C, 2 * N, pols, out=y, accumulate=True)
        assert _err(y, 2 * ref) <= 2 * bar


@pytest.mark.parametrize("F,S", [(256, 2), (257, 2), (384, 4), (383, 4), (103, 5), (103, 6)])
def test_4096_by_number_of_spectra(F, S):
    """Both kernels of the rate, on each side of their bounds."""
    x = _rand(F + S, 1, F, S * 4096, 2)
    assert _err(ops.channelizer(x, 4096), _spectra(x, 4096)) <= _bar(4096)
