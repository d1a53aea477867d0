"""Channelizer and detector at the bounds of their kernels' index types.

Blocks of zeros with a few spectra of noise: every other output must be zero
(the buffer starts as NaN, so an output that nothing wrote shows too).
"""

import math

import pytest
import torch

from blade_amd import ops

pytestmark = pytest.mark.gpu


def _powers(spec, pols):
    """FP64 powers of spectra [n, C, 2], fftshifted: [C, n, pols]."""
    X = torch.fft.fftshift(torch.fft.fft(spec.to(torch.complex128), dim=1), dim=1)
    a, b = X[..., 0], X[..., 1]
    if pols == 1:
        return (a.abs().square() + b.abs().square()).T[..., None]
    xy = a * b.conj()
    return torch.stack((a.abs().square(), b.abs().square(), xy.real, xy.imag), -1).transpose(0, 1)


def _needs(gib):
    free, _ = torch.cuda.mem_get_info()
    if free < gib * 2 ** 30:
        pytest.skip(f"needs {gib} GiB of device memory")


def _sparse_block(C, S, at, seed):
    """One channel of S spectra, zero but for those numbered `at`."""
    x = torch.zeros((1, 1, S * C, 2), dtype=torch.complex64, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    noise = torch.randn((len(at), C, 2), dtype=torch.complex64, device="cuda", generator=gen)
    for i, s in enumerate(at):
        x[0, 0, s * C:(s + 1) * C] = noise[i]
    return x, noise


def _check_single_spectra(C, S, pols, at):
    """Integrations of one spectrum."""
    x, noise = _sparse_block(C, S, at, 1)
    out = torch.full((1, C, S, pols), float("nan"), dtype=torch.float32, device="cuda")
    ops.channelizer_detector(x, C, 1, pols, out=out)
    del x
    ref = _powers(noise, pols)
    got = out[0][:, at].double()
    err = float((got - ref).norm() / ref.norm())
    assert err <= (4 * math.log2(max(C, 2)) + 5) * 2.0 ** -24
    out[0][:, at] = 0
    for k in range(C):
        row = out[0, k].view(-1)
        for i in range(0, row.numel(), 1 << 28):
            assert not (row[i:i + (1 << 28)] != 0).any(), f"channel {k}"
    del out
    torch.cuda.empty_cache()


def test_outputs_past_32_bits_of_a_channel():
    """C * integrations * 4 past 2^32: the last rows' offsets."""
    C, S = 256, 4_600_000
    _needs(48)
    _check_single_spectra(C, S, 4, [0, 1, S // 2, S - 1])


def test_integrations_past_31_bits():
    """More than 2^31 integrations of one channel."""
    S = 2 ** 31 + 8
    _needs(64)
    _check_single_spectra(1, S, 1, [0, 1, 2 ** 31 - 1, 2 ** 31, S - 1])


@pytest.mark.parametrize("C", [1, 4, 64, 96, 256, 1000, 4096, 4374, 4802, 8100, 8192])
@pytest.mark.parametrize("S", [3, 70])
@pytest.mark.parametrize("pols", [1, 4])
def test_adding_a_block_rounds_once(C, S, pols):
    """An integration over several blocks: each call adds its block's sums in one
    FP32 addition.  On outputs 2^20 times the block's, adding them in parts
    rounds by many times more than half a unit in the last place."""
    gen = torch.Generator(device="cuda").manual_seed(C + S)
    x = torch.randn((1, 5, S * C, 2), dtype=torch.complex64, device="cuda", generator=gen)
    y = ops.channelizer_detector(x, C, S, pols)
    start = 2.0 ** (20 + round(math.log2(4 * C * S)))
    out = torch.full_like(y, start)
    ops.channelizer_detector(x, C, 3 * S, pols, out=out, accumulate=True)
    err = float((out.double() - (start + y.double())).abs().max())
    assert err <= start * 2.0 ** -24 * (1 + 2.0 ** -10)


def _check_sparse_spectra(C, S, at):
    x, noise = _sparse_block(C, S, at, C)
    y = torch.full((1, C, S, 2), complex("nan"), dtype=torch.complex64, device="cuda")
    ops.channelizer(x, C, out=y)
    X = torch.fft.fftshift(torch.fft.fft(noise.to(torch.complex128), dim=1), dim=1).transpose(0, 1)
    err = float((y[0][:, at] - X).norm() / X.norm())
    assert err <= 2 * math.log2(C) * 2.0 ** -24
    y[0][:, at] = 0
    for k in range(C):
        assert not (y[0, k] != 0).any(), f"channel {k}"


@pytest.mark.parametrize("C", [64, 256, 2048, 4096, 8192])
def test_channels_past_63_million_samples(C):
    """Spectra of one long channel, and their powers in integrations of one."""
    S = 2 ** 26 // C + 16
    _needs(8)
    at = [0, 7, S // 2, S - 1]
    _check_sparse_spectra(C, S, at)
    for pols in (1, 4):
        _check_single_spectra(C, S, pols, at)


def test_channel_past_31_bits_of_samples():
    S = 2 ** 31 // 64 + 24
    _needs(80)
    _check_sparse_spectra(64, S, [0, S // 2, S - 2, S - 1])
    torch.cuda.empty_cache()


@pytest.mark.parametrize("F,S", [(256, 2), (257, 2), (416, 2), (417, 2), (208, 4), (209, 4)])
def test_4096_by_rounds_of_workgroups(F, S):
    """512 and 832 spectra on 256 compute units: both kernels, on each side."""
    gen = torch.Generator(device="cuda").manual_seed(F)
    x = torch.randn((1, F, S * 4096, 2), dtype=torch.complex64, device="cuda", generator=gen)
    v = x.to(torch.complex128).reshape(1, F, S, 4096, 2)
    ref = torch.fft.fftshift(torch.fft.fft(v, dim=3), dim=3).permute(0, 1, 3, 2, 4).reshape(1, F * 4096, S, 2)
    err = float((ops.channelizer(x, 4096) - ref).norm() / ref.norm())
    assert err <= 2 * 12 * 2.0 ** -24
