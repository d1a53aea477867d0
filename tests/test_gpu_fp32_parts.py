"""FP32 beamforming of CI8 voltages on three exact BF16 phasor parts.

Elementwise bar: with exact products, only the FP32 accumulation of the 2A
real terms rounds (unit roundoff 2^-24; the matrix core's own summation is
allowed a factor of two), so |y - ref| <= 2 (2A + 2) 2^-24 sum_a |w| |x|,
with (|Re w| + |Im w|) (|Re x| + |Im x|) bounding each antenna's terms.
"""

import numpy as np
import pytest
import torch

import oracle as O
from blade_amd import ops
from blade_amd._lib import BladeError

pytestmark = pytest.mark.gpu


def _case(A, F, T, B, seed):
    rng = np.random.default_rng(seed)
    x8 = rng.integers(-128, 128, size=(A, F, T, 2, 2), dtype=np.int8)
    # phasor magnitudes from 1e-20 to 1e20 over the beams: no scale is shared
    mag = 10.0 ** rng.uniform(-20, 20, size=(B, 1, 1, 1, 1))
    w = (mag * (rng.normal(size=(B, A, F, 1, 2)) + 1j * rng.normal(size=(B, A, F, 1, 2)))).astype(np.complex64)
    return x8, w


def _check(y, x8, w, A, B):
    ref = O.beamformer_ata(x8, w, False, False)
    x = np.abs(x8[..., 0].astype(np.float64)) + np.abs(x8[..., 1].astype(np.float64))
    ww = np.abs(w[:, :, :, 0].real.astype(np.float64)) + np.abs(w[:, :, :, 0].imag.astype(np.float64))
    bound = 2 * (2 * A + 2) * 2.0 ** -24 * np.einsum("bafp,aftp->bftp", ww, x)
    d = y[:B] - ref
    assert (np.maximum(np.abs(d.real), np.abs(d.imag)) <= bound).all()


@pytest.mark.parametrize("A,B", [(1, 1), (15, 8), (16, 9), (17, 16), (33, 5), (176, 16), (177, 16), (193, 9),
                                 (240, 17), (400, 8)])
@pytest.mark.parametrize("T", [64, 132, 70])
def test_fp32_parts_match_oracle_elementwise(A, B, T):
    x8, w = _case(A, 2, T, B, A * 100 + B)
    y = ops.beamformer(torch.from_numpy(x8).cuda(), torch.from_numpy(w).cuda()).cpu().numpy()
    _check(y, x8, w, A, B)


def test_antenna_limits():
    for A, B, ok in ((240, 9, True), (241, 9, False), (400, 8, True), (401, 8, False)):
        x = torch.zeros((A, 1, 64, 2, 2), dtype=torch.int8, device="cuda")
        w = torch.zeros((B, A, 1, 1, 2), dtype=torch.complex64, device="cuda")
        y = torch.empty((B, 1, 64, 2), dtype=torch.complex64, device="cuda")
        if ok:
            ops.beamformer(x, w)
            ops.BatchedBeamformer([(x, w, y)], tuning={"beam_tiles": 2 if B > 8 else 1})()
        else:
            with pytest.raises(BladeError, match="too many antennas"):
                ops.beamformer(x, w)
            with pytest.raises(BladeError, match="too many antennas"):
                ops.BatchedBeamformer([(x, w, y)])()


def test_nonfinite_phasors_stay_in_their_beam():
    x8, w = _case(20, 1, 64, 4, 3)
    w[1, 3, 0, 0, 0] = np.inf
    w[2, 5, 0, 0, 1] = np.nan
    with np.errstate(invalid="ignore"):
        y = ops.beamformer(torch.from_numpy(x8).cuda(), torch.from_numpy(w).cuda()).cpu().numpy()
    assert not np.isfinite(y[1, :, :, 0]).any() and not np.isfinite(y[2, :, :, 1]).any()
    assert np.isfinite(y[[0, 3]]).all() and np.isfinite(y[1, :, :, 1]).all() and np.isfinite(y[2, :, :, 0]).all()


@pytest.mark.parametrize("A,B", [(1, 1), (16, 8), (17, 9), (42, 4), (64, 3), (80, 2), (96, 5), (128, 17)])
@pytest.mark.parametrize("T,offset", [(1, 0), (31, 0), (32, 0), (132, 0), (130, 0), (260, 1)])
def test_adjoint_matches_oracle_elementwise(A, B, T, offset):
    """sum_t gy conj(x): 2T exact products accumulated in FP32, the sums of the
    four waves and of the time splits after them; ``offset`` float2s shift the
    gradient off 16-byte alignment (single loads)."""
    rng = np.random.default_rng(A + 10 * T)
    x8 = rng.integers(-128, 128, size=(A, 3, T, 2, 2), dtype=np.int8)
    gy = (10.0 ** rng.uniform(-6, 6, size=(B, 1, 1, 1)) *
          (rng.normal(size=(B, 3, T, 2)) + 1j * rng.normal(size=(B, 3, T, 2)))).astype(np.complex64)
    buf = torch.empty(gy.size + offset, dtype=torch.complex64, device="cuda")
    gyd = buf[offset:].view(gy.shape)
    gyd.copy_(torch.from_numpy(gy))
    got = ops.beamformer_adjoint(torch.from_numpy(x8).cuda(), gyd).cpu().numpy()
    ref = O.beamformer_adjoint(x8, gy)
    g1 = np.abs(gy.real.astype(np.float64)) + np.abs(gy.imag.astype(np.float64))
    x1 = np.abs(x8[..., 0].astype(np.float64)) + np.abs(x8[..., 1].astype(np.float64))
    bound = 2 * (2 * T + 16) * 2.0 ** -24 * np.einsum("bftp,aftp->bafp", g1, x1)[:, :, :, None]
    d = got - ref
    assert (np.maximum(np.abs(d.real), np.abs(d.imag)) <= bound).all()
    again = ops.beamformer_adjoint(torch.from_numpy(x8).cuda(), gyd).cpu().numpy()
    assert (again == got).all()


@pytest.mark.parametrize("precision", ["f32", "f16x2"])
@pytest.mark.parametrize("A,B", [(1, 1), (16, 8), (17, 9), (42, 4), (48, 3), (64, 5), (65, 2), (96, 2), (128, 17)])
@pytest.mark.parametrize("T,offset", [(1, 0), (63, 0), (64, 0), (68, 0), (260, 0), (261, 0), (512, 1)])
def test_stokes_gradient_matches_oracle_elementwise(A, B, T, offset, precision):
    """y as in the forward test (error ey); gy = -lambda y rounds once; the
    adjoint accumulates 2T terms and the partial sums.  ``offset`` shifts the
    voltages off 16-byte alignment (single loads).  Split FP16 phasors are
    off by 2^-22 of themselves, or by half the smallest FP16 step (2^-25) of
    a scale below twice the largest of the pol and beam group of 8."""
    rng = np.random.default_rng(A + 10 * T)
    x8 = rng.integers(-128, 128, size=(A, 2, T, 2, 2), dtype=np.int8)
    w = (10.0 ** rng.uniform(-4, 4, size=(B, 1, 1, 1, 1)) *
         (rng.normal(size=(B, A, 2, 1, 2)) + 1j * rng.normal(size=(B, A, 2, 1, 2)))).astype(np.complex64)
    lam = [float(np.float32(v)) for v in rng.uniform(0.1, 1.0, size=B)]
    buf = torch.empty(x8.size + 4 * offset, dtype=torch.int8, device="cuda")
    xd = buf[4 * offset:].view(x8.shape)
    xd.copy_(torch.from_numpy(x8))
    loss, got = ops.stokes_i_loss_and_grad(xd, torch.from_numpy(w).cuda(), lam, precision=precision)
    got = got.cpu().numpy()[:, :, :, 0]
    x = x8[..., 0].astype(np.float64) + 1j * x8[..., 1]
    y = np.einsum("bafp,aftp->bftp", w[:, :, :, 0].astype(np.complex128), x)
    L = np.array(lam)[:, None, None, None]
    ref = np.einsum("bftp,aftp->bafp", -L * y, x.conj())
    x1 = np.abs(x.real) + np.abs(x.imag)
    w1 = np.abs(w.real[:, :, :, 0].astype(np.float64)) + np.abs(w.imag[:, :, :, 0].astype(np.float64))
    u = 2.0 ** -24
    ey = 2 * (2 * A + 2) * u * np.einsum("bafp,aftp->bftp", w1, x1)
    if precision == "f16x2":
        ew = 2.0 ** -22 * w1
        for b in range(0, B, 8):
            top = np.maximum(np.abs(w.real[b:b + 8]), np.abs(w.imag[b:b + 8])).astype(np.float64)[:, :, :, 0]
            ew[b:b + 8] += 2 * 2.0 ** -25 * 2 * top.max((0, 1))
        ey += np.einsum("bafp,aftp->bftp", ew, x1)
    y1 = np.abs(y.real) + np.abs(y.imag) + 2 * ey
    bound = np.einsum("bftp,aftp->bafp", L * (2 * ey + (2 * (2 * T + 16) + 2) * u * y1), x1)
    d = got - ref
    assert (np.maximum(np.abs(d.real), np.abs(d.imag)) <= bound).all()
    power = float((L * np.abs(y) ** 2).sum())
    assert abs(float(loss) + power) <= float((L * (2 * np.sqrt(2) * np.abs(y) * ey + ey ** 2 + 64 * u * np.abs(y) ** 2)).sum())


def test_stokes_gradient_keeps_nonfinite_values_in_their_beam():
    rng = np.random.default_rng(1)
    x8 = rng.integers(-128, 128, size=(20, 1, 128, 2, 2), dtype=np.int8)
    w = (rng.normal(size=(3, 20, 1, 1, 2)) + 1j * rng.normal(size=(3, 20, 1, 1, 2))).astype(np.complex64)
    w[1, 4, 0, 0, 0] = np.inf
    _, got = ops.stokes_i_loss_and_grad(torch.from_numpy(x8).cuda(), torch.from_numpy(w).cuda(), [1.0, 1.0, 1.0])
    got = got.cpu().numpy()
    assert np.isfinite(got[[0, 2]]).all() and np.isfinite(got[1, ..., 1]).all()
    assert not np.isfinite(got[1, ..., 0]).any()


@pytest.mark.parametrize("kind", ["ci8-f32", "ci8-f16x2", "cf32"])
@pytest.mark.parametrize("A,F,T,B,inc,polarize", [(3, 2, 1, 2, False, False), (5, 2, 65, 9, True, True),
                                                  (20, 3, 255, 8, True, False), (7, 300, 1021, 17, False, True),
                                                  (6, 3, 1023, 6, True, True), (18, 2, 2046, 12, True, False)])
def test_sample_counts_no_multiple_of_four(kind, A, F, T, B, inc, polarize):
    """Lanes of one sample, and lanes of four with a bound each; normwise, the
    FP32 bar of the forward bound above."""
    rng = np.random.default_rng(T)
    x8 = rng.integers(-128, 128, size=(A, F, T, 2, 2), dtype=np.int8)
    w = (rng.normal(size=(B, A, F, 1, 2)) + 1j * rng.normal(size=(B, A, F, 1, 2))).astype(np.complex64)
    ref = O.beamformer_ata(x8, w, inc, False)
    ref = O.polarizer(ref) if polarize else ref
    x = torch.from_numpy(x8).cuda() if kind != "cf32" else torch.from_numpy(O.ci8_to_complex(x8).astype(np.complex64)).cuda()
    y = ops.beamform_chain(x, torch.from_numpy(w).cuda(), inc, False, 1, polarize,
                           "f16x2" if kind == "ci8-f16x2" else "f32").cpu().numpy()
    assert O.norm_rel_err(y[:B], ref[:B]) <= 2 * (2 * A + 4) * 2.0 ** -24
    if inc:
        assert O.norm_rel_err(y[B], ref[B]) <= 2 * (2 * A + 4) * 2.0 ** -24


@pytest.mark.parametrize("kind", ["ci8-f32", "ci8-f16x2", "cf32"])
@pytest.mark.parametrize("rate,polarize,B,inc", [(4, True, 5, False), (4, True, 16, False), (2, False, 9, True)])
@pytest.mark.parametrize("T", [4, 8, 12, 260, 264, 268, 272])
def test_integrated_rows_at_every_alignment(kind, rate, polarize, B, inc, T):
    """Rows of T / rate samples on and off 64-byte sectors take different
    stores; normwise, the same bar."""
    rng = np.random.default_rng(T)
    A, F = 6, 3
    x8 = rng.integers(-128, 128, size=(A, F, T, 2, 2), dtype=np.int8)
    w = (rng.normal(size=(B, A, F, 1, 2)) + 1j * rng.normal(size=(B, A, F, 1, 2))).astype(np.complex64)
    ref = O.channelizer(O.beamformer_ata(x8, w, inc, False), rate)
    ref = O.polarizer(ref) if polarize else ref
    x = torch.from_numpy(x8).cuda() if kind != "cf32" else torch.from_numpy(O.ci8_to_complex(x8).astype(np.complex64)).cuda()
    got = ops.beamform_chain(x, torch.from_numpy(w).cuda(), inc, False, rate, polarize,
                             "f16x2" if kind == "ci8-f16x2" else "f32").cpu().numpy()
    assert got.shape == ref.shape and O.norm_rel_err(got, ref) <= 1e-6


@pytest.mark.parametrize("kind", ["f32", "f16x2", "adjoint"])
@pytest.mark.parametrize("A,B", [(1, 1), (16, 2), (42, 4), (64, 3), (17, 9), (128, 17)])
@pytest.mark.parametrize("T", [4, 8, 64, 260])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -100])
def test_gradients_keep_the_third_part(kind, A, B, T, scale):
    """Normwise per beam.  Without their third part the operands are cut at 16
    bits: each is off by up to 2^-16 of itself, 7e-6 in the norm.  FP32
    accumulation (and the 22 bits of split-FP16 phasors) leave 16 units of
    2^-24."""
    rng = np.random.default_rng(A + 10 * T)
    x8 = rng.integers(-128, 128, size=(A, 2, T, 2, 2), dtype=np.int8)
    x = x8[..., 0].astype(np.float64) + 1j * x8[..., 1]
    xd = torch.from_numpy(x8).cuda()
    if kind == "adjoint":
        gy = (scale * (rng.normal(size=(B, 2, T, 2)) + 1j * rng.normal(size=(B, 2, T, 2)))).astype(np.complex64)
        got = ops.beamformer_adjoint(xd, torch.from_numpy(gy).cuda())
        ref = np.einsum("bftp,aftp->bafp", gy.astype(np.complex128), x.conj())
    else:
        w = (scale * (rng.normal(size=(B, A, 2, 1, 2)) + 1j * rng.normal(size=(B, A, 2, 1, 2)))).astype(np.complex64)
        lam = [float(np.float32(v)) for v in rng.uniform(0.5, 1.0, size=B)]
        _, got = ops.stokes_i_loss_and_grad(xd, torch.from_numpy(w).cuda(), lam, precision=kind)
        y = np.einsum("bafp,aftp->bftp", w[:, :, :, 0].astype(np.complex128), x)
        ref = np.einsum("bftp,aftp->bafp", -np.array(lam)[:, None, None, None] * y, x.conj())
    got = got.cpu().numpy()[:, :, :, 0].astype(np.complex128)
    for b in range(B):
        assert np.linalg.norm(got[b] - ref[b]) <= 16 * 2.0 ** -24 * np.linalg.norm(ref[b]), b


@pytest.mark.parametrize("precision", ["f32", "f16x2"])
@pytest.mark.parametrize("A,F,T,B", [(6, 37, 4100, 16), (5, 41, 4108, 13), (3, 19, 8204, 33), (4, 50, 2052, 24)])
def test_mode_b_rows_off_sectors_past_the_caches(A, F, T, B, precision):
    """Outputs past 32 MiB with rows off 64-byte sectors: workgroups in XCD order,
    their number a multiple of 8 and not."""
    rng = np.random.default_rng(F)
    x8 = rng.integers(-128, 128, size=(A, F, T, 2, 2), dtype=np.int8)
    w = (rng.normal(size=(B, A, F, 1, 2)) + 1j * rng.normal(size=(B, A, F, 1, 2))).astype(np.complex64)
    assert T % 16 and B * F * T * 16 > 2 ** 25
    out = torch.full((B, F * 4, T // 4, 2), complex("nan"), dtype=torch.complex64, device="cuda")
    ops.beamform_chain(torch.from_numpy(x8).cuda(), torch.from_numpy(w).cuda(), False, False, 4, True, precision, out=out)
    ref = O.polarizer(O.channelizer(O.beamformer_ata(x8, w, False, False), 4))
    for b in range(B):
        assert O.norm_rel_err(out[b].cpu().numpy(), ref[b]) <= 1e-6
