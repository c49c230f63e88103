"""Smooth lengths (multiples of 4 without a prime factor above 7, 36 to 640): the direct two-pass
transform in every kernel that takes it, against float64.  Its error is that of the power-of-two
transforms, so the bound is theirs, 1e-6 log2 n; the general path (Bluestein) at the same lengths is the
oracle's, whose distance is bounded by the parity tolerance in the other test files."""

from __future__ import annotations

import pytest
import torch

import trnfft_amd
from conftest import rel_l2, tol_pow2
from trnfft_amd import ComplexTensor

pytestmark = pytest.mark.gpu


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


LENGTHS = [n for n in range(36, 641, 4) if _smooth(n) and n & (n - 1)]


def _randn(seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, generator=g, device="cuda")


def _z(re, im):
    return torch.complex(re.double().cpu(), im.double().cpu())


@pytest.mark.parametrize("n", LENGTHS)
def test_smooth_rows_and_strided_axis(n):
    # ragged row counts on both workgroup shapes (the wider one from 8192 // n * 256 rows at most), real
    # input, and a strided axis of ragged width
    for rows in ((8192 // n + 1) * 256 + 3, 1, 37):
        re, im = _randn(n, rows, n), _randn(n + 1, rows, n)
        z = _z(re, im)
        y, x = trnfft_amd.fft(ComplexTensor(re, im)), trnfft_amd.ifft(ComplexTensor(re, im))
        ref, refi = torch.fft.fft(z), torch.fft.ifft(z)
        assert rel_l2(y.real, y.imag, ref.real, ref.imag) <= tol_pow2(n)
        assert rel_l2(x.real, x.imag, refi.real, refi.imag) <= tol_pow2(n)
    y, x = trnfft_amd.fft(re), trnfft_amd.ifft(re)
    ref, refi = torch.fft.fft(_z(re, 0 * re)), torch.fft.ifft(_z(re, 0 * re))
    assert rel_l2(y.real, y.imag, ref.real, ref.imag) <= tol_pow2(n)
    assert rel_l2(x.real, x.imag, refi.real, refi.imag) <= tol_pow2(n)
    for width in (1, 21):
        re, im = _randn(n + 2, 3, n, width), _randn(n + 3, 3, n, width)
        z = _z(re, im)
        y, x = trnfft_amd.fftn(ComplexTensor(re, im), dim=(1,)), trnfft_amd.ifftn(ComplexTensor(re, im), dim=(1,))
        ref, refi = torch.fft.fft(z, dim=1), torch.fft.ifft(z, dim=1)
        assert rel_l2(y.real, y.imag, ref.real, ref.imag) <= tol_pow2(n)
        assert rel_l2(x.real, x.imag, refi.real, refi.imag) <= tol_pow2(n)


def test_smooth_in_place_and_unaligned_planes():
    from trnfft_amd import _lib
    from trnfft_amd.dispatch import ptr, stream_handle
    from trnfft_amd.plan import native_plan

    for inverse in (False, True):
        buf = _randn(5, 2, 50 * 300 + 1)
        re, im = buf[0, 1:], buf[1, :-1]  # one plane 4 bytes off a 16-byte boundary
        z = _z(re, im).reshape(50, 300)
        plan = native_plan(_lib.KIND_BLUESTEIN, 300, inverse, buf.device.index)
        rc = _lib.lib().tfa_execute(plan.handle, 50, ptr(re), ptr(im), ptr(re), ptr(im), None, stream_handle(buf.device))
        _lib.check(rc, "tfa_execute")
        ref = torch.fft.ifft(z) if inverse else torch.fft.fft(z)
        assert rel_l2(re.reshape(50, 300), im.reshape(50, 300), ref.real, ref.imag) <= tol_pow2(300)
        re, im = _randn(6, 2, 300, 40), _randn(7, 2, 300, 40)
        z = _z(re, im)
        rc = _lib.lib().tfa_execute_strided(plan.handle, 2, 40, ptr(re), ptr(im), ptr(re), ptr(im),
                                            stream_handle(buf.device))
        _lib.check(rc, "tfa_execute_strided")
        ref = torch.fft.ifft(z, dim=1) if inverse else torch.fft.fft(z, dim=1)
        assert rel_l2(re, im, ref.real, ref.imag) <= tol_pow2(300)


def _stft64(x, n, hop, win):
    pad = torch.nn.functional.pad(x, (n // 2, n // 2), mode="reflect")
    return torch.fft.rfft(pad.unfold(-1, n, hop) * win, dim=-1).transpose(-2, -1)


@pytest.mark.parametrize("n", LENGTHS)
def test_smooth_stft_inverse_and_gradient(n):
    # 70 frames of two signals: the forward kernel's quarter tiles (the full ones below), a whole and a partial tile of
    # the inverse and the gradient; the signal short enough that both edges reflect
    hop = (2 * n) // 5
    x = _randn(n, 2, 69 * hop + 3)
    win = torch.hann_window(n, device="cuda") + 0.05
    w64 = win.double().cpu()
    x64 = x.double().cpu().requires_grad_()
    ref = _stft64(x64, n, hop, w64)
    a = x.clone().requires_grad_()
    y = trnfft_amd.stft(a, n, hop, window=win)
    assert y.real.shape == ref.shape
    assert rel_l2(y.real, y.imag, ref.detach().real, ref.detach().imag) <= tol_pow2(n)
    g = _randn(n + 1, 2, *y.real.shape)
    (got,) = torch.autograd.grad((y.real, y.imag), (a,), (g[0], g[1]))
    (want,) = torch.autograd.grad((ref.real, ref.imag), (x64,), (g[0].double().cpu(), g[1].double().cpu()))
    assert rel_l2(got, torch.zeros_like(got), want, torch.zeros_like(want)) <= 2 * tol_pow2(n)
    # inverse: bins 0 and n/2 keep imaginary parts that must not reach the signal
    with torch.no_grad():
        spec = ComplexTensor(g[0], g[1])
        got = trnfft_amd.istft(spec, n, hop, window=win)
        frames = torch.fft.irfft(_z(g[0], g[1]).transpose(-2, -1), n=n, dim=-1) * w64
        total = n + (frames.shape[-2] - 1) * hop
        pos = (torch.arange(frames.shape[-2])[:, None] * hop + torch.arange(n)).reshape(-1)
        out = torch.zeros(2, total, dtype=torch.float64).index_add_(1, pos, frames.reshape(2, -1))
        env = torch.zeros(total, dtype=torch.float64).index_add_(0, pos, (w64 * w64).repeat(frames.shape[-2]))
        want = (out / env)[:, n // 2 : total - n // 2]
        assert rel_l2(got, torch.zeros_like(got), want, torch.zeros_like(want)) <= 2 * tol_pow2(n)


@pytest.mark.parametrize("n,hop", [(400, 160), (60, 15), (640, 200)])
def test_smooth_stft_layouts_and_options(n, hop):
    x = _randn(n, 3, 5001)
    win = torch.hann_window(n, device="cuda")
    full = torch.fft.fft(torch.nn.functional.pad(x.double().cpu(), (n // 2, n // 2), mode="reflect")
                         .unfold(-1, n, hop) * win.double().cpu(), dim=-1).transpose(-2, -1)
    two = trnfft_amd.stft(x, n, hop, window=win, onesided=False)
    assert rel_l2(two.real, two.imag, full.real, full.imag) <= tol_pow2(n)
    half = trnfft_amd.stft(x, n, hop, window=win)
    fm = trnfft_amd.stft(x, n, hop, window=win, frames_major=True)
    assert torch.equal(half.real, fm.real) and torch.equal(half.imag, fm.imag)
    norm = trnfft_amd.stft(x, n, hop, window=win, normalized=True, center=False)
    ref = torch.fft.rfft(x.double().cpu().unfold(-1, n, hop) * win.double().cpu(), dim=-1).transpose(-2, -1) / n**0.5
    assert rel_l2(norm.real, norm.imag, ref.real, ref.imag) <= tol_pow2(n)
    back = trnfft_amd.istft(half, n, hop, window=win, length=5200)
    back_fm = trnfft_amd.istft(fm, n, hop, window=win, length=5200)
    assert torch.equal(back, back_fm)
    covered = hop * (half.real.shape[-1] - 1)
    assert rel_l2(back[:, :covered], torch.zeros_like(x)[:, :covered], x[:, :covered],
                  torch.zeros_like(x)[:, :covered]) <= 4 * tol_pow2(n)


def test_smooth_stft_nan_stays_in_its_frames():
    n, hop = 400, 160
    x = _randn(1, 1, 16000).reshape(1, -1).repeat(2, 1)
    x[1, 8000] = float("nan")
    y = trnfft_amd.stft(x, n, hop)
    hit = torch.isnan(y.real[1]).any(0).nonzero().flatten().tolist()
    # window ends are zero at sample 0 of a frame, but 0 * NaN is NaN: every covering frame is hit, no other
    assert hit == [f for f in range(y.real.shape[-1]) if 0 <= 8000 + n // 2 - f * hop < n]
    assert not torch.isnan(y.real[0]).any()
    s = ComplexTensor(y.real.clone(), y.imag.clone())
    out = trnfft_amd.istft(s, n, hop)
    bad = torch.isnan(out[1]).nonzero().flatten()
    assert bad.min() >= hit[0] * hop - n // 2 and bad.max() < hit[-1] * hop + n - n // 2
    assert not torch.isnan(out[0]).any()


def _frames_per_tile(n):
    return 64 if n <= 128 else 32 if n <= 448 else 16


@pytest.mark.parametrize("n", LENGTHS)
def test_smooth_stft_full_tiles(n):
    # calls of 256 tiles or more take the full tile: one whole and one of five frames per signal, 260 in all; a hop whose
    # span the areas hold, and one whose frames are read one by one
    fr = _frames_per_tile(n)
    win = torch.hann_window(n, device="cuda") + 0.05
    for hop in ((2 * n) // 5 + 1, 2 * n + 3):
        x = _randn(n + hop, 130, (fr + 4) * hop + 3)
        ref = _stft64(x.double(), n, hop, win.double())
        assert ref.shape[-1] == fr + 5
        y = trnfft_amd.stft(x, n, hop, window=win)
        assert rel_l2(y.real, y.imag, ref.real, ref.imag) <= tol_pow2(n)
        if n not in (36, 60, 120, 140, 196, 384, 392, 400, 432, 448, 480, 640):
            continue
        fm = trnfft_amd.stft(x, n, hop, window=win, frames_major=True)
        assert torch.equal(fm.real, y.real) and torch.equal(fm.imag, y.imag)
        for frames_major in (False, True):
            two = trnfft_amd.stft(x, n, hop, window=win, onesided=False, frames_major=frames_major)
            h = n // 2 + 1
            assert torch.equal(two.real[:, :h], y.real) and torch.equal(two.imag[:, :h], y.imag)
            assert torch.equal(two.real[:, h:], y.real[:, 1 : h - 1].flip(1))
            assert torch.equal(two.imag[:, h:], -y.imag[:, 1 : h - 1].flip(1))


@pytest.mark.parametrize("frames_major", [False, True])
@pytest.mark.parametrize("n,hop", [(36, 4), (60, 7), (96, 3), (96, 11), (120, 15), (120, 23), (140, 17), (200, 25), (200, 39), (400, 50),
                                   (400, 99), (448, 56), (480, 60), (480, 96), (600, 120), (640, 130), (640, 150)])
def test_smooth_inverse_and_gradient_of_many_overlaps(n, hop, frames_major):
    # five to 32 frames over each sample (halos of 4 and more): the overlap-add's general form, over several tiles
    halo = (n - 1) // hop
    assert halo >= 4
    frames = 3 * _frames_per_tile(n) + 7
    win = torch.hann_window(n, device="cuda") + 0.05
    w64 = win.double()
    shape = (2, 2, frames, n // 2 + 1) if frames_major else (2, 2, n // 2 + 1, frames)
    g = _randn(n + hop, *shape)
    g = g.transpose(-2, -1) if frames_major else g
    g64 = torch.complex(g[0].double(), g[1].double())
    spec = ComplexTensor._wrap(g[0], g[1])
    got = trnfft_amd.istft(spec, n, hop, window=win)
    assert trnfft_amd.api._istft_fused(spec, n, hop, n, win, True, False, True, None) is not None
    y = torch.fft.irfft(g64.transpose(-2, -1), n=n, dim=-1) * w64
    total = n + (frames - 1) * hop
    pos = (torch.arange(frames, device="cuda")[:, None] * hop + torch.arange(n, device="cuda")).reshape(-1)
    out = torch.zeros(2, total, dtype=torch.float64, device="cuda").index_add_(1, pos, y.reshape(2, -1))
    env = torch.zeros(total, dtype=torch.float64, device="cuda").index_add_(0, pos, (w64 * w64).repeat(frames))
    want = (out / env)[:, n // 2 : total - n // 2]
    assert rel_l2(got, torch.zeros_like(got), want, torch.zeros_like(want)) <= 2 * tol_pow2(n)
    # the gradient (the composed adjoint where the kernel's tile has no room for the halo)
    x = _randn(n, 2, (frames - 1) * hop).requires_grad_()
    x64 = x.detach().double().requires_grad_()
    z = trnfft_amd.stft(x, n, hop, window=win, frames_major=frames_major)
    ref = _stft64(x64, n, hop, w64)
    assert z.real.shape == ref.shape == g[0].shape
    (got,) = torch.autograd.grad((z.real, z.imag), (x,), (g[0], g[1]))
    (want,) = torch.autograd.grad((ref.real, ref.imag), (x64,), (g64.real, g64.imag))
    assert rel_l2(got, torch.zeros_like(got), want, torch.zeros_like(want)) <= 2 * tol_pow2(n)


@pytest.mark.parametrize("n", LENGTHS)
def test_smooth_rows_of_tones(n):
    # the direct transform of tones, on and between bins, is the exact one too (the reference's fp32 chirp errs most there)
    f = torch.cat([torch.arange(0, n, max(1, n // 20)).double(), torch.rand(20, generator=torch.Generator().manual_seed(n)).double() * n])
    z = torch.exp(2j * torch.pi * f[:, None] * torch.arange(n) / n)
    x = ComplexTensor(z.real.float().cuda(), z.imag.float().cuda())
    ref = torch.fft.fft(_z(x.real, x.imag))
    y = trnfft_amd.fft(x)
    for i in range(len(f)):
        assert rel_l2(y.real[i], y.imag[i], ref.real[i], ref.imag[i]) <= tol_pow2(n)


@pytest.mark.parametrize("n", [96, 400, 600])
@pytest.mark.parametrize("hop", [2**31 + 7, 2**32 + 5, 2**40 + 1])
def test_smooth_single_frame_at_a_hop_past_int(n, hop):
    # one frame: the hop's value plays no part, in the inverse and in the gradient (cut to 32 bits it is negative, 5 and 1)
    win = torch.hann_window(n, device="cuda") + 0.05
    s = _randn(n, 2, 2, n // 2 + 1, 1)
    spec = ComplexTensor(s[0], s[1])
    got, want = (trnfft_amd.istft(spec, n, h, window=win, center=False) for h in (hop, n))
    zero = torch.zeros_like(got)
    assert got.shape == (2, n) and rel_l2(got, zero, want, zero) <= 2.0**-22  # (a quotient, or a product with the reciprocal)
    grads = []
    for h in (hop, n):
        x = _randn(n + 1, 2, n + 3).requires_grad_()
        y = trnfft_amd.stft(x, n, h, window=win, center=False)
        grads += torch.autograd.grad((y.real, y.imag), (x,), (s[0], s[1]))
    assert torch.equal(grads[0], grads[1])
