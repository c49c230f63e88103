"""What a user of this package has it do, as cases that can be timed and checked.

Every case goes through the package's public functions (``fft``, ``ifft``, ``rfft``, ``irfft``, ``fft2``,
``fftn``, ``stft``, ``istft``, ``ComplexLinear``) on device-resident fp32 data, as a program that keeps
its tensors on the GPU calls them.  The sizes come from the package's benchmark, README and tests:

* batched 1-D transforms, from a few short rows (latency) to 16 rows of 2^20 points, powers of two and
  any other length, forward and inverse;
* real rows (rfft / irfft);
* short-time transforms of batches of 10 s signals at 16 kHz: analysis, analysis + synthesis, and the
  forward + backward pass of a loss on spectra;
* images (real 2-D) and 3-D volumes / stacks of images (complex, strided axes);
* the complex linear layer's training pass.
"""

from __future__ import annotations

import math

import torch

import trnfft_amd
from trnfft_amd import ComplexTensor
from trnfft_amd.nn import ComplexLinear


def listed():
    return [
        # a few short rows: a filter bank or a small spectrum inside a larger program, bound by the call itself
        {"name": "fft_32x1024", "kind": "c2c", "rows": 32, "n": 1024, "inverse": False},
        # the headline batch of the benchmark: rows of 1024, the ordinary bulk transform
        {"name": "fft_4096x1024", "kind": "c2c", "rows": 4096, "n": 1024, "inverse": False},
        # long rows (wide-band spectra, fast convolution): 2^20 points, inverse direction
        {"name": "ifft_16x1048576", "kind": "c2c", "rows": 16, "n": 1 << 20, "inverse": True},
        # a decimal length, as data that nobody padded has it
        {"name": "fft_1024x1000", "kind": "c2c", "rows": 1024, "n": 1000, "inverse": False},
        # a prime length just past a power of two
        {"name": "ifft_256x4099", "kind": "c2c", "rows": 256, "n": 4099, "inverse": True},
        # real rows forward and back: spectra of real signals and the signals of filtered spectra
        {"name": "rfft_irfft_4096x1024", "kind": "real", "rows": 4096, "n": 1024},
        # spectrograms of 64 signals of 10 s at 16 kHz, 32 ms frames, half overlap
        {"name": "stft_64x160000_512", "kind": "stft", "rows": 64, "samples": 160000, "n_fft": 512, "hop": 256},
        # speech enhancement: 25 ms frames every 10 ms (n_fft 400, hop 160), spectra masked and resynthesised
        {"name": "mask_64x160000_400", "kind": "mask", "rows": 64, "samples": 160000, "n_fft": 400, "hop": 160},
        # the gradient of a loss on spectra with respect to the signal (vocoder training), quarter overlap
        {"name": "stft_grad_32x64000_1024", "kind": "stft_grad", "rows": 32, "samples": 64000, "n_fft": 1024,
         "hop": 256},
        # a batch of large real images
        {"name": "fft2_32x2048x2048", "kind": "fft2", "rows": 32, "h": 2048, "w": 2048},
        # a stack of camera-sized complex images: neither axis a power of two
        {"name": "ifftn_16x480x640", "kind": "fftn", "shape": "16x480x640", "axes": 2, "inverse": True},
        # a hidden layer's training pass: forward, input gradient, weight and bias gradients
        {"name": "linear_8192x1024x1024", "kind": "linear", "m": 8192, "k": 1024, "n": 1024},
    ]


_SPEECH_NFFT = (200, 240, 320, 400, 441, 480, 512, 600, 640, 800, 1000, 1024, 2048, 256)


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["c2c_pow2", "c2c_any", "real", "stft", "mask", "stft_grad", "fft2", "fftn", "linear"])
    if kind == "c2c_pow2":
        n = 1 << rng.randint(6, 20)
        rows = _log_int(rng, 1, max(2, (1 << 24) // n))
        return {"kind": "c2c", "rows": rows, "n": n, "inverse": rng.random() < 0.5}
    if kind == "c2c_any":
        n = _log_int(rng, 12, 12000)
        if n & (n - 1) == 0:
            n += 1
        return {"kind": "c2c", "rows": _log_int(rng, 1, max(2, (1 << 22) // n)), "n": n, "inverse": rng.random() < 0.5}
    if kind == "real":
        n = 1 << rng.randint(6, 14)
        if rng.random() < 0.4:
            n = 2 * _log_int(rng, 50, 2000)
        return {"kind": "real", "rows": _log_int(rng, 1, (1 << 23) // n), "n": n}
    if kind in ("stft", "mask", "stft_grad"):
        n_fft = rng.choice(_SPEECH_NFFT)
        hop = rng.choice([n_fft // 4, n_fft // 2, (2 * n_fft) // 5])
        samples = _log_int(rng, 4 * n_fft, 200000)
        rows = _log_int(rng, 1, max(2, min(128, 6000000 // samples)))
        return {"kind": kind, "rows": rows, "samples": samples, "n_fft": n_fft, "hop": hop}
    if kind == "fft2":
        h, w = 1 << rng.randint(5, 11), 1 << rng.randint(5, 11)
        return {"kind": "fft2", "rows": _log_int(rng, 1, max(2, (1 << 24) // (h * w))), "h": h, "w": w}
    if kind == "fftn":
        axes = rng.choice([2, 3])
        top = 1024 if axes == 2 else 160
        dims = [_log_int(rng, 16, top) if rng.random() < 0.6 else 1 << rng.randint(4, int(math.log2(top)))
                for _ in range(axes)]
        rows = _log_int(rng, 1, max(2, (1 << 22) // math.prod(dims)))
        return {"kind": "fftn", "shape": "x".join(str(v) for v in [rows, *dims]), "axes": axes,
                "inverse": rng.random() < 0.5}
    m, k, n = (_log_int(rng, 33, 4096) for _ in range(3))
    return {"kind": "linear", "m": m, "k": min(k, 2048), "n": min(n, 2048)}


# --- inputs ----------------------------------------------------------------------------------------


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _gen(seed):
    return torch.Generator(device=_device()).manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=g.device)


def _signals(g, rows, samples):
    """Three sinusoids of random frequency per signal and N(0, 0.1) noise, 16 kHz."""
    t = torch.arange(samples, device=g.device, dtype=torch.float32) / 16000.0
    x = 0.1 * _normal(g, rows, samples)
    for _ in range(3):
        f = 100.0 + 6900.0 * torch.rand(rows, 1, generator=g, device=g.device)
        p = 2.0 * math.pi * torch.rand(rows, 1, generator=g, device=g.device)
        x += torch.sin(2.0 * math.pi * f * t + p)
    return x


def _shape(case):
    return [int(v) for v in case["shape"].split("x")]


def _frames(case):
    return 1 + (case["samples"] + 2 * (case["n_fft"] // 2) - case["n_fft"]) // case["hop"]


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind == "c2c":
        return {"re": _normal(g, case["rows"], case["n"]), "im": _normal(g, case["rows"], case["n"])}
    if kind == "real":
        bins = case["n"] // 2 + 1
        return {"x": _normal(g, case["rows"], case["n"]), "re": _normal(g, case["rows"], bins),
                "im": _normal(g, case["rows"], bins)}
    if kind in ("stft", "mask", "stft_grad"):
        d = {"x": _signals(g, case["rows"], case["samples"]),
             "window": torch.hann_window(case["n_fft"], device=g.device)}
        spec = (case["rows"], case["n_fft"] // 2 + 1, _frames(case))
        if case["rows"] == 1:  # one signal: a vector, as a program with one signal has it
            d["x"], spec = d["x"][0], spec[1:]
        if kind == "mask":
            d["mask"] = torch.rand(case["n_fft"] // 2 + 1, 1, generator=g, device=g.device) + 0.1
        if kind == "stft_grad":
            d["g_re"], d["g_im"] = _normal(g, *spec), _normal(g, *spec)
        return d
    if kind == "fft2":
        return {"x": torch.rand(case["rows"], case["h"], case["w"], generator=g, device=g.device)}
    if kind == "fftn":
        return {"re": _normal(g, *_shape(case)), "im": _normal(g, *_shape(case))}
    m, k, n = case["m"], case["k"], case["n"]
    bound = 1.0 / math.sqrt(k)

    def uniform(*shape):
        return bound * (2.0 * torch.rand(*shape, generator=g, device=g.device) - 1.0)

    return {"w_re": uniform(n, k), "w_im": uniform(n, k), "b_re": uniform(n), "b_im": uniform(n),
            "re": _normal(g, m, k), "im": _normal(g, m, k), "g_re": _normal(g, m, n), "g_im": _normal(g, m, n)}


def prepare(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    state = {"case": case}
    if kind in ("c2c", "fftn"):
        state["x"] = ComplexTensor(d["re"], d["im"])
    elif kind == "real":
        state["x"], state["spec"] = d["x"], ComplexTensor(d["re"], d["im"])
    elif kind == "linear":
        layer = ComplexLinear(case["k"], case["n"]).to(d["re"].device)
        with torch.no_grad():
            layer.W_re.weight.copy_(d["w_re"])
            layer.W_im.weight.copy_(d["w_im"])
            layer.bias_re.copy_(d["b_re"])
            layer.bias_im.copy_(d["b_im"])
        x = ComplexTensor(d["re"].requires_grad_(), d["im"].requires_grad_())
        state.update(layer=layer, x=x, grads=(d["g_re"], d["g_im"]),
                     leaves=(x.real, x.imag, layer.W_re.weight, layer.W_im.weight, layer.bias_re, layer.bias_im))
    else:
        state.update(d)
        if kind == "stft_grad":
            state["x"].requires_grad_()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "c2c":
        out = (trnfft_amd.ifft if case["inverse"] else trnfft_amd.fft)(state["x"])
        return out.real, out.imag
    if kind == "real":
        spec = trnfft_amd.rfft(state["x"])
        return spec.real, spec.imag, trnfft_amd.irfft(state["spec"])
    if kind == "fft2":
        out = trnfft_amd.fft2(state["x"])
        return out.real, out.imag
    if kind == "fftn":
        dims = tuple(range(-case["axes"], 0))
        out = (trnfft_amd.ifftn if case["inverse"] else trnfft_amd.fftn)(state["x"], dim=dims)
        return out.real, out.imag
    if kind == "linear":
        y = state["layer"](state["x"])
        grads = torch.autograd.grad((y.real, y.imag), state["leaves"], state["grads"])
        return (y.real.detach(), y.imag.detach(), *grads)
    n_fft, hop = case["n_fft"], case["hop"]
    spec = trnfft_amd.stft(state["x"], n_fft, hop, window=state["window"])
    if kind == "mask":
        masked = spec * state["mask"]
        return spec.real, spec.imag, trnfft_amd.istft(masked, n_fft, hop, window=state["window"])
    if kind == "stft_grad":
        (grad,) = torch.autograd.grad((spec.real, spec.imag), (state["x"],), (state["g_re"], state["g_im"]))
        return spec.real.detach(), spec.imag.detach(), grad
    return spec.real, spec.imag


# --- what a pass cannot do without -----------------------------------------------------------------


def _fft_flops(n):
    return 5.0 * n * math.log2(n)


def work(case):
    kind = case["kind"]
    if kind == "c2c":
        return {"bytes": 16.0 * case["rows"] * case["n"], "flops": case["rows"] * _fft_flops(case["n"])}
    if kind == "real":
        row = 4 * case["n"] + 8 * (case["n"] // 2 + 1)
        return {"bytes": 2.0 * case["rows"] * row, "flops": case["rows"] * _fft_flops(case["n"])}
    if kind == "fft2":
        size = case["rows"] * case["h"] * case["w"]
        return {"bytes": 12.0 * size, "flops": 2.5 * size * math.log2(case["h"] * case["w"])}
    if kind == "fftn":
        shape = _shape(case)
        size = math.prod(shape)
        return {"bytes": 16.0 * size, "flops": 5.0 * size * math.log2(math.prod(shape[1:]))}
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        # read x, W, bias, dy once; write y, dx, dW, db once; three complex products
        return {"bytes": 8.0 * (2 * m * k + 2 * n * k + 2 * m * n + 2 * n), "flops": 24.0 * m * n * k}
    samples, rows = case["samples"], case["rows"]
    spec = rows * (case["n_fft"] // 2 + 1) * _frames(case)
    flops = rows * _frames(case) * 0.5 * _fft_flops(case["n_fft"])
    if kind == "stft":
        return {"bytes": 4.0 * rows * samples + 8.0 * spec, "flops": flops}
    # mask: the spectra are a result, and the masked ones only pass through; grad: cotangents in, gradient out
    extra = 8.0 * spec if kind == "stft_grad" else 0.0
    return {"bytes": 8.0 * rows * samples + 8.0 * spec + extra, "flops": 2.0 * flops}


# --- how far two correct results may be apart ------------------------------------------------------


def _length_error(n):
    # powers of two: fp32 butterflies, measured 1.1e-7 to 2.9e-7 from the exact transform.  Other lengths:
    # the interface's results follow a chirp whose angle pi k^2 / n is rounded to fp32, measured 1.15e-7 n
    # from it (1.2e-4 at 1000, 4.7e-4 at 4099).  Four times either
    return 1.2e-6 if n & (n - 1) == 0 else 1.2e-6 + 4.6e-7 * n


def _frame_error(n):
    # windowed frames weigh the chirp's worst angles less: measured 5.5e-8 n (2.2e-5 at 400)
    return 1.2e-6 if n & (n - 1) == 0 else 1.2e-6 + 2.2e-7 * n


def tolerance(case):
    kind = case["kind"]
    if kind in ("c2c", "real"):
        return {"rel": _length_error(case["n"])}
    if kind == "fft2":
        return {"rel": 1.2e-6}
    if kind == "fftn":
        return {"rel": sum(_length_error(n) for n in _shape(case)[1:])}
    if kind == "linear":
        # sums of up to 8192 fp32 products: measured 2.3e-6 from 64 bits
        return {"rel": 1e-5}
    return {"rel": _frame_error(case["n_fft"])}


# --- 64-bit results --------------------------------------------------------------------------------


def _stft64(x, case, window):
    # any odd or even n_fft: reflect-padded by n_fft // 2, framed, windowed, transformed
    n, hop = case["n_fft"], case["hop"]
    padded = torch.nn.functional.pad(x.reshape(-1, x.shape[-1]), (n // 2, n // 2), mode="reflect")
    padded = padded.reshape(*x.shape[:-1], -1)
    return torch.fft.rfft(padded.unfold(-1, n, hop) * window, dim=-1).transpose(-2, -1)


def _istft64(spec, case, window):
    n, hop = case["n_fft"], case["hop"]
    frames = torch.fft.irfft(spec.transpose(-2, -1), n=n, dim=-1) * window
    count = frames.shape[-2]
    total = n + (count - 1) * hop
    pos = (torch.arange(count, device=spec.device)[:, None] * hop + torch.arange(n, device=spec.device)).reshape(-1)
    out = torch.zeros(*frames.shape[:-2], total, dtype=frames.dtype, device=spec.device)
    out.index_add_(-1, pos, frames.flatten(-2))
    env = torch.zeros(total, dtype=frames.dtype, device=spec.device)
    env.index_add_(0, pos, (window * window).repeat(count))
    return (out / env)[..., n // 2 : total - n // 2]


def exact(case, seed):
    d, kind = {k: v.double() for k, v in _inputs(case, seed).items()}, case["kind"]
    if kind == "c2c":
        z = torch.complex(d["re"], d["im"])
        z = torch.fft.ifft(z) if case["inverse"] else torch.fft.fft(z)
        return z.real, z.imag
    if kind == "real":
        z, spec = torch.fft.rfft(d["x"]), torch.complex(d["re"], d["im"])
        return z.real, z.imag, torch.fft.irfft(spec, n=case["n"])
    if kind == "fft2":
        z = torch.fft.fft2(d["x"])
        return z.real, z.imag
    if kind == "fftn":
        z = torch.complex(d["re"], d["im"])
        dims = tuple(range(-case["axes"], 0))
        z = torch.fft.ifftn(z, dim=dims) if case["inverse"] else torch.fft.fftn(z, dim=dims)
        return z.real, z.imag
    if kind == "linear":
        x_re, x_im, w_re, w_im, g_re, g_im = (d[k] for k in ("re", "im", "w_re", "w_im", "g_re", "g_im"))
        return (x_re @ w_re.T - x_im @ w_im.T + d["b_re"], x_re @ w_im.T + x_im @ w_re.T + d["b_im"],
                g_re @ w_re + g_im @ w_im, g_im @ w_re - g_re @ w_im,
                g_re.T @ x_re + g_im.T @ x_im, g_im.T @ x_re - g_re.T @ x_im, g_re.sum(0), g_im.sum(0))
    x, window = d["x"], d["window"]
    if kind == "stft_grad":
        x.requires_grad_()
        z = _stft64(x, case, window)
        (grad,) = torch.autograd.grad((z.real, z.imag), (x,), (d["g_re"], d["g_im"]))
        return z.real.detach().contiguous(), z.imag.detach().contiguous(), grad
    z = _stft64(x, case, window)
    if kind == "mask":
        return z.real.contiguous(), z.imag.contiguous(), _istft64(z * d["mask"], case, window)
    return z.real.contiguous(), z.imag.contiguous()
