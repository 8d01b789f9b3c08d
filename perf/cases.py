"""Timed cases: what a program that uses FourierTransformer has it do.

Each case is a dict of plain values.  `op` is the work of one pass:

  roundtrip   FwdFFT of a zero padded image, then InvFFT of the whole frame
  fwd         FwdFFT, with or without padding (2-D or 3-D)
  inv         InvFFT, whole or trimmed to a window (2-D or 3-D)
  search      one padded and trimmed cross-correlation; 2-D ones with the peak of the window
  batch       many templates correlated with one spectrum in one call, a map and a peak of each

Sizes are (x, y) or (x, y, z): `small` is the forward input (image or template), `n` the
power-of-two transform, `window` the kept part of the inverse and `origin` its first lag.
"""
from __future__ import annotations

import math
import random

import torch

import fastfft_amd as F

AXES = ("x", "y", "z")


def _case(name, op, n, small=None, window=None, origin=None, dtype="f32", counts=1, least=0, precision="fp32"):
    """Sizes as plain numbers: n_x, small_x, ..., and the number of templates (the sizes of an uneven batch run from
    `least` to `small`)."""
    c = {"op": op, "rank": len(n), "dtype": dtype, "templates": counts, "least": least, "precision": precision}
    if name:
        c["name"] = name
    small, window = small or n, window or n
    origin = origin or tuple(0 for _ in n)
    for a, ax in enumerate(AXES[: len(n)]):
        c[f"n_{ax}"], c[f"small_{ax}"], c[f"window_{ax}"], c[f"origin_{ax}"] = n[a], small[a], window[a], origin[a]
    return c


def _get(case, what):
    return tuple(case[f"{what}_{ax}"] for ax in AXES[: case["rank"]])


def _centred(window):
    return tuple(-(w // 2) for w in window)


def listed():
    return [
        # a small image padded to a frame and back: latency and launches
        _case("roundtrip_64_in_512", "roundtrip", (512, 512), (64, 64)),
        # a micrograph to its spectrum, the producer of every search
        _case("fwd_4096", "fwd", (4096, 4096)),
        # a filtered spectrum back to a micrograph
        _case("inv_4096", "inv", (4096, 4096)),
        # a camera frame of no round size, kept in FP16, padded to the next power of two
        _case("fwd_ragged_f16", "fwd", (4096, 4096), (3001, 2750), dtype="f16"),
        # a region cut out of a micrograph's spectrum, off the origin, sizes of no power of two
        _case("inv_crop_ragged", "inv", (4096, 4096), window=(1001, 900), origin=(1203, -317)),
        # one template against a micrograph, as the drop-in's FwdImageInvFFT is called
        _case("search_one", "search", (4096, 4096), (384, 384), (512, 512), (-256, -256)),
        # one volume against another, template and window of no power of two
        _case("search_3d", "search", (256, 256, 256), (51, 47, 49), (90, 90, 90), (-45, -45, -45)),
        # the batched search: 64 templates of one size
        _case("batch_64", "batch", (4096, 4096), (384, 384), (512, 512), (-256, -256), counts=64),
        # the batched search over templates of uneven sizes
        _case("batch_256_uneven", "batch", (4096, 4096), (384, 384), (512, 512), (-256, -256), counts=256, least=128),
        # FP16 storage of templates, spectrum and maps, the matrix-core correlation pass
        _case("batch_256_f16_split", "batch", (4096, 4096), (512, 512), (512, 512), (-256, -256), dtype="f16", counts=256,
              precision="split_bf16"),
        # a padded volume to its spectrum
        _case("fwd_3d_64_in_256", "fwd", (256, 256, 256), (64, 64, 64)),
        # a sub-volume cut out of a large spectrum
        _case("inv_3d_512_to_128", "inv", (512, 512, 512), window=(128, 128, 128), origin=(-64, -64, -64)),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    """One more case: the operation, then its sizes, spread over their logarithm, any parity, x and y apart."""
    op = rng.choice(["roundtrip", "fwd", "fwd", "inv", "inv", "search", "search", "batch", "fwd3", "inv3", "search3"])
    if op.endswith("3"):
        top = 512 if op == "inv3" else 256
        n = [rng.choice([v for v in (64, 128, 256, 512) if v <= top]) for _ in range(3)]
        if min(n) == 512:  # no larger than the listed 512-cubed inverse
            n[rng.randrange(3)] = 256
        n = tuple(n)
        small, window, origin = n, n, (0, 0, 0)
        if op == "search3":
            small = tuple(_log_int(rng, v // 8, v // 4) for v in n)
            window = tuple(_log_int(rng, v // 4, v // 2) for v in n)
            origin = _centred(window)
        elif op == "fwd3" and rng.random() < 0.8:
            small = tuple(_log_int(rng, v // 4, v - 1) for v in n)
        elif op == "inv3":
            window = tuple(_log_int(rng, v // 4, v - 1) for v in n)
            origin = tuple(rng.randrange(-v // 2, v // 2) for v in n)
        return _case(None, {"fwd3": "fwd", "inv3": "inv", "search3": "search"}[op], n, small, window, origin)
    if op == "batch":
        n = rng.choice([1024, 2048, 4096])
        n = (n, rng.choice([n, n // 2, n]))
        size = _log_int(rng, min(n) // 16, min(n) // 8)
        window = tuple(_log_int(rng, v // 16, v // 8) for v in n)
        count = _log_int(rng, 4, 64)
        return _case(None, op, n, (size, size), window, _centred(window), counts=count,
                     least=rng.choice([0, max(8, size // 3)]), dtype=rng.choice(["f32", "f32", "f16"]))
    n = rng.choice([256, 512, 1024, 2048, 4096])
    n = (n, rng.choice([n, n, max(256, n // 2)]))
    if op == "search":
        small = tuple(_log_int(rng, v // 16, v // 4) for v in n)
        window = tuple(_log_int(rng, v // 8, v // 2) for v in n)
        return _case(None, op, n, small, window, _centred(window))
    dtype = rng.choice(["f32", "f32", "f16"])
    if op == "roundtrip":
        return _case(None, op, n, tuple(_log_int(rng, v // 8, v - 1) for v in n))
    if op == "fwd":
        return _case(None, op, n, tuple(_log_int(rng, v // 8, v - 1) for v in n) if rng.random() < 0.8 else n, dtype=dtype)
    if rng.random() < 0.2:
        return _case(None, op, n, dtype=dtype)
    return _case(None, op, n, window=tuple(_log_int(rng, v // 8, v - 1) for v in n),
                 origin=tuple(rng.randrange(-v // 2, v // 2) for v in n), dtype=dtype)


# ------------------------------------------------------------------------------------------ inputs


def _sizes(case):
    """(x, y) of every template of a batch: three sizes in turn from `least` to `small`, or all of one size."""
    big = case["small_x"]
    if not case["least"]:
        return [(big, big)] * case["templates"]
    three = [case["least"], (case["least"] + big) // 2, big]
    return [(three[i % 3],) * 2 for i in range(case["templates"])]


def _spectrum(real, dtype, scale=1.0):
    """Half spectrum C[kz][kx][ky] (C[kx][ky] in 2-D) of a real array [z][y][x], computed in 64 bits, stored in `dtype`."""
    s = torch.fft.rfftn(real.double()) * scale
    s = s.transpose(-1, -2).contiguous()
    return torch.view_as_real(s).to(dtype).contiguous()


def _template(size_x, size_y, gen, dev):
    """N(0,1) values within a disc, as masked projections are."""
    t = torch.randn(size_y, size_x, generator=gen, device=dev)
    y = (torch.arange(size_y, device=dev) - (size_y - 1) / 2) / size_y
    x = (torch.arange(size_x, device=dev) - (size_x - 1) / 2) / size_x
    return t * ((x[None, :] ** 2 + y[:, None] ** 2) <= (160.0 / 384.0) ** 2)


def _inputs(case, seed):
    """The inputs of a case on the GPU, in the case's storage types: real arrays [z][y][x] and spectra as (re, im) pairs."""
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)
    lag = random.Random(seed)
    half = case["dtype"] == "f16"
    dt = torch.float16 if half else torch.float32
    n, small = _get(case, "n"), _get(case, "small")
    if case["op"] in ("roundtrip", "fwd"):
        return {"real": [torch.randn(*small[::-1], generator=gen, device=dev).to(dt)]}
    # FP16 spectra are kept near one, below the largest FP16 value
    scale = 1.0 / math.sqrt(math.prod(n)) if half else 1.0
    image = torch.randn(*n[::-1], generator=gen, device=dev)
    if case["op"] == "inv":
        return {"spectrum": _spectrum(image, dt, scale)}
    templates = []
    window, origin = _get(case, "window"), _get(case, "origin")
    sizes = _sizes(case) if case["op"] == "batch" else [small]
    for size in sizes:  # a copy of every template, half its amplitude, at a lag within the window
        if case["rank"] == 2:
            t = _template(*size, gen, dev).to(dt)
        else:
            t = torch.randn(*size[::-1], generator=gen, device=dev).to(dt)
        at = []
        for a in range(case["rank"]):
            d = origin[a] + lag.randrange(window[a] // 8, window[a] - window[a] // 8)
            at.append((torch.arange(size[a], device=dev) + d) % n[a])
        image[torch.meshgrid(*at[::-1], indexing="ij")] += 0.5 * t.float()
        templates.append(t)
    return {"real": templates, "spectrum": _spectrum(image, dt, scale)}


def _padded(real):
    """FFTW padding: rows of 2 (x / 2 + 1) elements."""
    out = torch.zeros(*real.shape[:-1], F.padded_pitch(real.shape[-1]), dtype=real.dtype, device=real.device)
    out[..., : real.shape[-1]] = real
    return out


def _scales(case):
    """Operator scales (pre of a forward, post of an inverse or a search) that keep FP16 results in range."""
    if case["dtype"] == "f32":
        return 1.0, 1.0
    root = math.sqrt(math.prod(_get(case, "n")))
    return 1.0 / root, 1.0 / (root * (math.prod(_get(case, "small")) if case["op"] == "batch" else 1.0))


# ------------------------------------------------------------------------------------------ one pass


def _three(size):
    return tuple(size) + (1,) * (3 - len(size))


def _plan(case, fwd_in, n, inv_out, origin):
    half = case["dtype"] == "f16"
    ft = F.FourierTransformer("f16" if half else "f32", "c32h" if half else "c64", case["rank"])
    ft.SetForwardFFTPlan(*_three(fwd_in), *_three(n))
    ft.SetInverseFFTPlan(*_three(n), *_three(inv_out))
    if any(origin):
        ft.SetOutputWindow(*(tuple(origin) + (0,) * (3 - len(origin))))
    return ft


def prepare(case, seed):
    dev = torch.device("cuda:0")
    dt = torch.float16 if case["dtype"] == "f16" else torch.float32
    op = case["op"]
    n, small, window, origin = (_get(case, k) for k in ("n", "small", "window", "origin"))
    data = _inputs(case, seed)
    pre, post = _scales(case)
    state = {"op": op, "pre": F.Scale(pre) if pre != 1.0 else F.Noop(), "post": F.Scale(post) if post != 1.0 else F.Noop()}
    state["plan"] = _plan(case, small, n, window, origin)
    state["in"] = [_padded(r) for r in data.get("real", [])]
    state["spectrum"] = data.get("spectrum")
    if op in ("roundtrip", "fwd"):
        planes = (n[2],) if case["rank"] == 3 else ()
        state["out_spectrum"] = torch.zeros(*planes, n[0] // 2 + 1, n[1], 2, dtype=dt, device=dev)
    if op != "fwd":
        rows = (case["templates"],) if op == "batch" else ()
        out = torch.zeros(*rows, *window[:0:-1], F.padded_pitch(window[0]), dtype=dt, device=dev)
        state["out"], state["window"] = out, out[..., : window[0]]
    if op == "search" and case["rank"] == 2 or op == "batch":
        state["peaks"] = torch.zeros(case["templates"], 2, dtype=torch.int32, device=dev)
        state["values"] = torch.zeros(case["templates"], dtype=torch.float32, device=dev)
    if op == "batch":
        state["plan"].SetPrecision(case["precision"])
        state["plan"].SetBatch(state["in"], _sizes(case), list(state["out"]), state["peaks"], state["values"])
    return state


def run(state):
    op, plan = state["op"], state["plan"]
    if op == "fwd":
        plan.FwdFFT(state["in"][0], state["out_spectrum"], pre_op=state["pre"])
        return state["out_spectrum"]
    if op == "roundtrip":
        plan.FwdFFT(state["in"][0], state["out_spectrum"], pre_op=state["pre"])
        plan.InvFFT(state["out_spectrum"], state["out"], post_op=state["post"])
        return state["out_spectrum"], state["window"]
    if op == "inv":
        plan.InvFFT(state["spectrum"], state["out"], post_op=state["post"])
        return state["window"]
    if op == "batch":
        plan.FwdImageInvFFTBatch(state["spectrum"], post_op=state["post"])
        return state["window"], state["peaks"], state["values"]
    if "peaks" in state:
        plan.FwdImageInvFFTArgMax(state["in"][0], state["spectrum"], state["out"], state["peaks"], state["values"],
                                  post_op=state["post"])
        return state["window"], state["peaks"], state["values"]
    plan.FwdImageInvFFT(state["in"][0], state["spectrum"], state["out"], post_op=state["post"])
    return state["window"]


# ------------------------------------------------------------------------------------------ what a pass needs


def _line(n):
    return 5.0 * n * math.log2(n)


def _forward_flops(small, n):
    """Padded real forward: the x lines that hold data, then whole lines of the half spectrum along each further axis."""
    lines = [math.prod(small[1:]) / 2] + [(n[0] // 2 + 1) * math.prod(n[1:a]) * math.prod(small[a + 1:]) for a in range(1, len(n))]
    return sum(m * _line(v) for m, v in zip(lines, n))


def work(case):
    n, small, window = (_get(case, k) for k in ("n", "small", "window"))
    el = 2 if case["dtype"] == "f16" else 4
    spectrum = 2 * el * (n[0] // 2 + 1) * math.prod(n[1:])
    out = el * math.prod(window)
    op = case["op"]
    if op == "fwd":
        return {"bytes": el * math.prod(small) + spectrum, "flops": _forward_flops(small, n)}
    if op == "inv":
        return {"bytes": spectrum + out, "flops": _forward_flops(window, n)}
    if op == "roundtrip":
        return {"bytes": el * math.prod(small) + 2 * spectrum + out, "flops": _forward_flops(small, n) + _forward_flops(window, n)}
    sizes = _sizes(case) if op == "batch" else [small]
    total = sum(math.prod(s) for s in sizes)
    # a correlation of s with a window w needs transforms of s + w - 1 points per axis, not of the whole frame
    flops = 0.0
    for s in sizes:
        frame = tuple(min(v, 1 << (a + b - 2).bit_length()) for v, a, b in zip(n, s, window))
        flops += _forward_flops(s, frame) + _forward_flops(window, frame) + 6.0 * (frame[0] // 2 + 1) * math.prod(frame[1:])
    return {"bytes": spectrum + el * total + len(sizes) * out, "flops": flops}


# ------------------------------------------------------------------------------------------ the same in 64 bits


def _crop(real, window, origin):
    """The window [..][y][x] of a periodic array, its first element at `origin`."""
    idx = [(torch.arange(w, device=real.device) + o) % s for w, o, s in zip(window[::-1], origin[::-1], real.shape)]
    return real[torch.meshgrid(*idx, indexing="ij")]


def exact(case, seed):
    data = _inputs(case, seed)
    n, window, origin = (_get(case, k) for k in ("n", "window", "origin"))
    pre, post = _scales(case)
    shape, op = n[::-1], case["op"]

    def inverse(half):  # unnormalised
        return torch.fft.irfftn(half, s=shape, norm="forward")

    if op in ("fwd", "roundtrip"):
        s = torch.fft.rfftn(data["real"][0].double() * pre, s=shape)
        out = torch.view_as_real(s.transpose(-1, -2).contiguous())
        return out if op == "fwd" else (out, inverse(s) * post)
    image = torch.view_as_complex(data["spectrum"].double().contiguous()).transpose(-1, -2).contiguous()
    if op == "inv":
        return _crop(inverse(image), window, origin) * post
    maps = [_crop(inverse(image * torch.fft.rfftn(t.double(), s=shape).conj()), window, origin) * post for t in data["real"]]
    if op == "search":
        return (maps[0], None, maps[0].amax().reshape(1)) if case["rank"] == 2 else maps[0]
    maps = torch.stack(maps)
    return maps, None, maps.amax(dim=(1, 2))
