"""Line passes of 64 to 512 points (3-D transforms, and the 256- and 512-point passes of 2-D ones) against
the FP64 oracle: line counts that leave a workgroup partly filled, two-index maps whose groups do, odd row
counts of the paired C2R rows, the shortest and longest lengths and windows, origins that wrap, both storage
types, and the fused z-pass."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

TOL = 2e-6  # FP32 against FP64
TOL_F16 = 2.0 ** -11 + TOL  # one rounding of every stored value to FP16 on top
NP = {"f32": np.float32, "f16": np.float16}
IMG = {"f32": "c64", "f16": "c32h"}
TOLS = {"f32": TOL, "f16": TOL_F16}


def _vol(shape_zyx, seed, dtype="f32"):
    return np.random.default_rng(seed).standard_normal(shape_zyx).astype(NP[dtype])


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("vin,n", [((64, 64, 64), (64, 64, 64)), ((33, 17, 5), (64, 128, 64)), ((1, 1, 1), (256, 64, 128)),
                                   ((100, 255, 3), (128, 256, 64)), ((65, 30, 47), (256, 512, 64)), ((511, 3, 7), (512, 64, 128)),
                                   ((64, 64, 16), (64, 64, 512)), ((128, 128, 128), (128, 128, 128))])
def test_fwd_3d_lines(vin, n, dtype):
    H.log(f"3d fwd lines {vin} -> {n} {dtype}")
    v = _vol(vin[::-1], sum(vin), dtype)
    scale = 1.0 if dtype == "f32" else 1.0 / np.sqrt(np.prod(vin))
    ft = H.make_plan(vin, n, n, n, input_type=dtype, image_type=IMG[dtype], rank=3)
    out = H.dev_poison(ft.ReturnFwdOutputMemorySize(), dtype)
    ft.FwdFFT(H.to_dev(H.padded_real(v, vin[0], NP[dtype]).reshape(-1)), out, pre_op=H.F.Scale(scale))
    got = H.complex_from_f32(H.to_host(out).astype(np.float32), (n[2], n[0] // 2 + 1, n[1]))
    want = O.fwd_3d(H.padded_real(v.astype(np.float32), vin[0]), vin[0], *n, pre_scale=scale)
    assert O.rel_l2(got, want) < TOLS[dtype]


def _inv(n, nout, origin, dtype):
    rank = len(n)
    rng = np.random.default_rng(sum(n) + sum(nout))
    shape = (n[2], n[0] // 2 + 1, n[1]) if rank == 3 else (n[0] // 2 + 1, n[1])
    spec = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
    for kx in (0, n[0] // 2):  # the half spectrum of a real array
        p = spec[..., kx, :]
        spec[..., kx, :] = 0.5 * (p + np.conj(np.roll(np.flip(p, axis=tuple(range(p.ndim))), 1, axis=tuple(range(p.ndim)))))
    raw = H.complex_to_f32(spec).astype(NP[dtype])
    post = 1.0 if dtype == "f32" else 1.0 / np.sqrt(np.prod(n))
    three = lambda s, f: tuple(s) + (f,) * (3 - len(s))
    ft = H.make_plan(three(n, 1), three(n, 1), three(n, 1), three(nout, 1), origin=three(origin, 0), input_type=dtype,
                     image_type=IMG[dtype], rank=rank)
    out = H.dev_poison(ft.ReturnInvOutputMemorySize(), dtype)
    ft.InvFFT(H.to_dev(raw), out, post_op=H.F.Scale(post))
    got = H.real_window(H.to_host(out).astype(np.float32), *nout)
    spec = raw.astype(np.float32).view(np.complex64).reshape(shape)
    want = (O.inv_3d if rank == 3 else O.inv_2d)(spec, *n, *nout, *origin, post_scale=post)
    assert O.rel_l2(got, want) < TOLS[dtype]


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("n,nout,origin", [((64, 64, 64), (64, 64, 64), (0, 0, 0)), ((128, 64, 256), (33, 17, 90), (-16, 5, -45)),
                                           ((256, 512, 64), (1, 511, 3), (255, -1, 60)), ((512, 64, 128), (101, 63, 1), (-50, 1, 127)),
                                           ((64, 128, 512), (63, 100, 401), (2, -50, -200)),
                                           ((256, 128, 128), (256, 128, 128), (0, 0, 0))])
def test_inv_3d_lines(n, nout, origin, dtype):
    H.log(f"3d inv lines {n} -> {nout} at {origin} {dtype}")
    _inv(n, nout, origin, dtype)


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("n,nout,origin", [((256, 256), (255, 1), (-3, 250)), ((512, 256), (301, 203), (-100, 7)),
                                           ((256, 4096), (77, 4095), (0, -1)), ((512, 512), (512, 512), (0, 0))])
def test_inv_2d_lines(n, nout, origin, dtype):
    H.log(f"2d inv lines {n} -> {nout} at {origin} {dtype}")
    _inv(n, nout, origin, dtype)


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("fin,n", [((1, 1), (256, 256)), ((255, 203), (256, 512)), ((511, 4095), (512, 4096)), ((300, 17), (512, 32))])
def test_fwd_2d_lines(fin, n, dtype):
    H.log(f"2d fwd lines {fin} -> {n} {dtype}")
    img = _vol(fin[::-1], sum(fin), dtype)
    scale = 1.0 if dtype == "f32" else 1.0 / np.sqrt(np.prod(fin))
    ft = H.make_plan((*fin, 1), (*n, 1), (*n, 1), (*n, 1), input_type=dtype, image_type=IMG[dtype])
    out = H.dev_poison(ft.ReturnFwdOutputMemorySize(), dtype)
    ft.FwdFFT(H.to_dev(H.padded_real(img, fin[0], NP[dtype]).reshape(-1)), out, pre_op=H.F.Scale(scale))
    got = H.complex_from_f32(H.to_host(out).astype(np.float32), (n[0] // 2 + 1, n[1]))
    want = O.fwd_2d(H.padded_real(img.astype(np.float32), fin[0]), fin[0], *n, pre_scale=scale)
    assert O.rel_l2(got, want) < TOLS[dtype]


@pytest.mark.parametrize("image", ["c64", "c32h"])
@pytest.mark.parametrize("tin,n,nout,origin", [((13, 11, 9), (64, 64, 64), (31, 30, 29), (-15, -15, -14)),
                                               ((50, 20, 49), (128, 64, 256), (20, 33, 90), (-10, -16, -45)),
                                               ((8, 8, 100), (64, 64, 512), (16, 16, 413), (0, 0, -200)),
                                               ((64, 64, 128), (64, 64, 128), (64, 64, 128), (0, 0, 0)),
                                               ((1, 1, 1), (64, 128, 64), (1, 1, 1), (5, 6, 63))])
def test_xcorr_3d_lines(tin, n, nout, origin, image):
    H.log(f"3d xcorr lines {tin} in {n} -> {nout} at {origin} {image}")
    t = _vol(tin[::-1], seed=21)
    store = np.float32 if image == "c64" else np.float16
    spec = O.fwd_3d(H.padded_real(_vol(n[::-1], seed=22), n[0]), n[0], *n, pre_scale=1.0 / np.sqrt(np.prod(n)))
    raw = H.complex_to_f32(spec).astype(store)
    ft = H.make_plan(tin, n, n, nout, origin=origin, image_type=image, rank=3)
    out = H.dev_poison(ft.ReturnInvOutputMemorySize())
    ft.FwdImageInvFFT(H.to_dev(H.padded_real(t, tin[0]).reshape(-1)), H.to_dev(raw), out)
    got = H.real_window(H.to_host(out), *nout)
    spec = raw.astype(np.float32).view(np.complex64).reshape(n[2], n[0] // 2 + 1, n[1]).astype(np.complex128)
    want = O.inv_3d(spec * np.conj(O.fwd_3d(H.padded_real(t, tin[0]), tin[0], *n)), *n, *nout, *origin)
    assert O.rel_l2(got, want) < TOL
