"""Inverse columns of one, two and four waves (unit-stride complex lines read from memory by every wave, and
eight waves through LDS), whole and windowed at odd, even and wrapping origins, against the FP64 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

TOL = 2e-6  # FP32 against FP64


@pytest.mark.parametrize("image_type", ["c64", "c32h"])  # half2 spectra keep the LDS form
@pytest.mark.parametrize("nx,ny,window,origin", [(16, 256, (16, 256), (0, 0)), (16, 256, (9, 101), (-4, 77)),
                                                 (8, 512, (8, 512), (0, 0)), (8, 512, (8, 511), (0, -3)),
                                                 (64, 1024, (64, 1024), (0, 0)), (64, 1024, (33, 1), (5, 1023)),
                                                 (64, 1024, (64, 700), (0, -350)), (32, 2048, (32, 2048), (0, 0)),
                                                 (32, 2048, (31, 1025), (1, -513)), (16, 4096, (16, 4096), (0, 0)),
                                                 (16, 4096, (16, 1001), (0, -99))])
def test_inverse_columns(monkeypatch, nx, ny, window, origin, image_type):
    H.log(f"inverse columns {nx}x{ny} -> {window} at {origin} {image_type}")
    monkeypatch.setenv("FASTFFT_NO_TILE_LINES", "1")  # the 256- and 512-point columns too
    w = nx // 2 + 1
    np_t = np.float32 if image_type == "c64" else np.float16
    spec = np.random.default_rng(ny + window[1]).standard_normal((w, ny, 2)).astype(np_t)
    post = 1.0 / np.sqrt(nx * ny)
    ft = H.make_plan((nx, ny, 1), (nx, ny, 1), (nx, ny, 1), (*window, 1), origin=(*origin, 0),
                     input_type="f32" if image_type == "c64" else "f16", image_type=image_type)
    out = H.dev_poison(ft.ReturnInvOutputMemorySize(), "f32" if image_type == "c64" else "f16")
    ft.InvFFT(H.to_dev(spec.reshape(-1)), out, post_op=H.F.Scale(post))
    got = H.real_window(H.to_host(out).astype(np.float32), *window)
    want = O.inv_2d(spec.astype(np.float32).view(np.complex64).reshape(w, ny), nx, ny, *window, *origin, post_scale=post)
    assert O.rel_l2(got, want) < (TOL if image_type == "c64" else 2.0 ** -11 + TOL)
