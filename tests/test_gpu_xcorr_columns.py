"""One-template correlation columns of 512, 1024 and 8192 points against the FP64 oracle: lengths of one value, one
sub-transform, one more and the whole column, windows on either side of the quarter where the outputs' sum changes
form, with and without the shared DC and Nyquist columns, FP32 and FP16 images."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

TOL = 2e-6


@pytest.mark.parametrize("image", ["c64", "c32h"])
@pytest.mark.parametrize("pack", ["1", "0"])
@pytest.mark.parametrize("ny,length,window,origin", [(512, 256, 128, -3), (512, 257, 129, 500), (512, 1, 1, 511), (512, 512, 512, 0),
                                                     (1024, 256, 256, -100), (1024, 257, 257, 1023), (1024, 1, 2, 7), (1024, 1024, 1000, 13),
                                                     (8192, 1024, 2048, -1000), (8192, 1025, 2049, 8191), (8192, 1, 1, 1), (8192, 8192, 500, 4095)])
def test_columns(ny, length, window, origin, pack, image, monkeypatch):
    monkeypatch.setenv("FASTFFT_XCORR_PACK", pack)
    H.log(f"xcorr columns {ny} {length} -> {window} at {origin} pack={pack} {image}")
    tin, n, nout = (9, length), (16, ny), (12, window)
    rng = np.random.default_rng(ny + length)
    t = rng.standard_normal(tin[::-1]).astype(np.float32)
    raw = rng.standard_normal((n[0] // 2 + 1, ny, 2)).astype(np.float32 if image == "c64" else np.float16)
    ft = H.make_plan((*tin, 1), (*n, 1), (*n, 1), (*nout, 1), origin=(-5, origin, 0), image_type=image)
    out = H.dev_poison(ft.ReturnInvOutputMemorySize())
    ft.FwdImageInvFFT(H.to_dev(H.padded_real(t, tin[0]).reshape(-1)), H.to_dev(raw.reshape(-1)), out)
    spec = raw.astype(np.float32).view(np.complex64).reshape(n[0] // 2 + 1, ny)
    # (a whole axis starts at lag 0)
    want = O.xcorr_2d(H.padded_real(t, tin[0]), tin[0], spec, *n, *nout, -5, origin if window < ny else 0)
    assert O.rel_l2(H.real_window(H.to_host(out), *nout), want) < TOL
