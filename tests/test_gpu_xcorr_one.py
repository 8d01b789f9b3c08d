"""The correlation column kernel of one template against the FP64 oracle: lengths and windows of one value,
beyond the 512-point sub-transforms and of the whole column, origins off the 64-lane grid that wrap, with and
without the shared DC and Nyquist columns, FP32 and FP16 images; and its templates' rows of at most 128 and of
more than 1024 points."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

TOL = 2e-6


@pytest.mark.parametrize("image", ["c64", "c32h"])
@pytest.mark.parametrize("pack", ["1", "0"])
@pytest.mark.parametrize("tin,n,nout,origin", [((30, 30), (256, 256), (60, 61), (-30, -31)), ((1, 1), (256, 256), (1, 1), (255, -1)),
                                               ((101, 512), (512, 512), (128, 512), (-64, 0)), ((20, 513), (32, 1024), (16, 600), (3, -301)),
                                               ((300, 1025), (1024, 2048), (700, 1100), (-350, 777)),
                                               ((40, 129), (64, 4096), (32, 2047), (-16, -1033)), ((17, 4096), (32, 4096), (32, 4096), (0, 0)),
                                               ((24, 1500), (32, 8192), (16, 3001), (-8, 8000)), ((128, 7), (2048, 256), (256, 9), (-128, -4)),
                                               ((1300, 5), (4096, 256), (100, 100), (-50, -50)), ((60, 4), (8192, 256), (9, 30), (1, 2))])
def test_xcorr_one_vs_oracle(tin, n, nout, origin, pack, image, monkeypatch):
    monkeypatch.setenv("FASTFFT_XCORR_PACK", pack)
    H.log(f"xcorr one {tin} in {n} -> {nout} at {origin} pack={pack} {image}")
    rng = np.random.default_rng(tin[0] * 3 + n[1])
    t = rng.standard_normal((tin[1], tin[0])).astype(np.float32)
    w = n[0] // 2 + 1
    raw = rng.standard_normal((w, n[1], 2)).astype(np.float32 if image == "c64" else np.float16)
    ft = H.make_plan((*tin, 1), (*n, 1), (*n, 1), (*nout, 1), origin=(*origin, 0), image_type=image)
    out = H.dev_poison(ft.ReturnInvOutputMemorySize())
    ft.FwdImageInvFFT(H.to_dev(H.padded_real(t, tin[0]).reshape(-1)), H.to_dev(raw.reshape(-1)), out)
    got = H.real_window(H.to_host(out), *nout)
    spec = raw.astype(np.float32).view(np.complex64).reshape(w, n[1])
    want = O.xcorr_2d(H.padded_real(t, tin[0]), tin[0], spec, n[0], n[1], *nout, *origin)
    assert O.rel_l2(got, want) < TOL
