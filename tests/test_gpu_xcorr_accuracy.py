"""Accuracy of the one-template correlation columns: the lags of a small window, whose outputs are summed from the
sub-transforms one by one, are as accurate as the same lags out of a window that takes whole passes."""
import numpy as np
import pytest

from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# Both windows share the rows, the forward transform, the product and the sub-transforms' inverse, some 2 log2 N
# roundings of a value; the sum of Q <= 16 shares adds log2 Q = 4 products: an error of at most sqrt(1 + 4 / 26) =
# 1.08 times that of the whole pass.
RATIO = 1.1


@pytest.mark.parametrize("n", [(64, 2048), (64, 4096), (64, 8192)])
def test_small_window_is_as_accurate_as_a_large_one(n):
    H.log(f"xcorr accuracy {n}")
    tin, small, large, origin = (32, n[1] // 16), (64, n[1] // 5), (64, n[1] // 2 + 3), (0, -77)
    rng = np.random.default_rng(n[1])
    t = rng.standard_normal(tin[::-1]).astype(np.float32)
    spec = np.ascontiguousarray(np.fft.rfft2(rng.standard_normal(n[::-1])).T.astype(np.complex64))
    maps = np.fft.irfft2(spec.astype(np.complex128).T * np.conj(np.fft.rfft2(t.astype(np.float64), s=n[::-1])), s=n[::-1]) * (n[0] * n[1])
    want = np.roll(maps, (-origin[1], -origin[0]), (0, 1))[: small[1], : small[0]]
    errors = []
    for window in (small, large):
        ft = H.make_plan((*tin, 1), (*n, 1), (*n, 1), (*window, 1), origin=(*origin, 0))
        out = H.dev_poison(ft.ReturnInvOutputMemorySize())
        ft.FwdImageInvFFT(H.to_dev(H.padded_real(t, tin[0]).reshape(-1)), H.to_dev(spec.view(np.float32).reshape(-1)), out)
        got = H.real_window(H.to_host(out), *window)[: small[1], : small[0]]
        errors.append(np.linalg.norm(got - want) / np.linalg.norm(want))
    assert errors[1] < 2e-6 and errors[0] < RATIO * errors[1], errors
