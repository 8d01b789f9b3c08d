"""2-D passes of 256-point lines on either side of the counts at which they change kernels, and of 128-point lines at
counts that leave a workgroup partly filled, against the FP64 oracle, both storage types."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

NP = {"f32": np.float32, "f16": np.float16}
IMG = {"f32": "c64", "f16": "c32h"}
TOLS = {"f32": 2e-6, "f16": 2.0 ** -11 + 2e-6}  # one rounding of every stored value to FP16 on top


@pytest.mark.parametrize("dtype", ["f32", "f16"])
# rows of 256 points, padded and whole; columns of 256 points (1025 and 2049 lines); rows and columns of 128 points
@pytest.mark.parametrize("fin,n", [((255, 256), (256, 512)), ((256, 257), (256, 512)), ((100, 256), (2048, 256)), ((2048, 255), (2048, 256)),
                                   ((4096, 256), (4096, 256)), ((127, 33), (128, 64)), ((128, 1), (128, 128)), ((3, 127), (128, 128)),
                                   ((60, 128), (512, 128))])
def test_forward(fin, n, dtype):
    H.log(f"short lines forward {fin} -> {n} {dtype}")
    img = np.random.default_rng(sum(fin)).standard_normal(fin[::-1]).astype(NP[dtype])
    scale = 1.0 if dtype == "f32" else 1.0 / np.sqrt(np.prod(fin))
    ft = H.make_plan((*fin, 1), (*n, 1), (*n, 1), (*n, 1), input_type=dtype, image_type=IMG[dtype])
    inp, out = H.to_dev(H.padded_real(img, fin[0], NP[dtype]).reshape(-1)), H.dev_poison(ft.ReturnFwdOutputMemorySize(), dtype)
    ft.FwdFFT(inp, out, pre_op=H.F.Scale(scale))
    got = H.complex_from_f32(H.to_host(out).astype(np.float32), (n[0] // 2 + 1, n[1]))
    want = O.fwd_2d(H.padded_real(img.astype(np.float32), fin[0]), fin[0], *n, pre_scale=scale)
    assert O.rel_l2(got, want) < TOLS[dtype]


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("n,window,origin", [((256, 512), (255, 256), (-3, 250)), ((256, 512), (256, 257), (0, -1)), ((256, 256), (256, 256), (0, 0)),
                                             ((256, 256), (61, 59), (200, -30)), ((2048, 256), (2048, 256), (0, 0)), ((2048, 256), (77, 255), (-9, 3)),
                                             ((4096, 256), (99, 31), (5, 255)), ((128, 64), (127, 33), (-3, 60)), ((128, 128), (128, 128), (0, 0)),
                                             ((128, 128), (1, 1), (127, -1)), ((512, 128), (60, 127), (500, 1))])
def test_inverse(n, window, origin, dtype):
    H.log(f"short lines inverse {n} -> {window} at {origin} {dtype}")
    w = n[0] // 2 + 1
    spec = np.random.default_rng(sum(n) + window[0]).standard_normal((w, n[1], 2)).astype(NP[dtype])
    post = 1.0 if dtype == "f32" else 1.0 / np.sqrt(np.prod(n))
    ft = H.make_plan((*n, 1), (*n, 1), (*n, 1), (*window, 1), origin=(*origin, 0), input_type=dtype, image_type=IMG[dtype])
    inp, out = H.to_dev(spec.reshape(-1)), H.dev_poison(ft.ReturnInvOutputMemorySize(), dtype)
    ft.InvFFT(inp, out, post_op=H.F.Scale(post))
    got = H.real_window(H.to_host(out).astype(np.float32), *window)
    want = O.inv_2d(spec.astype(np.float32).view(np.complex64).reshape(w, n[1]), *n, *window, *origin, post_scale=post)
    assert O.rel_l2(got, want) < TOLS[dtype]
