"""Padded forward lines: the C2C y-pass of a 2-D FwdFFT whose columns hold L < N values, on one workgroup
per line (256 to 8192 points), against the FP64 oracle in both storage types of the spectrum."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

TOL = 2e-6  # FP32 against FP64
TOL_F16 = 2.0 ** -11 + TOL  # one rounding of every stored value to FP16 on top


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("length,n", [(1, 256), (255, 256), (47, 512), (511, 512), (512, 1024), (1023, 1024), (3, 2048),
                                      (1025, 2048), (2751, 4096), (8191, 8192), (4096, 8192)])
def test_padded_columns(length, n, dtype):
    H.log(f"padded columns {length} -> {n} {dtype}")
    x, nx = 15, 32
    np_t = {"f32": np.float32, "f16": np.float16}[dtype]
    scale = 1.0 if dtype == "f32" else 1.0 / np.sqrt(x * length)
    img = np.random.default_rng(length + n).standard_normal((length, x)).astype(np_t)
    ft = H.make_plan((x, length, 1), (nx, n, 1), (nx, n, 1), (nx, n, 1), input_type=dtype,
                     image_type="c64" if dtype == "f32" else "c32h")
    inp = H.to_dev(H.padded_real(img, x, np_t).reshape(-1))
    out = H.dev_poison(ft.ReturnFwdOutputMemorySize(), dtype)
    ft.FwdFFT(inp, out, pre_op=H.F.Scale(scale))
    got = H.complex_from_f32(H.to_host(out).astype(np.float32), (nx // 2 + 1, n))
    want = O.fwd_2d(H.padded_real(img.astype(np.float32), x), x, nx, n, pre_scale=scale)
    assert O.rel_l2(got, want) < (TOL if dtype == "f32" else TOL_F16)
