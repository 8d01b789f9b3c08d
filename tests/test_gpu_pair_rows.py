"""Real rows of 1024 to 8192 points as pairs (the R2C and C2R x-passes of 2-D FwdFFT and InvFFT), against
the FP64 oracle: one, two and four pairs per workgroup, odd row counts (a last pair of one row), the
shortest and longest non-zero lengths and windows, origins that wrap, both storage types."""
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


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("length,n,rows,ny", [(1, 1024, 1, 2), (1023, 1024, 511, 512), (1024, 1024, 255, 256),
                                              (1025, 2048, 3, 4), (2047, 2048, 513, 1024), (2751, 4096, 255, 256),
                                              (4096, 4096, 2, 2), (4095, 4096, 519, 1024), (8192, 8192, 5, 8),
                                              (4097, 8192, 257, 512)])
def test_r2c_pair_rows(length, n, rows, ny, dtype):
    H.log(f"r2c pair rows {length} -> {n}, {rows} rows {dtype}")
    scale = 1.0 if dtype == "f32" else 1.0 / np.sqrt(length * rows)
    img = np.random.default_rng(length + rows).standard_normal((rows, length)).astype(NP[dtype])
    ft = H.make_plan((length, rows, 1), (n, ny, 1), (n, ny, 1), (n, ny, 1), input_type=dtype, image_type=IMG[dtype])
    inp = H.to_dev(H.padded_real(img, length, NP[dtype]).reshape(-1))
    out = H.dev_poison(ft.ReturnFwdOutputMemorySize(), dtype)
    ft.FwdFFT(inp, out, pre_op=H.F.Scale(scale))
    got = H.complex_from_f32(H.to_host(out).astype(np.float32), (n // 2 + 1, ny))
    want = O.fwd_2d(H.padded_real(img.astype(np.float32), length), length, n, ny, pre_scale=scale)
    assert O.rel_l2(got, want) < TOLS[dtype]


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("n,ny,window,origin", [(1024, 2, (1, 1), (-1, 0)), (1024, 512, (1023, 511), (700, 3)),
                                                (1024, 256, (1024, 256), (0, 0)), (2048, 4, (777, 3), (-2000, 1)),
                                                (2048, 1024, (2047, 513), (1, -9)), (4096, 256, (1001, 255), (1203, -317)),
                                                (4096, 2, (4096, 2), (0, 0)), (4096, 1024, (64, 519), (-32, 0)),
                                                (8192, 8, (8191, 5), (5, 0)), (8192, 512, (3000, 257), (-1500, -128))])
def test_c2r_pair_rows(n, ny, window, origin, dtype):
    H.log(f"c2r pair rows {n}x{ny} -> {window} at {origin} {dtype}")
    rng = np.random.default_rng(n + window[0])
    w = n // 2 + 1
    spec = rng.standard_normal((w, ny, 2)).astype(NP[dtype])  # not Hermitian at kx = 0 and n/2: the oracle drops the same parts
    post = 1.0 if dtype == "f32" else 1.0 / np.sqrt(n * ny)
    ft = H.make_plan((n, ny, 1), (n, ny, 1), (n, ny, 1), (*window, 1), origin=(*origin, 0), input_type=dtype, image_type=IMG[dtype])
    inp = H.to_dev(spec.reshape(-1))
    out = H.dev_poison(ft.ReturnInvOutputMemorySize(), dtype)
    ft.InvFFT(inp, out, post_op=H.F.Scale(post))
    got = H.real_window(H.to_host(out).astype(np.float32), *window)
    want = O.inv_2d(spec.astype(np.float32).view(np.complex64).reshape(w, ny), n, ny, *window, *origin, post_scale=post)
    assert O.rel_l2(got, want) < TOLS[dtype]


@pytest.mark.parametrize("group", [1, 2, 4])
@pytest.mark.parametrize("n", [1024, 2048, 4096, 8192])
def test_pair_rows_of_every_group(monkeypatch, n, group):
    """Every workgroup shape (whole values or their parts through LDS) at row counts and lengths that the
    launch rule gives to other shapes or kernels: seven rows are a last pair of one row, and a last
    workgroup of fewer pairs than its group."""
    H.log(f"pair rows {n} group {group}")
    monkeypatch.setenv("FASTFFT_PAIR_MIN", "1")
    monkeypatch.setenv("FASTFFT_PAIR_GROUP", str(group))
    rows = 256 * group + 7  # above every rule that halves a group
    length, ny, window, origin = n - n // 3, 2048, (n // 2 + 5, rows), (n - 9, 3)
    img = np.random.default_rng(n + group).standard_normal((rows, length)).astype(np.float32)
    ft = H.make_plan((length, rows, 1), (n, ny, 1), (n, ny, 1), (*window, 1), origin=(*origin, 0))
    inp = H.to_dev(H.padded_real(img, length).reshape(-1))
    spec = H.dev_poison(ft.ReturnFwdOutputMemorySize())
    ft.FwdFFT(inp, spec)
    got = H.complex_from_f32(H.to_host(spec), (n // 2 + 1, ny))
    want = O.fwd_2d(H.padded_real(img, length), length, n, ny)
    assert O.rel_l2(got, want) < TOL
    out = H.dev_poison(ft.ReturnInvOutputMemorySize())
    post = 1.0 / (n * ny)
    ft.InvFFT(spec, out, post_op=H.F.Scale(post))
    want = O.inv_2d(got, n, ny, *window, *origin, post_scale=post)
    assert O.rel_l2(H.real_window(H.to_host(out), *window), want) < TOL
