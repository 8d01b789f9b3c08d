"""Pairs of real rows in workgroups of one, two and four pairs, as the launch rule takes them by the number of rows,
with a last workgroup that is partly filled (fewer pairs than its group, and a last pair of one row): the R2C and C2R
x-passes of 2-D FwdFFT and InvFFT against the FP64 oracle, and the kernels that run, from the launch log."""
import os
import re
import subprocess
import sys

import numpy as np
import pytest

from oracle import oracle as O
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

TOL = 2e-6  # FP32 against FP64, as in the other pair-row tests
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NY = 2048

# rows of a forward, padded and whole (160 workgroups' worth of pairs keep a group): 161, 321 and 641 pairs
FORWARD = [(n, rows, length, group) for n in (1024, 2048, 4096, 8192) for rows, group in ((321, 1), (641, 2), (1281, 4))
           for length in (n - n // 5, n)]
# rows and window of an inverse, windows of over half a row and of less (rows of over 1024 points come as pairs from 160
# pairs on)
INVERSE = [(n, rows, n // 2 if half else n // 2 + 3, group) for n in (1024, 2048, 4096, 8192)
           for rows, half, group in ((321, False, 1), (641, False, 2), (1281, False, 4), (199, True, 1), (401, True, 1), (801, True, 2))
           if rows > 199 or n == 1024]


def _forward(n, rows, length):
    ft = H.make_plan((length, rows, 1), (n, NY, 1), (n, NY, 1), (n, NY, 1))
    img = np.random.default_rng(n + rows).standard_normal((rows, length)).astype(np.float32)
    out = H.dev_poison(ft.ReturnFwdOutputMemorySize())
    ft.FwdFFT(H.to_dev(H.padded_real(img, length).reshape(-1)), out)
    return img, H.complex_from_f32(H.to_host(out), (n // 2 + 1, NY))


def _inverse(n, rows, window):
    ft = H.make_plan((n, NY, 1), (n, NY, 1), (n, NY, 1), (window, rows, 1), origin=(n - 7, 5, 0))
    spec = np.random.default_rng(n + rows).standard_normal((n // 2 + 1, NY, 2)).astype(np.float32)
    out = H.dev_poison(ft.ReturnInvOutputMemorySize())
    ft.InvFFT(H.to_dev(spec.reshape(-1)), out)
    return spec, H.real_window(H.to_host(out), window, rows)


@pytest.mark.parametrize("n,rows,length,group", FORWARD)
def test_forward_groups(n, rows, length, group):
    H.log(f"pair groups forward {length} -> {n}, {rows} rows")
    img, got = _forward(n, rows, length)
    want = O.fwd_2d(H.padded_real(img, img.shape[1]), img.shape[1], n, NY)
    assert O.rel_l2(got, want) < TOL


@pytest.mark.parametrize("n,rows,window,group", INVERSE)
def test_inverse_groups(n, rows, window, group):
    H.log(f"pair groups inverse {n}, {rows} rows of {window}")
    spec, got = _inverse(n, rows, window)
    want = O.inv_2d(spec.view(np.complex64).reshape(n // 2 + 1, NY), n, NY, window, rows, n - 7, 5)
    assert O.rel_l2(got, want) < TOL


def test_groups_of_the_launch_rule():
    """The pairs per workgroup named above are those that run (8192-point rows: two above 512 pairs, else one)."""
    H.log("pair groups from the launch log")
    code = ("from tests import test_gpu_pair_groups as T\n"
            "for n, rows, length, _ in T.FORWARD: T._forward(n, rows, length)\n"
            "for n, rows, window, _ in T.INVERSE: T._inverse(n, rows, window)\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=110,
                       env=dict(os.environ, FASTFFT_LOG="1"))
    assert r.returncode == 0, r.stderr[-2000:]
    got = [(int(n), int(g)) for n, g in re.findall(r"launch k_(?:r2c|c2r)_pair_rows<(\d+), (\d+),", r.stderr)]
    assert got == [(n, group if n < 8192 else 2 if rows > 1024 else 1) for n, rows, _, group in FORWARD + INVERSE]
