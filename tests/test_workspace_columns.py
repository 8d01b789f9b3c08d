"""Leading dimension of the column workspaces of 2-D FwdFFT and InvFFT: a multiple of 8 where the x-pass moves
segments of neighbouring rows, the plain row count where a row kernel gathers one row at a time (CPU)."""
import re

import pytest

import fastfft_amd as F


def _maps(small, n, window, op):
    ft = F.FourierTransformer("f32", "c64", 2)
    ft.SetForwardFFTPlan(*small, 1, *n, 1)
    ft.SetInverseFFTPlan(*n, 1, *window, 1)
    x, y = [line for line in ft.Describe(op).splitlines() if " ref=" in line][:: 1 if op == "fwd" else -1]
    out_of_x = re.search(r"om=\((\d+),\d+,(\d+)," if op == "fwd" else r"im=\((\d+),\d+,(\d+),", x).groups()
    of_y = re.search(r"im=\((\d+)," if op == "fwd" else r"om=\((\d+),", y).group(1)
    assert out_of_x[0] == "1" and out_of_x[1] == of_y
    return int(of_y)


@pytest.mark.parametrize("n,rows,ld", [(8192, 251, 251), (8192, 319, 320), (4096, 123, 123), (2048, 318, 318), (1024, 251, 256),
                                       (1024, 1, 8), (512, 59, 64), (256, 61, 64), (4096, 1024, 1024)])
def test_inverse_columns(n, rows, ld):
    assert _maps((n, 2048), (n, 2048), (n // 4 + 1, rows), "inv") == ld


@pytest.mark.parametrize("n,rows,ld", [(4096, 128, 128), (4096, 127, 127), (4096, 129, 136), (2048, 100, 100), (1024, 99, 104), (256, 100, 104)])
def test_forward_columns(n, rows, ld):
    assert _maps((n - 5, rows), (n, 2048), (n, 2048), "fwd") == ld
