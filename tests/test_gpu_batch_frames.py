"""Batches of small templates on the shortest frame the batched kernels take (512 x 256 points), against the
FP64 oracle of the whole pipeline: frames as long as the plan along one or both axes, windows off the 64-lane
grid, at wrapping origins and as long as the plan along an axis (where a plan has no origin), 256- and
512-point columns of one sub-transform, uneven sizes, FP16, and peaks."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

TOL = 2e-6
TOL_F16 = 2e-3  # FP16 storage of templates, spectrum and maps
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("sizes,n,nout,origin,frame", [
    ([(34, 30), (11, 34), (20, 7), (1, 1), (34, 34)], (1024, 512), (113, 43), (-56, -21), "512x256"),
    ([(68, 68)] * 4, (512, 256), (81, 137), (500, -68), "512x256"),
    ([(90, 60), (40, 90), (90, 90), (3, 3)], (512, 512), (301, 333), (-150, 77), "512x512"),
    ([(50, 50), (20, 50), (50, 20), (9, 8), (50, 1), (2, 50)], (512, 256), (512, 100), (-3, -50), "512x256"),
    ([(50, 50), (20, 50), (50, 20), (9, 8)], (1024, 256), (100, 256), (-3, -50), "full"),
    ([(100, 101), (64, 64), (100, 1), (30, 100)], (2048, 512), (400, 101), (-201, -50), "512x256"),
    ([(300, 290), (64, 64), (100, 1), (30, 100)], (1024, 1024), (150, 201), (-75, -100), "512x512")])
def test_small_template_batch(sizes, n, nout, origin, frame, dtype):
    H.log(f"small template batch {sizes} in {n} -> {nout} at {origin} {dtype}")
    rng = np.random.default_rng(n[0] + nout[1] + len(sizes))
    np_t = {"f32": np.float32, "f16": np.float16}[dtype]
    big = (max(s[0] for s in sizes), max(s[1] for s in sizes))
    w = n[0] // 2 + 1
    spec = O.fwd_2d(H.padded_real(rng.standard_normal(n[::-1]).astype(np.float32), n[0]), n[0], *n, pre_scale=1.0 / np.sqrt(n[0] * n[1]))
    raw = H.complex_to_f32(spec).astype(np_t)
    ft = H.make_plan((*big, 1), (*n, 1), (*n, 1), (*nout, 1), origin=(*origin, 0), input_type=dtype,
                     image_type="c64" if dtype == "f32" else "c32h")
    post = 1.0 / (np.sqrt(n[0] * n[1]) * big[0] * big[1])
    tmpl = [rng.standard_normal(s[::-1]).astype(np_t) for s in sizes]
    bufs = [H.to_dev(H.padded_real(t, t.shape[1], np_t).reshape(-1)) for t in tmpl]
    outs = [H.dev_poison(ft.ReturnInvOutputMemorySize(), dtype) for _ in sizes]
    peaks = torch.zeros(2 * len(sizes), dtype=torch.int32, device="cuda:0")
    vals = torch.zeros(len(sizes), dtype=torch.float32, device="cuda:0")
    ft.SetBatch(bufs, sizes, outs, peaks, vals)
    assert f"frame={frame}" in ft.Describe("batch").splitlines()[0]
    img = H.to_dev(raw)
    for _ in range(2):  # the call, then its graph again
        ft.FwdImageInvFFTBatch(img, post_op=H.F.Scale(post))
    lag = [o if m < v else 0 for o, m, v in zip(origin, nout, n)]  # a whole axis starts at lag 0, as in a single correlation
    spec32 = raw.astype(np.float32).view(np.complex64).reshape(w, n[1])
    for i, t in enumerate(tmpl):
        got = H.real_window(H.to_host(outs[i]).astype(np.float32), *nout)
        want = O.xcorr_2d(H.padded_real(t.astype(np.float32), t.shape[1]), t.shape[1], spec32, *n, *nout, *lag, post_scale=post)
        assert O.rel_l2(got, want) < (TOL if dtype == "f32" else TOL_F16), i
        gx, gy, gv = O.argmax_2d(got)
        px, py = (int(v) for v in H.to_host(peaks)[2 * i: 2 * i + 2])
        assert (px, py) == (gx, gy) and abs(float(H.to_host(vals)[i]) - gv) <= 1e-6 * abs(gv)


def test_small_frame_answers_as_the_plan():
    """A frame that only these small templates get leaves what the plan's own stages answer: no statistics or
    stage timing where those have no batched kernels, and FP32 whatever the precision asked for."""
    n, nout, size, count = (2048, 1024), (500, 500), (300, 300), 4
    ft = H.make_plan((*size, 1), (*n, 1), (*n, 1), (*nout, 1), origin=(-250, -250, 0))
    rng = np.random.default_rng(5)
    bufs = [H.to_dev(H.padded_real(rng.standard_normal(size[::-1]).astype(np.float32), size[0]).reshape(-1)) for _ in range(count)]
    outs = [H.dev_poison(ft.ReturnInvOutputMemorySize()) for _ in range(count)]
    ft.SetPrecision("split_bf16")
    ft.SetBatch(bufs, [size] * count, outs)
    line = ft.Describe("batch").splitlines()[0]
    assert "frame=1024x1024" in line and "precision=fp32" in line
    maps = [torch.zeros(nout[0] * nout[1], dtype=t, device="cuda:0") for t in (torch.float32, torch.int32, torch.float32, torch.float32)]
    with pytest.raises(H.F.FastFFTError, match="UNSUPPORTED"):
        ft.SetBatchStats(*maps)
