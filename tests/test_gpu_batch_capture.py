"""A batch of small templates set while the plan's stream is being captured: nothing is allocated there, so the batch
runs per template, and the graph's replays give the maps of the batch set outside a capture."""
import numpy as np
import pytest

from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,size,window,origin", [((1024, 512), (60, 50), (80, 90), (-40, -45)),  # a raised frame
                                                  ((1024, 1024), (300, 300), (200, 200), (-100, -100)),  # a frame of 512-point columns
                                                  ((512, 512), (300, 300), (200, 200), (-100, 0))])  # the plan's own 512-point columns
def test_batch_set_under_capture(n, size, window, origin):
    H.log(f"batch set under capture {n} {size} -> {window}")
    count, rng = 4, np.random.default_rng(n[1] + size[0])
    img = H.to_dev(rng.standard_normal(2 * (n[0] // 2 + 1) * n[1]).astype(np.float32))
    bufs = [H.to_dev(H.padded_real(rng.standard_normal(size[::-1]).astype(np.float32), size[0]).reshape(-1)) for _ in range(count)]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        ft = H.make_plan((*size, 1), (*n, 1), (*n, 1), (*window, 1), origin=(*origin, 0))
        outs = [H.dev_poison(ft.ReturnInvOutputMemorySize()) for _ in range(count)]
        ft.FwdImageInvFFT(bufs[0], img, outs[0])  # the plan's workspace
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ft.SetBatch(bufs, [size] * count, outs)
            assert "chunk=0" in ft.Describe("batch").splitlines()[0]
            ft.FwdImageInvFFTBatch(img)
        got = []
        for _ in range(3):
            for o in outs:
                o.fill_(float("nan"))
            graph.replay()
            stream.synchronize()
            got.append([H.real_window(H.to_host(o), *window) for o in outs])
        ft.SetBatch(bufs, [size] * count, outs)
        assert "chunk=0" not in ft.Describe("batch").splitlines()[0]
        ft.FwdImageInvFFTBatch(img)
        want = [H.real_window(H.to_host(o), *window) for o in outs]
    for maps in got:
        for a, b in zip(maps, want):
            assert np.linalg.norm(a - b) < 2e-6 * np.linalg.norm(b)
