"""What a batch answers besides its maps (statistics, stage timing), and which frame it takes: batches whose columns
are one short sub-transform (on a frame, or on the plan's own stages) answer as the plan's own stages do, where the
batched kernels take those with longer or more sub-transforms, and else as per-template launches do."""
import pytest

from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _batch(n, size, window, origin, count):
    H.log(f"batch answers {n} {size} -> {window} at {origin} x{count}")
    ft = H.make_plan((*size, 1), (*n, 1), (*n, 1), (*window, 1), origin=(*origin, 0))
    bufs = [H.dev_zeros(ft.ReturnInputMemorySize()) for _ in range(count)]
    outs = [H.dev_poison(ft.ReturnInvOutputMemorySize()) for _ in range(count)]
    ft.SetBatch(bufs, [size] * count, outs)
    return ft, dict(v.split("=") for v in ft.Describe("batch").splitlines()[0].split() if "=" in v)


@pytest.mark.parametrize("n,size,window,origin,count,frame,answers", [
    ((1024, 1024), (300, 300), (200, 200), (-100, -100), 4, "512x512", False),  # own stages: an origin off the lane grid
    ((2048, 2048), (300, 140), (200, 110), (-64, -64), 4, "512x256", False),
    ((512, 512), (300, 300), (200, 200), (-100, 0), 4, "full", False),  # own stages: 512-point columns at origin 0
    ((1024, 1024), (300, 300), (200, 200), (-100, 0), 4, "512x512", True),  # own stages: 1024 = 2 x 512
    ((1024, 1024), (384, 384), (500, 500), (-250, 0), 4, "full", True),
    ((2048, 2048), (300, 500), (200, 500), (-100, -250), 4, "512x1024", True)])  # long columns
def test_answers_of_short_columns(n, size, window, origin, count, frame, answers):
    ft, d = _batch(n, size, window, origin, count)
    assert d["frame"] == frame
    img = H.dev_zeros(2 * (n[0] // 2 + 1) * n[1])
    maps = [torch.zeros(window[0] * window[1], dtype=t, device="cuda:0") for t in (torch.float32, torch.int32, torch.float32, torch.float32)]
    for call in (lambda: ft.RunBatchStage(2, img), lambda: ft.SetBatchStats(*maps)):
        if answers:
            call()
        else:
            with pytest.raises(H.F.FastFFTError, match="UNSUPPORTED"):
                call()
    ft.FwdImageInvFFTBatch(img)
    torch.cuda.synchronize()


@pytest.mark.parametrize("size,window,count,frame", [((300, 300), (200, 200), 1, "full"), ((300, 300), (200, 200), 2, "512x512"),
                                                     ((300, 100), (200, 100), 1, "full"), ((300, 100), (200, 100), 2, "512x256")])
def test_one_template_runs_on_the_plans_stages(size, window, count, frame):
    assert _batch((2048, 2048), size, window, (-100, -50), count)[1]["frame"] == frame


@pytest.mark.parametrize("n,count,frame", [((2048, 2048), 4, "full"), ((2048, 2048), 5, "2048x2048"), ((4096, 2048), 4, "2048x2048"),
                                           ((4096, 2048), 3, "full")])
def test_four_templates_do_not_pay_for_a_whole_plan_frame(n, count, frame):
    """Templates of 1000^2 whose lags need 2048 x 2048 points: the frame is the plan's own size, or half of it."""
    assert _batch(n, (1000, 1000), (1000, 500), (-500, -250), count)[1]["frame"] == frame
