"""Which search a batch runs with, as it reports it."""
import numpy as np
import pytest

from vszipcu import device, synth

pytestmark = pytest.mark.gpu

PLANES = [(97, 50, 97, 8.0), (64, 64, 64, 5.0), (40, 131, 40, 12.0)]


def _run(torch, planes, **kw):
    noisy = [torch.from_numpy(synth.noisy(synth.clean_luma(w, h, i), sg, i + 9)).cuda() for i, (w, h, _, sg) in enumerate(planes)]
    b = device.Batch(planes, block_step=4, extractor_exp=3, **kw)
    outs = [torch.zeros_like(t) for t in noisy]
    work = torch.zeros(b.workspace_size, dtype=torch.uint8, device="cuda")
    b.run(noisy, outs, work)
    torch.cuda.synchronize()
    b.check()
    return b, [o.cpu().numpy() for o in outs]


@pytest.mark.parametrize("schedule,bm_range,metric,screened", [
    ("staged", 12, "ssd", True), ("persistent", 12, "ssd", False), ("staged", 7, "ssd", False), ("staged", 12, "sad", False)])
def test_batch_reports_its_search(torch_gpu, schedule, bm_range, metric, screened):
    print(f"batch search: {schedule} R={bm_range} {metric}", flush=True)
    b, _ = _run(torch_gpu, PLANES, bm_range=bm_range, metric=metric, schedule=schedule, autotune=False)
    assert b.schedule() == (schedule, "rows")     # the exhaustive matcher
    assert b.screened() is screened
