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


def test_small_planes_screen_together(orc, torch_gpu):
    """The rule sees all planes' tiles, since they are one launch: few enough for the screened search from bm_range 9."""
    print("batch search: small planes R=9", flush=True)
    b, outs = _run(torch_gpu, PLANES, bm_range=9, schedule="staged", autotune=False, two_pass=False)
    assert b.screened()
    for i, ((w, h, _, sg), out) in enumerate(zip(PLANES, outs)):
        op = orc.make_params(w, h, sigma=tuple(device.scaled_sigma([sg] * 3, False)), block_step=4, bm_range=9, extractor_exp=3)
        res, _, _ = orc.bm3d(op, synth.noisy(synth.clean_luma(w, h, i), sg, i + 9)[None, None, None])
        assert np.array_equal(out, orc.aggregate(res[:, 0], w)[0])


@pytest.mark.parametrize("schedule", ["staged", "auto"])
@pytest.mark.parametrize("planes", [PLANES, PLANES[1:]])      # with and without the shared-column matcher among the pairs
def test_tuned_batches_give_the_same(torch_gpu, planes, schedule):
    print(f"batch search: tuned {schedule}, {len(planes)} planes", flush=True)
    _, want = _run(torch_gpu, planes, bm_range=12, schedule="staged", autotune=False)
    b, got = _run(torch_gpu, planes, bm_range=12, schedule=schedule, autotune=True)
    assert b.schedule()[0] == "staged" or not b.screened()
    for a, c in zip(want, got):
        assert np.array_equal(a, c)


def test_large_shared_column_planes_screen_only_if_timed(torch_gpu):
    """Above 2048 tiles the shared-column scan is preferred at bm_range 12; the autotuner may find the screen faster."""
    print("batch search: shared columns, 960x720", flush=True)
    planes = [(960, 720, 960, 8.0)]
    b, want = _run(torch_gpu, planes, bm_range=12, schedule="staged", autotune=False)
    assert b.schedule() == ("staged", "shared-column") and not b.screened()
    b, got = _run(torch_gpu, planes, bm_range=12, schedule="staged", autotune=True)
    assert np.array_equal(want[0], got[0])
