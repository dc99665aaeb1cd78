"""The exhaustive ssd matchers on searches that the screened one does not take, each named by the plan, against the FP32
oracle: single planes, the centre frame of a temporal pass, and the staged batch."""
import numpy as np
import pytest

from gpu_util import assert_matches_equal, gpu_pass, kp_and_op
from vszipcu import device, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,bs,rng,plan", [
    # shared columns: several 15 x 16-block tiles, partial tiles, clamped rows, windows larger than the plane
    (200, 150, 4, 8, "lds4"), (68, 70, 4, 8, "lds4"), (236, 101, 4, 7, "lds4"), (20, 60, 4, 8, "lds4"),
    (1920, 1080, 4, 12, "lds4"),
    # search rows split over 4, 2 and 1 lanes
    (200, 150, 8, 8, "lds_rows4"), (140, 260, 7, 8, "lds_rows4"), (333, 121, 5, 8, "lds_rows4"),
    (1101, 600, 3, 9, "lds_rows2"), (1001, 560, 2, 9, "lds_rows1")])
def test_single_planes(orc, torch_gpu, w, h, bs, rng, plan):
    torch = torch_gpu
    print(f"exhaustive ssd: {w}x{h} bs={bs} R={rng} ({plan})", flush=True)
    img = synth.noisy(synth.clean_luma(w, h, 3), 10.0, w + h)
    img[: h // 4] = 0.25                              # exact ties: order by position
    kp, op = kp_and_op(orc, w, h, bs=bs, rng=rng)
    assert device.match_plan(kp) == plan and not device.match_screened(kp)
    nbx, nby = device.num_blocks(kp)
    m = torch.zeros((nby, nbx, 8, 4), dtype=torch.int32, device="cuda")
    device.match(kp, torch.from_numpy(img[None]).cuda(), m)
    torch.cuda.synchronize()
    gm = m.cpu().numpy().reshape(-1, 8, 4)
    ids = np.arange(nbx * nby, dtype=np.int32)
    if len(ids) > 20000:                              # the borders and a sample
        by, bx = np.divmod(ids, nbx)
        edge = (by < 2) | (by >= nby - 2) | (bx < 2) | (bx >= nbx - 2)
        ids = np.flatnonzero(edge | (np.random.default_rng(bs).random(len(ids)) < 0.05)).astype(np.int32)
    om, oe = orc.match_blocks(op, img[None], ids)
    assert_matches_equal(gm[ids], om, oe)


@pytest.mark.parametrize("bs,rng,plan", [(8, 8, "lds_rows4+temporal"), (4, 8, "lds4+temporal")])
def test_centre_frame_before_the_temporal_stage(orc, torch_gpu, bs, rng, plan):
    print(f"exhaustive ssd, temporal: bs={bs} R={rng}", flush=True)
    _, seq = synth.moving_sequence(72, 64, 5, 8.0, seed=43)
    kp, op = kp_and_op(orc, 72, 64, bs=bs, rng=rng, radius=2, sigma=device.scaled_sigma([8.0] * 3, False))
    assert device.match_plan(kp) == plan and not device.match_screened(kp)
    src = np.stack(seq)[None, None]
    ores, om, oe = orc.bm3d(op, src)
    gres, gm = gpu_pass(torch_gpu, kp, src, 1)
    assert_matches_equal(gm, om, oe)
    assert np.array_equal(gres, ores)


@pytest.mark.parametrize("sizes,matcher", [([(97, 50), (64, 64), (40, 131)], "rows"), ([(96, 48), (64, 64), (40, 132)], "shared-column")])
def test_staged_batch(orc, torch_gpu, sizes, matcher):
    torch = torch_gpu
    print(f"exhaustive ssd, staged batch: {matcher}", flush=True)
    kw = dict(block_step=4, bm_range=7, extractor_exp=3)
    noisy = [synth.noisy(synth.clean_luma(w, h, i), 8.0, 70 + i) for i, (w, h) in enumerate(sizes)]
    b = device.Batch([(w, h, w, 8.0) for w, h in sizes], autotune=False, schedule="staged", two_pass=False, **kw)
    outs = [torch.zeros((h, w), device="cuda") for w, h in sizes]
    work = torch.zeros(b.workspace_size, dtype=torch.uint8, device="cuda")
    b.run([torch.from_numpy(t).cuda() for t in noisy], outs, work)
    torch.cuda.synchronize()
    assert b.schedule() == ("staged", matcher) and not b.screened()
    for (w, h), img, out in zip(sizes, noisy, outs):
        op = orc.make_params(w, h, sigma=tuple(device.scaled_sigma([8.0] * 3, False)), **kw)
        res, _, _ = orc.bm3d(op, img[None, None, None])
        assert np.array_equal(out.cpu().numpy(), orc.aggregate(res[:, 0], w)[0])
