"""The screened ssd search (half-precision products on the matrix cores, exact evaluation of what passes)
against the FP32 oracle: match lists and distances bit for bit. Sizes at the edges of its 4 x 4-block
tiles, 4-row groups and 16-column tiles, windows of one and of several column passes, and the
contents where its bounds or queues work hardest: flat and half-flat planes (ties), periodic ones, tiny and
huge ranges, values that are not finite."""
import numpy as np
import pytest

from gpu_util import assert_matches_equal, kp_and_op
from vszipcu import device, synth

pytestmark = pytest.mark.gpu


def _content(kind, w, h):
    rng = np.random.default_rng(w * 131 + h)
    noise = rng.normal(0, 0.02, (h, w)).astype(np.float32)
    clean = synth.clean_luma(w, h, 5)
    if kind == "video":
        return clean + noise
    if kind == "flat":
        return np.full((h, w), 0.25, np.float32)
    if kind == "bars":                       # a letterbox: exact ties beside noise
        img = clean + noise
        img[: h // 3] = 0.0
        return img
    if kind == "quiet":                      # flat areas at two levels, nearly free of noise
        img = np.where(np.arange(w)[None, :] < w // 2, 0.1, 0.9).astype(np.float32) + noise * 1e-4
        return img.astype(np.float32)
    if kind == "periodic":                   # exact repetitions: ties all over the window
        return np.tile(rng.random((4, 8), dtype=np.float32), (h // 4 + 1, w // 8 + 1))[:h, :w].copy()
    if kind == "tiny":                       # a range far below that of video
        return ((clean + noise) * np.float32(1e-18)).astype(np.float32)
    if kind == "huge":                       # beyond the range of halves
        return ((clean + noise) * np.float32(1e6)).astype(np.float32)
    img = clean + noise                      # "nan": some values are not finite
    img[h // 2, w // 2] = np.nan
    img[3, 5] = np.inf
    return img


def _check(orc, torch, img, w, h, stride, bs, rng):
    kp, op = kp_and_op(orc, w, h, bs=bs, rng=rng, stride=stride, sigma=device.scaled_sigma([10.0] * 3, False))
    padded = np.full((h, stride), np.nan, np.float32)       # padding must never be read
    padded[:, :w] = img
    _, om, oe = orc.bm3d(op, padded[None, None, None])
    nbx, nby = device.num_blocks(kp)
    m = torch.zeros((nby, nbx, 8, 4), dtype=torch.int32, device="cuda")
    device.match(kp, torch.from_numpy(padded[None]).cuda(), m)
    torch.cuda.synchronize()
    assert_matches_equal(m.cpu().numpy(), om, oe)


@pytest.mark.parametrize("w,h,pad,bs,rng", [
    (8, 8, 0, 8, 6), (9, 11, 3, 1, 9), (21, 40, 0, 4, 16), (64, 48, 0, 8, 9), (77, 61, 19, 3, 12),
    (100, 50, 1, 5, 8), (133, 70, 0, 8, 20), (57, 90, 0, 2, 24), (120, 96, 0, 6, 19), (96, 64, 0, 7, 23)])
def test_sizes(orc, torch_gpu, w, h, pad, bs, rng):
    print(f"screened search: {w}x{h}+{pad} bs={bs} R={rng}", flush=True)
    _check(orc, torch_gpu, _content("video", w, h), w, h, w + pad, bs, rng)


@pytest.mark.parametrize("bs,rng", [(4, 16), (8, 20)])      # one column pass, two column passes
@pytest.mark.parametrize("kind", ["flat", "bars", "quiet", "periodic", "tiny", "huge", "nan"])
def test_contents(orc, torch_gpu, kind, bs, rng):
    print(f"screened search: {kind} bs={bs} R={rng}", flush=True)
    w, h = 90, 75
    _check(orc, torch_gpu, _content(kind, w, h), w, h, w, bs, rng)


def test_batch_screens_like_single_planes(orc, torch_gpu):
    """Uneven planes in one staged plan (the batched kernel) against the oracle's chain per plane."""
    torch = torch_gpu
    sizes = [(97, 50), (64, 64), (40, 131)]
    print("screened search: batch", flush=True)
    kw = dict(block_step=4, bm_range=12, extractor_exp=3)
    noisy = [_content("bars" if i else "video", w, h) for i, (w, h) in enumerate(sizes)]
    b = device.Batch([(w, h, w, 8.0) for w, h in sizes], autotune=False, schedule="staged", two_pass=False, **kw)
    outs = [torch.zeros((h, w), device="cuda") for w, h in sizes]
    work = torch.zeros(b.workspace_size, dtype=torch.uint8, device="cuda")
    b.run([torch.from_numpy(t).cuda() for t in noisy], outs, work)
    torch.cuda.synchronize()
    for (w, h), img, out in zip(sizes, noisy, outs):
        op = orc.make_params(w, h, sigma=tuple(device.scaled_sigma([8.0] * 3, False)), **kw)
        res, _, _ = orc.bm3d(op, img[None, None, None])
        assert np.array_equal(out.cpu().numpy(), orc.aggregate(res[:, 0], w)[0])
