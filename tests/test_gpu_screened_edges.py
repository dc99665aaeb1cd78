"""The screened ssd search at the edges of what it accepts, against the FP32 oracle: match lists and distances bit for
bit."""
import numpy as np
import pytest

from gpu_util import assert_matches_equal, kp_and_op
from vszipcu import device, synth

pytestmark = pytest.mark.gpu


def _match(torch, kp, img):
    nbx, nby = device.num_blocks(kp)
    m = torch.zeros((nby, nbx, 8, 4), dtype=torch.int32, device="cuda")
    device.match(kp, img, m)
    torch.cuda.synchronize()
    return m.cpu().numpy()


@pytest.mark.parametrize("bs,rng", [(5, 20), (3, 15)])
def test_tall_plane(orc, torch_gpu, bs, rng):
    """Rows beyond 32640, whose packed positions would be infinities and NaNs if they were read as floats; 4 rows divide
    both windows, so the last searched row reads past the norms' pitch. The lower end of the plane is compared with the
    oracle's search of that end alone."""
    torch = torch_gpu
    print(f"screened search: 64x32800 bs={bs} R={rng}", flush=True)
    W, H, y0 = 64, 32800, 32400                     # 32400 is a multiple of both block steps
    img = np.random.default_rng(bs).random((H, W), dtype=np.float32)
    kp, _ = kp_and_op(orc, W, H, bs=bs, rng=rng)
    _, op = kp_and_op(orc, W, H - y0, bs=bs, rng=rng)
    om, oe = orc.match(op, np.ascontiguousarray(img[None, y0:]))
    gm = _match(torch, kp, torch.from_numpy(img[None]).cuda())[y0 // bs:]
    first = -(-rng // bs)                           # block rows whose windows stay inside the end
    gm[..., 1] -= y0
    assert_matches_equal(gm[first:], om[first:], oe[first:])


@pytest.mark.parametrize("stride", [(1 << 24) - 8, (1 << 24) + 8])
def test_wide_stride(orc, torch_gpu, stride):
    """Strides at both sides of 24 bits (a plane of 604 MB of which 64 columns are used)."""
    torch = torch_gpu
    print(f"screened search: 64x9 stride {stride}", flush=True)
    W, H = 64, 9
    img = np.random.default_rng(9).random((H, W), dtype=np.float32)
    kp, _ = kp_and_op(orc, W, H, bs=1, rng=9, stride=stride)
    _, op = kp_and_op(orc, W, H, bs=1, rng=9)
    plane = torch.zeros((1, H, stride), device="cuda")
    plane[0, :, :W] = torch.from_numpy(img).cuda()
    om, oe = orc.match(op, img[None])
    assert_matches_equal(_match(torch, kp, plane), om, oe)


@pytest.mark.parametrize("bs,rng", [(4, 16), (8, 20)])
@pytest.mark.parametrize("level", [1.0, 50.0])
def test_isolated_bright_pixels(orc, torch_gpu, bs, rng, level):
    """Pixels far above a window of low contrast: one term of a product outweighs the others, and the window's halves have
    coarse steps."""
    torch = torch_gpu
    print(f"screened search: bright pixels {level} bs={bs} R={rng}", flush=True)
    W, H = 132, 110
    r = np.random.default_rng(4)
    img = (0.2 + r.normal(0, 0.002, (H, W))).astype(np.float32)
    img[r.integers(0, H, 12), r.integers(0, W, 12)] = level
    kp, op = kp_and_op(orc, W, H, bs=bs, rng=rng)
    om, oe = orc.match(op, img[None])
    assert_matches_equal(_match(torch, kp, torch.from_numpy(img[None]).cuda()), om, oe)
