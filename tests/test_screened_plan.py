"""Which searches the screened ssd search takes (vsz_bm3d_match_screened, the rule of the launch itself): both sides of each
line of the rule. The parity tests of the screened and of the exhaustive matchers rely on it."""
import pytest

from vszipcu import _lib, device


@pytest.mark.parametrize("kw,screened", [
    # up to 256 tiles of 4 x 4 blocks: from bm_range 9
    (dict(width=640, height=360, block_step=8, bm_range=9), True),
    (dict(width=640, height=360, block_step=8, bm_range=8), False),
    (dict(width=128, height=96, block_step=8, bm_range=9), True),
    # up to 512: from 12
    (dict(width=960, height=540, block_step=8, bm_range=12), True),
    (dict(width=960, height=540, block_step=8, bm_range=11), False),
    # above: from 12 where eight waves share a CU's LDS
    (dict(width=640, height=360, block_step=4, bm_range=12), True),
    (dict(width=640, height=360, block_step=4, bm_range=11), False),
    (dict(width=1920, height=1080, block_step=4, bm_range=16), True),
    (dict(width=1920, height=1080, block_step=2, bm_range=12), True),
    (dict(width=1920, height=1080, block_step=8, bm_range=9), False),
    # the shared-column scan, which is the faster one, keeps its large planes up to 15
    (dict(width=1920, height=1080, block_step=4, bm_range=15), False),
    (dict(width=1921, height=1080, block_step=4, bm_range=12), True),
    # larger windows: from 16, on large planes where enough of the products are candidates
    (dict(width=960, height=540, block_step=5, bm_range=16), True),
    (dict(width=960, height=540, block_step=7, bm_range=15), False),
    (dict(width=1280, height=720, block_step=8, bm_range=16), True),
    (dict(width=1920, height=1080, block_step=8, bm_range=16), False),
    (dict(width=1920, height=1080, block_step=6, bm_range=16), True),
    # beyond its LDS budget, other metrics, wide strides
    (dict(width=640, height=480, block_step=8, bm_range=48), False),
    (dict(width=640, height=360, block_step=4, bm_range=16, metric="sad"), False),
    (dict(width=640, height=360, block_step=4, bm_range=16, metric="zssd"), False),
    (dict(width=64, height=9, stride=1 << 24, block_step=1, bm_range=9), False),
    (dict(width=64, height=9, stride=(1 << 24) - 1, block_step=1, bm_range=9), True),
    # the centre frame's search of a temporal pass
    (dict(width=72, height=64, block_step=4, bm_range=16, radius=2), True),
    (dict(width=1920, height=1080, block_step=8, bm_range=9, radius=2), False),
])
def test_match_screened(kw, screened):
    kw = dict(kw)
    w, h = kw.pop("width"), kw.pop("height")
    assert device.match_screened(device.kparams(w, h, kw.pop("stride", None), **kw)) is screened


def test_match_screened_rejects_invalid_parameters():
    with pytest.raises(RuntimeError, match="vsz_bm3d_match_screened: invalid arguments"):
        device.match_screened(device.kparams(4, 4))
    assert _lib.load().vsz_bm3d_match_screened(None, None) != 0
    assert _lib.load().vsz_bm3d_batch_screened(None, None) != 0


def test_screened_parity_cases_run_the_screen():
    """The parameters of the screened search's parity tests."""
    for w, h, bs, rng in [(9, 11, 1, 9), (21, 40, 4, 16), (77, 61, 3, 12), (57, 90, 2, 24), (90, 75, 4, 16), (90, 75, 8, 20),
                          (64, 32800, 5, 20), (64, 32800, 3, 15), (400, 330, 4, 20), (600, 560, 3, 20)]:
        assert device.match_screened(device.kparams(w, h, block_step=bs, bm_range=rng)), (w, h, bs, rng)
