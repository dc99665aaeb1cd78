"""The reductions of the learned estimate's training step (weight gradient, bias gradient, loss) at the sizes
where their shares are uneven: fewer tiles than workgroups, more, partial tiles and single pixels.

Tolerance: inputs are bf16 and products exact in FP32, so only the order of the FP32 sums differs from the 64-bit
sums of the same values: |error| <= n * 2^-24 * sum |term| with n the longest chain of additions (below 2^13 here; the
rest are trees), taken as 5e-4 * sum |term|. A misplaced or doubled pixel is off by about 1 / sqrt(pixels) of the sum of squares."""
import numpy as np
import pytest

from vszipcu import _lib, cnn

CH = 32


def _bits(torch, v):
    return torch.from_numpy(v).to(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("n,h,w", [(1, 1, 1), (1, 16, 16), (2, 17, 33), (5, 15, 128), (3, 200, 180), (1, 1, 2048)])
def test_gradient_sums(torch_gpu, n, h, w):
    torch = torch_gpu
    print(f"cnn gradient sums: {n}x{h}x{w}", flush=True)
    L = _lib.load()
    rng = np.random.default_rng(n * 1000 + h + w)
    x = _bits(torch, rng.normal(0, 1, (n, h, w, CH)).astype(np.float32))
    dz = _bits(torch, rng.normal(0, 1, (n, h, w, CH)).astype(np.float32))
    out, tgt = (rng.random((n * h * w,), dtype=np.float32) for _ in range(2))
    dw, db, loss = (torch.zeros(k, dtype=torch.float32, device="cuda") for k in (9 * CH * CH, CH, 1))
    grad = torch.full((n * h * w, CH), 7.0, dtype=torch.bfloat16, device="cuda")
    xd, dzd = x.view(torch.int16).cuda(), dz.view(torch.int16).cuda()
    outd, tgtd = torch.from_numpy(out).cuda(), torch.from_numpy(tgt).cuda()
    cnn._check(L.vsz_cnn_conv3x3_dw(cnn._p(xd), cnn._p(dzd), n, h, w, cnn._p(dw), cnn._s(None)))
    cnn._check(L.vsz_cnn_bias_grad(cnn._p(dzd), n * h * w, cnn._p(db), cnn._s(None)))
    cnn._check(L.vsz_cnn_loss_grad(cnn._p(outd), cnn._p(tgtd), n * h * w, cnn._p(grad), cnn._p(loss), cnn._s(None)))
    torch.cuda.synchronize()
    xv, zv = x.double().numpy(), dz.double().numpy()
    pad = np.pad(xv, ((0, 0), (1, 1), (1, 1), (0, 0)))
    for t in range(9):
        s = pad[:, t // 3:t // 3 + h, t % 3:t % 3 + w].reshape(-1, CH)
        ref, big = zv.reshape(-1, CH).T @ s, np.abs(zv).reshape(-1, CH).T @ np.abs(s)
        assert np.all(np.abs(dw.cpu().numpy().reshape(9, CH, CH)[t] - ref) <= 5e-4 * big), t
    zf = zv.reshape(-1, CH)
    assert np.all(np.abs(db.cpu().numpy() - zf.sum(0)) <= 5e-4 * np.abs(zf).sum(0))
    d = out.astype(np.float64) - tgt
    assert abs(float(loss) - float((d * d).mean())) <= 5e-4 * float((d * d).mean()) + 1e-12
    g = grad.float().cpu().numpy()
    assert np.all(g[:, 1:] == 0.0)
    scale = np.float32(1.0) / np.float32(n * h * w)
    want = torch.from_numpy((np.float32(2.0) * scale) * (out - tgt)).to(torch.bfloat16).float().numpy()
    assert np.array_equal(g[:, 0], want)
