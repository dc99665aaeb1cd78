"""The rounding that the screened search's limits allow its half-precision products (kScrC in csrc/bm3d_kernels.hip), on the
instruction itself: three chained 16x16x32 products from an accumulator of -n_b/2, as a row of the search computes
a.b - n_b/2, against 64-bit sums of the same halves.

Limit: |S' - S_q| <= c (n_a + n_b) with c = 8e-6 and S' = n_a - 2 (a.b - n_b/2). Of it the squared norms' own rounding, 7 roundings
of 2^-24 of a sum of positive terms, takes 4.2e-7 (n_a + n_b); twice the products' error has to stay below the other 7.5e-6.
A subnormal half may count as 0, which the limits allow apart from c."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "mfma_error", "_build", "libmfma_error.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        subprocess.run(["make", "-s", "-C", os.path.dirname(os.path.dirname(LIB))], check=True)
    f = C.CDLL(LIB).mfma_error_run
    f.argtypes = [C.c_void_p] * 4 + [C.c_int, C.c_void_p]
    return f


def _patches(kind, n):
    """[n, 16, 64] blocks and candidates, in the screen's scale (values up to 1024)."""
    rng = np.random.default_rng(len(kind))
    a, b = rng.normal(0, 100, (n, 16, 64)), rng.normal(0, 100, (n, 16, 64))
    if kind == "one large term":              # 2^12 times the others, which are all below its last places
        a, b = rng.uniform(0.5, 1, (n, 16, 64)) * 16, rng.uniform(0.5, 1, (n, 16, 64)) * 16
        at = rng.integers(0, 64, (n, 16, 1))
        np.put_along_axis(a, at, 1000.0, 2)
        np.put_along_axis(b, at, 1000.0, 2)
    elif kind == "one large in each row":     # every product of eight has one
        a, b = rng.uniform(0.5, 1, (n, 16, 64)), rng.uniform(0.5, 1, (n, 16, 64))
        a[..., ::8] = b[..., ::8] = 64.0
    elif kind == "cancelling":                # the sum is far below its terms
        a = np.repeat(rng.normal(0, 300, (n, 16, 32)), 2, axis=2)
        b = np.repeat(rng.normal(0, 300, (n, 16, 32)), 2, axis=2) * np.tile([1.0, -1.0], 32)
        b += rng.normal(0, 0.5, b.shape)
    elif kind == "equal":                     # a candidate like its block: a.b - n_b/2 is half of n_a
        b = a + rng.normal(0, 0.5, a.shape)
    elif kind == "small block":               # the accumulator outweighs the products
        a *= 1e-3
    elif kind == "edge of the subnormals":
        a, b = rng.normal(0, 6e-5, a.shape), rng.normal(0, 100, b.shape)
    elif kind == "same sign":
        a, b = rng.uniform(500, 1024, a.shape), rng.uniform(500, 1024, b.shape)
    return a.astype(np.float16), b.astype(np.float16)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["noise", "one large term", "one large in each row", "cancelling", "equal", "small block",
                                  "edge of the subnormals", "same sign"])
def test_product_rounding_stays_within_the_limit(torch_gpu, lib, kind):
    torch = torch_gpu
    n = 512
    a, b = _patches(kind, n)
    worst = 0.0
    for s in range(4):                        # the block's rows start at slot row s of twelve
        fa, fb = np.zeros((n, 16, 96), np.float16), np.random.default_rng(s).normal(0, 100, (n, 16, 96)).astype(np.float16)
        fa[..., 8 * s:8 * s + 64], fb[..., 8 * s:8 * s + 64] = a, b
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        na, nb = (a64 ** 2).sum(-1), (b64 ** 2).sum(-1)
        c = (-0.5 * nb).astype(np.float32)
        dev = [torch.from_numpy(v).cuda() for v in (fa, fb, c)]
        d = torch.zeros((n, 16, 16), device="cuda")
        assert lib(*[C.c_void_p(t.data_ptr()) for t in (*dev, d)], n, C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        torch.cuda.synchronize()
        exact = a64 @ b64.transpose(0, 2, 1) + c.astype(np.float64)[:, None, :]
        sub = np.where(np.abs(a64) < 2.0 ** -14, np.abs(a64), 0) @ np.abs(b64).transpose(0, 2, 1)
        sub += np.abs(a64) @ np.where(np.abs(b64) < 2.0 ** -14, np.abs(b64), 0).transpose(0, 2, 1)
        err = 2 * np.maximum(np.abs(d.cpu().numpy() - exact) - sub, 0)
        worst = max(worst, float((err / (na[:, :, None] + nb[:, None, :])).max()))
    print(f"product rounding: {kind}: {worst:.2e} (n_a + n_b)", flush=True)
    assert worst <= 7.5e-6
