"""The standalone operand preparation (cmolhip_act_prepare), bit for bit
against numpy: high and low f16 parts per (block, k-group, vector) in each
format's input order, and the sums of squares per block."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def expected(x, w, q8):
    """[block][k-group][2 vectors][8] halves of x (times w) / 256."""
    n, cols = x.shape
    f = np.float32
    t = (x if w is None else w * x) * f(1 / 256)
    b = t.reshape(n, cols // 32, 32)
    if q8:
        g = b.reshape(n, -1, 4, 8)
    else:   # inputs 4g .. 4g+3 and 16+4g .. +3, each four in the order 0, 2, 1, 3
        g = b.reshape(n, -1, 2, 4, 4)[..., [0, 2, 1, 3]].transpose(0, 1, 3, 2, 4).reshape(n, -1, 4, 8)
    hi = g.astype(np.float16)
    lo = ((g - hi.astype(f)) * f(2048)).astype(np.float16)
    return np.stack([hi, lo], 0).transpose(2, 3, 1, 0, 4).reshape(cols // 32, 4, 2 * n, 8)


# one vector, the last count of the one-vector waves, the first of the
# 16-vector ones, and a ragged last group; one block, and block counts that
# leave a work-group partly idle
@pytest.mark.parametrize("dtype", [2, 8, 12])
@pytest.mark.parametrize("n,cols", [(1, 32), (1, 2048), (3, 2080), (15, 288), (16, 32), (17, 2080), (33, 576)])
@pytest.mark.parametrize("norm,shift", [(False, 0), (True, 0), (True, 1)])
def test_act_prepare_bit_exact(gpu, dtype, n, cols, norm, shift):
    if dtype == 12:
        cols = (cols + 255) // 256 * 256
    rng = np.random.default_rng(n * 10000 + cols + dtype)
    x = (rng.standard_normal((n, cols)) * 3).astype(np.float32)
    w = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32) if norm else None
    ctx = gpu.Ctx(64 << 20)
    L = gpu.lib()
    # vectors and norm weights at addresses with a float's alignment only
    dx = ctx.alloc(x.nbytes + 4 * shift) + 4 * shift
    ctx.h2d(dx, x)
    dw = None
    if norm:
        dw = ctx.alloc(w.nbytes + 4 * shift) + 4 * shift
        ctx.h2d(dw, w)
    op = ctx.alloc(L.cmolhip_act_bytes(cols, n))
    ss = ctx.alloc(n * cols // 32 * 4)
    gpu.check(L.cmolhip_act_prepare(ctx.h, C.c_void_p(dx), n, cols, dtype, C.c_void_p(dw) if norm else None,
                                    C.c_void_p(op), C.c_void_p(ss) if norm else None), "act_prepare")
    gpu.check(L.cmolhip_synchronize(ctx.h), "sync")
    got = ctx.d2h(op, (cols // 32, 4, 2 * n, 8), np.uint16)
    assert np.array_equal(got, expected(x, w, dtype == 8).view(np.uint16))
    if norm:
        want = (x.astype(np.float64) ** 2).reshape(n, -1, 32).sum(2)
        s = ctx.d2h(ss, (n, cols // 32), np.float32)
        # 32 rounded squares and 31 rounded additions of positive terms
        assert np.all(np.abs(s - want) <= 32 * 2.0 ** -24 * want)
    ctx.close()
