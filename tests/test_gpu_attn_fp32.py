"""Lock-step decode attention over fp32 caches on balanced ranges
(attn_piece_fw) against the oracle, and its route against the split grid's."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_kernels import attention_case

pytestmark = pytest.mark.gpu

_R = np.random.default_rng(7)


@pytest.fixture(scope="module")
def ctx(gpu):
    c = gpu.Ctx(1 << 30)
    yield c
    c.close()


# one to four query heads per kv head at both head sizes; contexts around the
# wave's 16 positions, the work-group's 64 and the smallest range of 128, cut
# into several pieces and several contexts in one range (bal: total
# work-groups, see attn_bal_wgs; None: the default, which leaves small grids
# to the split kernel)
@pytest.mark.parametrize("n_heads,n_kv,d_head,lens,split,bal", [
    (16, 4, 128, [4096, 1, 257, 1500], 64, "100"), (16, 4, 128, [1, 15, 16, 17, 63, 64, 65, 127, 128, 129], 64, "60"),
    (9, 3, 64, [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 700], 64, "60"), (15, 5, 64, [1024, 64, 300], 64, "1000"),
    (4, 4, 128, [333, 2], 64, "12"), (4, 2, 64, [500, 77, 900], 128, "20"),
    (16, 4, 128, [int(x) for x in _R.integers(64, 4096, 8)], 64, None),
    (15, 5, 64, [int(x) for x in _R.integers(64, 1024, 16)], 64, None),
    (4, 2, 64, [int(x) for x in _R.integers(1, 300, 70)], 64, "200"), (2, 2, 128, [1000, 3], 64, None)])
@pytest.mark.parametrize("q_scale", [1.0, 8.0])
def test_fp32_balanced_attention_matches_oracle(ctx, gpu, monkeypatch, n_heads, n_kv, d_head, lens, split, bal, q_scale):
    if bal is None:
        monkeypatch.delenv("CMOL_ATTN_BAL", raising=False)
    else:
        monkeypatch.setenv("CMOL_ATTN_BAL", bal)
    attention_case(ctx, gpu, n_heads, n_kv, d_head, lens, split, 0, seed=len(lens) + d_head, q_scale=q_scale)


def test_fp32_balanced_equals_split_grid_closely(ctx, gpu, monkeypatch):
    """Same inputs through both routes: fp32 sums in another order."""
    n_heads, n_kv, d_head = 16, 4, 128
    lens = [5000, 17, 900, 2600, 1, 128]
    n, max_ctx = len(lens), max(lens)
    rng = np.random.default_rng(5)
    q = rng.standard_normal((n, n_heads * d_head)).astype(np.float32)
    kc = rng.standard_normal((n, n_kv, max_ctx, d_head)).astype(np.float32)
    vc = rng.standard_normal((n, n_kv, max_ctx, d_head)).astype(np.float32)
    dk, dv, dq = ctx.upload(kc), ctx.upload(vc), ctx.upload(q)
    ds = ctx.upload(np.array(lens, np.int32))
    outs = []
    for bal in ("0", "200", "2000"):
        monkeypatch.setenv("CMOL_ATTN_BAL", bal)
        dout = ctx.alloc(q.nbytes)
        gpu.check(gpu.lib().cmolhip_attn_decode(ctx.h, n, C.c_void_p(dq), C.c_void_p(dk), C.c_void_p(dv),
                                                C.c_void_p(ds), n_heads, n_kv, d_head, max_ctx, 0, 64,
                                                C.c_void_p(dout)), "attn")
        outs.append(ctx.d2h(dout, q.shape, np.float32))
    for o in outs[1:]:
        assert np.allclose(outs[0], o, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("kv_f16", [0, 1])
def test_contexts_without_positions_change_no_other(ctx, gpu, monkeypatch, kv_f16):
    """Lengths of zero and below among others, on balanced ranges: those
    contexts' outputs stay as they were, the others equal a call without them."""
    n_heads, n_kv, d_head, max_ctx = 16, 4, 128, 1024
    lens = [700, -900, 0, 1024, -1, -(1 << 31), 300]
    real = [i for i, m in enumerate(lens) if m > 0]
    rng = np.random.default_rng(11)
    n = len(lens)
    q = rng.standard_normal((n, n_heads * d_head)).astype(np.float32)
    kc, vc = (rng.standard_normal((n, n_kv, max_ctx, d_head)).astype(np.float16 if kv_f16 else np.float32)
              for _ in range(2))
    monkeypatch.setenv("CMOL_ATTN_BAL", "200")

    def run(rows):
        m = len(rows)
        out = np.full((m, n_heads * d_head), 7.0, np.float32)
        dq, dk, dv, dout = ctx.upload(q[rows]), ctx.upload(kc[rows]), ctx.upload(vc[rows]), ctx.upload(out)
        ds = ctx.upload(np.array([lens[i] for i in rows], np.int32))
        gpu.check(gpu.lib().cmolhip_attn_decode(ctx.h, m, *(C.c_void_p(p) for p in (dq, dk, dv, ds)), n_heads, n_kv,
                                                d_head, max_ctx, kv_f16, 64, C.c_void_p(dout)), "attn")
        return ctx.d2h(dout, out.shape, np.float32)

    got, want = run(list(range(n))), run(real)
    # fp32 sums over ranges cut elsewhere
    assert np.allclose(got[real], want, rtol=1e-5, atol=1e-6)
    assert (got[[i for i in range(n) if i not in real]] == 7.0).all()
