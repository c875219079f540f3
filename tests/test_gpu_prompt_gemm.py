"""The prompt GEMM's fused epilogues (RoPE and cache write, residual and next
operand, SwiGLU) at the edges of their tiles, against the oracle."""
import numpy as np
import pytest

import libcmol_amd.native as native
from libcmol_amd import synth
from oracle import oracle as O
from tests.qdata import random_blocks

pytestmark = pytest.mark.gpu
ATOL, RTOL = 1e-4, 1e-3


# token counts around a 16-vector group and the 32- and 64-vector tiles;
# widths that end inside a 128-row tile (576 = 4.5, 320 = 2.5), a q|k|v row
# count with heads of 64 and of 32, and a feed-forward width of odd blocks
# (1056: 2112 interleaved rows = 16.5 tiles; 2080: the down projection also
# splits k); the K-quants, whose widths are whole tiles
@pytest.mark.parametrize("wtype,heads,kv,d_model,d_ffn", [
    (w, *shape) for shape in [(9, 3, 576, 1056), (10, 2, 320, 2080)] for w in (synth.Q4_0, synth.Q5_0, synth.Q8_0)
] + [(synth.Q4_K, 12, 4, 768, 1792), (synth.Q6_K, 12, 4, 768, 1792)])
@pytest.mark.parametrize("n", [9, 17, 33, 64, 65, 129])
def test_prompt_epilogues_match_oracle(gpu, model_dir, wtype, heads, kv, d_model, d_ffn, n):
    spec = synth.ModelSpec(2, d_model, heads, kv, d_ffn, 512, ctx_len=192, wtype=wtype, embd_type=wtype, wstd=0.05,
                           seed=d_model + wtype)
    path = synth.model_file(spec, model_dir)
    prompt = synth.tokens(n, 5, spec.vocab)
    m = native.Model(path, max_ctx=160, max_sessions=1)
    s = m.acquire()
    am, lg = s.prefill(prompt, spec.vocab)
    om = O.Model(path, 160)
    for p, t in enumerate(prompt):
        want = om.forward(int(t), p)
    assert np.all(np.abs(lg - want) <= ATOL + RTOL * np.abs(want))
    assert am == int(np.argmax(want))
    ok, ov = om.kv()
    kvd = spec.n_kv_heads * spec.d_head
    for layer in range(spec.n_layers):
        k, v = native.kv_download(m, s.slot, layer, n, kvd)
        for got, ref in ((k, ok[layer, :n].reshape(n, kvd)), (v, ov[layer, :n].reshape(n, kvd))):
            assert np.all(np.abs(got - ref) <= ATOL + RTOL * np.abs(ref))
    m.close()
    om.close()


def check_gemm(ctx, dtype, rows, cols, fold, n, norm):
    raw = random_blocks(dtype, rows, cols, seed=rows + 3 * cols + n)
    rng = np.random.default_rng(n + rows)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    w = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32) if norm else None
    t = ctx.qtensor([raw], dtype, cols, [rows], fold=fold)
    got = ctx.gemm(t, x, w)
    if norm:
        x64 = x.astype(np.float64)
        x = (x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-5) * w).astype(np.float32)
    want = O.matmul(raw, np.ascontiguousarray(x.T), rows, cols, dtype, O.AVX512).T
    # Both sides sum thousands of terms in fp32, in their own orders: rounding
    # of each partial sum (2^-24 of it, the sums growing to the outputs' rms
    # over up to 512 blocks) adds up to 2..5e-7 of the rms per output, whatever
    # the output's own size; the largest of some thousands stays below 10 sigma
    tol = ATOL + RTOL * np.abs(want) + 5e-6 * np.sqrt(np.mean(want.astype(np.float64) ** 2))
    assert np.all(np.abs(got - want) <= tol), f"{dtype} {rows}x{cols} fold {fold} n {n}"


# k ranges 1 (one quad pair), 2, 4, 8 and 16, the last range short or empty
# (20 quads in 8 ranges of 3), ranges summed in one chain and in two halves,
# folded tensors, and row counts that are no multiple of 4 with partial sums
@pytest.mark.parametrize("dtype", [2, 8, 12])
@pytest.mark.parametrize("rows,cols,fold,n,norm", [
    (128, 256, 1, 33, True), (130, 512, 1, 40, False), (131, 1024, 1, 33, True), (257, 2560, 1, 64, True),
    (129, 8192, 1, 35, False), (96, 16384, 1, 33, True), (512, 2048, 2, 65, True), (512, 2048, 4, 100, False),
    (4096, 512, 1, 1056, False), (4096, 512, 1, 1024, True)])
def test_gemm_k_ranges_match_oracle(gpu, dtype, rows, cols, fold, n, norm):
    ctx = gpu.Ctx(512 << 20)
    check_gemm(ctx, dtype, rows, cols, fold, n, norm)
    ctx.close()


# vector tiles that do not divide by eight, in one, two and four slices per the
# grid's row tiles, the last row tile ragged; split k and not
@pytest.mark.parametrize("rows,cols,n", [(2500, 256, 160), (2500, 256, 188), (2500, 256, 300), (5000, 128, 350),
                                         (2500, 512, 600), (520, 4096, 188)])
def test_gemm_slices_match_oracle(gpu, rows, cols, n):
    ctx = gpu.Ctx(512 << 20)
    check_gemm(ctx, 2, rows, cols, 1, n, True)
    ctx.close()


# three to four work-groups per CU, whose first half's sums are kept half in
# registers: 10 vector tiles x 101 row tiles, the last ragged, and a single
# vector tile (there only the formats that spill nothing); five quads, so the
# second half is the shorter one
@pytest.mark.parametrize("dtype,cols", [(2, 640), (6, 640), (8, 640), (12, 768), (14, 768)])
@pytest.mark.parametrize("rows,n", [(12805, 300), (125000, 20)])
def test_gemm_kept_sums_match_oracle(gpu, dtype, cols, rows, n):
    ctx = gpu.Ctx(1 << 30)
    check_gemm(ctx, dtype, rows, cols, 1, n, n == 300)
    ctx.close()


def test_gemm_small_arena_takes_fewer_ranges(gpu):
    """An arena with room for fewer k ranges' partial sums than the product
    would take: the call still runs, on fewer ranges."""
    rows, cols, n = 256, 4096, 64
    sizes = [gpu.lib().cmolhip_qtensor_bytes(2, rows, cols, 1), rows * cols // 32 * 18, n * cols * 4, n * rows * 4,
             gpu.lib().cmolhip_act_bytes(cols, n)]
    # 32 quads on two 128-row tiles x two 32-vector tiles: 16 ranges of two,
    # 1 MiB of partial sums; the arena has room for four, 256 KiB
    ctx = gpu.Ctx(sum(sizes) + 4 * n * rows * 4 + 4096)
    check_gemm(ctx, 2, rows, cols, 1, n, False)
    ctx.close()


# batches of 9..32 that the tiled GEMM takes from the matvec: rows at and past
# the first such tile count (one tile per CU above 16 vectors, two up to 16),
# a ragged last tile, and K-quants by their size; with the counts on either
# side of 16 vectors
@pytest.mark.parametrize("dtype,rows,cols,n,norm", [
    (2, 32768, 96, 17, True), (8, 32770, 64, 32, False), (6, 32900, 64, 24, True), (8, 65540, 32, 9, True),
    (2, 65540, 64, 16, False), (12, 16384, 2048, 17, True), (14, 4224, 4096, 32, False)])
def test_batches_through_the_gemm_match_oracle(gpu, dtype, rows, cols, n, norm):
    ctx = gpu.Ctx(512 << 20)
    check_gemm(ctx, dtype, rows, cols, 1, n, norm)
    ctx.close()


@pytest.mark.parametrize("n", [17, 20])
def test_batch_logits_and_argmax_of_a_wide_head(gpu, model_dir, n):
    """A head of 33000 rows (258 tiles, the last ragged) for more than 16
    sessions: the GEMM's logits against each session's own step, and its
    argmax (combined over work-groups) exactly the largest of its logits."""
    spec = synth.ModelSpec(1, 256, 4, 2, 512, 33000, ctx_len=64, wtype=synth.Q8_0, embd_type=synth.Q8_0, wstd=0.08,
                           seed=3)
    m = native.Model(synth.model_file(spec, model_dir), max_ctx=32, max_sessions=n)
    ss = [m.acquire() for _ in range(n)]
    toks = synth.tokens(n, 9, spec.vocab)
    ids, lg = native.decode_batch_logits(m, ss, toks, [0] * n, spec.vocab)
    for i in range(n):
        _, want = ss[i].forward(int(toks[i]), 0, spec.vocab)
        assert np.all(np.abs(lg[i] - want) <= ATOL + RTOL * np.abs(want))
        assert ids[i] == int(np.argmax(lg[i]))
    m.close()
