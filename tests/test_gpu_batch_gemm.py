"""Lock-step decode steps whose projections run the tiled GEMM with its fused
epilogues (K-quant matrices large enough for more than 16 sessions, see
batch_by_gemm): logits, cached rows and choices of every session against its
own single step."""
import numpy as np
import pytest

import libcmol_amd.native as native
from libcmol_amd import synth

pytestmark = pytest.mark.gpu
ATOL, RTOL = 1e-4, 1e-3

# gate/up (SwiGLU) and down (residual, split k) of the SmolLM3-3B Q4_K_M mix;
# Q6_K with hidden 4096: q|k|v (RoPE and cache write into each session's own
# slot and position), gate/up and down
MIX = dict(n_layers=1, d_model=2048, n_heads=16, n_kv_heads=4, d_ffn=11008, vocab=512, wtype=synth.Q4_K,
           embd_type=synth.Q6_K, v_type=synth.Q6_K, down_type=synth.Q6_K)
WIDE = dict(n_layers=2, d_model=4096, n_heads=32, n_kv_heads=8, d_ffn=4352, vocab=512, wtype=synth.Q6_K,
            embd_type=synth.Q6_K)


@pytest.mark.parametrize("shape,f16", [(MIX, "0"), (WIDE, "0"), (WIDE, "1")], ids=["q4_k_m", "q6_k", "q6_k-f16"])
@pytest.mark.parametrize("n", [17, 32])
def test_lock_step_through_the_gemm_matches_single_steps(gpu, model_dir, monkeypatch, shape, f16, n):
    monkeypatch.setenv("CMOL_KV_F16", f16)
    spec = synth.ModelSpec(ctx_len=128, wstd=0.02, seed=5, **shape)
    m = native.Model(synth.model_file(spec, model_dir), max_ctx=96, max_sessions=32)
    ss = [m.acquire() for _ in range(32)][32 - n:]   # (slots other than the vectors' numbers)
    pos = [(7 * i) % 80 for i in range(n)]
    for i, s in enumerate(ss):
        if pos[i]:
            s.fill_kv(pos[i], seed=50 + i)
    toks = synth.tokens(n, 9, spec.vocab)
    ids, lg = native.decode_batch_logits(m, ss, toks, pos, spec.vocab)
    kvd = spec.n_kv_heads * spec.d_head
    rows = [[native.kv_download(m, s.slot, l, p + 1, kvd) for l in range(spec.n_layers)] for s, p in zip(ss, pos)]
    # fp16 caches: a new value next to a rounding boundary may fall to either
    # side (2^-11 of it), which the attention of this one row of p + 1 passes on
    rtol = RTOL if f16 == "0" else 2 * RTOL
    for i, s in enumerate(ss):
        _, want = s.forward(int(toks[i]), pos[i], spec.vocab)
        assert np.all(np.abs(lg[i] - want) <= ATOL + rtol * np.abs(want))
        assert ids[i] == int(np.argmax(lg[i]))
        for l in range(spec.n_layers):
            for got, ref in zip(rows[i][l], native.kv_download(m, s.slot, l, pos[i] + 1, kvd)):
                assert np.all(np.abs(got - ref) <= ATOL + rtol * np.abs(ref))
    m.close()
