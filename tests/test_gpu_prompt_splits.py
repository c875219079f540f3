"""Prompt passes behind long contexts, whose attention is cut into many splits:
the logits and cached rows against the same tokens decoded one by one."""
import numpy as np
import pytest

import libcmol_amd.native as native
from libcmol_amd import synth

pytestmark = pytest.mark.gpu


# 12 splits of 256 positions (the merge takes eight at a time), then, in passes
# of 64, as many as the partials of a model with so short a pass have room for
# (fp16 caches: 6 of 512); 7 splits; fewer tokens than a block
@pytest.mark.parametrize("f16", ["1", "0"])
@pytest.mark.parametrize("heads,kv,d_model", [(4, 1, 512), (9, 3, 576)])
@pytest.mark.parametrize("past,n,chunk", [(2900, 64, 512), (2900, 130, 64), (1700, 65, 512), (2050, 11, 512)])
def test_prompt_behind_a_long_context_matches_decode(gpu, model_dir, monkeypatch, f16, heads, kv, d_model, past, n, chunk):
    monkeypatch.setenv("CMOL_KV_F16", f16)
    spec = synth.ModelSpec(2, d_model, heads, kv, 2 * d_model, 512, ctx_len=4096, wtype=synth.Q8_0,
                           embd_type=synth.Q8_0, wstd=0.08, seed=heads + kv)
    m = native.Model(synth.model_file(spec, model_dir), max_ctx=3072, max_sessions=2, prefill_chunk=chunk)
    s, t = m.acquire(), m.acquire()
    for x in (s, t):
        x.fill_kv(past, seed=5)
    prompt = synth.tokens(n, 31, spec.vocab)
    am, lg = s.prefill(prompt, spec.vocab)
    for p, tok in enumerate(prompt):
        want_id, want = t.forward(int(tok), past + p, spec.vocab)
    # as in test_gpu_prompt_f16.py: 3e-5 from new rows next to an fp16 rounding
    # boundary, 1e-6 over fp32; three times that
    rel = 1e-4 if f16 == "1" else 5e-6
    assert np.linalg.norm(lg - want) <= rel * np.linalg.norm(want)
    assert am == want_id or abs(want[am] - want[want_id]) <= rel * np.abs(want).max()
    kvd = spec.n_kv_heads * spec.d_head
    for layer in range(spec.n_layers):
        for a, b in zip(native.kv_download(m, s.slot, layer, past + n, kvd),
                        native.kv_download(m, t.slot, layer, past + n, kvd)):
            assert np.linalg.norm(a[past:] - b[past:]) <= rel * np.linalg.norm(b[past:])
    m.close()
