"""Prompt passes over fp16 caches (flash-style attention straight from the
cache): the logits and cached rows of a chunked prompt against the same
tokens decoded one by one, whose attention kernels the oracle pins
(test_gpu_kernels.py, test_gpu_configs.py)."""
import numpy as np
import pytest

import libcmol_amd.native as native
from libcmol_amd import synth

pytestmark = pytest.mark.gpu


# 1, 2, 3, 4 and 8 query heads per kv head (3: 63 of a work-group's 64 query
# rows used) at d_head 64 and 128; one pass within a split, one over a split
# boundary (256), and later passes behind cached positions; lengths around
# the 64-position tile
@pytest.mark.parametrize("heads,kv,d_model", [(2, 2, 256), (4, 2, 256), (9, 3, 576), (4, 1, 512), (8, 1, 512)])
@pytest.mark.parametrize("n,chunk", [(63, 512), (65, 512), (300, 512), (300, 128), (321, 64)])
def test_prompt_over_f16_cache_matches_decode(gpu, model_dir, monkeypatch, heads, kv, d_model, n, chunk):
    monkeypatch.setenv("CMOL_KV_F16", "1")
    spec = synth.ModelSpec(2, d_model, heads, kv, 2 * d_model, 1024, ctx_len=512, wtype=synth.Q8_0,
                           embd_type=synth.Q8_0, wstd=0.08, seed=heads * 10 + kv)
    path = synth.model_file(spec, model_dir)
    prompt = synth.tokens(n, 31, spec.vocab)
    m = native.Model(path, max_ctx=330, max_sessions=2, prefill_chunk=chunk)
    s, t = m.acquire(), m.acquire()
    am, lg = s.prefill(prompt, spec.vocab)
    for p, tok in enumerate(prompt):
        want_id, want = t.forward(int(tok), p, spec.vocab)
    # The passes sum in different fp32 orders (about 1e-6), so a new K/V
    # value next to an fp16 rounding boundary may fall to either side: about
    # 2 * 1e-6 / 2^-11 = 0.4 % of the rows' values move by 2^-11, 3e-5 of the
    # rows in the 2-norm; three times that for the logits
    assert np.linalg.norm(lg - want) <= 1e-4 * np.linalg.norm(want)
    assert am == want_id or abs(want[am] - want[want_id]) <= 1e-4 * np.abs(want).max()
    kvd = spec.n_kv_heads * spec.d_head
    for layer in range(spec.n_layers):
        for a, b in zip(native.kv_download(m, s.slot, layer, n, kvd), native.kv_download(m, t.slot, layer, n, kvd)):
            assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b)
    m.close()
