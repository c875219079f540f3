"""The prompt GEMM's fused epilogues (RoPE and cache write, residual and next
operand, SwiGLU) at the edges of their tiles, against the oracle."""
import numpy as np
import pytest

import libcmol_amd.native as native
from libcmol_amd import synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu
ATOL, RTOL = 1e-4, 1e-3


# token counts around a 16-vector group and the 32- and 64-vector tiles;
# widths that end inside a 128-row tile (576 = 4.5, 320 = 2.5), a q|k|v row
# count with heads of 64 and of 32, and a feed-forward width of odd blocks
# (1056: 2112 interleaved rows = 16.5 tiles; 2080: the down projection also
# splits k)
@pytest.mark.parametrize("wtype", [synth.Q4_0, synth.Q5_0, synth.Q8_0])
@pytest.mark.parametrize("heads,kv,d_model,d_ffn", [(9, 3, 576, 1056), (10, 2, 320, 2080)])
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
