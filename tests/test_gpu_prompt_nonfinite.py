"""Prompt passes with a token whose V row is not finite in the cache (beyond
fp16): as when the tokens are decoded one by one, the tokens before it keep
their values and only those that attend to it lose theirs."""
import ctypes as C

import numpy as np
import pytest

import libcmol_amd.native as native
from libcmol_amd import synth

pytestmark = pytest.mark.gpu
VOCAB, HUGE = 256, 0   # token HUGE overflows


class Model:
    """Two layers of random Q8_0 weights; dimension 0 of the embedding is zero
    for every token but HUGE, and layer 0's V rows weigh it by 12700."""

    def __init__(self, heads, kv, d, f16, chunk, max_ctx):
        rng = np.random.default_rng(heads * 100 + d)
        dh, f, self.keep = d // heads, 2 * d, []
        self.kvd = kv * dh

        def ten(x, dt=0):
            rows, cols = x.shape if x.ndim == 2 else (1, x.size)
            a = synth.quantize(dt, x) if dt else np.ascontiguousarray(x, np.float32)
            self.keep.append(a)
            return native.HostTensor(C.c_void_p(a.ctypes.data), dt, rows, cols)

        def mat(rows, cols):
            return (0.08 * rng.standard_normal((rows, cols))).astype(np.float32)

        layers = (native.LayerTensors * 2)()
        for i, L in enumerate(layers):
            v = mat(self.kvd, d)
            if i == 0:
                v[:, 0] = 12700.0
            for name, x in (("q", mat(d, d)), ("k", mat(self.kvd, d)), ("v", v), ("o", mat(d, d)),
                            ("gate", mat(f, d)), ("up", mat(f, d)), ("down", mat(d, f))):
                setattr(L, name, ten(x, synth.Q8_0))
            L.attn_norm, L.ffn_norm = ten(np.ones(d)), ten(np.ones(d))
        embd = rng.standard_normal((VOCAB, d)).astype(np.float32)
        embd[:, 0] = 0.0
        embd[HUGE, 0] = 30.0
        ang = np.arange(max_ctx)[:, None] / 1e4 ** (np.arange(dh // 2) * 2.0 / dh)
        rope = np.ascontiguousarray(np.stack([np.cos(ang), np.sin(ang)], 2).astype(np.float32))
        desc = native.ModelDesc()
        desc.hp = native.HParams(2, heads, kv, d, dh, f, VOCAB, max_ctx, 2, 0, int(f16), chunk, 1e4, 1e-5)
        desc.embd = ten(embd, synth.Q8_0)
        desc.out_norm = ten(np.ones(d))
        desc.layers = layers
        desc.rope_table = C.c_void_p(rope.ctypes.data)
        self.device = C.c_void_p()
        native.check(native.lib().cmolhip_model_create(C.byref(desc), 0, C.byref(self.device)), "model_create")
        self.logits = np.zeros(VOCAB, np.float32)
        self.id = C.c_int32()

    def close(self):
        native.lib().cmolhip_model_destroy(self.device)

    def prefill(self, slot, tokens):
        t = np.ascontiguousarray(tokens, np.int32)
        native.check(native.lib().cmolhip_prefill(self.device, slot, native.ptr(t), len(t), 0, native.ptr(self.logits),
                                                  C.byref(self.id)), "prefill")

    def decode(self, slot, tokens):
        for p, t in enumerate(tokens):
            native.check(native.lib().cmolhip_decode(self.device, slot, int(t), p, native.ptr(self.logits),
                                                     C.byref(self.id)), "decode")

    def rows(self, slot, layer, n):
        return native.kv_download(self, slot, layer, n, self.kvd)


# the overflowing token first, inside, at the edges of a 32- and a 64-position
# tile and last; alone in its tile, before a split's end (256) and behind whole
# passes; 1, 3 and 4 query heads per kv head at d_head 64 and 128
@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("heads,kv,d", [(4, 4, 256), (9, 3, 576), (4, 1, 512)])
@pytest.mark.parametrize("n,at,chunk", [(40, 0, 512), (40, 25, 512), (65, 64, 512), (130, 95, 512), (330, 300, 512),
                                        (330, 255, 128), (330, 329, 64)])
def test_prompt_keeps_the_tokens_before_an_overflow(gpu, f16, heads, kv, d, n, at, chunk):
    toks = 1 + synth.tokens(n, 7, VOCAB - 1)
    toks[at] = HUGE
    m = Model(heads, kv, d, f16, chunk, 352)
    m.prefill(0, toks)
    m.decode(1, toks)
    for layer in range(2):
        for got, want in zip(m.rows(0, layer, n), m.rows(1, layer, n)):
            # fp16 caches round new K/V rows whose fp32 sums differ by about
            # 1e-6 to either side of a boundary (test_gpu_prompt_f16.py: 3e-5
            # of the rows, three times that here)
            assert np.isfinite(want[:at]).all()
            assert np.linalg.norm(got[:at] - want[:at]) <= 1e-4 * np.linalg.norm(want[:at])
            if f16:
                assert np.array_equal(np.isfinite(got), np.isfinite(want))
    if f16:
        assert not np.isfinite(m.rows(1, 0, n)[1][at]).all() and not np.isfinite(m.logits).all()
    m.close()
