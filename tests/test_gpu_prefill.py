"""GPU parity of long prefills (wide f16 calls in passes of up to 2048 columns:
the large-tile GEMM's fused epilogues, the one-pass cm1 attention, the last
column's logits) against the oracle's wide mode, with the bounds of parity.py.
The lengths sit at the edges of the tiles: 32-column groups, 256-row blocks,
64-key blocks, 128-row attention workgroups, and past one pass."""
import numpy as np
import pytest

import oracle as O
from parity import WIDE_REL, logits_close, pair
from seeker_amd import synth as S
from seeker_amd._native import GGML_Q4_K, GGML_Q6_K

pytestmark = pytest.mark.gpu

SHAPES = {
    "hd128": S.LlamaShape(2, 1024, 8, 2, 2048, 4000, 4096, 1e-5, 5e5, 0.02, GGML_Q4_K, GGML_Q4_K),
    "hd64": S.LlamaShape(2, 512, 8, 4, 1024, 2000, 4096, 1e-5, 1e4, 0.02, GGML_Q4_K, GGML_Q4_K),
    "qwen3": S.LlamaShape(2, 512, 4, 2, 1024, 2000, 4096, 1e-6, 1e6, 0.02, GGML_Q4_K, GGML_Q4_K, False, arch=1,
                          head_dim=128, norm_jitter=0.1),
    "mix": S.LlamaShape(2, 512, 4, 2, 1024, 2000, 4096, 1e-5, 1e4, 0.02, GGML_Q4_K, GGML_Q4_K, mix=1,
                        out_type=GGML_Q6_K),
    "small": S.LlamaShape(1, 256, 4, 2, 512, 1000, 4096, 1e-5, 1e4, 0.02, GGML_Q4_K, GGML_Q4_K),
}


@pytest.mark.parametrize("name,P,L", [("hd128", 0, 33), ("hd128", 70, 130), ("hd128", 64, 321), ("hd64", 0, 193),
                                      ("hd64", 1, 449), ("qwen3", 0, 200), ("qwen3", 40, 290), ("mix", 33, 260),
                                      ("small", 0, 2100)])
def test_long_prefill(engine, name, P, L):
    with S.GgufImage(SHAPES[name], seed=5) as img:
        gm, om = engine.upload_weights(img), O.Model(img)
        pair(om, gm)
        V = gm.dims.n_vocab
        toks = S.tokens(77, P + L, V)
        gkv, okv = engine.allocate_kv_cache(gm, P + L + 8), O.KvCache(om, P + L + 8)
        if P:
            engine.prefill(gm, gkv, toks[:P], 0)
            O.forward(om, okv, toks[:P], 0, logits_mode=0)
        gl, gr = engine.forward_full_readback(gm, gkv, toks[P:], P, full_logits=False)
        ol, orr = O.forward(om, okv, toks[P:], P, logits_mode=1)
        err = logits_close(gl, ol, wide=True)
        rerr = np.abs(gr - orr).max() / np.abs(orr).max()
        print(f"{name} P={P} L={L}: max|dlogit| {err:.2e}, residual {rerr:.2e} of max", flush=True)
        assert rerr <= WIDE_REL, rerr
        assert gkv.position == P + L
        gkv.close(); okv.close(); gm.close(); om.close()
