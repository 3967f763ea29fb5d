"""COMPARE decided inside the chunked draw (vocabularies of 8192 and more, at most
64 rows) and by its own kernel, and REJECTION beside it, vs the oracle: both sides
of each limit, k = 1, 63 and 64, every draft accepted and mixed. Accepted lengths
and next tokens are integers and equal; each call runs twice on the same scratch,
so that the arrival counters have to come back to zero."""
import numpy as np
import pytest

import oracle as O
from seeker_amd._native import SH_SAMPLE_COMPARE, SH_SAMPLE_REJECTION
from test_gpu_accept import make_inputs, oracle_uniforms, run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,k,V,kind", [
    (1, 1, 8192, "mixed"), (1, 63, 8193, "all"), (1, 63, 8193, "mixed"), (1, 64, 8193, "all"), (2, 63, 8200, "all"),
    (32, 1, 8192, "mixed"), (16, 3, 8191, "mixed"), (13, 4, 8200, "mixed"), (32, 3, 300, "mixed"),
])
def test_accept_in_draw(engine, B, k, V, kind):
    print(f"accept in draw B={B} k={k} V={V} {kind}", flush=True)
    p, q, drafts = make_inputs(B, k, V, seed=31)
    U = oracle_uniforms(31, B, k)
    cfg = O.SamplerCfg(0.8, 0, 1.0, 0.0)
    cd = drafts.copy()  # COMPARE: drafts equal to the target's samples, every third one not ("mixed")
    for b in range(B):
        for i in range(k):
            if kind == "all" or (b + i) % 3:
                cd[b, i] = O.sample_vocab_order(p[b, i], 0.8, float(U[b, i, 1]))
    rq = p[:, :k].copy() if kind == "all" else q  # REJECTION: q = p accepts every draft (u < 1)
    for _ in range(2):
        a, n = run_gpu(engine, p, q, cd, SH_SAMPLE_COMPARE, 0.8, seed=31)
        for b in range(B):
            em = O.sample_and_compare(p[b], cd[b], cfg, U[b, :, 1].copy(), mode=1)
            assert (a[b], n[b]) == (len(em) - 1, em[-1]), b
        if kind == "all":
            assert np.all(a == k)
        a, n = run_gpu(engine, p, rq, drafts, SH_SAMPLE_REJECTION, 0.8, seed=31)
        for b in range(B):
            want = O.rejection(p[b], rq[b], drafts[b], 0.8, U[b, :k, 0].copy(), U[b, :, 1].copy())
            assert (a[b], n[b]) == want, b
        if kind == "all":
            assert np.all(a == k)
