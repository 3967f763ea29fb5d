"""Greedy ids of a batched verify (k_argmax) against its own logits: both block
sizes, a last block of one logit, every column count that one launch takes, and
twice on one workspace (the kernel clears its keys and counters itself)."""
import dataclasses

import numpy as np
import pytest

from seeker_amd import synth as S

pytestmark = pytest.mark.gpu


# 8192-logit blocks from 512 workgroups on (32769 x 192: 960, 32000 x 128: 512), else 2048-logit ones
@pytest.mark.parametrize("vocab,lens", [(32769, [48, 48, 48, 48]), (32000, [64, 64]), (32000, [61, 64]),
                                        (4097, [41, 41, 41, 41]), (32769, [1]), (500, [3, 7])])
def test_argmax_of_every_column(engine, vocab, lens):
    shape = dataclasses.replace(S.TINY_TARGET, n_vocab=vocab)
    print(f"argmax vocab={vocab} columns={sum(lens)}", flush=True)
    with S.GgufImage(shape, seed=3) as img:
        gm = engine.upload_weights(img)
        for seed in (1, 2):
            caches = [engine.allocate_kv_cache(gm, 128) for _ in lens]
            out = engine.verify_unified(gm, caches, S.tokens(seed, sum(lens), vocab), lens, want_logits=True)
            assert np.array_equal(out.sampled, out.logits.argmax(axis=1))
            for c in caches:
                c.close()
        gm.close()
