"""GPU: the batch-1 product that asks for everything at once, and the staged one beside it, through decode steps of whole models against their
oracles.  Widths and feed-forwards at the edges of its pieces (512 bf16 or 256 fp32 columns a wavefront, 8 wavefronts behind a norm, 16 of one, two or
four pieces on a plain input), vocabularies for 2 to 16 rows a workgroup, norms in groups, merges of two to sixteen splits."""
import numpy as np
import pytest

import lebelix_cases as sided
import nusilix_cases as grouped
import test_gpu_lebelix as lebelix
import test_gpu_nusilix as nusilix
from oracle import lebelix_oracle, nusilix_oracle

pytestmark = pytest.mark.gpu
DTYPES = ["float32", "bfloat16"]


# The head is behind a norm of one group, the input products of later layers behind a sum and a norm, the down projection takes its input as it is.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,ff,vocab", [(64, 64, 31), (256, 512, 1100), (257, 513, 300), (512, 1111, 2100), (1000, 255, 4200), (1030, 2049, 512), (96, 4097, 40),
                                            (72, 8193, 70), (96, 16384, 33), (40, 16385, 33), (2048, 300, 2600), (2064, 300, 40), (4096, 64, 64), (4160, 64, 40)])
def test_widths_and_feed_forwards(hip, width, ff, vocab, dtype):
    cfg = sided.model([sided.attention(2, 1, 16, 24, 8, 9, ff=ff), sided.delta(2, 1, 16, 16, ff=70), sided.latent(2, 16, 8, 16, 24, 7, ff=0)], width=width, vocab=vocab, side=min(width, 100))
    w = sided.weights(cfg, 8, 8, seed=width + ff)
    toks = sided.tokens(cfg, 5, seed=3)
    m = sided.device_model(hip, cfg, w, dtype)
    sided.check(lebelix.run(m, toks, [1] * 5), lebelix_oracle.forward(cfg, w, toks), dtype, (width, ff, vocab))
    m.free()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,groups", [(64, 8), (520, 5), (1024, 2), (1024, 8), (1032, 3), (1040, 8), (2048, 4), (2304, 6), (144, 9)])
def test_norms_in_groups(hip, width, groups, dtype):
    cfg = grouped.model([grouped.attention(2, 1, 16, ff=1300), grouped.delta(2, 24, ff=90)], width=width, vocab=70, groups=groups)
    w = grouped.weights(cfg, 4, seed=width)
    toks = grouped.tokens(cfg, 5, seed=2)
    m = grouped.device_model(hip, cfg, w, dtype)
    grouped.check(nusilix.run(m, toks, [1] * 5), nusilix_oracle.forward(cfg, w, toks), dtype, (width, groups))
    m.free()


# (heads of 20 elements are no whole requests of bf16 lanes; with 33 heads of 128 the merged input is more than eight wavefronts have)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,dim,context", [(4, 2, 64, 150), (8, 8, 64, 500), (2, 1, 128, 900), (6, 3, 20, 500), (33, 1, 128, 300), (1, 1, 256, 900)])
def test_merges_of_attention_splits(hip, heads, kv_heads, dim, context, dtype):
    """An output product that merges the splits of its attention: with a sink and a gate (ranged attention), and with neither."""
    for cases, run, oracle, layer in ((sided, lebelix.run, lebelix_oracle, sided.attention(heads, kv_heads, dim, dim, 16, 4096, ff=64)),
                                      (grouped, nusilix.run, nusilix_oracle, grouped.attention(heads, kv_heads, dim, ff=1300))):
        cfg = cases.model([layer], width=192, vocab=50)
        w = cases.weights(cfg, 4, 4, seed=heads) if cases is sided else cases.weights(cfg, 4, seed=heads)
        toks = cases.tokens(cfg, context + 3, seed=4)
        m = cases.device_model(hip, cfg, w, dtype, max_tokens=1024)
        last = list(range(context, context + 3))
        cases.check(run(m, toks, [context, 1, 1, 1], want=last), oracle.forward(cfg, w, toks)[last], dtype, (heads, dim, context))
        m.free()
