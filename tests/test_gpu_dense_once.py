"""GPU: the batch-1 product that asks for everything at once, and the staged one beside it, through decode steps of whole models against their
oracles.  Widths and feed-forwards at the edges of its pieces (512 bf16 or 256 fp32 columns a wavefront, 8 wavefronts behind a norm, 16 of one, two or
four pieces on a plain input), vocabularies for 2 to 16 rows a workgroup, norms in groups, merges of two to sixteen splits; test_dense_plan.py asks the plan which
forms these lists reach.  And that the library runs what the plan says, by the workgroups of a step."""
import pytest

import lebelix_cases as sided
import nusilix_cases as grouped
import test_gpu_lebelix as lebelix
import test_gpu_nusilix as nusilix
from oracle import lebelix_oracle, nusilix_oracle

pytestmark = pytest.mark.gpu
DTYPES = ["float32", "bfloat16"]


# width, feed-forward, vocabulary
WIDTHS = [(64, 64, 31), (256, 512, 1100), (257, 513, 300), (512, 1111, 2100), (1000, 255, 4200), (1000, 255, 960), (1030, 2049, 512), (96, 4097, 40),
          (72, 8193, 70), (96, 16384, 33), (40, 16385, 33), (2048, 300, 2600), (2064, 300, 40), (4096, 64, 64), (4160, 64, 40)]
# width, norm groups, vocabulary
GROUPS = [(64, 8, 70), (520, 5, 70), (1024, 2, 1000), (1024, 8, 3000), (1032, 3, 2600), (1040, 8, 70), (2048, 4, 2000), (2304, 6, 70), (144, 9, 70)]
# heads, key heads, elements of a head, width, tokens of context, splits of 32768 / (elements padded to 64, 128 or 256) tokens of the next power of two
MERGES = [(4, 2, 64, 192, 150, 1), (4, 2, 64, 192, 600, 2), (8, 8, 64, 192, 600, 2), (2, 1, 128, 192, 900, 4), (2, 1, 128, 1100, 900, 4), (6, 3, 20, 192, 600, 2),
          (33, 1, 128, 192, 300, 2), (1, 1, 256, 192, 900, 8), (1, 1, 256, 192, 1500, 16), (1, 1, 256, 1100, 1500, 16)]


# The head is behind a sum and a norm, as the input products of later layers are; the feed-forward's behind a norm; the down projection takes its input as it is.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,ff,vocab", WIDTHS)
def test_widths_and_feed_forwards(hip, width, ff, vocab, dtype):
    cfg = sided.model([sided.attention(2, 1, 16, 24, 8, 9, ff=ff), sided.delta(2, 1, 16, 16, ff=70), sided.latent(2, 16, 8, 16, 24, 7, ff=0)], width=width, vocab=vocab, side=min(width, 100))
    w = sided.weights(cfg, 8, 8, seed=width + ff)
    toks = sided.tokens(cfg, 5, seed=3)
    m = sided.device_model(hip, cfg, w, dtype)
    sided.check(lebelix.run(m, toks, [1] * 5), lebelix_oracle.forward(cfg, w, toks), dtype, (width, ff, vocab))
    m.free()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,groups,vocab", GROUPS)
def test_norms_in_groups(hip, width, groups, vocab, dtype):
    cfg = grouped.model([grouped.attention(2, 1, 16, ff=1300), grouped.delta(2, 24, ff=90)], width=width, vocab=vocab, groups=groups)
    w = grouped.weights(cfg, 4, seed=width)
    toks = grouped.tokens(cfg, 5, seed=2)
    m = grouped.device_model(hip, cfg, w, dtype)
    grouped.check(nusilix.run(m, toks, [1] * 5), nusilix_oracle.forward(cfg, w, toks), dtype, (width, groups))
    m.free()


# (heads of 20 elements are no whole requests of bf16 lanes; with 33 heads of 128 the merged input is more than eight wavefronts have)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,dim,width,context,splits", MERGES)
def test_merges_of_attention_splits(hip, heads, kv_heads, dim, width, context, splits, dtype):
    """An output product that merges the splits of its attention: with a sink and a gate (ranged attention), and with neither."""
    for cases, run, oracle, layer in ((sided, lebelix.run, lebelix_oracle, sided.attention(heads, kv_heads, dim, dim, 16, 4096, ff=64)),
                                      (grouped, nusilix.run, nusilix_oracle, grouped.attention(heads, kv_heads, dim, ff=1300))):
        cfg = cases.model([layer], width=width, vocab=50, **({"groups": 2} if cases is grouped else {}))
        w = cases.weights(cfg, 4, 4, seed=heads) if cases is sided else cases.weights(cfg, 4, seed=heads)
        toks = cases.tokens(cfg, context + 3, seed=4)
        m = cases.device_model(hip, cfg, w, dtype, max_tokens=1536)
        last = list(range(context, context + 3))
        cases.check(run(m, toks, [context, 1, 1, 1], want=last), oracle.forward(cfg, w, toks)[last], dtype, (heads, dim, context))
        m.free()


def _step_workgroups(hip, cases, cfg, dtype, context=1):
    """of a decode step's launches, counted while it is captured"""
    w = cases.weights(cfg, 4, 4) if cases is sided else cases.weights(cfg, 4)
    toks = cases.tokens(cfg, context + 1, seed=4)
    m = cases.device_model(hip, cfg, w, dtype, max_tokens=1536)
    if context > 1:
        m.extend(toks[:context], [])
    before = hip.stat("workgroups")
    m.extend(toks[context:], [])
    took = hip.stat("workgroups") - before
    m.free()
    return took


# Steps that differ in the head's rows alone, 8192 and 64: 8 rows a workgroup (16 in fp32 of 512 columns) and 2 of the kernel that asks for everything
# at once; the staged kernel has three workgroups a compute unit, and 8 rows each of 64.
@pytest.mark.parametrize("design,width,groups,dtype,more", [(grouped, 512, 2, "bfloat16", 1024 - 32), (grouped, 512, 2, "float32", 512 - 32), (grouped, 576, 9, "bfloat16", 768 - 8),
                                                            (sided, 512, 1, "bfloat16", 1024 - 32), (sided, 512, 1, "float32", 512 - 32), (sided, 4160, 1, "bfloat16", 768 - 8)])
def test_kernel_of_the_head(hip, design, width, groups, dtype, more):
    assert hip.device_info()["compute_units"] == 256, "the numbers are for 256 compute units"
    layer = grouped.attention(1, 1, 16, ff=0) if design is grouped else sided.attention(1, 1, 16, 16, 16, 64, ff=0)
    took = [_step_workgroups(hip, design, design.model([layer], width=width, vocab=vocab, **({"groups": groups} if design is grouped else {})), dtype) for vocab in (64, 8192)]
    assert took[1] - took[0] == more


# Steps that differ in the output product's rows alone, 960 and 1024: four rows a workgroup of the kernel that asks for everything at once, eight of the staged one
@pytest.mark.parametrize("heads,dim,dtype,more", [(2, 64, "bfloat16", 64 // 4), (2, 64, "float32", 64 // 4), (6, 20, "bfloat16", 64 // 8), (6, 20, "float32", 64 // 4),
                                                  (33, 128, "bfloat16", 64 // 8)])
def test_kernel_of_a_merge(hip, heads, dim, dtype, more):
    took = [_step_workgroups(hip, grouped, grouped.model([grouped.attention(heads, 1, dim, ff=0)], width=width, vocab=64, groups=2), dtype, context=600) for width in (960, 1024)]
    assert took[1] - took[0] == more


# the attention's workgroups of one key head are its splits
@pytest.mark.parametrize("design", [sided, grouped])
def test_number_of_splits(hip, design):
    layer = grouped.attention(1, 1, 256, ff=0) if design is grouped else sided.attention(1, 1, 256, 256, 16, 4096, ff=0)
    took = [_step_workgroups(hip, design, design.model([layer], width=192, vocab=64), "bfloat16", context) for context in (200, 400, 900, 1500)]
    assert [b - a for a, b in zip(took, took[1:])] == [2, 4, 8]
