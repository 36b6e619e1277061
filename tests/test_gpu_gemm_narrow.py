"""GPU: Q4_K products on 256 x 96 tiles (a matrix's columns in blocks of 32, the blocks of a launch's matrices one after the other, three to a
tile) against the 256 x 128 tiles of the same kernel, whose arithmetic and order per element they share: the same bits."""
import numpy as np
import pytest

import test_gpu_llama_conditioned as conditioned
from oracle import oracle_c, oracle_np
from skainet_amd import llama, synth

pytestmark = pytest.mark.gpu
Q4_K = synth.Q4_K
TOL = 1e-3


def _with_tile(hip, tile, call):
    hip.set_option("gemm.tile", tile)
    try:
        return call()
    finally:
        hip.set_option("gemm.tile", 0)


# columns at the edges of blocks and tiles; one superblock, two, and a number that three buffers do not divide; rows at the edges of a tile and its
# consumers' 64
@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (63, 31, 512), (65, 33, 256), (256, 96, 768), (257, 97, 1024), (300, 95, 2816), (200, 128, 512), (512, 288, 4096),
                                   (130, 320, 11008)])
def test_tiles_of_96_columns_equal_those_of_128(hip, m, n, k):
    raw, a = synth.weight(Q4_K, n, k, seed=n + k), synth.activation_bf16((m, k), seed=m)
    hip.set_option("gemm.split", 1)  # (k of a tile undivided in both)
    try:
        wide, narrow = (_with_tile(hip, t, lambda: hip.gemm_q_host(Q4_K, raw, n, k, a, m)) for t in (3, 4))
    finally:
        hip.set_option("gemm.split", 0)
    assert np.array_equal(wide.view(np.uint32), narrow.view(np.uint32))
    assert oracle_np.rel_err(narrow, oracle_c.gemm_q(Q4_K, raw, n, k, a, m)) <= TOL


@pytest.mark.parametrize("case", ["q4_k", "q4_k_kv2", "q4_k_kv1", "mixed"])
def test_tiles_that_hold_the_columns_of_two_and_three_matrices(hip, case):
    """q, k and v in one launch (512, 256 or 128 columns of k and v: tiles that end in another matrix's columns), residuals added by the store."""
    cfg = conditioned.CASES[case]
    prompt, first, _, _ = conditioned._oracle_prompt(case, 41, 12)

    def logits():
        model = llama.LlamaModel(hip, cfg, weights=llama.conditioned_weights(cfg, conditioned.SEED))
        model.prefill(prompt)
        out = model.logits()
        model.free()
        return out

    assert conditioned.logit_err(_with_tile(hip, 4, logits), first) <= conditioned.PROMPT_TOL


# Tiles of 256 x 128 and of 256 x 96 for 256 compute units: 192 and 256, one round each; 194 and 258, one and two; 352 and 472, two each (short rows, whose last
# tiles are not shared); 388 and 516, two and three; 564 and 750, three each; 1288 and 1720, six and seven.
@pytest.mark.parametrize("m,n,k,narrow", [(512, 12288, 256, True), (512, 12288 + 32, 256, False), (1024, 11264, 1024, True), (1024, 12288 + 32, 512, False), (768, 24000, 512, True),
                                          (2048, 20608, 256, True)])
def test_where_the_library_picks_them(hip, m, n, k, narrow):
    assert hip.device_info()["compute_units"] == 256, "the widths are chosen for 256 compute units"
    raw, a = synth.weight(Q4_K, n, k, seed=5), synth.activation_bf16((m, k), seed=6)

    def product(tile):
        before = hip.stat("workgroups")
        got = _with_tile(hip, tile, lambda: hip.gemm_q_host(Q4_K, raw, n, k, a, m))
        return got, hip.stat("workgroups") - before

    (got, took), (wide, wide_took), (_, narrow_took) = product(0), product(3), product(4)
    assert narrow_took - wide_took == -(-m // 256) * (-(-n // 96) - -(-n // 128))
    assert took == (narrow_took if narrow else wide_took)
    assert np.array_equal(wide.view(np.uint32), got.view(np.uint32))
