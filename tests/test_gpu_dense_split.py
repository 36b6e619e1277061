"""GPU: 128 x 128 tiles of the dense GEMM whose slices two groups of wavefronts share, through whole models against their oracles (even and odd
numbers of slices, one slice, last tiles of 300, 129 and 1 tokens), and where the library picks them."""
import pytest

import nusilix_cases as cases
import test_gpu_dense_tiles as tiles
import test_gpu_lebelix as lebelix

pytestmark = pytest.mark.gpu
DTYPES = tiles.DTYPES


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tokens", [1, 129, 256, 300])
def test_tiles_with_shared_slices(hip, tokens, dtype):
    tiles.test_tiles_of_192_weight_rows(hip, 8, tokens, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_tiles_with_shared_slices_behind_a_side_table(hip, dtype):
    lebelix.test_every_tile_of_the_gemm(hip, 8, dtype)


# 2048 columns of output from 4160 of input: one round of 128 x 128 tiles with shared slices for 2048 tokens, 128 x 64 tiles for 1000, 32 x 64 with k in four for 100;
# 4224 columns from 2048: 256 x 192, 128 x 128 and 64 x 64 (test_dense_plan.py has these choices).  The head is one tile in each.  more: workgroups beside 64 x 64 tiles
@pytest.mark.parametrize("tokens,more", [(100, 4 * 32 - 2 * 32), (1000, 8 * 33 + 8 * 32 - 16 * 66 - 16 * 32), (2048, 8 * 22 + 16 * 16 - 32 * 66 - 32 * 32)])
def test_what_the_library_picks_agrees_with_the_smallest_tiles(hip, tokens, more):
    assert hip.device_info()["compute_units"] == 256, "the numbers are for 256 compute units"
    cfg = cases.model([cases.attention(1, 1, 64, ff=4096)], width=2048, vocab=31, groups=2)
    w = cases.weights(cfg, 1)
    toks = cases.tokens(cfg, tokens, seed=5)
    m = cases.device_model(hip, cfg, w, "bfloat16", max_tokens=2048)
    got, took = {}, {}
    for tile in (0, 1):
        hip.set_option("dense.tile", tile)
        try:
            m.reset()
            before = hip.stat("workgroups")
            got[tile] = m.extend(toks, [tokens - 1])
            took[tile] = hip.stat("workgroups") - before
        finally:
            hip.set_option("dense.tile", 0)
    m.free()
    assert cases.logit_error(got[0], got[1]).max() < cases.TOLERANCE["bfloat16"] / 4
    assert took[0] - took[1] == more
