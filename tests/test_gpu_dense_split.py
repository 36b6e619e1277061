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


# 2048 columns of output from 4160 of input: one round of 128 x 128 tiles for 2048 tokens, half of one for 1000, few outputs for 100
@pytest.mark.parametrize("tokens", [100, 1000, 2048])
def test_what_the_library_picks_agrees_with_the_smallest_tiles(hip, tokens):
    cfg = cases.model([cases.attention(1, 1, 64, ff=4096)], width=2048, vocab=31, groups=2)
    w = cases.weights(cfg, 1)
    toks = cases.tokens(cfg, tokens, seed=5)
    m = cases.device_model(hip, cfg, w, "bfloat16", max_tokens=2048)
    got = {}
    for tile in (0, 1):
        hip.set_option("dense.tile", tile)
        try:
            m.reset()
            got[tile] = m.extend(toks, [tokens - 1])
        finally:
            hip.set_option("dense.tile", 0)
    m.free()
    assert cases.logit_error(got[0], got[1]).max() < cases.TOLERANCE["bfloat16"] / 4
