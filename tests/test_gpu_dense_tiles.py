"""GPU: the 192-row tiles of the dense GEMM, through whole models against their oracles (a last tile of 300 tokens, widths that are no
multiple of 192, products with a side table), and where the library picks them itself."""
import pytest

import nusilix_cases as cases
import test_gpu_lebelix as lebelix
from oracle import nusilix_oracle as orc
from test_gpu_nusilix import DTYPES, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tile,tokens", [(6, 300), (6, 256), (7, 300), (7, 129)])
def test_tiles_of_192_weight_rows(hip, tile, tokens, dtype):
    cfg, rank = cases.MODELS["mixed"]
    w = cases.weights(cfg, rank)
    toks = cases.tokens(cfg, tokens, seed=5)
    want = orc.forward(cfg, w, toks)
    m = cases.device_model(hip, cfg, w, dtype)
    hip.set_option("dense.tile", tile)
    try:
        err = cases.logit_error(run(m, toks, [tokens]), want)
    finally:
        hip.set_option("dense.tile", 0)
    assert err.max() < cases.TOLERANCE[dtype]
    m.free()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tile", [6, 7])
def test_tiles_of_192_weight_rows_behind_a_side_table(hip, tile, dtype):
    lebelix.test_every_tile_of_the_gemm(hip, tile, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_the_library_picks_them_where_they_fill_their_last_round(hip, dtype):
    """An input projection of 13248 or 15360 rows and 536 tokens: three row tiles by 69 or 80 column tiles of 256 x 192 for 256 compute units,
    their number rounded up to whole turns of eight XCDs (128 x 128 tiles would be 520 and 600, 256 x 256 tiles 160 and 184)."""
    assert hip.device_info()["compute_units"] == 256, "the widths are chosen for 256 compute units"
    tokens, took = 536, []
    for ff in (13056, 13056 + 2112):
        cfg = cases.model([cases.attention(2, 2, 32, ff=ff)], width=64, vocab=31, groups=2)
        w = cases.weights(cfg, 1)
        toks = cases.tokens(cfg, tokens, seed=5)
        m = cases.device_model(hip, cfg, w, dtype, max_tokens=tokens)
        m.extend(toks, [tokens - 1])
        m.reset()
        before = hip.stat("workgroups")
        got = m.extend(toks, [tokens - 1])
        took.append(hip.stat("workgroups") - before)
        assert cases.logit_error(got, orc.forward(cfg, w, toks)[-1:]).max() < cases.TOLERANCE[dtype]
        m.free()
    assert took[1] - took[0] == 240 - 208
