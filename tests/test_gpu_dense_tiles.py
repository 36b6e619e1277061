"""GPU: the 192-row tiles of the dense GEMM, through a whole model against its oracle (a last tile of 300 tokens, widths that are no
multiple of 192)."""
import pytest

import nusilix_cases as cases
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
