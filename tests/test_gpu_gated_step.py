"""GPU: the gated delta rule's step in decoding, which asks for everything before it waits, against the oracle token by token: heads of every padded
size, value channels of one and of several turns, ranks at and past the two pieces of 64 that are asked for ahead, convolutions of one tap to
eight with fewer tokens behind them than taps and more."""
import pytest

import lebelix_cases as cases
import test_gpu_lebelix as lebelix
from oracle import lebelix_oracle

pytestmark = pytest.mark.gpu
DTYPES = ["float32", "bfloat16"]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,taps,rank,rank_gate", [(2, 1, 16, 24, 1, 1, 1), (2, 2, 32, 32, 2, 64, 65), (3, 3, 33, 70, 8, 129, 200),
                                                                         (4, 2, 64, 64, 4, 128, 130), (2, 1, 100, 128, 5, 300, 64), (1, 1, 128, 256, 8, 128, 128),
                                                                         (2, 2, 130, 40, 3, 64, 64), (1, 1, 256, 256, 4, 190, 70), (4, 1, 24, 256, 8, 20, 20)])
def test_steps(hip, heads, kv_heads, dim, vdim, taps, rank, rank_gate, dtype):
    cfg = cases.model([cases.delta(heads, kv_heads, dim, vdim, taps=taps, ff=40)], width=96, vocab=61, side=8)
    w = cases.weights(cfg, rank, rank_gate, seed=dim + vdim)
    toks = cases.tokens(cfg, 12, seed=taps)
    m = cases.device_model(hip, cfg, w, dtype)
    cases.check(lebelix.run(m, toks, [1] * 12), lebelix_oracle.forward(cfg, w, toks), dtype, (dim, vdim, taps))
    m.free()
