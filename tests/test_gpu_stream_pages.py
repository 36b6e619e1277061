"""GPU: attention over ranges, latents and shared caches of more pages than ride in a register, in portions and token by token."""
import pytest

import lebelix_cases as cases
import nusilix_cases
import test_gpu_lebelix as lebelix
import test_gpu_nusilix as nusilix
from oracle import lebelix_oracle, nusilix_oracle

pytestmark = pytest.mark.gpu
DTYPES = ["float32", "bfloat16"]


# pages of sixteen tokens: 1100 tokens are more than 64 pages, in whole rounds of requests and not
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tokens", [1023, 1100])
def test_more_pages_than_ride_in_a_register(hip, tokens, dtype):
    cfg = cases.model([cases.attention(2, 1, 32, 32, 16, 5000, ff=0), cases.latent(2, 24, 8, 16, 40, 5000, ff=0)], width=64, vocab=61, side=8)
    w = cases.weights(cfg, 1, 1, seed=3)
    toks = cases.tokens(cfg, tokens, seed=4)
    m = cases.device_model(hip, cfg, w, dtype, max_tokens=tokens, page_tokens=16)
    cases.check(lebelix.run(m, toks, [tokens - 3, 1, 1, 1]), lebelix_oracle.forward(cfg, w, toks), dtype, tokens)
    m.free()
    cfg = nusilix_cases.model([nusilix_cases.attention(2, 1, 32, ff=40)], width=64, vocab=61, groups=2)
    w = nusilix_cases.weights(cfg, 1)
    m = nusilix_cases.device_model(hip, cfg, w, dtype, max_tokens=tokens, page_tokens=16)
    nusilix_cases.check(nusilix.run(m, toks, [tokens - 3, 1, 1, 1]), nusilix_oracle.forward(cfg, w, toks), dtype, tokens)
    m.free()
