"""GPU parity of the product of formats in blocks of 32 on 96-row tiles, against the oracle."""
import pytest

from oracle import oracle_c, oracle_np
from skainet_amd import synth

pytestmark = pytest.mark.gpu
FORMATS = {"q8_0": synth.Q8_0, "q4_0": synth.Q4_0, "q4_1": synth.Q4_1, "q5_0": synth.Q5_0, "q5_1": synth.Q5_1, "q5_k": synth.Q5_K}
# fp32 sums of exact products: 2^-24 per addition, of which a chain has k / 4 / 32 blocks of two; 1e-5 of the largest output holds
# for k = 16384, and the floor of the metric is a thousandth of that output
TOL = 1e-3


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("m,n,k", [(65, 16321, 256), (96, 8250, 1280), (289, 4090, 1024), (200, 5000, 768), (1250, 700, 2304)])
def test_tiles_of_96_rows(hip, name, m, n, k):
    """One to fourteen tiles of 96 rows with 1 to 96 of them in the last and 1 to 64 columns; as many superblocks as pairs of wavefronts,
    fewer, and a remainder.  All are sizes that 64-row tiles would take more than one round of 256 compute units for: those, with
    \"gemm.split\" set, give the same to the tolerance."""
    assert hip.device_info()["compute_units"] == 256, "the shapes are chosen for 256 compute units"
    t = FORMATS[name]
    raw = synth.weight(t, n, k, seed=n + k + t)
    a = synth.activation_bf16((m, k), seed=m + 1)
    want = oracle_c.gemm_q(t, raw, n, k, a, m)
    for splits in (0, 1):
        hip.set_option("gemm.split", splits)
        try:
            got = hip.gemm_q_host(t, raw, n, k, a, m)
        finally:
            hip.set_option("gemm.split", 0)
        err = oracle_np.rel_err(got, want)
        assert err <= TOL, f"{splits}: rel err {err}"
