"""GPU: the preparation pass of the Q4_K and Q6_K products with four rows a workgroup (512 rows and more), against the one with two rows: the same bits
of every row; and behind a norm, whose squares are added in the order of fewer rows."""
import numpy as np
import pytest

import test_gpu_prompt_norm as prompt_norm
from oracle import oracle_c, oracle_np
from skainet_amd import synth

pytestmark = pytest.mark.gpu
Q4_K, Q6_K = synth.Q4_K, synth.Q6_K


# rows at the edges of quads and row blocks; elements at the edges of what a thread holds, and on either side of what four rows a workgroup take
@pytest.mark.parametrize("m", [512, 515, 1000])
@pytest.mark.parametrize("k", [256, 768, 1024, 2048, 2304, 4096, 4352, 8192, 8448, 12288, 12544])
def test_rows_do_not_depend_on_how_many_a_workgroup_has(hip, m, k):
    n = 40
    raw, a = synth.weight(Q4_K, n, k, seed=k), synth.activation_bf16((m, k), seed=m)
    hip.set_option("gemm.tile", 2)  # (128-row tiles with k undivided: a row's sums are the same whatever the rows beside it)
    hip.set_option("gemm.split", 1)
    hip.set_option("gemm.few", 0)
    try:
        before = hip.stat("workgroups")
        got = hip.gemm_q_host(Q4_K, raw, n, k, a, m)
        took = hip.stat("workgroups") - before
        want = np.concatenate([hip.gemm_q_host(Q4_K, raw, n, k, np.ascontiguousarray(a[i:i + 256]), len(a[i:i + 256])) for i in range(0, m, 256)])
    finally:
        hip.set_option("gemm.tile", 0)
        hip.set_option("gemm.split", 0)
        hip.set_option("gemm.few", 1)
    rows = -(-m // 128) * 128
    assert took == rows // (4 if 1024 <= k <= 12288 else 2) + rows // 128  # (the pass and the tiles)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert oracle_np.rel_err(hip.gemm_q_host(Q6_K, synth.weight(Q6_K, n, k, seed=k), n, k, a, m), oracle_c.gemm_q(Q6_K, synth.weight(Q6_K, n, k, seed=k), n, k, a, m)) <= 1e-3


@pytest.mark.parametrize("hidden", [1280, 4096])
def test_rows_behind_a_norm_round_as_few_rows_do(hip, hidden):
    prompt_norm.check_rounding(hip, hidden, tokens=1000, max_tokens=1008)
