"""GPU parity of the prompt GEMM that unpacks formats in blocks of 32 itself, against the oracle."""
import numpy as np
import pytest

from oracle import oracle_c, oracle_np
from skainet_amd import synth

pytestmark = pytest.mark.gpu
FORMATS = {"q8_0": synth.Q8_0, "q4_0": synth.Q4_0, "q4_1": synth.Q4_1, "q5_0": synth.Q5_0, "q5_1": synth.Q5_1, "q5_k": synth.Q5_K}
# fp32 sums of exact products: 2^-24 per addition, of which a chain has k / 4 / 32 blocks of two; 1e-5 of the largest output holds
# for k = 16384, and the floor of the metric is a thousandth of that output
TOL = 1e-3


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (32, 64, 256), (33, 65, 512), (64, 63, 1280), (65, 100, 768), (128, 130, 2816), (129, 64, 1024), (3, 600, 16384)])
def test_every_tile_height_and_remainder(hip, name, m, n, k):
    """One row and column to ragged tiles of 32 and 64 rows; fewer superblocks than a workgroup has k-parts, unequal
    parts, and the longest row the path takes; with k divided over workgroups as the library chooses, not at all, in unequal
    parts and superblock by superblock."""
    t = FORMATS[name]
    raw = synth.weight(t, n, k, seed=n + k + t)
    a = synth.activation_bf16((m, k), seed=m + 1)
    want = oracle_c.gemm_q(t, raw, n, k, a, m)
    for splits in (0, 1, 3, 64):
        hip.set_option("gemm.split", splits)
        try:
            got = hip.gemm_q_host(t, raw, n, k, a, m)
        finally:
            hip.set_option("gemm.split", 0)
        err = oracle_np.rel_err(got, want)
        assert err <= TOL, f"{splits} parts: rel err {err}"


@pytest.mark.parametrize("name", list(FORMATS))
def test_whole_range_of_fields_and_rows_far_apart(hip, name):
    """Random bytes in every field but the scales (zero, subnormal and of both signs among them), rows of 1e6 beside rows of
    1e-6 and a row of zeros."""
    t = FORMATS[name]
    m, n, k = 70, 96, 1024
    be, bb = synth.BLOCK[t]
    rng = np.random.default_rng(t)
    raw = rng.integers(0, 256, (n * k // be, bb), dtype=np.uint8)
    d = (rng.standard_normal(len(raw)) * 0.01).astype(np.float16)
    d[::5], d[3::11] = 0.0, np.float16(6e-8)
    raw[:, 0:2] = d.view(np.uint8).reshape(-1, 2)
    if name in ("q4_1", "q5_1", "q5_k"):
        raw[:, 2:4] = (rng.standard_normal(len(raw)) * 0.02).astype(np.float16).view(np.uint8).reshape(-1, 2)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0] *= 1e6
    x[1] *= 1e-6
    x[2] = 0.0
    a = synth.f32_to_bf16_bits(x)
    got = hip.gemm_q_host(t, raw.reshape(-1), n, k, a, m)
    want = oracle_c.gemm_q(t, raw.reshape(-1), n, k, a, m)
    for r in range(m):
        assert oracle_np.rel_err(got[r], want[r]) <= TOL if np.any(want[r]) else not np.any(got[r]), r


def test_weights_off_the_16_byte_grid_take_the_general_path(hip):
    m, n, k = 5, 70, 512
    raw = synth.weight(synth.Q8_0, n, k, seed=4)
    buf = hip.alloc(raw.nbytes + 16)
    buf.upload(raw, offset=2)
    a = synth.activation_bf16((m, k), seed=5)
    c = hip.alloc(4 * m * n)
    hip.gemm_q(synth.Q8_0, buf.ptr + 2, n, k, hip.to_device(a), m, c)
    got = c.download(np.float32, m * n).reshape(m, n)
    assert oracle_np.rel_err(got, oracle_c.gemm_q(synth.Q8_0, raw, n, k, a, m)) <= TOL


@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (32, 64, 256), (32, 65, 512), (17, 63, 1280), (31, 130, 2816), (3, 600, 16384)])
def test_q4_k_of_up_to_32_rows(hip, m, n, k):
    """Few rows of Q4_K take the same kernel: divisions of k as above, no row or column of a tile left over or missing."""
    raw = synth.weight(synth.Q4_K, n, k, seed=n + k)
    a = synth.activation_bf16((m, k), seed=m + 1)
    want = oracle_c.gemm_q(synth.Q4_K, raw, n, k, a, m)
    for splits in (0, 1, 3, 64):
        hip.set_option("gemm.split", splits)
        try:
            got = hip.gemm_q_host(synth.Q4_K, raw, n, k, a, m)
        finally:
            hip.set_option("gemm.split", 0)
        err = oracle_np.rel_err(got, want)
        assert err <= TOL, f"{splits} parts: rel err {err}"


@pytest.mark.parametrize("name,t", [("q4_k", synth.Q4_K), ("q5_k", synth.Q5_K)])
def test_superblock_scales_far_apart(hip, name, t):
    """d and dmin zero, negative, subnormal, from 2^-20 to 2^20 of each other and of the next superblock's, up to 32 rows (rows of
    1e6, of 1e-6 and of zeros among them): each block's sum joins the total in fp32 with its own scale."""
    m, n, k = 20, 64, 4096
    nb = k // 256
    rng = np.random.default_rng(92)
    raw = synth.weight(t, n, k, seed=91).reshape(n, nb, -1).copy()
    cases = [(0.0, 0.01), (0.0, 0.0), (-0.02, 0.01), (0.02, -0.01), (0.01, 0.0), (6e-8, 1e-7), (1e-5, 10.0), (1e-6, 1.0), (10.0, 1e-5), (500.0, 0.5),
             (3e-5, 0.03), (0.03, 3e-5), (-1e-4, -20.0), (2e-7, 0.2)]
    for col in range(n):
        for sb in range(nb):
            d = np.array(cases[rng.integers(len(cases))] if col < 48 else cases[(col + sb) % len(cases)], dtype=np.float16)
            raw[col, sb, 0:4] = d.view(np.uint8)
    raw[49, :, 0:2] = 0  # a column with no live superblock but its minima
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0] *= 1e6
    x[1] *= 1e-6
    x[2] = 0.0
    a = synth.f32_to_bf16_bits(x)
    got = hip.gemm_q_host(t, raw.reshape(-1), n, k, a, m)
    want = oracle_c.gemm_q(t, raw.reshape(-1), n, k, a, m)
    assert np.all(np.isfinite(got)) and not np.any(got[2])
    for r in (0, 1):
        for col in range(n):
            # a product of fp32 sums of exact terms: 2^-24 per addition of a chain of 2 * 128 of them and of the minima's sixteen, relative to
            # the sum of the terms' magnitudes
            w = oracle_c.dequant(t, raw[col].reshape(-1)).astype(np.float64)
            size = np.sum(np.abs(w) * np.abs(oracle_np.bf16_to_f32(a).reshape(m, k)[r]))
            assert abs(got[r, col] - want[r, col]) <= 300 * 2.0**-24 * size + 1e-30, (r, col)
    for col in range(n):
        assert oracle_np.rel_err(got[3:, col], want[3:, col]) <= TOL, col


@pytest.mark.parametrize("name,m,n,k,direct", [("q5_1", 1400, 70, 512, True), ("q5_1", 1401, 70, 512, False), ("q4_1", 1850, 2560, 4096, True),
                                               ("q4_1", 1851, 2560, 4096, False), ("q4_1", 1851, 2559, 4096, True), ("q4_1", 1851, 2560, 3840, True),
                                               ("q4_1", 3300, 2560, 4096, False), ("q4_1", 3301, 2560, 4096, True), ("q5_0", 2000, 2560, 4096, True)])
def test_many_rows_of_the_formats_that_unpack_slowest_take_the_weight_pass(hip, name, m, n, k, direct):
    """Preparation and product where the kernel unpacks the blocks itself, a pass over the weights more where many rows share it; either
    against the oracle, first and last rows, sampled columns."""
    t = FORMATS[name]
    raw, a = synth.weight(t, n, k, seed=n), synth.activation_bf16((m, k), seed=m)
    w, x, c = hip.to_device(raw), hip.to_device(a), hip.alloc(4 * m * n)
    hip.memset(c, 0xFF, 4 * m * n)
    before = hip.stat("launches")
    hip.gemm_q(t, w, n, k, x, m, c)
    assert hip.stat("launches") - before == (2 if direct else 3)
    got = c.download(np.float32, m * n).reshape(m, n)
    assert np.all(np.isfinite(got))
    cols = np.unique(np.concatenate([np.arange(0, n, 97), [n - 1]]))
    rows = np.concatenate([np.arange(8), np.arange(m - 70, m)])
    want = oracle_c.gemm_q(t, raw.reshape(n, -1)[cols].reshape(-1), len(cols), k, a.reshape(m, k)[rows], len(rows))
    assert oracle_np.rel_err(got[np.ix_(rows, cols)], want) <= TOL


def test_long_prompt_of_a_format_that_unpacks_slowest(hip):
    """A prompt keeps the direct products of Q5_1 up to 1800 rows and for short rows; the others' results agree with them to the rounding
    of the activations that a prompt's passes do one by one."""
    from skainet_amd import llama

    cfg = llama.Config(n_layer=1, hidden=512, ffn=4096, n_head=4, head_dim=128, vocab=256, max_tokens=1824, page_tokens=32, type_embd=synth.Q6_K,
                       matrix_types={w: synth.Q5_1 for w in ("wq", "wk", "wv", "wo", "w_gate", "w_up", "w_down")})
    model = llama.LlamaModel(hip, cfg, weights=llama.random_weights(cfg, seed=11))
    ids = np.random.default_rng(3).integers(0, cfg.vocab, 1801).tolist()
    took, logits = [], []
    for tokens, fused in ((1800, 1), (1801, 1), (1801, 0)):
        hip.set_option("gemm.q6k_fused", fused)
        try:
            model.reset()
            before = hip.stat("launches")
            model.prefill(ids[:tokens])
            took.append(hip.stat("launches") - before)
            logits.append(model.logits())
        finally:
            hip.set_option("gemm.q6k_fused", 1)
    # the down projection alone has rows of 4096: a conversion, three launches and an addition instead of a preparation and a product
    assert took[1] - took[0] == 3
    assert np.abs(logits[1] - logits[2]).max() <= 5e-3 * np.abs(logits[2]).max()
    model.free()
