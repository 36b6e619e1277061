"""GPU: the rounding of a prompt's rows behind a norm, pinned to the order in which a row's squares are added (two equal prompts of
different builds give the same bits, however many wavefronts a row has)."""
import numpy as np
import pytest

from oracle import oracle_np
from skainet_amd import llama, synth

pytestmark = pytest.mark.gpu
F32 = np.float32
EPS = 1e-5


def _inverse_rms(x, chains):
    """In fp32: tasks of four elements and four 32 further on; tasks u, u + chains, ... in turn; the lanes of 64 in pairs of pairs; the
    wavefronts in pairs."""
    k = x.size
    sq = (x * x).reshape(k // 64, 2, 8, 4)
    four = (sq[..., 0] + sq[..., 1]) + (sq[..., 2] + sq[..., 3])
    tasks = (four[:, 0] + four[:, 1]).reshape(-1)
    lanes = np.zeros(chains, F32)
    for u in range(chains):
        for v in tasks[u::chains]:
            lanes[u] += v
    at = np.arange(chains)
    for mirror in (1, 2, 7, 15):
        lanes = lanes + lanes[at ^ mirror]
    rows = lanes[::16]
    while rows.size > 1:
        rows = rows[0::2] + rows[1::2]
    return F32(1.0) / np.sqrt(rows[0] / F32(k) + F32(EPS), dtype=F32)


def _bf16(y):
    return oracle_np.bf16_to_f32(synth.f32_to_bf16_bits(y))


def _one_hot_q4k(rows, k, places):
    """[rows, k]: 1 at each (row, element) of places, 0 elsewhere."""
    w = np.zeros((rows, k // 256, 144), np.uint8)
    for row, e in places:
        block, i = w[row, e // 256], e % 256
        block[0:2] = np.array([1.0], np.float16).view(np.uint8)
        sub = i // 32
        block[4 + sub if sub < 4 else 8 + sub] |= 1  # (its scale: 1; the minima stay 0)
        block[16 + 32 * (sub // 2) + i % 32] |= 1 << (4 * (sub % 2))
    return w.reshape(-1)


def check_rounding(hip, hidden, tokens, max_tokens):
    """Norm weights for which one bit of the sum decides bf16 roundings, through a layer of one-hot matrices: values, attention over
    equal tokens, residual, head.  Elements of odd places in the rounding, others beside them as a measure."""
    rng, probes = np.random.default_rng(hidden), 32
    for _ in range(1000):  # (squares of eleven bits and their pairs are exact: only the order of the sums rounds)
        x = (rng.integers(256, 2048, hidden) * rng.choice([-1, 1], hidden) / 512).astype(F32)
        two, four = _inverse_rms(x, 128), _inverse_rms(x, 256)
        if two != four:
            break
    assert two != four
    at = rng.choice(hidden, probes, replace=False)
    g, decided = np.ones(hidden, F32), 0
    for j, e in enumerate(at):
        tries = (64 * (1 + rng.random(1 << 20))).astype(F32)
        here = _bf16(x[e] * two * tries) != _bf16(x[e] * four * tries)
        if j % 2 == 0 and here.any():
            g[e], decided = tries[np.argmax(here)], decided + 1
        else:
            g[e] = tries[np.argmin(here)]
    assert decided >= 8
    value = _bf16(x[at] * two * g[at])
    cfg = llama.Config(n_layer=1, hidden=hidden, ffn=256, n_head=hidden // 128, n_kv_head=1, head_dim=128, vocab=probes, max_tokens=max_tokens, page_tokens=16,
                       rms_eps=EPS, type_embd=0, type_head=0)
    ones, q4 = np.ones(hidden, F32), synth.Q4_K
    head = np.zeros((probes, hidden), F32)
    head[np.arange(probes), at] = 1.0
    square = np.zeros(hidden * hidden // 256 * 144, np.uint8)
    short = np.zeros(256 * hidden // 256 * 144, np.uint8)
    w = {"tok_embd": (0, np.tile(x, (probes, 1)).reshape(-1)), "out_head": (0, head.reshape(-1)), "out_norm": (None, ones), "l0.wq": (q4, square),
         "l0.wk": (q4, short[: short.size // 2]), "l0.wv": (q4, _one_hot_q4k(128, hidden, [(j, e) for j, e in enumerate(at)])),
         "l0.wo": (q4, _one_hot_q4k(hidden, hidden, [(e, j) for j, e in enumerate(at)])), "l0.w_gate": (q4, short), "l0.w_up": (q4, short), "l0.w_down": (q4, short),
         "l0.attn_norm": (None, g), "l0.ffn_norm": (None, ones)}
    model = llama.LlamaModel(hip, cfg, weights=w)
    model.prefill([0] * tokens)
    got = model.logits()
    model.free()
    y = x.astype(np.float64)
    y[at] += value
    want = y[at] / np.sqrt(np.mean(y * y) + EPS)
    # a rounding the other way moves its element by a part in 512 at least (and the norm, if all go that way, by half as much)
    assert np.all(np.abs(got - want) <= 2.0**-12 * np.abs(want)), np.abs(got / want - 1).max()


@pytest.mark.parametrize("hidden", [1280, 4096, 5120])
def test_rows_behind_a_norm_round_as_two_wavefronts_sum_them(hip, hidden):
    check_rounding(hip, hidden, tokens=2, max_tokens=16)
