"""GPU parity of the product of formats in blocks of 32 on 96-row tiles, against the oracle.  The option "gemm.few" is off: at some of the
sizes skn_gemm_q would take the path for few rows, which prompts do not."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle_c, oracle_np
from skainet_amd import synth

pytestmark = pytest.mark.gpu
FORMATS = {"q8_0": synth.Q8_0, "q4_0": synth.Q4_0, "q4_1": synth.Q4_1, "q5_0": synth.Q5_0, "q5_1": synth.Q5_1, "q5_k": synth.Q5_K}
MINIMA = ("q4_1", "q5_1", "q5_k")
BF16, F32, RMSNORM = 0, 1, 2


@pytest.fixture
def passes(hip):
    assert hip.device_info()["compute_units"] == 256, "the shapes are chosen for 256 compute units"
    hip.set_option("gemm.few", 0)
    yield hip
    hip.set_option("gemm.few", 1)
    hip.set_option("gemm.split", 0)


def grid(m, n, rows):
    """Workgroups of a product: its 64-column tiles go out in groups of eight."""
    return -(-n // 512) * 8 * -(-m // rows)


def weights(name, n, k, seed):
    raw = synth.weight(FORMATS[name], n, k, seed=seed)
    return raw, oracle_c.dequant(FORMATS[name], raw, n * k).reshape(n, k)


def bf16(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32)


def bound(name, w, a):
    """Of |result - exact| per output: the products of a block are exact, the matrix core adds 32 of them in fp32, a chain of k / 128 blocks and
    three parts follow, and the minima come as pairs of 22 bits -- each addition at most 2^-24 of the sum of magnitudes.  That is |a| |w|; a
    format with minima adds the scaled quants and the minimum of a block apart, each up to four times its largest element."""
    k = w.shape[1]
    size = np.abs(w)
    if name in MINIMA:
        size = np.repeat(4 * size.reshape(len(w), -1, 32).max(2), 32, axis=1)
    return (k // 128 + 48) * 2.0**-24 * (np.abs(a) @ size.T).astype(np.float64)


def check(name, got, want, w, a):
    over = np.abs(got.astype(np.float64) - want) - bound(name, w, a)
    assert np.max(over) <= 0, f"off by {np.max(over)} more than the bound at {np.unravel_index(np.argmax(over), over.shape)}"


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("m,n,k", [(65, 16321, 256), (96, 8250, 1280), (289, 4090, 1024), (200, 5000, 768), (1250, 700, 2304)])
def test_tiles_of_96_rows(passes, name, m, n, k):
    """One to fourteen tiles of 96 rows with 1 to 96 of them in the last, some past the rows that the operands are padded to, and 1 to 64
    columns; as many superblocks as pairs of wavefronts, fewer, and a remainder.  All are sizes that 64-row tiles would take more than one
    round of 256 compute units for: those come with "gemm.split" set."""
    t = FORMATS[name]
    raw, w = weights(name, n, k, n + k + t)
    a = synth.activation_bf16((m, k), seed=m + 1)
    want = oracle_c.gemm_q(t, raw, n, k, a, m).reshape(m, n)
    for splits, rows in ((0, 96), (1, 64)):
        passes.set_option("gemm.split", splits)
        before = passes.stat("workgroups")
        got = passes.gemm_q_host(t, raw, n, k, a, m).reshape(m, n)
        assert passes.stat("workgroups") - before == -(-m // 64) * 64 + grid(m, n, rows), "another kernel than meant"
        assert oracle_np.rel_err(got, want) <= 1e-3  # (the bar of the other products)
        check(name, got, bf16(a).astype(np.float64) @ w.T.astype(np.float64), w, bf16(a))


class Seg(C.Structure):  # skn_gemm_seg
    _fields_ = [("w", C.c_void_p), ("n", C.c_int), ("c", C.c_void_p), ("accumulate", C.c_int)]


class Src(C.Structure):  # skn_gemm_src
    _fields_ = [("kind", C.c_int), ("a", C.c_void_p), ("b", C.c_void_p), ("eps", C.c_float), ("ahead", C.c_bool)]


def blocks_multi(ctx, types, segs, k, src, m):
    """skn_gemm_blocks_multi, which decoders' prompts call."""
    fn = ctx.lib._Z21skn_gemm_blocks_multiP7skn_ctxPKiPK12skn_gemm_segiiRK12skn_gemm_srci
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p, C.POINTER(C.c_int), C.POINTER(Seg), C.c_int, C.c_int, C.POINTER(Src), C.c_int]
    ctx._check(fn(ctx.handle, (C.c_int * len(types))(*types), (Seg * len(segs))(*segs), len(segs), k, C.byref(src), m))


def source(to_device, kind, m, k):
    """-> (the source, the bf16 rows it stands for).  The normed rows are a power of two each, so that their mean square and its root are exact and
    the norm has one rounding only, that to bf16."""
    rng = np.random.default_rng(m + k + kind)
    if kind == BF16:
        bits = synth.activation_bf16((m, k), seed=m)
        return Src(BF16, to_device(bits).ptr, None, 0.0, False), bits
    x, g = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal(k).astype(np.float32)
    if kind == F32:
        return Src(F32, to_device(x).ptr, None, 0.0, False), synth.f32_to_bf16_bits(x)
    sign = np.where(x < 0, np.float32(-1), np.float32(1))
    rows = sign * np.ldexp(np.float32(1), rng.integers(-8, 8, (m, 1))).astype(np.float32)
    return Src(RMSNORM, to_device(rows).ptr, to_device(g).ptr, 0.0, False), synth.f32_to_bf16_bits(sign * g)


@pytest.mark.parametrize("kind", [BF16, F32, RMSNORM])
def test_several_matrices_and_sources(passes, kind):
    """One call whose matrices take 96-row tiles, divided k on 64-row tiles and whole 64-row tiles, all from one preparation of rows that the two
    heights pad differently; the first and the second added to what is there."""
    m, k = 200, 1536
    keep = []  # (buffers live until the results are there)

    def to_device(x):
        keep.append(passes.to_device(x))
        return keep[-1]

    src, bits = source(to_device, kind, m, k)
    a = bf16(bits)
    mats = [("q5_k", 5000, 1), ("q8_0", 700, 1), ("q4_1", 6000, 0)]
    segs, outs, olds = [], [], []
    for i, (name, n, acc) in enumerate(mats):
        raw, w = weights(name, n, k, 7 * i + 1)
        old = np.random.default_rng(i).standard_normal((m, n)).astype(np.float32)
        c = to_device(old)
        segs.append(Seg(to_device(raw).ptr, n, c.ptr, acc)), outs.append((name, n, w, c)), olds.append(old if acc else 0)
    before, launches = passes.stat("workgroups"), passes.stat("launches")
    blocks_multi(passes, [FORMATS[name] for name, _, _ in mats], segs, k, src, m)
    assert passes.stat("launches") - launches == 1 + 1 + 2 + 1  # (divided k: the addition too)
    wide = 256 + grid(m, 5000, 96) + grid(m, 6000, 64)
    assert passes.stat("workgroups") - before > wide and grid(m, 700, 64) * 2 <= passes.stat("workgroups") - before - wide
    for (name, n, w, c), old in zip(outs, olds):
        got = c.download(np.float32, m * n).reshape(m, n)
        exact = a.astype(np.float64) @ w.T.astype(np.float64) + old
        over = np.abs(got - exact) - bound(name, w, a) - 2.0**-23 * (np.abs(exact) + np.abs(old))  # (scaling, addition, store)
        assert np.max(over) <= 0, (name, float(np.max(over)))


@pytest.mark.parametrize("name", ["q8_0", "q5_1"])
def test_an_infinite_or_undefined_activation_reaches_its_row_alone(passes, name):
    """In a full tile and in the last, whose rows past the end repeat others."""
    m, n, k = 200, 5000, 512
    raw, w = weights(name, n, k, 9)
    bits = synth.activation_bf16((m, k), seed=3).reshape(m, k).copy()
    bits[17, 77], bits[195, 300], bits[199, 511] = 0x7F80, 0x7FC0, 0xFF80
    before = passes.stat("workgroups")
    got = passes.gemm_q_host(FORMATS[name], raw, n, k, bits, m).reshape(m, n)
    assert passes.stat("workgroups") - before == 256 + grid(m, n, 96)
    bad = np.isin(np.arange(m), [17, 195, 199])
    assert np.all(np.isfinite(got[~bad])) and not np.any(np.isfinite(got[bad]))
    a = bf16(bits[~bad])
    check(name, got[~bad], a.astype(np.float64) @ w.T.astype(np.float64), w, a)
