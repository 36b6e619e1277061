"""GPU: products of few rows, and of more with a small matrix, that take one launch (two where k is divided) behind the activations as they
are, against 64-bit sums of the oracle's weights."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle_c, oracle_np
from skainet_amd import runtime, synth

pytestmark = pytest.mark.gpu
FORMATS = {"q4_k": synth.Q4_K, "q5_k": synth.Q5_K, "q6_k": synth.Q6_K, "q8_0": synth.Q8_0, "q4_0": synth.Q4_0}
# 2^-24 of the sum of the terms' magnitudes per rounding: up to 32 in a matrix instruction, 16 in a superblock, then one for each of
# a wavefront's superblocks (8 at most here) and of the wavefronts and parts (12)
ROUNDINGS = 32 + 16 + 8 + 12


def _launches(hip, t, w, n, k, x, m, c):
    before = hip.stat("launches")
    hip.gemm_q(t, w, n, k, x, m, c)
    return hip.stat("launches") - before


def _check(hip, t, raw, n, k, a, m, launches=None):
    c = hip.alloc(4 * m * n)
    w, x = hip.to_device(raw), hip.to_device(a)
    hip.set_option("gemm.few", 0)
    try:
        passes = _launches(hip, t, w, n, k, x, m, c)
    finally:
        hip.set_option("gemm.few", 1)
    hip.memset(c, 0xFF, 4 * m * n)
    took = _launches(hip, t, w, n, k, x, m, c)
    assert took < passes, "the shape takes the passes: nothing was tested"
    assert launches is None or took == launches
    got = c.download(np.float32, m * n).reshape(m, n)
    wd = oracle_c.dequant(t, raw).astype(np.float64).reshape(n, k)
    xd = oracle_np.bf16_to_f32(a).astype(np.float64).reshape(m, k)
    size = np.abs(xd) @ np.abs(wd).T
    if t in (synth.Q4_K, synth.Q5_K):  # d sc q and dmin m are terms of their own
        size = size * 4
    # (and half of the least subnormal, where the result is one)
    assert np.all(np.abs(got - xd @ wd.T) <= ROUNDINGS * 2.0**-24 * size + 2.0**-150)
    return got


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (2, 15, 512), (15, 16, 2048), (16, 17, 2304), (17, 100, 1280), (32, 31, 4096), (33, 48, 4352), (48, 33, 6144),
                                   (64, 20, 8192), (5, 40, 11008), (33, 4090, 4352), (30, 4200, 512)])
def test_row_blocks_ragged_tiles_and_divided_k(hip, name, m, n, k):
    """One to four row blocks, full and ragged; fewer superblocks than wavefronts, as many, one more; few columns with k over
    workgroups; more tiles than compute units."""
    t = FORMATS[name]
    _check(hip, t, synth.weight(t, n, k, seed=n + k + t), n, k, synth.activation_bf16((m, k), seed=m + 1), m)


@pytest.mark.parametrize("name", ["q4_k", "q6_k", "q8_0"])
def test_four_row_blocks_of_more_tiles_than_compute_units(hip, name):
    t, m, n, k = FORMATS[name], 49, 4100, 4352
    _check(hip, t, synth.weight(t, n, k, seed=n + k + t), n, k, synth.activation_bf16((m, k), seed=m + 1), m)


@pytest.mark.parametrize("name", ["q5_k", "q8_0", "q4_0"])
@pytest.mark.parametrize("m,n,k", [(33, 48, 2304), (48, 33, 256), (49, 16, 2048), (64, 65, 768), (40, 4200, 512), (50, 4200, 768)])
def test_three_and_four_row_blocks_of_short_rows(hip, name, m, n, k):
    t = FORMATS[name]
    _check(hip, t, synth.weight(t, n, k, seed=n + k + t), n, k, synth.activation_bf16((m, k), seed=m + 1), m)


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("m,n,k", [(65, 33, 512), (127, 40, 2304), (128, 16, 256), (129, 200, 1024), (333, 500, 512)])
def test_more_rows_in_groups(hip, name, m, n, k):
    """Groups of 48 and 64 rows, the last one ragged or nearly empty."""
    t = FORMATS[name]
    _check(hip, t, synth.weight(t, n, k, seed=n + k + t), n, k, synth.activation_bf16((m, k), seed=m + 1), m)


@pytest.mark.parametrize("name", list(FORMATS))
def test_rows_far_apart_and_fields_over_their_range(hip, name):
    """Random bytes in every field but the scales (zero, subnormal and of both signs among them); rows of 1e30, of 1e-30 and of zeros,
    elements 2^40 apart in one row: the activations are taken as they are."""
    t = FORMATS[name]
    m, n, k = 21, 40, 1024
    be, bb = synth.BLOCK[t]
    rng = np.random.default_rng(t)
    raw = rng.integers(0, 256, (n * k // be, bb), dtype=np.uint8)
    d = (rng.standard_normal(len(raw)) * 0.01).astype(np.float16)
    d[::5], d[3::11] = 0.0, np.float16(6e-8)
    at = 208 if name == "q6_k" else 0
    raw[:, at:at + 2] = d.view(np.uint8).reshape(-1, 2)
    if name in ("q4_k", "q5_k"):
        raw[:, 2:4] = (rng.standard_normal(len(raw)) * 0.02).astype(np.float16).view(np.uint8).reshape(-1, 2)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0] *= 1e30
    x[1] *= 1e-30
    x[2] = 0.0
    x[3, ::2] *= 2.0**40
    _check(hip, t, raw.reshape(-1), n, k, synth.f32_to_bf16_bits(x), m)


@pytest.mark.parametrize("name,m,n,k,few", [("q4_0", 31, 30269, 512, False), ("q4_k", 252, 6683, 256, False), ("q5_k", 32, 29393, 512, False), ("q6_k", 370, 13269, 256, False),
                                            ("q8_0", 248, 24474, 256, False), ("q5_k", 49, 4296, 3072, False), ("q4_0", 49, 4555, 4096, False), ("q5_k", 58, 13285, 1536, False),
                                            ("q8_0", 507, 8812, 256, True), ("q4_k", 16, 30000, 512, True), ("q5_k", 57, 7844, 1536, True), ("q4_0", 57, 6795, 2048, True)])
def test_many_short_tiles_take_the_passes(hip, name, m, n, k, few):
    """Shapes on both sides of where so many rounds of short workgroups cost more than the launches they save."""
    assert hip.device_info()["compute_units"] == 256, "the rounds are counted for 256 compute units"
    t = FORMATS[name]
    w, x, c = hip.alloc(synth.weight(t, 16, k, seed=1).nbytes // 16 * n), hip.alloc(2 * m * k), hip.alloc(4 * m * n)
    took = []
    for value in (1, 0):
        hip.set_option("gemm.few", value)
        try:
            took.append(_launches(hip, t, w, n, k, x, m, c))
        finally:
            hip.set_option("gemm.few", 1)
    assert (took[0] == 1 and took[1] >= 2) if few else took[0] == took[1]


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("m", [7, 40])
def test_without_room_for_parts_k_is_undivided(hip, name, m):
    """The same bits as from a matrix of so many more columns that no unit is left to divide k; others than with k divided."""
    assert hip.device_info()["compute_units"] == 256, "k is divided for 256 compute units"
    t, n, wide, k = FORMATS[name], 192, 2304, 11008
    raw, a = synth.weight(t, wide, k, seed=m), synth.activation_bf16((m, k), seed=m + 1)
    w, x, c = hip.to_device(raw), hip.to_device(a), hip.alloc(4 * m * wide)
    assert _launches(hip, t, w, wide, k, x, m, c) == 1
    want = c.download(np.float32, m * wide).reshape(m, wide)[:, :n]
    assert _launches(hip, t, w, n, k, x, m, c) == 2
    divided = c.download(np.float32, m * n).reshape(m, n)
    hip.set_option("test.gemm_no_parts", 2)
    try:
        assert _launches(hip, t, w, n, k, x, m, c) == 1
    finally:
        hip.set_option("test.gemm_no_parts", 0)
    got = c.download(np.float32, m * n).reshape(m, n)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)) and not np.array_equal(got, divided)


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("size", [2.0**127, 2.0**-125])
def test_activations_at_either_end_of_their_range(hip, name, size):
    """Largest finite activations with weights that bring the sums back into range (a block's sum of quants alone would leave it);
    least normal ones with scales as large as the format has."""
    t = FORMATS[name]
    m, n, k = 18, 33, 512
    be, bb = synth.BLOCK[t]
    raw = np.frombuffer(synth.weight(t, n, k, seed=9).tobytes(), np.uint8).reshape(-1, bb).copy()
    scale = np.float16(2.0**-20 if size > 1 else 1000.0)
    at = 208 if name == "q6_k" else 0
    for f in ((0, 2) if name in ("q4_k", "q5_k") else (at,)):
        raw[:, f:f + 2] = np.full(len(raw), scale).view(np.uint8).reshape(-1, 2)
    x = np.random.default_rng(t).uniform(0.5, 1.9, (m, k)).astype(np.float32) * np.float32(size)
    a = synth.f32_to_bf16_bits(x)
    got = hip.gemm_q_host(t, raw.reshape(-1), n, k, a, m).reshape(m, n)
    wd = oracle_c.dequant(t, raw.reshape(-1)).astype(np.float64).reshape(n, k)
    xd = oracle_np.bf16_to_f32(a).astype(np.float64).reshape(m, k)
    bound = np.abs(xd) @ np.abs(wd).T * (4 if name in ("q4_k", "q5_k") else 1)
    assert np.all(np.abs(got - xd @ wd.T) <= ROUNDINGS * 2.0**-24 * bound)


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("k,launches", [(512, 1), (10752, 2)])
def test_sums_that_leave_the_range_on_their_way(hip, name, k, launches):
    """Results of every size beside each other, k in one piece and divided: a row of 2^124 whose halves cancel (over wavefronts, over parts;
    minima against scales in a block), rows of 2^60 and 2^100, of elements 2^40 apart, of zeros, of the least normal and of subnormal
    activations, ordinary ones."""
    assert hip.device_info()["compute_units"] == 256, "k is divided for 256 compute units"
    t = FORMATS[name]
    m, n = 20, 33
    half = synth.weight(t, n, k // 2, seed=k + t).reshape(n, -1)
    raw = np.concatenate([half, half], axis=1).reshape(-1)
    rng = np.random.default_rng(t)
    x = rng.standard_normal((m, k))
    x[0] = 2.0**124 * (1 + rng.random(k))
    x[0, k // 2:] = -x[0, : k // 2]
    x[1] *= 2.0**60
    x[2] *= 2.0**100
    x[3] = 0.0
    x[4] *= 2.0**100
    x[4, ::2] *= 2.0**-40
    x[5] = rng.uniform(1, 2, k) * 2.0**-126 * rng.choice([-1, 1], k)
    x[6] = rng.integers(-127, 128, k) * 2.0**-133
    a = synth.f32_to_bf16_bits(x.astype(np.float32)).reshape(m, k)
    assert np.array_equal(a[0, k // 2:], a[0, : k // 2] ^ 0x8000)
    got = _check(hip, t, raw, n, k, a, m, launches)
    assert np.all(np.isfinite(got)) and np.all(got[3] == 0) and np.any(got[6])


@pytest.mark.parametrize("name", list(FORMATS))
def test_an_infinite_activation_reaches_its_row_alone(hip, name):
    t = FORMATS[name]
    m, n, k = 18, 33, 512
    raw = synth.weight(t, n, k, seed=3)
    a = synth.activation_bf16((m, k), seed=4).reshape(m, k).copy()
    a[17, 77], a[5, 300] = 0x7F80, 0x7FC0
    got = hip.gemm_q_host(t, raw, n, k, a, m)
    bad = np.zeros(m, bool)
    bad[[5, 17]] = True
    assert np.all(np.isfinite(got[~bad])) and not np.any(np.isfinite(got[bad]))
    want = oracle_c.gemm_q(t, raw, n, k, a.reshape(m, k)[~bad], m - 2)
    assert oracle_np.rel_err(got[~bad], want) <= 1e-3


def test_weights_and_activations_on_their_least_alignment(hip):
    """Q6_K weights from any even address, activations from any multiple of eight."""
    m, n, k = 20, 35, 768
    raw, a = synth.weight(synth.Q6_K, n, k, seed=4), synth.activation_bf16((m, k), seed=5)
    w, x, c = hip.alloc(raw.nbytes + 16), hip.alloc(a.nbytes + 16), hip.alloc(4 * m * n)
    w.upload(raw, offset=2)
    x.upload(a, offset=8)
    hip.gemm_q(synth.Q6_K, w.ptr + 2, n, k, x.ptr + 8, m, c)
    got = c.download(np.float32, m * n).reshape(m, n)
    assert oracle_np.rel_err(got, oracle_c.gemm_q(synth.Q6_K, raw, n, k, a, m)) <= 1e-3


@pytest.mark.parametrize("name,m,n,wide,k", [("q8_0", 333, 1024, 4096, 4096), ("q5_k", 41, 512, 20000, 4096), ("q6_k", 33, 512, 20000, 4096), ("q4_k", 48, 512, 20000, 4096),
                                             ("q4_k", 17, 256, 20000, 4096), ("q8_0", 200, 1024, 5000, 4096), ("q5_k", 200, 960, 5000, 4096), ("q4_k", 300, 1024, 14336, 1024), ("q6_k", 300, 1024, 14336, 1024)])
def test_a_call_of_few_rows_readies_a_captured_one_of_more_columns(name, m, n, wide, k):
    """A caller that captures its calls runs one of the same activations first: what that one does not need itself is there for the
    captured one, which takes three launches.  Every replay against the eager result, with other work between."""
    t = FORMATS[name]
    rt = runtime.load_library()  # (the HIP runtime's functions too)

    def call(fn, *args):
        assert getattr(rt, fn)(*args) == 0, fn

    stream, graph, replay = C.c_void_p(), C.c_void_p(), C.c_void_p()
    with runtime.Context(0) as ctx:
        call("hipStreamCreate", C.byref(stream))
        ctx.set_stream(stream)
        w, x = ctx.to_device(synth.weight(t, wide, k, seed=n)), ctx.to_device(synth.activation_bf16((m, k), seed=m))
        c = ctx.alloc(4 * m * wide)
        few = _launches(ctx, t, w, n, k, x, m, c)
        ctx.sync()
        before = ctx.stat("launches")
        call("hipStreamBeginCapture", stream, 1)  # (of this thread's calls)
        try:
            ctx.gemm_q(t, w, wide, k, x, m, c)
        finally:
            ended = rt.hipStreamEndCapture(stream, C.byref(graph))
        assert ended == 0
        assert few == 1 and ctx.stat("launches") - before >= 2, "both take the same path: nothing was tested"
        call("hipGraphInstantiate", C.byref(replay), graph, None, None, C.c_size_t(0))
        ctx.gemm_q(t, w, wide, k, x, m, c)
        ctx.sync()
        want = c.download(np.float32, m * wide).view(np.uint32)
        for _ in range(3):
            ctx.memset(c, 0xFF, 4 * m * wide)
            ctx.sync()
            call("hipGraphLaunch", replay, stream)
            ctx.sync()
            assert np.array_equal(c.download(np.float32, m * wide).view(np.uint32), want)
            ctx.gemm_q(t, w, n, k, x, m, c)
        call("hipGraphExecDestroy", replay)
        call("hipGraphDestroy", graph)
        ctx.set_stream(None)
        call("hipStreamDestroy", stream)


def test_a_workspace_that_a_capture_uses_is_not_grown_for_other_matrices_of_its_rows():
    """A call captured without one of its type before, in a workspace that is enough for its tiles but not for the highest of its rows: the same
    call outside the capture leaves that workspace where it is."""
    m, n, k, t = 300, 2048, 1024, synth.Q6_K
    rt = runtime.load_library()
    stream, graph, replay = C.c_void_p(), C.c_void_p(), C.c_void_p()
    with runtime.Context(0) as ctx:
        assert rt.hipStreamCreate(C.byref(stream)) == 0
        ctx.set_stream(stream)
        ctx.set_option("gemm.few", 0)
        w8, x8 = ctx.to_device(synth.weight(synth.Q8_0, n, k, seed=1)), ctx.to_device(synth.activation_bf16((384, k), seed=2))
        w, x = ctx.to_device(synth.weight(t, n, k, seed=3)), ctx.to_device(synth.activation_bf16((m, k), seed=4))
        c = ctx.alloc(4 * 384 * n)
        ctx.gemm_q(synth.Q8_0, w8, n, k, x8, 384, c)  # (operands of 384 rows: what 128-row tiles of 300 take, 256-row ones 512)
        ctx.sync()
        assert rt.hipStreamBeginCapture(stream, 1) == 0
        try:
            ctx.gemm_q(t, w, n, k, x, m, c)
        finally:
            ended = rt.hipStreamEndCapture(stream, C.byref(graph))
        assert ended == 0 and rt.hipGraphInstantiate(C.byref(replay), graph, None, None, C.c_size_t(0)) == 0
        free, total = C.c_size_t(), C.c_size_t()
        assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        ctx.gemm_q(t, w, n, k, x, m, c)
        ctx.sync()
        want, before = c.download(np.float32, m * n).view(np.uint32), free.value
        assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0 and free.value == before
        for _ in range(3):
            ctx.memset(c, 0xFF, 4 * m * n)
            ctx.sync()
            assert rt.hipGraphLaunch(replay, stream) == 0
            ctx.sync()
            assert np.array_equal(c.download(np.float32, m * n).view(np.uint32), want)
        assert rt.hipGraphExecDestroy(replay) == 0 and rt.hipGraphDestroy(graph) == 0
        ctx.set_stream(None)
        assert rt.hipStreamDestroy(stream) == 0
