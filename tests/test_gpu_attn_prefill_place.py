"""GPU: prompt attention at the counts of heads for which its workgroups are placed differently -- the cached heads, else the query heads, else neither
a multiple of eight -- with ragged blocks of queries, and the rows of q in blocks that are not full."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle_c, oracle_np
from skainet_amd import runtime, synth
from test_gpu_lebelix_ops import ranged_case, ranged_oracle, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("heads,n", [(8, 1), (8, 33), (16, 70), (24, 40), (12, 70), (7, 33)])
def test_heads_and_blocks(hip, heads, n, dim):
    rng = np.random.default_rng(heads * n + dim)
    q = rng.standard_normal((n, heads, dim)).astype(np.float32)
    k, v = (rng.standard_normal((1, n, heads, dim)).astype(np.float16).view(np.uint16) for _ in range(2))
    kv = hip.kv_cache(1, heads, dim, 16, n + 16)
    kv.append_run(0, hip.to_device(k[0]), hip.to_device(v[0]), n)
    out = hip.alloc(q.nbytes)
    out.upload(np.full(q.shape, np.nan, np.float32))
    kv.attn_prefill(0, hip.to_device(q), n, out, dim ** -0.5)
    got = out.download(np.float32, q.size).reshape(q.shape)
    kk, vv = (np.ascontiguousarray(np.broadcast_to(a, (n,) + a.shape[1:])) for a in (k, v))
    want = oracle_c.attn_decode(q, kk, vv, [t + 1 for t in range(n)], dim ** -0.5)
    for t in range(n):
        assert oracle_np.rel_err(got[t], want[t]) <= 1e-3, t  # (the bar of the other attention tests)
    kv.free()


@pytest.mark.parametrize("heads,kv_heads", [(16, 8), (24, 8), (64, 16), (8, 2), (24, 12), (12, 4), (8, 1)])
def test_grouped_heads(hip, heads, kv_heads):
    n, dim, vdim = 70, 64, 64
    q, k, v, gate, p = ranged_case(heads, kv_heads, dim, vdim, n, seed=heads + kv_heads)
    want = ranged_oracle(q, k, v, gate, p, kv_heads, dim, vdim)
    kv = runtime.RangedKVCache(hip, 1, kv_heads, dim, vdim, 16, 96, runtime.F16)
    got = kv.attend(0, p, q, k, v, gate)
    assert rel(got, want) < 5e-3  # (fp16 rows: the bar of the other ranged tests)
    kv.free()


@pytest.mark.parametrize("heads,n,dim", [(8, 33, 64), (7, 70, 128), (16, 1, 128)])
def test_rows_in_bf16_are_the_fp32_rows_rounded(hip, heads, n, dim):
    """What a decoder's prompt asks of it (skn_attn_prefill_launch with an output type) against the public call on the same cache."""
    rng = np.random.default_rng(heads + n)
    q = rng.standard_normal((n, heads, dim)).astype(np.float32)
    kv = hip.kv_cache(1, heads, dim, 16, n + 16)
    kv.append_run(0, hip.to_device(synth.kv_f16((n, heads, dim), seed=1)), hip.to_device(synth.kv_f16((n, heads, dim), seed=2)), n)
    q_dev, wide, narrow = hip.to_device(q), hip.alloc(q.nbytes), hip.alloc(q.nbytes)
    kv.attn_prefill(0, q_dev, n, wide, dim ** -0.5)
    hip.memset(narrow, 0xFF, q.nbytes)
    fn = hip.lib._Z23skn_attn_prefill_launchP7skn_ctxP6skn_kviPKfiifPvii
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_float, C.c_void_p, C.c_int, C.c_int]
    hip._check(fn(hip.handle, kv.handle, 0, q_dev.ptr, n, 1, dim ** -0.5, narrow.ptr, heads, runtime.BF16))
    got, want = narrow.download(np.uint16, 2 * q.size), synth.f32_to_bf16_bits(wide.download(np.float32, q.size))
    assert np.array_equal(got[: q.size], want)
    assert np.all(got[q.size :] == 0xFFFF)  # (nothing behind them)
    kv.free()
