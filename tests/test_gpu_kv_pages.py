"""GPU: a cache's page table on the device after sequences have given their pages back: started again in the same order, in another
one, longer and shorter than before, alone or all at once.  (Which entries are uploaded: tests/test_kv_table.py.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_pages_given_back_and_mapped_again(hip):
    heads, dim, page = 2, 64, 4
    kv = hip.kv_cache(3, heads, dim, page, 24)
    rng = np.random.default_rng(3)

    def fill(order):
        rows = {}
        for seq, n in order:
            k, v = (rng.standard_normal((n, heads, dim)).astype(np.float16).view(np.uint16) for _ in range(2))
            kv.append_run(seq, hip.to_device(k), hip.to_device(v), n)
            old = rows.get(seq)
            rows[seq] = (k, v) if old is None else tuple(np.concatenate([a, b]) for a, b in zip(old, (k, v)))
        for seq, (k, v) in rows.items():
            n = len(k)
            kb, vb = hip.alloc(k.nbytes), hip.alloc(v.nbytes)
            kv.gather(seq, 0, n, kb, vb)
            assert np.array_equal(kb.download(np.uint16, k.size).reshape(k.shape), k), (order, seq)
            assert np.array_equal(vb.download(np.uint16, v.size).reshape(v.shape), v), (order, seq)

    same = [(0, 5), (1, 9), (0, 6), (2, 1)]
    for order in (same, same, [(2, 20), (0, 3)], [(1, 24), (2, 24), (0, 24)], same, [(0, 24)], [(0, 1), (0, 1), (0, 22), (1, 2)]):
        fill(order)
        kv.reset()
    fill([(1, 10), (2, 10)])
    kv.reset(1)
    fill([(0, 7), (1, 12)])
    kv.free()
