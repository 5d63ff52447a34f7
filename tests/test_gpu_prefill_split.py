"""GPU parity of the short-grid prefill launch (prefill_split_kernel: 16 or 32 query rows per
workgroup, the keys shared out over its waves) against the oracle, at the edges of its query
tiles (one query; a tile, a tile and one; the largest 16-row and the smallest and largest
32-row grids of one sequence), with fewer batches of keys than waves, windows, block sizes and
ragged counts; bad tables, inactive sequences and, with the 128-row kernel beside it, pool rows
outside the attended keys that are not finite.
Same tolerance as the other prefill tests (2e-2, tests/parity.py)."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from pkv import BF16, LayerSpec, hip, lib
from pkv.engine import make_params
from pkv.workloads import PrefillChunk
from tests.test_gpu_prefill import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,prefix,counts,window", [
    (16, 8, [0], [1], 0), (16, 8, [3], [8], 0), (16, 8, [120], [9], 0), (16, 8, [700], [17], 30),
    (16, 8, [1000], [256], 0), (16, 8, [333], [257], 100), (16, 8, [50], [512], 0),
    (16, 8, [0, 640], [1, 120], 0), (16, 8, [31, 250], [250, 33], 64), (8, 8, [77], [300], 0),
    (8, 8, [900], [40], 128), (16, 4, [129], [100], 0), (16, 4, [260], [250], 90),
    (16, 8, [16, 5, 900, 0], [7, 32, 1, 12], 0), (16, 8, [0, 9], [17, 3], 0), (16, 8, [0] * 8, [33] * 8, 0),
])
def test_prefill_split_matches_oracle(gpu, hq, hkv, prefix, counts, window):
    print(f"[prefill split] {hq}q/{hkv}kv prefix={prefix} counts={counts} window={window}", flush=True)
    w = PrefillChunk(seed=hq + sum(counts), batch=len(prefix), chunk=max(counts), prefix_max=max(prefix), hq=hq,
                     hkv=hkv, window=window, prefix=prefix)
    if w.max_pos < 128:  # so few keys take the 128-row kernel, unless the bound allows more
        _run(w, q_counts=counts)
        w.max_pos = 128
    _run(w, q_counts=counts)


@pytest.mark.parametrize("bs", [8, 32, 64])
def test_prefill_split_block_sizes(gpu, bs):
    print(f"[prefill split] block size {bs}", flush=True)

    class Chunk(PrefillChunk):
        BS = bs

    _run(Chunk(seed=bs, batch=1, chunk=90, prefix_max=205, prefix=[205]))
    _run(Chunk(seed=bs + 1, batch=1, chunk=300, prefix_max=13, prefix=[13]))


@pytest.mark.parametrize("n", [12, 300], ids=["16-rows", "32-rows"])
def test_prefill_split_contract_and_unwritten_rows(gpu, n):
    print(f"[prefill split] contract, {n} queries", flush=True)
    rng = np.random.default_rng(n)
    hq, hkv, d, bs, nb, stride = 16, 8, 256, 16, 64, 40
    p = make_params(LayerSpec(hq, hkv, d, kv_dtype=BF16), bs, nb, 0.0625)
    q = hip.DeviceArray.from_numpy(O.to_bf16(rng.standard_normal((n, hq, d), dtype=np.float32)))
    k = hip.DeviceArray((nb * bs, hkv * d), np.uint16, zero=True)
    v = np.full((nb, bs, hkv * d), 0x7FC0, np.uint16)  # NaN in every row no key was written to
    tables = rng.permutation(nb)[:stride].astype(np.int32).reshape(1, stride)
    pos = 37
    for t in range(pos + n):
        v[tables[0, t // bs], t % bs] = 0x3F80  # 1.0
    dv, out = hip.DeviceArray.from_numpy(v), hip.DeviceArray((n, hq, d), np.float32)
    off = hip.DeviceArray.from_numpy(np.array([0, n], np.int32))

    def call(tab, at, max_pos):
        dt, dp = hip.DeviceArray.from_numpy(tab), hip.DeviceArray.from_numpy(np.array([at], np.int32))
        lib.call("pkv_prefill", None, ctypes.byref(p), q.ptr, k.ptr, dv.ptr, dt.ptr, stride, dp.ptr, off.ptr, n, 1,
                 max_pos, out.ptr)
        return out.numpy()

    assert np.allclose(call(tables, pos, 600), 1.0, atol=1e-6)  # equal weights of rows of ones
    assert np.all(call(tables, -1, 600) == 0.0)                 # inactive
    assert np.all(np.isnan(call(tables, pos, pos + n - 2)))     # past max_pos
    bad = tables.copy()
    bad[0, 1] = nb
    assert np.all(np.isnan(call(bad, pos, 600)))                # an entry outside the pool


@pytest.mark.parametrize("batch", [1, 40], ids=["16-rows", "128-rows"])
@pytest.mark.parametrize("bs,window,pos,n", [
    (8, 4, 13, 1), (8, 4, 14, 3), (8, 0, 13, 1), (16, 5, 20, 1), (16, 0, 3, 2), (64, 20, 100, 9), (8, 70, 150, 5),
])
def test_prefill_rows_outside_the_range(gpu, batch, bs, window, pos, n):
    # Every pool row but those of the keys the queries attend is NaN in V: the copies round
    # the range down and up to whole batches and tiles, in the rows of its first and last block.
    print(f"[prefill split] NaN outside the keys, batch {batch} bs {bs} window {window} pos {pos}", flush=True)
    rng = np.random.default_rng(bs + pos)
    hq, hkv, d = 16, 8, 256
    stride = (pos + n + bs - 1) // bs + 1
    p = make_params(LayerSpec(hq, hkv, d, window=window, kv_dtype=BF16), bs, batch * stride, 0.0625)
    tables = rng.permutation(batch * stride).astype(np.int32).reshape(batch, stride)
    v = np.full((batch * stride, bs, hkv * d), 0x7FC0, np.uint16)
    for t in range(max(0, pos - window + 1) if window else 0, pos + n):
        v[tables[:, t // bs], t % bs] = 0x3F80  # 1.0
    q = hip.DeviceArray.from_numpy(O.to_bf16(rng.standard_normal((batch * n, hq, d), dtype=np.float32)))
    k, out = hip.DeviceArray(v.shape, np.uint16, zero=True), hip.DeviceArray((batch * n, hq, d), np.float32)
    dv, dt = hip.DeviceArray.from_numpy(v), hip.DeviceArray.from_numpy(tables)
    dp = hip.DeviceArray.from_numpy(np.full(batch, pos, np.int32))
    off = hip.DeviceArray.from_numpy((np.arange(batch + 1) * n).astype(np.int32))
    lib.call("pkv_prefill", None, ctypes.byref(p), q.ptr, k.ptr, dv.ptr, dt.ptr, stride, dp.ptr, off.ptr, n, batch,
             1000, out.ptr)
    assert np.allclose(out.numpy(), 1.0, atol=1e-6)  # equal weights of rows of ones


@pytest.mark.parametrize("n,pos", [(40, 900), (333, 900)], ids=["16-rows", "32-rows"])
def test_prefill_split_precision(gpu, n, pos):
    # Q, K and V are bf16 and exact; P enters as P_hi + P_lo, off by at most 2^-16 of p, and
    # fp32 sums add less. The keys' errors are independent, so the output's relative error
    # (2-norm) stays below 2^-16; without P_lo it would be about 3e-3 (P_hi truncates).
    print(f"[prefill split] precision, {n} queries over {pos}", flush=True)
    rng = np.random.default_rng(n)
    hq, hkv, d, bs = 16, 8, 256, 16
    nb = (pos + n + bs - 1) // bs
    p = make_params(LayerSpec(hq, hkv, d, kv_dtype=BF16), bs, nb, 0.0625)
    tables = rng.permutation(nb).astype(np.int32).reshape(1, nb)
    q, k, v = (O.to_bf16(rng.standard_normal(s, dtype=np.float32)) for s in ((n, hq, d), (nb * bs * hkv * d,),
                                                                            (nb * bs * hkv * d,)))
    dq, dk, dv, dt, dp, off = (hip.DeviceArray.from_numpy(x) for x in (
        q, k, v, tables, np.array([pos], np.int32), np.array([0, n], np.int32)))
    out = hip.DeviceArray((n, hq, d), np.float32)
    lib.call("pkv_prefill", None, ctypes.byref(p), dq.ptr, dk.ptr, dv.ptr, dt.ptr, nb, dp.ptr, off.ptr, n, 1,
             pos + n - 1, out.ptr)
    exact = O.attend_f64(O.bf16_to_f32(q)[None], O.bf16_to_f32(k), O.bf16_to_f32(v), tables, np.array([pos], np.int32),
                         n, hq, hkv, d, bs, 0, scale=0.0625)[0]
    err = np.linalg.norm(out.numpy() - exact) / np.linalg.norm(exact)
    print(f"[prefill split] relative error {err:.2e}", flush=True)
    assert err <= 2.0 ** -16
