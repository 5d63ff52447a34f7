"""GPU parity of the 9..32-rows-per-kv-head attention launch (stream_rows_kernel, fp32 pools)
against the oracle: row tiles (9, 16, 17, 32 rows, and one query group past 32), piece and
batch edges (contexts 0 .. 33 and long ones, one sequence cut into many pieces), windows
that open inside a batch, ring pools, and values that are not finite in keys some rows mask.
Tolerances: tests/parity.py (sums in double, so 1e-5 against float64). Beside them the bf16 form
for 9..16 rows: values that are not finite, precision, and pieces of one batch."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from pkv import BF16, F32, LayerSpec, hip, lib
from pkv.engine import make_params
from tests import parity
from tests.test_gpu_attend import _batched_case

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 14, 15, 16, 17, 31, 32, 33, 1500]


@pytest.mark.parametrize("hq,hkv,d,q_len,window", [
    (16, 8, 256, 5, 0), (16, 8, 256, 8, 20), (16, 8, 256, 9, 1024), (16, 8, 256, 16, 0),
    (16, 8, 256, 17, 40), (12, 4, 256, 4, 0), (16, 2, 512, 2, 0), (16, 2, 512, 4, 0), (16, 2, 512, 3, 25),
    (8, 8, 512, 9, 0), (16, 2, 512, 5, 1024),
])
def test_rows_match_oracle(gpu, hq, hkv, d, q_len, window):
    print(f"[rows] {hq}q/{hkv}kv/{d} q_len={q_len} window={window}", flush=True)
    rng = np.random.default_rng(hq + 31 * d + q_len)
    _batched_case(rng, len(EDGES), q_len, np.array(EDGES), hq, hkv, d, 16, window, F32, 0.0625)


@pytest.mark.parametrize("bs", [1, 4, 64])
def test_rows_block_sizes(gpu, bs):
    print(f"[rows] block size {bs}", flush=True)
    rng = np.random.default_rng(bs)
    _batched_case(rng, 3, 5, np.array([3, 130, 700]), 16, 8, 256, bs, 0, F32, 0.0625)


def test_rows_one_long_sequence(gpu):
    print("[rows] one sequence, 20000 keys over every workgroup", flush=True)
    _batched_case(np.random.default_rng(5), 1, 4, np.array([20000]), 16, 2, 512, 16, 0, F32, 0.0625)


def _call(name, p, q, k, v, tables, pos, q_lens=None, max_pos=None):
    B, q_len, hq, d = q.shape
    mp = int(pos.max()) + q_len - 1 if max_pos is None else max_pos
    ws = hip.DeviceArray((lib.load().pkv_workspace_size(ctypes.byref(p), B, q_len, mp),), np.uint8)
    a = [hip.DeviceArray.from_numpy(x) for x in (q, k, v, tables, pos)]
    out = hip.DeviceArray((B, q_len, hq, d), np.float32, zero=True)
    counts = [hip.DeviceArray.from_numpy(q_lens)] if q_lens is not None else []
    lib.call(name, None, ctypes.byref(p), a[0].ptr, a[1].ptr, a[2].ptr, a[3].ptr, tables.shape[1], a[4].ptr,
             *[c.ptr for c in counts], q_len, B, mp, out.ptr, ws.ptr, ws.nbytes)
    return out.numpy()


@pytest.mark.parametrize("hq,hkv,d,q_len", [(16, 8, 256, 5), (16, 8, 256, 9), (16, 2, 512, 4)])
def test_rows_ring(gpu, hq, hkv, d, q_len):
    # The same keys in a ring and in pages: the key split and every sum are the same.
    print(f"[rows] ring {hq}q/{hkv}kv/{d} q_len={q_len}", flush=True)
    rng = np.random.default_rng(q_len + d)
    window, ring, bs, B = 200, 200 + 8, 16, 5
    pos = np.array([0, 150, 203, 1000, 417], np.int32)
    slots = rng.permutation(B).astype(np.int32)
    nblk = (int(pos.max()) + q_len + bs - 1) // bs
    tables = rng.permutation(B * nblk).astype(np.int32).reshape(B, nblk)
    kv = rng.standard_normal((2, B, nblk * bs, hkv, d), dtype=np.float32)
    paged = np.zeros((2, B * nblk, bs, hkv, d), np.float32)
    rings = np.full((2, B, ring, hkv, d), np.nan, np.float32)
    for s in range(B):
        paged[:, tables[s]] = kv[:, s].reshape(2, nblk, bs, hkv, d)
        for t in range(max(0, pos[s] + q_len - ring), pos[s] + q_len):
            rings[:, slots[s], t % ring] = kv[:, s, t]
    rings[np.isnan(rings)] = 7.0
    q = rng.standard_normal((B, q_len, hq, d), dtype=np.float32)
    pp = make_params(LayerSpec(hq, hkv, d, window, F32), bs, B * nblk, 0.0625)
    pr = make_params(LayerSpec(hq, hkv, d, window, F32, ring), bs, B, 0.0625)
    a = _call("pkv_attend", pp, q, paged[0], paged[1], tables, pos)
    b = _call("pkv_attend", pr, q, rings[0], rings[1], slots.reshape(B, 1), pos)
    assert np.array_equal(a, b)
    lens = np.full(B, nblk, np.int32)
    args = (q_len, hq, hkv, d, bs, window)
    parity.check(a, O.attend(q, paged[0].ravel(), paged[1].ravel(), tables, lens, pos, *args, scale=0.0625),
                 O.attend_f64(q, paged[0].ravel(), paged[1].ravel(), tables, pos, *args, scale=0.0625))


@pytest.mark.parametrize("hq,hkv,q_len,window,ring", [
    (16, 8, 5, 0, 0), (16, 8, 5, 200, 208), (16, 16, 16, 100, 0), (12, 4, 3, 0, 0), (16, 8, 18, 0, 0),
    (16, 8, 16, 200, 216),
])
@pytest.mark.parametrize("many", [False, True], ids=["few", "many"])
def test_verify_large_step_by_counts(gpu, hq, hkv, q_len, window, ring, many):
    # A step whose bound on the keys is large (stream_verify_kernel: 65536 keys times kv heads): no
    # sequence with more than 8 rows, or two; sequences without queries, inactive ones and invalid
    # counts among them.
    print(f"[rows] counts {hq}q/{hkv}kv q_len {q_len} window {window} ring {ring} many {many}", flush=True)
    rng = np.random.default_rng(hq + q_len + window + many)
    d, bs, few = 256, 16, 8 * hkv // hq
    pos = np.array([0, 40, 7, -1, 300, 90, 33, 60, 12, 410, 15, 150] + [5, 260, 31] * 12, np.int32)
    q_lens = np.minimum(rng.integers(1, few + 1, pos.size), few).astype(np.int32)
    q_lens[:3] = few, 1, 0
    q_lens[6], q_lens[7] = -1, q_len + 1
    if many:
        q_lens[4], q_lens[10] = q_len, few + 1
    B, nblk = pos.size, (410 + q_len + bs - 1) // bs
    kv = rng.standard_normal((2, B, nblk * bs, hkv, d), dtype=np.float32)
    tables = rng.permutation(B * nblk).astype(np.int32).reshape(B, nblk)
    paged = np.zeros((2, B * nblk, bs, hkv, d), np.float32)
    for s in range(B):
        paged[:, tables[s]] = kv[:, s].reshape(2, nblk, bs, hkv, d)
    q = rng.standard_normal((B, q_len, hq, d), dtype=np.float32)
    max_pos = 1 << 16
    if ring:
        rings = np.zeros((2, B, ring, hkv, d), np.float32)
        slots = rng.permutation(B).astype(np.int32).reshape(B, 1)
        for s in range(B):
            for t in range(max(0, pos[s] + max(q_lens[s], 0) - ring), pos[s] + max(q_lens[s], 0)):
                rings[:, slots[s, 0], t % ring] = kv[:, s, t]
        p = make_params(LayerSpec(hq, hkv, d, window, F32, ring), bs, B, 0.0625)
        got = _call("pkv_verify", p, q, rings[0], rings[1], slots, pos, q_lens, max_pos)
    else:
        p = make_params(LayerSpec(hq, hkv, d, window, F32), bs, B * nblk, 0.0625)
        got = _call("pkv_verify", p, q, paged[0], paged[1], tables, pos, q_lens, max_pos)
    for s in range(B):
        n = int(q_lens[s])
        if n < 0 or n > q_len:
            assert np.all(np.isnan(got[s])), s
            continue
        assert np.all(got[s, n:] == 0), s  # rows past the count are not written
        if n == 0 or pos[s] < 0:
            assert np.all(got[s] == 0), s
            continue
        args = (n, hq, hkv, d, bs, window)
        qs, ts, ps = q[s:s + 1, :n].copy(), tables[s:s + 1], pos[s:s + 1]
        parity.check(got[s:s + 1, :n],
                     O.attend(qs, paged[0].ravel(), paged[1].ravel(), ts, np.array([nblk], np.int32), ps, *args,
                              scale=0.0625),
                     O.attend_f64(qs, paged[0].ravel(), paged[1].ravel(), ts, ps, *args, scale=0.0625), what=f"{s}")


@pytest.mark.parametrize("hq,hkv,d,q_len", [(16, 8, 256, 5), (16, 2, 512, 4)])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_rows_masked_values_not_finite(gpu, hq, hkv, d, q_len, value):
    # V of the last query's own key is not finite in dims 3 and d - 1: the rows
    # before it mask that key and must not change; its own row carries the value.
    print(f"[rows] {value} in a masked key, {hq}q/{hkv}kv/{d}", flush=True)
    rng = np.random.default_rng(9)
    bs, pos = 16, np.array([70, 29], np.int32)
    nblk = 6
    tables = rng.permutation(2 * nblk).astype(np.int32).reshape(2, nblk)
    k = rng.standard_normal((2 * nblk, bs, hkv, d), dtype=np.float32)
    v = rng.standard_normal((2 * nblk, bs, hkv, d), dtype=np.float32)
    q = rng.standard_normal((2, q_len, hq, d), dtype=np.float32)
    p = make_params(LayerSpec(hq, hkv, d, 0, F32), bs, 2 * nblk, 0.0625)
    clean = _call("pkv_attend", p, q, k, v, tables, pos)
    for s in range(2):
        t = int(pos[s]) + q_len - 1
        v[tables[s, t // bs], t % bs][:, [3, d - 1]] = value
    got = _call("pkv_attend", p, q, k, v, tables, pos)
    assert np.array_equal(got[:, :-1], clean[:, :-1])
    last = got[:, -1]
    assert np.array_equal(last[..., 4:d - 1], clean[:, -1][..., 4:d - 1])
    want = np.full(last[..., [3, d - 1]].shape, value, np.float32)
    assert np.array_equal(last[..., [3, d - 1]], want, equal_nan=True)


@pytest.mark.parametrize("hq,hkv,q_len", [(16, 8, 5), (16, 16, 16)])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_bf16_wide_values_not_finite(gpu, hq, hkv, q_len, value):
    # bf16 pools, 9..16 rows: a V value that is not finite reaches the rows that attend its
    # key and no other; a K value of -inf gives the key no weight, as a very negative one.
    print(f"[rows] bf16, {value} in a masked key, {hq}q/{hkv}kv q_len {q_len}", flush=True)
    rng = np.random.default_rng(9)
    bs, d, nblk, pos = 16, 256, 20, np.array([70, 29, 300], np.int32)
    tables = rng.permutation(3 * nblk).astype(np.int32).reshape(3, nblk)
    k = O.to_bf16(rng.standard_normal((3 * nblk, bs, hkv, d), dtype=np.float32))
    v = O.to_bf16(rng.standard_normal((3 * nblk, bs, hkv, d), dtype=np.float32))
    q = rng.standard_normal((3, q_len, hq, d), dtype=np.float32)
    q[..., 5] = np.abs(q[..., 5]) + 0.01
    q[..., 6] = 1.0  # parts 1 and 2 are zero
    p = make_params(LayerSpec(hq, hkv, d, 0, BF16), bs, 3 * nblk, 0.0625)
    bits = O.to_bf16(np.full(1, value, np.float32))[0]
    low, inf = (O.to_bf16(np.full(1, x, np.float32))[0] for x in (-1e30, -np.inf))
    clean = _call("pkv_attend", p, q, k, v, tables, pos)
    odd = v.copy()
    for s in range(3):
        t = int(pos[s]) + q_len - 1
        odd[tables[s, t // bs], t % bs][:, [3, d - 1]] = bits
    got = _call("pkv_attend", p, q, k, odd, tables, pos)
    assert np.array_equal(got[:, :-1], clean[:, :-1])
    last = got[:, -1]
    assert np.array_equal(last[..., 4:d - 1], clean[:, -1][..., 4:d - 1])
    want = np.full(last[..., [3, d - 1]].shape, value, np.float32)
    assert np.array_equal(last[..., [3, d - 1]], want, equal_nan=True)
    for dim in (5, 6):
        k1, k2 = k.copy(), k.copy()
        for s in range(3):
            k1[tables[s, 1], 4][:, dim], k2[tables[s, 1], 4][:, dim] = low, inf
        a, b = (_call("pkv_attend", p, q, x, v, tables, pos) for x in (k1, k2))
        assert np.all(np.isfinite(b)) and np.array_equal(a, b)


@pytest.mark.parametrize("hq,hkv,q_len", [(16, 8, 5), (16, 16, 16)])
def test_bf16_wide_precision(gpu, hq, hkv, q_len):
    # Q and P enter as three bf16 parts, which are exact, so only fp32 roundings are left: about
    # 24 in a score of size ~1 behind the scale, those of exp2 and of its argument, and the sums,
    # 2^-24 of their size each and independent: 4e-7 to 6e-7 of the output (2-norm). 2e-6 leaves
    # that four times; two parts of Q alone (off by 2^-17 of every element) give 4e-6.
    print(f"[rows] bf16 wide precision {hq}q/{hkv}kv q_len {q_len}", flush=True)
    rng = np.random.default_rng(q_len)
    d, bs, pos = 256, 16, np.array([600, 1500, 45, 3000], np.int32)
    nblk = (3000 + q_len + bs - 1) // bs
    tables = rng.permutation(4 * nblk).astype(np.int32).reshape(4, nblk)
    k, v = (O.to_bf16(rng.standard_normal((4 * nblk, bs, hkv, d), dtype=np.float32)) for _ in range(2))
    q = rng.standard_normal((4, q_len, hq, d), dtype=np.float32)
    p = make_params(LayerSpec(hq, hkv, d, 0, BF16), bs, 4 * nblk, 0.0625)
    got = _call("pkv_attend", p, q, k, v, tables, pos)
    exact = O.attend_f64(q, O.bf16_to_f32(k).ravel(), O.bf16_to_f32(v).ravel(), tables, pos, q_len, hq, hkv, d, bs, 0,
                         scale=0.0625)
    err = np.linalg.norm(got - exact) / np.linalg.norm(exact)
    print(f"[rows] relative error {err:.2e}", flush=True)
    assert err <= 2e-6


@pytest.mark.parametrize("q_len", [4, 5], ids=["8-rows", "10-rows"])
def test_bf16_pieces_of_one_batch(gpu, q_len):
    # A workgroup's pieces of a single batch of keys follow one another with nothing to exchange
    # between its waves; the next piece's Q must not reach LDS before every wave has read this one's.
    print(f"[rows] bf16, 300 sequences of 1..12 keys, q_len {q_len}", flush=True)
    rng = np.random.default_rng(q_len)
    _batched_case(rng, 300, q_len, rng.integers(0, 12, 300), 16, 8, 256, 16, 0, BF16, 0.0625)
