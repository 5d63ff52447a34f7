"""Performance cases of the paged KV-cache attention path.

Each case is the work of one layer, or of one whole step, as a serving program calls it
through the `pkv` package: PagedKVCache's append / attend / verify / prefill / rollback, the
producer step, LSA's key lists and the Wo projection. The sizes are those of the engine
this package serves and of the repository's benchmark:

  sliding layers   16 query / 8 kv heads, head_dim 256, window 1024 (paged, or in rings of
                   window + 8 rows, the engine's default)
  global layers    16 query / 2 kv heads, head_dim 512, full causal, V := K before the norms
  benchmark layers 16 query / 8 kv heads, head_dim 256, full causal

with blocks of 16 tokens, fp32 or bf16 pools, and a hidden size of 2816 behind Wo.

A case is a dict of plain values. "mix" seeds what decides the amount of work (context
lengths, draft counts, key lists); the seed of prepare() decides the values and where the
blocks lie in the pool.
"""
import math
import os
import random
import sys

import numpy as np
import torch

_REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_REPO, "llm-mojo_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_REPO, "llm-mojo_amd"))

BS = 16        # tokens per block
HQ = 16        # query heads of every layer
HIDDEN = 2816  # outputs of Wo
SCALE = 0.0625
WINDOW = 1024
EPS = 1e-6     # of the RMS norms

# name -> (kv heads, head_dim, window, ring rows)
LAYERS = {
    "sliding": (8, 256, WINDOW, 0),
    "ring": (8, 256, WINDOW, WINDOW + 8),
    "global": (2, 512, 0, 0),
    "full": (8, 256, 0, 0),
}

# The engine's LSA settings: up to 256 keys from 20 picked buckets of up to 32 members, a
# window of 128 keys and 4 sinks.
LSA_TOP_K, LSA_PICK, LSA_CAP, LSA_WINDOW, LSA_SINKS = 256, 20, 32, 128, 4


# ------------------------------------------------------------------------------ cases
def listed():
    return [
        # One chat turn's decode step on one layer: a single sequence, a few hundred keys.
        # Latency and launches are all there is.
        _case("decode", "decode_one", layers="full", batch=1, lo=512, hi=512),
        # Continuous batching: 32 sequences of mixed length, a sliding and a full layer.
        _case("decode", "decode_mixed", layers="sliding,full", batch=32, lo=128, hi=8192),
        # Long documents in bf16 pages: 8 sequences of 32K keys.
        _case("decode", "decode_long_bf16", layers="full", batch=8, lo=32767, hi=32767, dtype="bf16"),
        # The engine's chat mode: a sliding layer's whole decode step (norms + RoPE + append,
        # attention in the ring, Wo) for one sequence.
        _case("layer", "layer_ring_one", layers="ring", batch=1, lo=2900, hi=2900),
        # A global layer's whole decode step at a serving batch.
        _case("layer", "layer_global", layers="global", batch=32, lo=128, hi=8192),
        # Speculative decoding: four drafting reads of the target's pools on two layers, the
        # verify of four drafts, and the rollback of the rejected ones.
        _case("speculate", "speculate", layers="full,full", batch=16, lo=512, hi=4096, draft=4),
        # The engine's own verify: one to five tokens per sequence (the drafts and the token
        # before them) on a ring layer and a global layer, then the rollback.
        _case("verify", "verify_engine", layers="ring,global", batch=16, lo=512, hi=4096, draft=5),
        # The same on bf16 pages.
        _case("verify", "verify_bf16", layers="full", batch=16, lo=512, hi=4096, draft=5, dtype="bf16"),
        # Prompt processing at full load: 4 sequences x 2048 tokens over prefixes up to 6144.
        _case("prefill", "prefill_chunk", layers="full", batch=4, lo=0, hi=6144, chunk=2048, dtype="bf16"),
        # The ordinary prompt: one sequence, a few hundred tokens (a ragged number) behind an
        # earlier conversation, beside other sequences' decode steps.
        _case("prefill", "prefill_short", layers="full", batch=1, lo=3001, hi=3001, chunk=333, dtype="bf16"),
        # The producer step of the same prompt load: norms, RoPE and append of 4 x 2048 tokens.
        _case("produce", "produce_chunk", layers="full", batch=4, lo=0, hi=6144, chunk=2048, dtype="bf16"),
        # LSA decode on a global layer: key lists from the picked buckets, then the sparse
        # attention over them.
        _case("lsa", "lsa_decode", layers="global", batch=32, lo=128, hi=8192),
    ]


def _case(kind, name, layers, batch, lo, hi, dtype="f32", draft=1, chunk=1, mix=1):
    c = {"kind": kind, "layers": layers, "batch": batch, "lo": lo, "hi": hi, "dtype": dtype,
         "draft": draft, "chunk": chunk, "mix": mix}
    if name:
        c["name"] = name
    return c


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    """A case of the listed ones' ranges: batches 1 to 64, contexts 1 to 32K, chunks 1 to
    2048 tokens, one to five tokens to verify; what it reads is kept below the largest
    listed case's."""
    kind = rng.choice(["decode", "decode", "layer", "speculate", "verify", "prefill", "prefill",
                       "produce", "lsa"])
    mix = rng.randrange(1 << 30)
    while True:
        batch, draft, chunk, dtype = _log_int(rng, 1, 64), 1, 1, rng.choice(["f32", "bf16"])
        hi = _log_int(rng, 16, 32768)
        lo = rng.choice([0, hi // 8, hi])
        if kind == "decode":
            layers = rng.choice(["full", "global", "sliding", "ring", "sliding,full", "ring,global"])
        elif kind == "layer":
            layers, dtype = rng.choice(["ring", "global", "sliding"]), "f32"
        elif kind == "speculate":
            layers, draft, hi = rng.choice(["full", "global", "full,full"]), rng.randint(1, 4), min(hi, 8192)
            lo = max(1, min(lo, hi))
        elif kind == "verify":
            layers, draft = rng.choice(["ring", "global", "full", "ring,global"]), rng.randint(2, 5)
        elif kind == "prefill":
            layers, dtype = rng.choice(["full", "full", "sliding"]), "bf16"
            batch, chunk, hi = _log_int(rng, 1, 8), _log_int(rng, 8, 2048), min(hi, 8192)
            lo = min(lo, hi)
        elif kind == "produce":
            layers, batch = rng.choice(["full", "ring", "global"]), _log_int(rng, 1, 32)
            chunk = _log_int(rng, 1, 1000 if layers == "ring" else 2048)
        else:
            layers, dtype, hi = "global", "f32", max(hi, 256)
            lo = rng.choice([128, hi // 8 + 1, hi])
        c = _case(kind, None, layers, batch, lo, hi, dtype, draft, chunk, mix)
        w = work(c)
        if w["bytes"] <= 2.0e9 and w["flops"] <= 4.0e11 and _pool_bytes(c) <= 4.0e9:
            return c


# ----------------------------------------------------------------- what a case amounts to
def _lens(case):
    """Cached tokens of each sequence before the step."""
    rng = random.Random(case["mix"])
    return [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]


def _counts(case):
    """New tokens of each sequence."""
    if case["kind"] in ("prefill", "produce"):
        return [case["chunk"]] * case["batch"]
    if case["kind"] == "verify":
        rng = random.Random(case["mix"] + 1)
        return [rng.randint(1, case["draft"]) for _ in range(case["batch"])]
    return [case["draft"]] * case["batch"]


def _layers(case):
    return [LAYERS[n] for n in case["layers"].split(",")]


def _elt(case):
    return 2 if case["dtype"] == "bf16" else 4


def _blocks(case):
    """(blocks in each paged pool, table entries per sequence)"""
    need = [(n + m + BS - 1) // BS for n, m in zip(_lens(case), _counts(case))]
    return int(math.ceil(sum(need) * 1.1)) + 1, max(need) + 1


def _pool_bytes(case):
    nb = _blocks(case)[0]
    return sum(2 * (case["batch"] * r if r else nb * BS) * g * d * _elt(case) for g, d, _, r in _layers(case))


def _window_start(pos, window):
    return max(0, pos - window + 1) if window > 0 else 0


def work(case):
    kind, elt = case["kind"], _elt(case)
    nbytes = flops = 0
    lens, counts = _lens(case), _counts(case)
    rows = sum(counts)
    if kind == "lsa":
        g, d, _, _ = _layers(case)[0]
        lists = _lsa(case)["lists"]
        keys = sum(len(x) for x in lists)
        return {"bytes": keys * (2 * g * d * elt + 4) + 2 * len(lists) * HQ * d * 4, "flops": 4 * HQ * d * keys}
    for g, d, window, _ in _layers(case):
        new = 2 * rows * g * d * elt  # the new K and V rows as they lie in the pool
        if kind in ("layer", "produce"):
            v_in = 1 if (g, d) != (2, 512) else 0  # global layers take V from K
            nbytes += rows * (HQ + g * (1 + v_in)) * d * 4 + new
            if kind == "produce":
                nbytes += rows * HQ * d * elt
                flops += rows * (HQ + 2 * g) * d * 8
                continue
        else:
            nbytes += 2 * new
        q_elt = 2 if kind == "prefill" else 4
        if kind != "layer":
            nbytes += rows * HQ * d * q_elt
        nbytes += rows * HQ * d * 4
        for n, m in zip(lens, counts):
            span = n + m - _window_start(n, window)
            nbytes += (span - m) * 2 * g * d * elt + (span + BS - 1) // BS * 4
            full = sum(n + j + 1 - _window_start(n + j, window) for j in range(m))
            flops += 4 * d * HQ * full
            if kind == "speculate":  # the drafting reads, each over the same keys
                nbytes += case["draft"] * (n * 2 * g * d * elt + 2 * HQ * d * 4)
                flops += 4 * d * HQ * n * case["draft"]
        if kind == "layer":
            c_in = HQ * d
            nbytes += HIDDEN * (c_in // 2 + c_in // 32 * 4) + rows * HIDDEN * 4
            flops += 2 * rows * HIDDEN * c_in
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what this path shows against exact(); pool bytes, block tables, free
    lists, key lists and statuses are whole numbers and have to agree."""
    if case["kind"] == "produce":
        # bf16: a value near the middle of two neighbours may round to either (one unit is
        # 2^-8); fp32: the norms' fp32 factor.
        return {"rel": 2e-4, "max": 0.016} if case["dtype"] == "bf16" else {"rel": 5e-7}
    if case["kind"] == "layer":
        return {"rel": 8e-7}  # the norms' fp32 factor, fp32 sums over c_in behind the attention
    if case["dtype"] == "bf16":
        # fp32 sums; the matrix-core paths carry P (and the verify's Q) as two bf16 parts,
        # 2^-16 of each product.
        return {"rel": 2e-5}
    return {"rel": 1e-7}  # sums in double, rounded once to fp32


# ------------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _lsa(case):
    """Bucket cache, picks and key lists of an LSA step (numpy; decided by the case)."""
    rng = np.random.default_rng(case["mix"])
    lens = _lens(case)
    max_buckets = (max(lens) + 512 + 511) // 512 * 32
    b = case["batch"]
    sizes = np.zeros((b, max_buckets), np.int32)
    members = np.zeros((b, max_buckets, LSA_CAP), np.int32)
    picked = np.zeros((b, LSA_PICK), np.int32)
    n_picked = np.zeros(b, np.int32)
    lists = []
    for s, n in enumerate(lens):  # the query sits at position n - 1
        nbk = min(n // 16 + 1, max_buckets)
        sizes[s, :nbk] = np.minimum(rng.integers(8, LSA_CAP + 1, nbk), n)
        members[s, :nbk] = rng.integers(0, n, (nbk, LSA_CAP))
        pick = rng.choice(nbk, min(LSA_PICK, nbk), replace=False)
        picked[s, :pick.size], n_picked[s] = pick, pick.size
        start = max(0, n - LSA_WINDOW)
        cat = np.concatenate([members[s, p, :sizes[s, p]] for p in pick])
        cat = cat[(cat >= LSA_SINKS) & (cat < start)][:LSA_TOP_K]
        lists.append(np.concatenate([cat, np.arange(start, n), np.arange(min(LSA_SINKS, start))]).astype(np.int64))
    return {"sizes": sizes, "members": members, "picked": picked, "n_picked": n_picked, "lists": lists,
            "max_buckets": max_buckets}


def _inputs(case, seed):
    """What the seed decides: pools, block tables and the step's new values."""
    g = _gen(seed)
    host = np.random.default_rng(seed)
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    kind = case["kind"]
    lens, counts = _lens(case), _counts(case)
    b, rows = case["batch"], sum(counts)
    nb, stride = _blocks(case)
    perm = host.permutation(nb).astype(np.int32)
    tables, held = np.zeros((b, stride), np.int32), np.zeros(b, np.int32)
    at = 0
    for s, n in enumerate(lens):
        held[s] = (n + BS - 1) // BS
        tables[s, :held[s]] = perm[at:at + held[s]]
        at += held[s]
    x = {"lens": lens, "counts": counts, "tables": tables, "held": held, "free": np.sort(perm[at:]),
         "admit": host.permutation(b), "off": np.concatenate([[0], np.cumsum(counts)]).astype(np.int32),
         "num_blocks": nb, "stride": stride, "layers": []}
    for hkv, d, window, ring in _layers(case):
        y = {}
        shape = (b, ring, hkv, d) if ring else (nb, BS, hkv, d)
        y["k"], y["v"] = _normal(g, *shape, dtype=dt), _normal(g, *shape, dtype=dt)
        if kind in ("layer", "produce"):
            y["q"] = _normal(g, rows, HQ, d)
            y["k_new"] = _normal(g, rows, hkv, d)
            y["v_new"] = None if (hkv, d) == (2, 512) else _normal(g, rows, hkv, d)
            y["qw"], y["kw"] = 1 + 0.1 * _normal(g, d), 1 + 0.1 * _normal(g, d)
        else:
            per = case["draft"] if kind != "prefill" else 0
            y["q"] = _normal(g, rows, HQ, d, dtype=dt) if kind == "prefill" else _normal(g, b, per, HQ, d)
            y["k_new"], y["v_new"] = _normal(g, rows, hkv, d, dtype=dt), _normal(g, rows, hkv, d, dtype=dt)
        if kind == "speculate":
            y["reads"] = _normal(g, case["draft"], b, 1, HQ, d)
        if kind == "layer":
            c_in = HQ * d
            y["w"] = torch.randint(0, 256, (HIDDEN, c_in // 2), generator=g, device="cuda", dtype=torch.uint8)
            y["ws"] = 0.001 + 0.01 * torch.rand(HIDDEN, c_in // 32, generator=g, device="cuda")
        x["layers"].append(y)
    if kind in ("speculate", "verify"):
        # drafts accepted of each sequence
        x["accept"] = np.array([int(host.integers(0, m + 1)) for m in counts], np.int32)
    return x


# ------------------------------------------------------------------------------ prepare
class _Foreign:
    """Device memory of the package, as torch sees it."""

    def __init__(self, arr, shape, typestr):
        self.arr = arr  # keeps the allocation
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (arr.ptr, False),
                                         "strides": None, "version": 2}


def _view(arr, dtype):
    """A torch tensor over a hip.DeviceArray."""
    typestr = {torch.float32: "<f4", torch.int32: "<i4", torch.bfloat16: "<i2", torch.uint8: "|u1"}[dtype]
    t = torch.as_tensor(_Foreign(arr, arr.shape, typestr), device="cuda")
    return t.view(torch.bfloat16) if dtype == torch.bfloat16 else t


def _package():
    """The package, on the HIP runtime that torch has loaded (one runtime per process)."""
    import pkv

    old = os.environ.get("ROCM_PATH")
    os.environ["ROCM_PATH"] = os.path.dirname(torch.__file__)
    try:
        pkv.load()
    finally:
        if old is None:
            del os.environ["ROCM_PATH"]
        else:
            os.environ["ROCM_PATH"] = old
    return pkv


def _bits(t):
    """Pool bytes as whole numbers."""
    return t.view(torch.int64)


def prepare(case, seed):
    pkv = _package()
    from pkv import hip

    x = _inputs(case, seed)
    kind, b = case["kind"], case["batch"]
    bf16 = case["dtype"] == "bf16"
    kv = pkv.BF16 if bf16 else pkv.F32
    dt = torch.bfloat16 if bf16 else torch.float32
    specs = [pkv.LayerSpec(HQ, g, d, window=w, kv_dtype=kv, ring_size=r) for g, d, w, r in _layers(case)]
    cache = pkv.PagedKVCache(specs, block_size=BS, num_blocks=x["num_blocks"], max_seqs=b,
                             max_blocks_per_seq=x["stride"], max_q_len=max(1, case["draft"]), scale=SCALE)
    cache.tables.upload(x["tables"])
    cache.table_lens.upload(x["held"])
    cache.free_list.upload_at(0, x["free"])
    cache.free_count.upload(np.array([x["free"].size], np.int32))
    if any(s.ring_size for s in specs):
        cache.admit([int(s) for s in x["admit"]])

    def ints(v):
        return hip.DeviceArray.from_numpy(np.asarray(v, np.int32))

    st = {"kind": kind, "cache": cache, "batch": b, "pos": ints(x["lens"]), "off": ints(x["off"]),
          "most": max(x["counts"]), "rows": int(x["off"][-1]), "layers": [], "keep": x}
    res = {"status": _view(cache.status, torch.int32), "tables": _view(cache.tables, torch.int32),
           "lens": _view(cache.table_lens, torch.int32), "free": _view(cache.free_list, torch.int32),
           "free_count": _view(cache.free_count, torch.int32)}
    for i, y in enumerate(x["layers"]):
        pools = [_view(a, dt) for a in (cache.k_pools[i], cache.v_pools[i])]
        pools[0].copy_(y.pop("k"))
        pools[1].copy_(y.pop("v"))
        q = y["q"]
        z = {n: t.data_ptr() for n, t in y.items() if isinstance(t, torch.Tensor)}
        z.setdefault("v_new", None)
        if kind == "produce":
            out = torch.zeros(q.shape, dtype=dt, device="cuda")
            z["q_dtype"] = kv
        else:
            out = torch.zeros(q.shape, dtype=torch.float32, device="cuda")
        z["out"] = out.data_ptr()
        res["out%d" % i] = out
        # appended rows: copies, to the byte; the producer step's are computed
        computed = kind in ("layer", "produce")
        res["k%d" % i], res["v%d" % i] = pools if computed else [_bits(p) for p in pools]
        if kind == "layer":
            z["qn"] = torch.empty_like(q)
            y["qn"], z["qn"] = z["qn"], z["qn"].data_ptr()
            y["proj"] = torch.zeros(b, HIDDEN, device="cuda")
            z["proj"] = y["proj"].data_ptr()
            res["proj%d" % i] = y["proj"]
            z["c_in"] = HQ * specs[i].head_dim
            z["wo_ws"] = pkv.q4_matmul(z["w"], z["ws"], z["out"], z["proj"], z["c_in"], HIDDEN, b)
        if kind == "speculate":
            y["read_out"] = torch.zeros_like(y["reads"])
            z["read"] = [(y["reads"][j].data_ptr(), y["read_out"][j].data_ptr()) for j in range(case["draft"])]
            res["reads%d" % i] = y["read_out"]
        z["global"] = (specs[i].num_kv_heads, specs[i].head_dim) == (2, 512)
        st["layers"].append(z)
    st["prev"] = ints([n - 1 for n in x["lens"]])
    if kind in ("speculate", "verify"):
        st["counts"] = ints(x["counts"])
        st["new_len"] = ints(np.asarray(x["lens"], np.int32) + x["accept"])
    if kind == "lsa":
        e = _lsa(case)
        lsa = pkv.LSABucketCache(b, max_capacity=e["max_buckets"] // 32 * 512)
        lsa.sizes.upload(e["sizes"])
        lsa.members.upload(e["members"])
        per = lsa.max_keys(LSA_TOP_K, LSA_SINKS, LSA_WINDOW)
        st.update(lsa=lsa, index=ints(range(b)), picked=hip.DeviceArray.from_numpy(e["picked"]),
                  n_picked=ints(e["n_picked"]), max_keys=per, keys=hip.DeviceArray((b * per,), np.int32, zero=True),
                  key_off=hip.DeviceArray((b + 1,), np.int32, zero=True),
                  lsa_status=hip.DeviceArray((b,), np.int32, zero=True))
        res = {"out": res["out0"], "keys": _view(st["keys"], torch.int32), "key_off": _view(st["key_off"], torch.int32),
               "status": _view(st["lsa_status"], torch.int32)}
    st["results"] = res
    st["q4"] = pkv.q4_matmul
    return st


# ---------------------------------------------------------------------------------- run
def run(st):
    kind, cache, b, pos, off, most, rows = (st[n] for n in ("kind", "cache", "batch", "pos", "off", "most", "rows"))
    for i, z in enumerate(st["layers"]):
        if kind == "decode":
            cache.append_attend(i, pos.ptr, off.ptr, z["k_new"], z["v_new"], 1, rows, z["q"], 1, z["out"])
        elif kind == "layer":
            cache.append_qkv(i, pos.ptr, off.ptr, z["q"], z["k_new"], z["v_new"], z["qw"], z["kw"], z["qn"], 1, rows,
                             z["global"])
            cache.attend(i, z["qn"], pos.ptr, 1, z["out"])
            st["q4"](z["w"], z["ws"], z["out"], z["proj"], z["c_in"], HIDDEN, b, workspace=z["wo_ws"])
        elif kind == "speculate":
            for q, out in z["read"]:
                cache.attend(i, q, st["prev"].ptr, 1, out)
        elif kind == "verify":
            cache.append(i, pos.ptr, off.ptr, z["k_new"], z["v_new"], most, rows)
            cache.verify(i, z["q"], pos.ptr, st["counts"].ptr, cache.max_q_len, z["out"])
        elif kind == "prefill":
            cache.append(i, pos.ptr, off.ptr, z["k_new"], z["v_new"], most, rows)
            cache.prefill(i, z["q"], pos.ptr, off.ptr, most, z["out"])
        elif kind == "produce":
            cache.append_qkv(i, pos.ptr, off.ptr, z["q"], z["k_new"], z["v_new"], z["qw"], z["kw"], z["out"], most,
                             rows, z["global"], z["q_dtype"])
        else:
            st["lsa"].expand(st["index"], st["picked"], st["n_picked"], st["prev"], LSA_TOP_K, LSA_SINKS, LSA_WINDOW,
                             keys=st["keys"], key_off=st["key_off"], status=st["lsa_status"])
            cache.attend_sparse(i, z["q"], st["keys"], st["key_off"].ptr, st["max_keys"], z["out"])
    if kind == "speculate":
        for i, z in enumerate(st["layers"]):
            cache.append_attend(i, pos.ptr, off.ptr, z["k_new"], z["v_new"], most, rows, z["q"], most, z["out"])
    if kind in ("speculate", "verify"):
        cache.rollback(st["new_len"].ptr)
    return st["results"]


# -------------------------------------------------------------------------------- exact
def _attention64(q, k, v, t0, pos, window):
    """q [nq][HQ][d] at positions pos, pos + 1, ...; k, v [n][hkv][d] at t0, t0 + 1, ...
    (t0 None: every query attends every key)."""
    nq, hq, d = q.shape
    hkv = k.shape[1]
    grp = hq // hkv
    q = q.double() * SCALE
    out = torch.empty(nq, hq, d, dtype=torch.float64, device=q.device)
    if t0 is not None:
        t = torch.arange(t0, t0 + k.shape[0], device=q.device)[None, :]
        p = torch.arange(pos, pos + nq, device=q.device)[:, None]
        live = (t <= p) & (t > p - window if window > 0 else t >= 0)
    for g in range(hkv):
        kg, vg = k[:, g].double(), v[:, g].double()
        for h in range(g * grp, (g + 1) * grp):
            s = q[:, h] @ kg.t().contiguous()
            if t0 is not None:
                s = s.masked_fill(~live, -math.inf)
            e = torch.exp(s - s.max(dim=1, keepdim=True).values)
            out[:, h] = (e @ vg) / (e.sum(dim=1, keepdim=True) + 1e-10)
    return out


def _rms64(x, w):
    y = x.double() / torch.sqrt(x.double().square().mean(dim=-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _rope64(x, positions, is_global):
    """Rotation of pairs (i, i + d/2); the angles are the reference's fp32 quotients."""
    d = x.shape[-1]
    half = d // 2
    n, base, dim = (min(64, half), 1e6, 512) if is_global else (half, 1e4, 256)
    den = torch.tensor([np.float32(base ** (2.0 * i / dim)) for i in range(n)], dtype=torch.float32, device=x.device)
    ang = (positions.float()[:, None] / den[None, :]).double()
    c, s = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    y = x.clone()
    a, b = x[..., :n], x[..., half:half + n]
    y[..., :n] = a * c - b * s
    y[..., half:half + n] = b * c + a * s
    return y


def _produced64(y, x, is_global):
    pos = torch.tensor([n + j for n, m in zip(x["lens"], x["counts"]) for j in range(m)], device="cuda")
    v_in = y["k_new"] if y["v_new"] is None else y["v_new"]
    return (_rope64(_rms64(y["q"], y["qw"]), pos, is_global), _rope64(_rms64(y["k_new"], y["kw"]), pos, is_global),
            _rms64(v_in, None))


def _keys64(x, y, s, spec, lo, hi, slot_of, rows, new):
    """K and V of positions lo .. hi - 1 of sequence s: cached rows, then the new ones."""
    hkv, d, _, ring = spec
    n = x["lens"][s]
    t = torch.arange(lo, min(hi, n), device="cuda")
    if ring:
        at = int(slot_of[s]) * ring + t % ring
    else:
        table = torch.from_numpy(x["tables"][s].astype(np.int64)).cuda()
        at = table[t // BS] * BS + t % BS
    r0 = int(x["off"][s]) + max(lo - n, 0)
    r1 = int(x["off"][s]) + max(hi - n, 0)
    got = []
    for pool, fresh in ((y["k"], new[0]), (y["v"], new[1])):
        got.append(torch.cat([pool.reshape(-1, hkv, d)[at].double(), fresh[r0:r1].double()]))
    return got


def exact(case, seed):
    x = _inputs(case, seed)
    kind, lens, counts = case["kind"], x["lens"], x["counts"]
    slot_of = np.zeros(case["batch"], np.int64)
    for k, s in enumerate(x["admit"]):
        slot_of[s] = k
    res = {}
    for i, (y, spec) in enumerate(zip(x["layers"], _layers(case))):
        hkv, d, window, _ = spec
        is_global = (hkv, d) == (2, 512)
        q, new = y["q"], (y["k_new"], y["v_new"])
        if kind in ("layer", "produce"):
            q, *new = _produced64(y, x, is_global)
        if kind == "produce":
            res["out%d" % i] = q
            continue
        if kind == "lsa":
            out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
            for s, keys in enumerate(_lsa(case)["lists"]):
                k, v = _keys64(x, y, s, spec, 0, lens[s], slot_of, None, new)
                at = torch.from_numpy(keys).cuda()
                out[s] = _attention64(q[s], k[at], v[at], None, 0, 0)
            return {"out": out}
        out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
        reads = torch.zeros(y["reads"].shape, dtype=torch.float64, device="cuda") if kind == "speculate" else None
        for s, (n, m) in enumerate(zip(lens, counts)):
            lo = _window_start(n, window)
            k, v = _keys64(x, y, s, spec, lo, n + m, slot_of, None, new)
            if kind in ("prefill", "layer"):
                r0 = int(x["off"][s])
                out[r0:r0 + m] = _attention64(q[r0:r0 + m], k, v, lo, n, window)
            else:
                out[s, :m] = _attention64(q[s, :m], k, v, lo, n, window)
            if reads is not None:
                for j in range(case["draft"]):
                    reads[j, s] = _attention64(y["reads"][j, s], k[:n], v[:n], lo, n - 1, window)
        res["out%d" % i] = out
        if reads is not None:
            res["reads%d" % i] = reads
        if kind == "layer":
            w = torch.stack([(y["w"] & 15).double() - 8, (y["w"] >> 4).double() - 8], dim=-1).reshape(HIDDEN, -1)
            w *= y["ws"].double().repeat_interleave(32, dim=1)
            res["proj%d" % i] = out.reshape(case["batch"], -1) @ w.t().contiguous()
    return res
