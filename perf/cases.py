"""What this library is timed on: the calls a decode loop makes through the C ABI.

Geometry is fixed by the contract (32 query heads, 8 KV heads, 128 channels,
alpha-margin selection under a 20 % cap), so a case is a path through the
entry points, a number of tokens and the options a program really varies:
the pool's layout, the row map, the order of the ids, the number of
sequences, query positions and cold rows.  A workspace is sized by the cap,
so its slots past a smaller selection are padding, as in a running decode.

Inputs are RoPE-rotated Gaussian keys and Gaussian queries and values in F16,
as in the benchmark.  The calls are bound to their buffers once, as a decode
loop that reuses its buffers binds them, and every pass makes the whole call.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import hillserve_amd as hs

H, KH, D = 32, 8, 128
RATIO = 0.2
RATIO32 = float(np.float32(RATIO))
THETA = 500000.0
ROOT128 = np.float32(math.sqrt(128.0))


# ---- the cases -----------------------------------------------------------------

def listed():
    return [
        # one sparse layer of a decode step, alone: score, select, attend.
        # A short sequence, where five dependent launches count
        dict(name="layer_1k", path="layer", n=1024, layout="arrays", paged=False, alpha=5.0),
        # a paged hot pool of the reference's 4096 B KV records behind a row
        # map, at a token count that fills neither a tile nor a bitmap word
        dict(name="layer_8k_paged", path="layer", n=7919, layout="records", paged=True, alpha=5.0),
        # the benchmark's layer: K and V arrays at the V3 limit of 32768 tokens
        dict(name="layer_32k", path="layer", n=32768, layout="arrays", paged=False, alpha=5.0),
        # the scorer's largest call: beyond the V3 limit, selection below the cap
        dict(name="layer_64k", path="layer", n=65536, layout="arrays", paged=False, alpha=3.0),
        # the decode loop: the next layer's history scored beside this layer's
        # rank-order selection, which completes its current token, then attention
        dict(name="pipeline_8x32k", path="pipeline", n=32768, layers=8, alpha=5.0),
        # history cover of a long sequence and its union: what a prefetch reads
        dict(name="cover_48k", path="cover", n=48001, alpha=5.0),
        # the next layer's query for a full batch of sequences
        dict(name="rehearsal_16", path="rehearsal", batch=16),
        # scoring and rank-order selection of 16 sequences of mixed lengths
        dict(name="batch_16", path="batch", sequences=16, lowest=8192, highest=32768, step=64,
             lengths=5, alpha=5.0),
        # the union of a selection and its packed workspace: one query position
        # (decode), and a 64-token prompt chunk over a shorter context
        dict(name="pack_decode_32k", path="pack", n=32768, nq=1, alpha=5.0),
        dict(name="pack_chunk_8k", path="pack", n=8192, nq=64, alpha=5.0),
        # gather of prefetched and missed rows into the packed layout
        dict(name="gather_32k", path="gather", n=32768, missed=0.25, alpha=5.0),
        # half the 64-token blocks in pinned host memory: plan, fetch the
        # selected cold rows over the host link, attend over both tiers
        dict(name="tier_8k", path="tier", n=8192, cold=0.5, alpha=5.0),
    ]


def _log_uniform(rng, low, high):
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    return min(high, max(low, n))


def draw(rng):
    path = rng.choice(["layer", "layer", "layer", "pipeline", "cover", "rehearsal", "batch",
                       "pack", "gather", "tier"])
    alpha = rng.choice([3.0, 4.0, 5.0, 5.0])
    if path == "layer":
        return dict(path=path, n=_log_uniform(rng, 256, 65536), layout=rng.choice(["arrays", "records"]),
                    paged=rng.random() < 0.4, alpha=alpha)
    if path == "pipeline":
        return dict(path=path, n=_log_uniform(rng, 1024, 32768), layers=rng.randint(2, 8), alpha=alpha)
    if path == "cover":
        return dict(path=path, n=_log_uniform(rng, 1024, 65536), alpha=alpha)
    if path == "rehearsal":
        return dict(path=path, batch=rng.randint(1, 15), position=rng.randint(0, 65535))
    if path == "batch":
        low = _log_uniform(rng, 512, 16384)
        return dict(path=path, sequences=rng.randint(2, 16), lowest=low, highest=min(32768, 2 * low + rng.randint(0, 4095)),
                    step=rng.choice([1, 64]), lengths=rng.randint(0, 1 << 30), alpha=alpha)
    if path == "pack":
        nq = rng.choice([1, 1, rng.randint(2, 96)])
        return dict(path=path, n=_log_uniform(rng, 512, 32768 if nq == 1 else 12288), nq=nq, alpha=alpha)
    if path == "gather":
        return dict(path=path, n=_log_uniform(rng, 512, 32768), missed=rng.choice([0.0, 0.1, 0.5]), alpha=alpha)
    return dict(path=path, n=_log_uniform(rng, 1024, 8192), cold=rng.choice([0.25, 0.5]), alpha=alpha)


def _lengths(case):
    """Tokens of each sequence of a batch: fixed by the case."""
    g = np.random.default_rng(case["lengths"])
    lo, hi, step = case["lowest"], case["highest"], case["step"]
    return [int(x) * step for x in g.integers(-(-lo // step), hi // step + 1, size=case["sequences"])]


def _cap(n):
    return math.floor(n * RATIO32)


def _packed_slots(n):
    """Slots of the packed workspace: the cap, in whole multiples of 32."""
    return max(32, (_cap(n) + 31) // 32 * 32)


def _share(n, alpha):
    """Share of the tokens a head selects when scaled scores are N(0, 1)."""
    top = math.sqrt(2.0 * math.log(n))
    return min(RATIO32, 0.5 * math.erfc((top - alpha) / math.sqrt(2.0)))


def work(case):
    """Bytes and operations of one pass: each input once, each output once."""
    path = case["path"]
    if path == "rehearsal":
        b = case["batch"]
        return {"bytes": 2 * 4096 * 4096 + 4 * 4096 * b, "flops": 2 * 4096 * 4096 * b}
    if path == "batch":
        n = sum(_lengths(case))
        k = sum(int(m * _share(m, case["alpha"])) for m in _lengths(case))
        return {"bytes": n * (2048 + 64) + 4 * H * k, "flops": 8192 * n}
    n, f = case["n"], _share(case["n"], case["alpha"])
    k, union = int(f * n), 1.0 - (1.0 - f) ** 4  # of a KV head's four query heads
    any_head = 1.0 - (1.0 - f) ** H
    score = n * (2048 + 64)
    attend = 2 * 2 * H * D * k  # flops
    if path == "layer":
        return {"bytes": score + 4 * H * k + 256 * KH * union * n + 16384 + 24576,
                "flops": 8192 * n + attend}
    if path == "pipeline":
        one = score + 4 * H * k + 512 * KH * union * n + 24576
        return {"bytes": case["layers"] * one, "flops": case["layers"] * (8192 * n + attend)}
    if path == "cover":
        return {"bytes": score + 4 * H * k + 4 * any_head * n, "flops": 8192 * n}
    slots = _packed_slots(n)
    if path == "pack":
        qpad = -(-case["nq"] // 64) * 64
        return {"bytes": 4 * H * k + 4 * any_head * n + 512 * KH * union * n
                         + slots * H * (2 * 2 * D + 4 * qpad), "flops": 0}
    if path == "gather":
        return {"bytes": 4 * H * slots + 512 * KH * union * n + slots * H * 2 * 2 * D, "flops": 0}
    cold = case["cold"] * any_head * n  # records that cross the host link
    return {"bytes": 4 * H * n / 32 + 8 * n + 2 * 4128 * cold + 512 * KH * union * n + 32768, "flops": attend}


def tolerance(case):
    """Scores, ids, counts and copied bytes are the contract's, bit for bit
    (whole numbers may not differ at all).  Attention rounds its softmax
    weights to F16 and measures 1.7e-4 from 64 bits; the query is rounded to
    F16 once, 2.1e-4."""
    if case["path"] in ("layer", "pipeline", "tier", "rehearsal"):
        return {"rel": 8e-4, "max": 4e-3}
    return "exact"


# ---- inputs (torch, from the seed alone) ------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _keys(n, g):
    """K F16 [n][8][128]: N(0, 1), adjacent channel pairs rotated at position t."""
    x = torch.randn((n, KH, D // 2, 2), generator=g, device="cuda")
    freq = THETA ** (-torch.arange(D // 2, device="cuda", dtype=torch.float64) * 2.0 / D)
    angle = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] * freq
    c, s = angle.cos().float()[:, None, :], angle.sin().float()[:, None, :]
    out = torch.stack((x[..., 0] * c - x[..., 1] * s, x[..., 0] * s + x[..., 1] * c), dim=-1)
    return out.reshape(n, KH, D).half()


def _normal(shape, g, dtype=torch.float16):
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _queries(g):
    """The attention's query in F32 and the rehearsal's F16 estimate of it."""
    q32 = torch.randn((H, D), generator=g, device="cuda")
    return (q32 + 0.1 * torch.randn((H, D), generator=g, device="cuda")).half(), q32


def _slots(n, g, spare):
    """Pool rows of n tokens kept in 64-token blocks at shuffled places, with
    `spare` free blocks among them, and the pool's rows."""
    blocks = (n + 63) // 64
    place = torch.randperm(blocks + spare, generator=g, device="cuda")[:blocks]
    t = torch.arange(n, device="cuda")
    return (place[t // 64] * 64 + t % 64).int(), (blocks + spare) * 64


def _layer_inputs(case, seed):
    g = _generator(seed)
    n = case["n"]
    return dict(k=_keys(n, g), v=_normal((n, KH, D), g), q=_queries(g), g=g)


def _pipeline_inputs(case, seed):
    return [_layer_inputs(case, seed * 64 + l) for l in range(case["layers"])]


def _batch_inputs(case, seed):
    g = _generator(seed)
    return [(_keys(n, g), _normal((H, D), g)) for n in _lengths(case)]


def _rehearsal_inputs(case, seed):
    g = _generator(seed)
    b = case["batch"]
    first = case.get("position", 8192)
    return dict(hidden=_normal((b, 4096), g, torch.bfloat16),
                wq=(torch.randn((4096, 4096), generator=g, device="cuda") * 0.02).bfloat16(),
                positions=[first + 1531 * i for i in range(b)])


# ---- binding calls ---------------------------------------------------------------------

def _arg(x):
    return ctypes.c_void_p(x.data_ptr()) if isinstance(x, torch.Tensor) else x


def _bind(name, *args):
    """The entry point on fixed buffers and the current stream; raises on a
    nonzero status."""
    fn = getattr(hs.lib(), name)
    full = tuple(_arg(x) for x in args) + (ctypes.c_void_p(torch.cuda.current_stream().cuda_stream),)

    def call():
        rc = fn(*full)
        if rc:
            hs.check(rc)

    call.keep = args
    return call


def _table(kind, jobs):
    t = (kind * len(jobs))(*(kind(*(_arg(x) for x in j)) for j in jobs))
    t.keep = jobs
    return t


def _zeros(shape, dtype=torch.int32):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _bytes(n):
    return torch.empty(max(256, int(n)), dtype=torch.uint8, device="cuda")


def _select_buffers(n, cap):
    return dict(ids=_zeros((H, max(1, cap))), counts=_zeros(H), member=_zeros((H, (n + 31) // 32)),
                status=_zeros(4), ws=_bytes(hs.lib().hs_gqa_select_workspace_bytes(H, n)))


def _select_job(scores, stride, n, partial, b, q=None, key=None):
    return (scores, partial, b["ids"], b["counts"], b["member"], b["status"], b["ws"], stride, n,
            b["ids"].shape[1], 0, q, key)


def _selection(k, q16, alpha):
    """Ids [32][cap] in rank order and k, selected by the library."""
    n = k.shape[0]
    raw, part, b = _zeros((H, n), torch.float16), _zeros((n + 63) // 64), _select_buffers(n, _cap(n))
    _bind("hs_gqa_score", q16, k, 1024, None, 0, n, raw, n, part)()
    _bind("hs_gqa_select", raw, H, n, n, alpha, RATIO, hs.HS_SELECT_SCALE_RAW, part, b["ids"],
          b["ids"].shape[1], b["counts"], b["member"], b["status"], b["ws"])()
    status = b["status"].tolist()
    assert status[0] == 0 and status[1] > 0, status
    return b, status[1]


# ---- prepare -----------------------------------------------------------------------------

def _prepare_layer(case, seed):
    x = _layer_inputs(case, seed)
    n, (q16, q32) = case["n"], x["q"]
    cap, rows, pool_rows = _cap(n), None, n
    if case["paged"]:
        rows, pool_rows = _slots(n, x["g"], 16)
    at = rows.long() if rows is not None else torch.arange(n, device="cuda")
    if case["layout"] == "records":
        pool = _zeros((pool_rows, 2, KH, D), torch.float16)
        pool[at, 0], pool[at, 1] = x["k"], x["v"]
        kp, vp, row_bytes = pool, ctypes.c_void_p(pool.data_ptr() + 2048), 4096
        keep = pool
    else:
        kp, vp = _zeros((pool_rows, KH, D), torch.float16), _zeros((pool_rows, KH, D), torch.float16)
        kp[at], vp[at] = x["k"], x["v"]
        row_bytes, keep = 2048, (kp, vp)
    out = dict(scores=_zeros((H, n), torch.float16), ids=_zeros((H, cap)), counts=_zeros(H),
               out=_zeros((H, D), torch.float32), status=_zeros(4))
    ws = _bytes(hs.lib().hs_decode_layer_workspace_bytes(n))
    call = _bind("hs_decode_layer", q16, q32, kp, vp, row_bytes, rows, pool_rows, n, case["alpha"],
                 RATIO, 0, out["scores"], out["ids"], cap, out["counts"], out["out"], out["status"], ws)
    return dict(calls=[call], out=out, keep=(keep, ws))


def _prepare_pipeline(case, seed):
    layers = _pipeline_inputs(case, seed)
    n, alpha, count = case["n"], case["alpha"], case["layers"]
    stride, cap, flags = (n + 7) // 8 * 8, _cap(n), hs.HS_SELECT_SCALE_RAW
    raws = _zeros((count, H, stride), torch.float16)
    parts = _zeros((count, (n - 1 + 63) // 64))
    ids, outs = _zeros((count, H, cap)), _zeros((count, H, D), torch.float32)
    status = _zeros((count, 4))
    member = _zeros((H, (n + 31) // 32))
    sel_ws = _bytes(hs.lib().hs_gqa_select_workspace_bytes(H, n))
    att_ws = _bytes(hs.lib().hs_gqa_attention_workspace_bytes(n))
    hist, sel = [], []
    for l, x in enumerate(layers):
        b = dict(ids=ids[l], counts=_zeros(H), member=member, status=status[l], ws=sel_ws)
        hist.append((x["q"][0], x["k"], raws[l], parts[l], 1024, n - 1, stride, 0))
        sel.append(_table(hs.SelectJob, [_select_job(raws[l], stride, n, parts[l], b, x["q"][0], x["k"][n - 1])]))
    calls = [_bind("hs_gqa_score_batched", _pointer(_table(hs.ScoreJob, hist[:1])), 1)]
    for l, x in enumerate(layers):
        if l + 1 < count:
            calls.append(_bind("hs_gqa_select_then_score", _pointer(sel[l]), 1, H, alpha, RATIO, flags,
                               _pointer(_table(hs.ScoreJob, hist[l + 1:l + 2])), 1))
        else:
            calls.append(_bind("hs_gqa_select_batched", _pointer(sel[l]), 1, H, alpha, RATIO, flags))
        calls.append(_bind("hs_gqa_sparse_attention", x["q"][1], x["k"], x["v"], 2048, None, n, member, n,
                           outs[l], att_ws))
    return dict(calls=calls, out=dict(ids=ids, out=outs, raw=raws[:, :, :n], status=status),
                keep=(layers, sel, member, sel_ws, att_ws))


def _pointer(table):
    p = ctypes.cast(table, ctypes.c_void_p)
    p.keep = table
    return p


def _prepare_cover(case, seed):
    x = _layer_inputs(case, seed)
    n = case["n"]
    cap = min(n, _cap(n + 1))
    raw, part, b = _zeros((H, n), torch.float16), _zeros((n + 63) // 64), _select_buffers(n, cap)
    flags = hs.HS_SELECT_SCALE_RAW | hs.HS_SELECT_COVER
    score = _bind("hs_gqa_score", x["q"][0], x["k"], 1024, None, 0, n, raw, n, part)
    select = _bind("hs_gqa_select", raw, H, n, n, case["alpha"], RATIO, flags, part, b["ids"], cap,
                   b["counts"], b["member"], b["status"], b["ws"])
    score()
    select()
    lens = b["status"][1].repeat(H)  # the cover's bound, known before the union is asked for
    union, union_n, status = _zeros(n), _zeros(1), _zeros(4)
    ws = _bytes(hs.lib().hs_gqa_union_workspace_bytes(n))
    unite = _bind("hs_gqa_physical_union", b["ids"], lens, cap, n, union, union_n, status, ws)
    return dict(calls=[score, select, unite], keep=(x, b, part, lens, ws),
                out=dict(raw=raw, ids=b["ids"], status=b["status"], union=union, union_n=union_n,
                         union_status=status))


def _prepare_rehearsal(case, seed):
    x = _rehearsal_inputs(case, seed)
    b = case["batch"]
    pos = (ctypes.c_uint32 * b)(*x["positions"])
    q, status = _zeros((b, H, D), torch.float16), _zeros((b, 4))
    call = _bind("hs_rehearsal_query", x["hidden"], x["wq"], _pointer(pos), b, 1e-5, THETA, q, status, None)
    return dict(calls=[call], out=dict(q=q, code=status[:, 0]), keep=x)


def _prepare_batch(case, seed):
    x = _batch_inputs(case, seed)
    score, sel, out = [], [], []
    for k, q16 in x:
        n = k.shape[0]
        stride = (n + 7) // 8 * 8
        raw, part, b = _zeros((H, stride), torch.float16), _zeros((n + 63) // 64), _select_buffers(n, _cap(n))
        score.append((q16, k, raw, part, 1024, n, stride, 0))
        sel.append(_select_job(raw, stride, n, part, b))
        out += [raw[:, :n], b["ids"], b["status"]]
    calls = [_bind("hs_gqa_score_batched", _pointer(_table(hs.ScoreJob, score)), len(x)),
             _bind("hs_gqa_select_batched", _pointer(_table(hs.SelectJob, sel)), len(x), H, case["alpha"],
                   RATIO, hs.HS_SELECT_SCALE_RAW)]
    return dict(calls=calls, out=out, keep=x)


def _prepare_pack(case, seed):
    x = _layer_inputs(case, seed)
    n, nq = case["n"], case["nq"]
    b, k = _selection(x["k"], x["q"][0], case["alpha"])
    slots = _packed_slots(n)
    qpad = (nq + 63) // 64 * 64
    lens, cap = torch.full((H,), k, dtype=torch.int32, device="cuda"), b["ids"].shape[1]
    positions = torch.arange(n - nq, n, device="cuda")  # 64-bit, ascending
    out = dict(union=_zeros(n), union_n=_zeros(1), union_status=_zeros(4),
               k=_zeros((slots, H, D), torch.float16), v=_zeros((H, D, slots), torch.float16),
               mask=_zeros((H, qpad, slots), torch.float32))
    status = _zeros(4)
    ws = _bytes(hs.lib().hs_gqa_union_workspace_bytes(n))
    unite = _bind("hs_gqa_physical_union", b["ids"], lens, cap, n, out["union"], out["union_n"],
                  out["union_status"], ws)
    pack = _bind("hs_gqa_pack", x["k"], x["v"], 2048, n, None, n, b["ids"], lens, cap, positions, nq,
                 slots, out["k"], out["v"], out["mask"], status)
    return dict(calls=[unite, pack], out=dict(out, code=status[0]), keep=(x, b, lens, positions, ws))


def _prepare_gather(case, seed):
    x = _layer_inputs(case, seed)
    n = case["n"]
    b, k = _selection(x["k"], x["q"][0], case["alpha"])
    slots = _packed_slots(n)
    ids = b["ids"][:, :k].long()
    union = torch.unique(ids)
    miss = torch.rand(union.numel(), generator=x["g"], device="cuda") < case["missed"]
    row = torch.where(miss, -1 - torch.cumsum(miss, 0), torch.cumsum(~miss, 0) - 1)  # <= -2: miss row
    of_id = torch.full((n,), -1, dtype=torch.int64, device="cuda")
    of_id[union] = row
    table = torch.full((H, slots), -1, dtype=torch.int32, device="cuda")
    table[:, :k] = of_id[ids].int()
    rows = torch.stack((x["k"], x["v"]), dim=1)[union]  # 4096 B records
    pre, misses = rows[~miss].contiguous(), rows[miss].contiguous()
    kk, v, status = _zeros((slots, H, D), torch.float16), _zeros((H, D, slots), torch.float16), _zeros(4)
    call = _bind("hs_gqa_gather_rows", pre, pre.shape[0], misses if misses.numel() else None,
                 misses.shape[0], table, slots, kk, v, status)
    return dict(calls=[call], out=dict(k=kk, v=v, code=status[0]), keep=(pre, misses, table))


def _tier_inputs(case, seed):
    x = _layer_inputs(case, seed)
    n = case["n"]
    full = n // 64  # a last, partial block is still being written: hot
    is_cold = torch.zeros(full + 1, dtype=torch.bool, device="cuda")
    is_cold[torch.randperm(full, generator=x["g"], device="cuda")[:round(case["cold"] * full)]] = True
    x["cold"] = is_cold[torch.arange(n, device="cuda") // 64]
    return x


def _prepare_tier(case, seed):
    x = _tier_inputs(case, seed)
    n, cold = case["n"], x["cold"]
    b, _ = _selection(x["k"], x["q"][0], case["alpha"])
    hot_rows, cold_rows = int((~cold).sum()), int(cold.sum())
    slot = torch.where(cold, -1, torch.cumsum(~cold, 0) - 1).int()
    records = torch.stack((x["k"], x["v"]), dim=1).contiguous()  # [n][K | V]
    pool = _zeros((hot_rows + cold_rows, 2, KH, D), torch.float16)
    pool[:hot_rows] = records[~cold]
    lib = hs.lib()
    image = torch.empty(lib.hs_kv_store_bytes(1, n), dtype=torch.uint8, pin_memory=True)
    host = records.cpu()
    hs.check(lib.hs_kv_store_init(_arg(image), 77, 1, n))
    hs.check(lib.hs_kv_store_append(_arg(image), 0, 0, _arg(host), n))
    out = dict(positions=_zeros(cold_rows), rows=_zeros(n), count=_zeros(1), status=_zeros(4),
               staged=pool[hot_rows:], out=_zeros((H, D), torch.float32))
    staging = ctypes.c_void_p(pool.data_ptr() + 4096 * hot_rows)
    staging_v = ctypes.c_void_p(pool.data_ptr() + 4096 * hot_rows + 2048)
    fetch_ws = _bytes(lib.hs_kv_cold_fetch_workspace_bytes(cold_rows))
    att_ws = _bytes(lib.hs_gqa_attention_workspace_bytes(n))
    calls = [_bind("hs_gqa_cold_plan", b["member"], H, n, slot, hot_rows, cold_rows, out["positions"],
                   out["rows"], out["count"]),
             _bind("hs_kv_cold_fetch", image, 0, out["positions"], cold_rows, staging, staging_v, 4096,
                   out["status"], fetch_ws),
             _bind("hs_gqa_sparse_attention", x["q"][1], pool, ctypes.c_void_p(pool.data_ptr() + 2048), 4096,
                   out["rows"], hot_rows + cold_rows, b["member"], n, out["out"], att_ws)]
    return dict(calls=calls, out=out, keep=(x["q"], b, slot, pool, image, fetch_ws, att_ws))


def prepare(case, seed):
    return globals()["_prepare_" + case["path"]](case, seed)


def run(state):
    for call in state["calls"]:
        call()
    return state["out"]


# ---- the same results in 64 bits ------------------------------------------------------------

def _scores64(q16, k):
    """q.k per query head and token in 64 bits, [32][n]."""
    kt = k.double().permute(1, 2, 0)  # [8][128][n]
    q = q16.double().reshape(KH, 4, D)
    return torch.cat([q[g] @ kt[g] for g in range(KH)])


def _contract_scores(q16, k):
    """The contract's raw scores F16 [32][n]: channels summed in order in
    FP32, one F16 rounding.  They alone decide what is selected."""
    kt = k.float().permute(1, 2, 0).contiguous()  # [8][128][n]
    q = q16.float().reshape(KH, 4, D)
    s = torch.zeros((KH, 4, k.shape[0]), device=k.device)
    for c in range(D):
        s = s + q[:, :, c, None] * kt[:, None, c, :]  # F16 products are exact in FP32
    return s.reshape(H, -1).half()


def _contract_selection(raw, alpha):
    """Membership bool [32][n] of the contract's selection over raw scores."""
    n = raw.shape[1]
    scaled = (raw.float().cpu().numpy() / ROOT128).astype(np.float16)
    thr = np.float16(np.float32(scaled[0].max()) - np.float32(alpha))
    counts = (scaled >= thr).sum(axis=1).astype(np.float16).astype(np.float32)
    mean = np.float16(counts.sum(dtype=np.float32) / np.float32(H))
    k = min(int(mean), _cap(n))
    top = torch.from_numpy(scaled.astype(np.float32)).cuda().sort(dim=1, descending=True, stable=True).indices
    member = torch.zeros((H, n), dtype=torch.bool, device="cuda")
    return member.scatter_(1, top[:, :k], True)


def _attention64(q32, k, v, member):
    dots = _scores64(q32, k) / math.sqrt(128.0)
    p = torch.softmax(dots.masked_fill(~member, -math.inf), dim=1).reshape(KH, 4, -1)
    vt = v.double().permute(1, 0, 2).contiguous()  # [8][n][128]
    return torch.cat([p[g] @ vt[g] for g in range(KH)])


def _exact_layer(x, alpha):
    q16, q32 = x["q"]
    member = _contract_selection(_contract_scores(q16, x["k"]), alpha)
    return _scores64(q16, x["k"]), _attention64(q32, x["k"], x["v"], member)


def exact(case, seed):
    path = case["path"]
    if path == "layer":
        raw, out = _exact_layer(_layer_inputs(case, seed), case["alpha"])
        return dict(scores=raw, out=out)
    if path == "pipeline":
        got = [_exact_layer(x, case["alpha"]) for x in _pipeline_inputs(case, seed)]
        return dict(raw=torch.stack([g[0] for g in got]), out=torch.stack([g[1] for g in got]))
    if path == "cover":
        x = _layer_inputs(case, seed)
        return dict(raw=_scores64(x["q"][0], x["k"]))
    if path == "rehearsal":
        x = _rehearsal_inputs(case, seed)
        h = x["hidden"].double()
        h = h / torch.sqrt((h * h).mean(dim=1, keepdim=True) + 1e-5)
        y = (h @ x["wq"].double().t()).reshape(case["batch"], H, D // 2, 2)
        freq = THETA ** (-torch.arange(D // 2, device="cuda", dtype=torch.float64) * 2.0 / D)
        angle = torch.tensor(x["positions"], device="cuda", dtype=torch.float64)[:, None, None] * freq
        c, s = angle.cos(), angle.sin()
        q = torch.stack((y[..., 0] * c - y[..., 1] * s, y[..., 0] * s + y[..., 1] * c), dim=-1)
        return dict(q=q.reshape(case["batch"], H, D))
    if path == "batch":
        out = []
        for k, q16 in _batch_inputs(case, seed):
            out += [_scores64(q16, k), None, None]
        return out
    if path == "tier":
        x = _tier_inputs(case, seed)
        member = _contract_selection(_contract_scores(x["q"][0], x["k"]), case["alpha"])
        return dict(out=_attention64(x["q"][1], x["k"], x["v"], member))
    return None  # pack and gather copy bytes
