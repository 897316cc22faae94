"""Workloads of the sparse attention path, called as a program calls them.

Every case is one call of a public entry point: the attention forward over a block
index, a disjoint split merged by log-sum-exp, a decode step against a cache, the
backward, the once-per-forward relabelling of Q, K and V, and the build of a block index.
``listed`` holds the fixed ones, ``draw`` gives further ones of the same ranges.
``exact`` is the same result in float64 from plain torch.
"""
import math

import torch

from polyhedral_amd import attention, backward, decode, index, perm, split
from polyhedral_amd.polyattn import masks

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
ESIZE = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # the smallest attention call: one short float32 prompt, where latency and launches
        # count (causal window 128, 4 heads of 64)
        dict(name="window-f32-small", op="attn", dtype="f32", BH=4, N=1024, D=64, BQ=128, A=128, mask="window", p0=128,
             p1=0, stride=0, lse=False),
        # dense causal attention in the reference's own setting (float16, 8 heads of 64, 4096
        # tokens, 128x128 tiles), with the log-sum-exp that training keeps
        dict(name="causal-f16-d64", op="attn", dtype="f16", BH=8, N=4096, D=64, BQ=128, A=128, mask="causal", p0=0,
             p1=0, stride=0, lse=True),
        # the reference's re-indexing benchmark at its longest sequence: every 8th key, the
        # tensors relabelled by residue class beforehand, 128x32 tiles
        dict(name="dilated8-f16-d64", op="attn", dtype="f16", BH=8, N=16384, D=64, BQ=128, A=32, mask="dilated", p0=8,
             p1=0, stride=8, lse=False),
        # the same mask on the finest tiles (16x16), the reference's fastest setting for it
        dict(name="dilated8-f16-16x16", op="attn", dtype="f16", BH=8, N=8192, D=64, BQ=16, A=16, mask="dilated", p0=8,
             p1=0, stride=8, lse=False),
        # the headline workload: band-256 and every 16th key as two passes in two bases,
        # merged by log-sum-exp
        dict(name="bandlat-L16k", op="split", dtype="bf16", BH=32, N=16384, D=128, w=256, s=16),
        # the largest forward: 64 sink tokens and a 1024-token window over 32768 tokens
        dict(name="sinkwin-L32k", op="attn", dtype="bf16", BH=32, N=32768, D=128, BQ=128, A=32, mask="sinks", p0=1024,
             p1=64, stride=0, lse=False),
        # one sequence generating a token: append its key and value, attend the band and
        # lattice keys of a cache held in the residue-16 basis (a length of no round number)
        dict(name="decode-one", op="decode", dtype="bf16", BH=32, D=128, capacity=16384, length=16011, s=16,
             mask="local_strided", p0=256, p1=16, nq=1),
        # a serving batch (8 sequences x 32 heads) generating a token each over their whole
        # context: bound by the bytes of the cache
        dict(name="decode-batch", op="decode", dtype="bf16", BH=256, D=128, capacity=4096, length=3977, s=0,
             mask="causal", p0=0, p1=0, nq=1),
        # training: the gradients of the headline workload
        dict(name="bwd-bandlat-L16k", op="bwd", dtype="bf16", BH=32, N=16384, D=128, mask="local_strided", p0=256,
             p1=16),
        # training a small float16 model with dense causal attention (8 heads of 64; the
        # length is no multiple of 128)
        dict(name="bwd-causal-f16-d64", op="bwd", dtype="f16", BH=8, N=4032, D=64, mask="causal", p0=0, p1=0),
        # relabelling Q, K, V and the position ids once per forward
        dict(name="permute-qkv", op="permute", dtype="bf16", BH=32, N=16384, D=128, n=3, s=16),
        # a prefix-LM block index, rebuilt for each prompt (its length differs from prompt to
        # prompt and is drawn around 2048)
        dict(name="index-prefix", op="index", N=16256, BQ=128, A=32, mask="prefix", p0=2048, p1=0),
    ]


# ---- draws ---------------------------------------------------------------------------
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mask_draw(rng, N):
    kind = rng.choice(["causal", "window", "dilated", "local_strided", "sinks", "prefix"])
    if kind == "window":
        return kind, _log(rng, 16, max(17, N // 2)), 0
    if kind == "dilated":
        return kind, rng.choice([2, 4, 8, 16]), 0
    if kind == "local_strided":
        return kind, _log(rng, 32, 512), rng.choice([8, 16, 32])
    if kind == "sinks":
        return kind, _log(rng, 16, 1024), rng.choice([4, 16, 64])
    if kind == "prefix":
        return kind, _log(rng, 16, max(17, N // 2)), 0
    return kind, 0, 0


def draw(rng):
    op = rng.choice(["attn", "attn", "attn", "split", "decode", "decode", "bwd", "bwd", "permute", "index"])
    while True:
        c = _DRAW[op](rng)
        w = work(c)
        # below the listed largest: the forward over 32768 tokens, and for the finer tiles
        # and float32, whose rates are lower, the listed ones of their kind
        if op == "attn":
            most = 4e10 if c["BQ"] < 64 or c["dtype"] == "f32" else 2e11
        else:
            most = {"split": 3e11, "decode": 2e10, "bwd": 4e11, "permute": 1, "index": 1}[op]
        if w["flops"] <= most and w["bytes"] <= 9e8:
            return c


def _draw_attn(rng):
    dtype = rng.choice(["f16", "bf16", "f16", "bf16", "f32"])
    BQ, A = rng.choice([(128, 32), (128, 128), (128, 64), (64, 64), (64, 32), (32, 32), (16, 16)])
    N = 128 * _log(rng, 4, 128)
    mask, p0, p1 = _mask_draw(rng, N)
    # a lattice runs in its residue basis (the tensors relabelled), the rest as they are
    stride = p0 if mask == "dilated" and (N // p0) % A == 0 and rng.random() < 0.8 else 0
    return dict(op="attn", dtype=dtype, BH=_log(rng, 1, 32), N=N, D=rng.choice([64, 128]), BQ=BQ, A=A, mask=mask, p0=p0,
                p1=p1, stride=stride, lse=rng.random() < 0.5)


def _draw_split(rng):
    s = rng.choice([4, 8, 16, 32])
    return dict(op="split", dtype=rng.choice(["bf16", "f16"]), BH=_log(rng, 1, 32), N=s * rng.choice([256, 512, 1024]),
                D=rng.choice([128, 128, 64]), w=_log(rng, 16, 512), s=s)


def _draw_decode(rng):
    s = rng.choice([0, 0, 8, 16, 32])
    length = _log(rng, 64, 65536)
    capacity = -(-(length + rng.randrange(1, 2000)) // 64) * 64
    mask, p0, p1 = _mask_draw(rng, length)
    BH = min(_log(rng, 1, 256), max(1, (1 << 21) // capacity))
    nq = rng.choice([1, 1, 1, 2, 4, 7])
    return dict(op="decode", dtype=rng.choice(["bf16", "f16"]), BH=BH, D=rng.choice([64, 128]), capacity=capacity,
                length=length, s=s, mask=mask, p0=p0, p1=p1, nq=nq)


def _draw_bwd(rng):
    N = 64 * _log(rng, 8, 256)
    mask, p0, p1 = _mask_draw(rng, N)
    return dict(op="bwd", dtype=rng.choice(["bf16", "f16"]), BH=_log(rng, 1, 32), N=N, D=rng.choice([64, 128]),
                mask=mask, p0=p0, p1=p1)


def _draw_permute(rng):
    return dict(op="permute", dtype=rng.choice(["bf16", "f16", "f32"]), BH=_log(rng, 1, 32), N=_log(rng, 500, 20000),
                D=rng.choice([64, 128]), n=rng.choice([1, 3, 3, 5]), s=rng.choice([3, 4, 8, 16, 32]))


def _draw_index(rng):
    BQ, A = rng.choice([(128, 32), (128, 128), (64, 64), (16, 16)])
    N = 128 * _log(rng, 8, 127)
    return dict(op="index", N=N, BQ=BQ, A=A, mask="prefix", p0=_log(rng, 64, max(65, N // 2)), p1=0)


_DRAW = dict(attn=_draw_attn, split=_draw_split, decode=_draw_decode, bwd=_draw_bwd, permute=_draw_permute,
             index=_draw_index)


# ---- masks ---------------------------------------------------------------------------
_KIND = dict(causal=attention.CAUSAL, window=attention.WINDOW, dilated=attention.DILATED,
             local_strided=attention.LOCAL_STRIDED, sinks=attention.SINKS, prefix=attention.PREFIX_LM)


def _mask(case):
    """The mask object of a case."""
    k, p0, p1 = case["mask"], case["p0"], case["p1"]
    return {"causal": lambda: masks.Causal(), "window": lambda: masks.SlidingWindow(p0),
            "dilated": lambda: masks.Dilated(p0), "local_strided": lambda: masks.LocalStrided(p0, p1),
            "sinks": lambda: masks.SinksWindow(p1, p0), "prefix": lambda: masks.PrefixLM(p0)}[k]()


def _live(case, q, kv):
    """The same predicate on broadcast torch position tensors."""
    k, p0, p1 = case["mask"], case["p0"], case["p1"]
    d = q - kv
    if k == "causal":
        return d >= 0
    if k == "window":
        return (d >= 0) & (d < p0)
    if k == "dilated":
        return (d >= 0) & (d % p0 == 0)
    if k == "local_strided":
        return (d >= 0) & ((d < p0) | (d % p1 == 0))
    if k == "sinks":
        return (d >= 0) & ((d < p0) | (kv < p1))
    return (d >= 0) | ((q < p0) & (kv < p0))


def _as_local(case):
    """The union mask of a split case."""
    return dict(mask="local_strided", p0=case["w"], p1=case["s"])


def _pieces(w, s):
    """A band in index order and the lattice outside it in the residue basis."""
    band = masks.SlidingWindow(w)
    return [split.Piece(band, 128, 32), split.Piece(masks.Difference(masks.Dilated(s), band), 128, 32, residue=s)]


# ---- float64 (or float32) attention in plain torch -------------------------------------
def _attend(case, q, k, v, qpos, kpos, dtype):
    """(o, natural-log sum-exp) of q against k, v at positions qpos, kpos, in dtype."""
    BH, nq, D = q.shape
    n = k.shape[1]
    o = torch.empty(BH, nq, D, dtype=dtype, device=q.device)
    lse = torch.empty(BH, nq, dtype=dtype, device=q.device)
    step = max(1, min(nq, (1 << 27) // n))
    for r in range(0, nq, step):
        dead = ~_live(case, qpos[r:r + step, None], kpos[None, :])
        for h in range(BH):
            s = (q[h, r:r + step].to(dtype) @ k[h].to(dtype).t()) * D ** -0.5
            s.masked_fill_(dead, -math.inf)
            lse[h, r:r + step] = torch.logsumexp(s, 1)
            o[h, r:r + step] = torch.softmax(s, 1) @ v[h].to(dtype)
    return o, lse


def _gradients(case, q, k, v, o, lse, do):
    """dq, dk, dv in float64 of the attention whose output and log-sum-exp are o and lse."""
    f = torch.float64
    BH, n, D = q.shape
    scale = D ** -0.5
    dq, dk, dv = (torch.zeros(BH, n, D, dtype=f, device=q.device) for _ in range(3))
    pos = torch.arange(n, device=q.device, dtype=torch.int32)
    step = max(1, min(n, (1 << 26) // n))
    for r in range(0, n, step):
        dead = ~_live(case, pos[r:r + step, None], pos[None, :])
        for h in range(BH):
            qh, oh, doh, kh = (t[h, r:r + step].to(f) for t in (q, o, do, k))
            kh, vh = k[h].to(f), v[h].to(f)
            p = torch.exp((qh @ kh.t()) * scale - lse[h, r:r + step, None].to(f)).masked_fill_(dead, 0)
            dv[h] += p.t() @ doh
            ds = p * (doh @ vh.t() - (doh * oh).sum(1, keepdim=True))
            dq[h, r:r + step] = ds @ kh * scale
            dk[h] += ds.t() @ qh * scale
    return dq, dk, dv


# ---- inputs --------------------------------------------------------------------------
def _randn(seed, dtype, n, *shape):
    """n tensors of unit normal values in dtype, from the seed."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(*shape, generator=g, device="cuda").to(dtype) for _ in range(n)]


def _qkv(case, seed):
    """q, k, v in original order; sink tokens have larger keys, as trained models do."""
    q, k, v = _randn(seed, DTYPES[case["dtype"]], 3, case["BH"], case["N"], case["D"])
    if case.get("mask") == "sinks":
        k[:, :case["p1"]] *= 4
    return q, k, v


def _prompt(case, seed):
    """The prompt length of an index case: within an eighth of the nominal one."""
    g = torch.Generator().manual_seed(seed)
    p = case["p0"]
    return p + int(torch.randint(-(p // 8), p // 8 + 1, (1,), generator=g))


def _cached(case, seed):
    """q, the tokens already cached and the new ones of a decode case."""
    dt, BH, D, nq, n = DTYPES[case["dtype"]], case["BH"], case["D"], case["nq"], case["length"]
    k, v = _randn(seed, dt, 2, BH, n - nq, D)
    q, k_new, v_new = _randn(seed + 1000003, dt, 3, BH, nq, D)
    return q, k, v, k_new, v_new


def prepare(case, seed):
    op = case["op"]
    if op == "attn":
        q, k, v = _qkv(case, seed)
        table = None
        if case["stride"]:
            table = perm.residue_perm(case["N"], case["stride"])
        bi = index.build(_mask(case), case["N"], case["BQ"], case["A"], perm=table)
        if table is not None:
            table = torch.from_numpy(table).cuda()
            q, k, v = (perm.apply_perm(t, table) for t in (q, k, v))
        lse = torch.empty(case["BH"], case["N"], device="cuda") if case["lse"] else None
        return dict(case=case, q=q, k=k, v=v, index=bi, lists=index.to_cuda(bi), perm=table, lse=lse)
    if op == "split":
        q, k, v = _qkv(case, seed)
        return dict(case=case, q=q, k=k, v=v, plan=split.SplitPlan(_pieces(case["w"], case["s"]), case["N"]))
    if op == "decode":
        q, k, v, k_new, v_new = _cached(case, seed)
        cache = decode.KVCache(case["BH"], case["capacity"], case["D"], DTYPES[case["dtype"]], residue=case["s"])
        cache.append(k, v)
        return dict(case=case, q=q, k_new=k_new, v_new=v_new, cache=cache, mask=_mask(case), cached=cache.length)
    if op == "bwd":
        q, k, v = _qkv(case, seed)
        (do,) = _randn(seed + 1000003, q.dtype, 1, *q.shape)
        pos = torch.arange(case["N"], device="cuda", dtype=torch.int32)
        o, lse = _attend(case, q, k, v, pos, pos, torch.float32)
        if case["mask"] == "local_strided" and case["N"] % case["p1"] == 0:
            plan = backward.SplitBackward(_pieces(case["p0"], case["p1"]), case["N"])
        elif case["mask"] == "dilated" and case["N"] % case["p0"] == 0:
            plan = backward.SplitBackward([split.Piece(_mask(case), residue=case["p0"])], case["N"])
        else:
            plan = backward.BackwardPlan(_mask(case), case["N"])
        return dict(case=case, q=q, k=k, v=v, o=o.to(q.dtype), lse=lse, do=do, plan=plan)
    if op == "permute":
        xs = _randn(seed, DTYPES[case["dtype"]], case["n"], case["BH"], case["N"], case["D"])
        return dict(case=case, xs=xs, perm=torch.from_numpy(perm.residue_perm(case["N"], case["s"])).cuda())
    return dict(case=case, mask=_mask(dict(case, p0=_prompt(case, seed))))


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "attn":
        ext = {} if state["lse"] is None else dict(lse=state["lse"])
        p2 = 0
        o = attention.block_sparse_attention(state["q"], state["k"], state["v"], *state["lists"], _KIND[case["mask"]],
                                             case["p0"], case["p1"], p2, case["BQ"], case["A"], perm_q=state["perm"],
                                             **ext)
        return o if state["lse"] is None else (o, state["lse"])
    if op == "split":
        return state["plan"].forward(state["q"], state["k"], state["v"])
    if op == "decode":
        cache = state["cache"]
        cache.length = state["cached"]  # the step is taken again from the same context
        o = cache.attend(state["q"], state["mask"], k_new=state["k_new"], v_new=state["v_new"])
        return o, cache.k, cache.v
    if op == "bwd":
        return state["plan"].backward(state["q"], state["k"], state["v"], state["o"], state["lse"], state["do"])
    if op == "permute":
        return perm.permute_stack(state["xs"], state["perm"])
    bi = index.build(state["mask"], case["N"], case["BQ"], case["A"])
    return bi.kv_idx, bi.kv_num, bi.kv_partial, bi.kv_wave_bits.view("int32"), bi.elements, bi.live


def work(case):
    op, es = case["op"], ESIZE.get(case.get("dtype"), 0)
    if op == "attn":
        rows = case["BH"] * case["N"]
        return dict(flops=4.0 * case["D"] * case["BH"] * _mask(case).live_count(case["N"]),
                    bytes=4.0 * rows * case["D"] * es + (4.0 * rows if case["lse"] else 0))
    if op == "split":
        live = masks.LocalStrided(case["w"], case["s"]).live_count(case["N"])
        return dict(flops=4.0 * case["D"] * case["BH"] * live, bytes=4.0 * case["BH"] * case["N"] * case["D"] * es)
    if op == "decode":
        # the keys live for some of the new rows, each read once; the new rows read and written
        n, nq = case["length"], case["nq"]
        rows = [set(_mask(case).row_cols(n - nq + i, n).nonzero()[0].tolist()) for i in range(nq)]
        pairs, keys = sum(len(r) for r in rows), len(set().union(*rows))
        return dict(flops=4.0 * case["D"] * case["BH"] * pairs,
                    bytes=2.0 * es * case["D"] * case["BH"] * (keys + 2 * nq))
    if op == "bwd":
        rows = case["BH"] * case["N"]
        return dict(flops=10.0 * case["D"] * case["BH"] * _mask(case).live_count(case["N"]),
                    bytes=8.0 * rows * case["D"] * es + 4.0 * rows)
    if op == "permute":
        return dict(flops=0.0, bytes=2.0 * case["n"] * case["BH"] * case["N"] * case["D"] * es + 12.0 * case["N"])
    # the lists: a tile id, a flag and a code for each place of the padded rows
    nq, nk = case["N"] // case["BQ"], case["N"] // case["A"]
    return dict(flops=0.0, bytes=9.0 * nq * nk + 4.0 * nq)


def tolerance(case):
    # about four times the measured distance to float64; the backward also rounds P and dS to
    # 16 bits before their products
    op = case["op"]
    if op in ("permute", "index"):
        return "exact"
    if op == "bwd":
        return {"rel": {"f16": 1.5e-3, "bf16": 1.25e-2}[case["dtype"]]}
    return {"rel": {"f32": 2e-6, "f16": 1.2e-3, "bf16": 1e-2}[case["dtype"]]}


def exact(case, seed):
    op, f = case["op"], torch.float64
    if op == "attn":
        q, k, v = _qkv(case, seed)
        pos = torch.arange(case["N"], device="cuda", dtype=torch.int32)
        if case["stride"]:
            pos = torch.cat([pos[c::case["stride"]] for c in range(case["stride"])])
            q, k, v = (t[:, pos.long()] for t in (q, k, v))
        o, lse = _attend(case, q, k, v, pos, pos, f)
        return (o, lse) if case["lse"] else o
    if op == "split":
        q, k, v = _qkv(case, seed)
        pos = torch.arange(case["N"], device="cuda", dtype=torch.int32)
        return _attend(_as_local(case), q, k, v, pos, pos, f)[0]
    if op == "decode":
        q, k, v, k_new, v_new = _cached(case, seed)
        pos = torch.arange(case["length"], device="cuda", dtype=torch.int32)
        o = _attend(case, q, torch.cat([k, k_new], 1), torch.cat([v, v_new], 1), pos[-case["nq"]:], pos, f)[0]
        return o, None, None
    if op == "bwd":
        q, k, v = _qkv(case, seed)
        (do,) = _randn(seed + 1000003, q.dtype, 1, *q.shape)
        pos = torch.arange(case["N"], device="cuda", dtype=torch.int32)
        o, lse = _attend(case, q, k, v, pos, pos, torch.float32)
        return _gradients(case, q, k, v, o.to(q.dtype), lse, do)
    return None
