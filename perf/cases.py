"""The work that users of loom_infer_hip have it do, as timed cases.

A serving engine on one MI355X calls the library once per layer and step: it
keeps its K/V pool, its plans and its command queue (whose workspace it
reserved once), and enqueues commands back to back on its stream.  The cases
below are those calls over the range of sizes that such engines see, each
through the public entry points of the Python binding:

  decode    paged batch decode (BF16 or FP8 E4M3 pages, NHD or HND, 16/32/64 rows)
  single    contiguous single decode, one plan for a whole request
  split_k   the same with the split-K plan
  append    fused RoPE + paged K/V append of explicit tokens
  prefill   paged causal prefill: whole prompts, chunks behind a cached prefix,
            a few rows per request behind a long context (draft verification)
  ragged    ragged causal prefill over contiguous K/V rows
  step      one decode step (one-token append, then decode) replayed as a graph
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "loom-kernels_amd"))
import loom_infer_hip as L  # noqa: E402

D = 128
RESERVE = 32 << 20  # bytes of queue workspace an engine reserves
MAX_COMMANDS = 1 << 40
K_SCALE, V_SCALE = 0.0171, 0.0157  # FP8 page scales: N(0, 1) values reach 4.5 sigma below 448


def listed():
    return [
        # The first tokens of a few short chats (the reference's gqa4_b4_reuse
        # lengths): launch and latency, hardly any bytes.
        _paged("decode_b4_short", "decode", 4, 3, 41, 16, 4),
        # A chat server at moderate load: 16 requests of some hundred tokens.
        _paged("decode_b16_1k", "decode", 16, 256, 1536, 32, 8),
        # The headline decode: 64 ragged requests, context U[512, 8192], GQA4.
        _paged("decode_b64_ragged", "decode", 64, 512, 8192, 32, 8),
        # Long documents on FP8 pages: 8 requests of 32768 tokens, GQA8.
        _paged("decode_b8_32k_fp8", "decode", 8, 32768, 32768, 64, 8, dtype="fp8_e4m3"),
        # One request over a contiguous cache, the direct plan (4096 tokens, 32/4).
        dict(name="single_l4096", op="single", kv=4096, hq=32, hkv=4, parts=0),
        # Chunked prompts of 32 requests written into their pages: about 1000
        # tokens in one command.
        dict(_paged("append_b32_tokens", "append", 32, 64, 4160, 32, 8), rows_lo=1, rows_hi=64),
        # Draft verification: 4-8 new rows of each of 16 requests behind
        # contexts of up to 8192 tokens.
        dict(_paged("prefill_verify_b16", "prefill", 16, 1024, 8192, 32, 8), rows_lo=4, rows_hi=8),
        # The largest paged prefill shape the reference times (rows 32 and 64
        # behind 256 and 1024 tokens): a small append to two conversations.
        dict(_paged("prefill_append_b2", "prefill", 2, 256, 1024, 16, 4), rows_lo=32, rows_hi=64),
        # A whole 8192-token prompt.
        dict(_paged("prefill_8192", "prefill", 1, 8192, 8192, 32, 8), rows_lo=8192, rows_hi=8192),
        # Chunked prefill of 4 long prompts on FP8 pages: 512 rows each behind
        # prefixes of 2048-16384 tokens.
        dict(_paged("prefill_chunk_b4_fp8", "prefill", 4, 2048, 16384, 32, 8, dtype="fp8_e4m3"),
             rows_lo=512, rows_hi=512),
        # A batch of fresh prompts of about 2048 rows whose K/V lie contiguous.
        dict(name="ragged_b4_2048", op="ragged", batch=4, lo=1600, hi=2400, mix=5, hq=32, hkv=8,
             rows_lo=0, rows_hi=0),
        # A whole decode step at high load as an engine replays it: one-token
        # append, then decode, 256 requests of lognormal lengths around 2048.
        _paged("step_b256_graph", "step", 256, 16, 16384, 32, 8, dist="lognormal"),
    ]


def _paged(name, op, batch, lo, hi, hq, hkv, dtype="bf16", layout="NHD", page=16, dist="uniform",
           mix=3):
    return dict(name=name, op=op, batch=batch, lo=lo, hi=hi, hq=hq, hkv=hkv, dtype=dtype,
                layout=layout, page=page, dist=dist, mix=mix)


# Query and kv heads of the repository's configurations and fixtures, and one odd group.
HEADS = [(32, 8), (32, 8), (32, 8), (64, 8), (16, 4), (32, 32), (8, 1), (28, 4)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes log-uniform over what the listed cases span, within
    about 3 GB of K/V and 500 GFLOP."""
    op = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "chunk", "verify",
                     "ragged", "ragged", "append", "single", "step"])
    hq, hkv = rng.choice(HEADS)
    mix = rng.randrange(1 << 20)
    kv = dict(dtype=rng.choice(["bf16", "bf16", "fp8_e4m3"]),
              layout=rng.choice(["NHD", "NHD", "HND"]), page=rng.choice([16, 16, 32, 64]))
    if op == "single":
        n = _log(rng, 1, 16384)
        parts = rng.choice([0, min(64, max(1, n // 32))])
        return dict(op="split_k" if parts else "single", kv=n, hq=hq, hkv=hkv, parts=parts)
    # tokens of K/V that the call may hold
    most = int(2.8e9 / (hkv * D * 4))
    if op in ("decode", "step"):
        b = _log(rng, 1, 256)
        hi = max(16, min(_log(rng, 64, 32768), most // b))
        lo = max(1, int(hi * rng.choice([0.06, 0.5, 1.0])))
        if op == "step":
            kv["dtype"] = "bf16"
        return dict(op=op, batch=b, lo=lo, hi=hi, hq=hq, hkv=hkv, dist="uniform", mix=mix, **kv)
    if op == "append":
        b = _log(rng, 1, 128)
        rows = max(1, min(256, 6000 // b, _log(rng, 1, 256)))
        lo = rows + _log(rng, 1, 256)
        return dict(op=op, batch=b, lo=lo, hi=lo + _log(rng, 64, 4096), rows_lo=max(1, rows // 8),
                    rows_hi=rows, hq=hq, hkv=hkv, dist="uniform", mix=mix, **kv)
    b = _log(rng, 1, 16)
    if op in ("prompt", "ragged"):
        hi = _log(rng, 48, 8192)
        # causal work of the whole prompts: 2 * 128 * hq * rows^2 per request
        b = max(1, min(b, int(4.5e11 / (256.0 * hq * hi * hi))))
        case = dict(batch=b, lo=max(1, int(hi * rng.choice([0.4, 0.8, 1.0]))), hi=hi, mix=mix,
                    hq=hq, hkv=hkv, rows_lo=0, rows_hi=0)
        if op == "ragged":
            return dict(op="ragged", **case)
        return dict(op="prefill", dist="uniform", **case, **kv)
    rows = _log(rng, 1, 16) if op == "verify" else _log(rng, 64, 1024)
    hi = max(rows + 64, min(_log(rng, 512, 32768), most // b))
    b = max(1, min(b, int(3e11 / (512.0 * hq * rows * hi))))
    return dict(op="prefill", batch=b, lo=max(rows, hi // rng.choice([1, 2, 8])), hi=hi,
                rows_lo=max(1, rows // rng.choice([1, 2])), rows_hi=rows, hq=hq, hkv=hkv,
                dist="uniform", mix=mix, **kv)


# ---- lengths and tables ---------------------------------------------------------
def _lengths(case):
    """(K/V length, query or new rows) of every request: the case's own, whatever
    the inputs' seed.  The longest and the shortest of the range are among them."""
    r = random.Random(case["mix"])
    b, lo, hi = case["batch"], case["lo"], case["hi"]
    if case.get("dist") == "lognormal":
        lens = [min(hi, max(lo, int(r.lognormvariate(math.log(2048), 0.8)))) for _ in range(b)]
    else:
        lens = [r.randint(lo, hi) for _ in range(b)]
        lens[0] = hi
        lens[-1] = lo if b > 1 else hi
    if "rows_lo" not in case:
        return lens, [1] * b
    if case["rows_hi"] == 0:  # whole prompts
        return lens, list(lens)
    rows = [min(n, r.randint(case["rows_lo"], case["rows_hi"])) for n in lens]
    rows[0] = min(lens[0], case["rows_hi"])
    if b > 1:
        rows[-1] = min(lens[-1], case["rows_lo"])
    return lens, rows


def _table(case, lens, rng):
    """Every request's pages scattered over a pool an eighth larger than they need."""
    P = case["page"]
    pages = [-(-n // P) for n in lens]
    indptr = np.concatenate([[0], np.cumsum(pages)]).astype(np.int32)
    total = int(indptr[-1])
    pool = total + max(4, total // 8)
    indices = rng.permutation(pool)[:total].astype(np.int32)
    last = np.array([n - (p - 1) * P for n, p in zip(lens, pages)], np.int32)
    return pool, indptr, indices, last


def _starts(counts):
    return np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)


def _inputs(case, seed):
    """The inputs of one call on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rng = np.random.default_rng(seed)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.bfloat16)

    def ints(a):
        return torch.from_numpy(np.ascontiguousarray(np.asarray(a, np.int32))).cuda()

    hq, hkv = case["hq"], case["hkv"]
    x = {}
    if case["op"] in ("single", "split_k"):
        x["q"], x["k"], x["v"] = normal(hq, D), normal(case["kv"], hkv, D), normal(case["kv"], hkv, D)
        return x
    lens, rows = _lengths(case)
    n = sum(rows)
    x["q"] = normal(n, hq, D)
    if case["op"] == "ragged":
        x["k"], x["v"] = normal(sum(lens), hkv, D), normal(sum(lens), hkv, D)
        x["qo"], x["kvp"] = ints(_starts(rows)), ints(_starts(lens))
        return x
    pool, indptr, indices, last = _table(case, lens, rng)
    P = case["page"]
    shape = (pool, P, hkv, D) if case["layout"] == "NHD" else (pool, hkv, P, D)
    if case["dtype"] == "bf16":
        x["kp"], x["vp"] = normal(*shape), normal(*shape)
    else:
        x["kp"], x["vp"] = (
            torch.randn(shape, generator=g, device="cuda").div_(s).clamp_(-448, 448)
            .to(torch.float8_e4m3fn).view(torch.uint8) for s in (K_SCALE, V_SCALE))
        x["scales"] = torch.tensor([K_SCALE, V_SCALE], device="cuda")
    x["indptr"], x["indices"], x["last"] = ints(indptr), ints(indices), ints(last)
    x["pool"] = pool
    if case["op"] in ("append", "step"):
        x["nk"], x["nv"] = normal(n, hkv, D), normal(n, hkv, D)
    if case["op"] == "append":
        # each request's new tokens at the end of its pages, in a scheduler's mixed order
        req = np.repeat(np.arange(len(lens)), rows)
        pos = np.concatenate([np.arange(a - r, a) for a, r in zip(lens, rows)])
        order = rng.permutation(n)
        x["req"], x["pos"] = ints(req[order]), ints(pos[order])
    elif case["op"] == "prefill":
        x["qo"] = ints(_starts(rows))
    return x


# ---- a user's program -------------------------------------------------------------
class _Program:
    """What a caller keeps: inputs, outputs, plan, queue, bindings and the open
    scope that its commands go into."""

    def __init__(self, case, x):
        self.x = x
        self.queue = L.CommandQueue(torch.cuda.current_stream(), MAX_COMMANDS)
        self.queue.reserve_workspace(RESERVE)
        self.plan, self.out = None, {}

    def open(self, reads, writes, make):
        """Binds the operands and opens a scope; `make` builds the command's args."""
        b = self.queue.bindings(len(reads) + len(writes))
        r = [b.bind_read(t) for t in reads]
        w = [b.bind_read_write(t) for t in writes]
        self.args = make(r, [h.write() for h in w], w)
        self.scope = self.queue.begin(b)
        return self

    def __call__(self):
        self.plan.enqueue_into(self.scope, self.args)
        return self.out


class _Step:
    """The decode step as a captured graph."""

    def __init__(self, case, x, spec, append):
        b, hq = case["batch"], case["hq"]
        self.x = x
        self.plans = (append, L.DecodeProvider.load(0).plan_bf16_paged_batch(spec))
        qr, o, lse = _empty(b, hq)
        gq = L.GraphQueue(0, 2)
        gq.reserve_workspace(max(RESERVE, self.plans[1].workspace_bytes))
        bd = gq.bindings(12)
        q, nk, nv, ip, ix, ln = (bd.bind_read(x[k]) for k in
                                 ("q", "nk", "nv", "indptr", "indices", "last"))
        kp, vp, hqr, ho, hl = (bd.bind_read_write(t) for t in (x["kp"], x["vp"], qr, o, lse))
        first = L.Bf16RopePagedKvAppendArgs(q, nk, nv, ip, ix, ln, hqr.write(), kp.write(),
                                            vp.write())
        second = L.Bf16PagedBatchDecodeArgs(hqr.read(), kp.read(), vp.read(), ip, ix, ln,
                                            ho.write(), hl.write())

        def record(scope):
            self.plans[0].enqueue_into(scope, first)
            self.plans[1].enqueue_into(scope, second)

        self.graph = gq.capture(bd, record).instantiate()
        self.out = {"q": qr, "out": o, "lse": lse, "k_pages": x["kp"], "v_pages": x["vp"]}

    def __call__(self):
        self.graph.launch().wait()
        return self.out


def _empty(rows, hq):
    return (torch.zeros(rows, hq, D, device="cuda", dtype=torch.bfloat16),
            torch.zeros(rows, hq, D, device="cuda", dtype=torch.bfloat16),
            torch.zeros(rows, hq, device="cuda"))


def prepare(case, seed):
    x = _inputs(case, seed)
    op, hq, hkv = case["op"], case["hq"], case["hkv"]
    torch.cuda.synchronize()  # the graph of a step runs on a stream of its own
    if op in ("single", "split_k"):
        p = _Program(case, x)
        _, o, lse = _empty(1, hq)
        p.out = {"out": o, "lse": lse}
        spec = L.Bf16SingleDecodeSpec(case["kv"], hq, hkv)
        prov = L.DecodeProvider.load(0)
        reads = [x["q"], x["k"], x["v"]]
        if op == "single":
            p.plan = prov.plan_bf16(spec)
            return p.open(reads, [o, lse], lambda r, w, rw: L.Bf16SingleDecodeArgs(*r, *w))
        p.plan = prov.plan_bf16_split_k(L.Bf16SingleDecodeSplitKSpec(spec, case["parts"]))
        ws = torch.empty(p.plan.workspace_required_numel, device="cuda")
        return p.open(reads, [ws, o, lse],
                      lambda r, w, rw: L.Bf16SingleDecodeSplitKArgs(*r, rw[0], w[1], w[2]))
    if op == "ragged":
        p = _Program(case, x)
        n, nkv = x["q"].shape[0], x["k"].shape[0]
        _, o, lse = _empty(n, hq)
        p.out = {"out": o, "lse": lse}
        p.plan = L.PrefillProvider.load(0).plan_bf16_ragged(
            L.Bf16RaggedPrefillSpec(case["batch"], n, nkv, hq, hkv))
        return p.open([x["q"], x["k"], x["v"], x["qo"], x["kvp"]], [o, lse],
                      lambda r, w, rw: L.Bf16RaggedPrefillArgs(*r, *w))
    form = dict(kv_layout=case["layout"], kv_dtype=case["dtype"], kv_page_size=case["page"])
    fp8 = case["dtype"] != "bf16"
    scales = [x["scales"]] if fp8 else []
    n, b = x["q"].shape[0], case["batch"]
    if op == "step":
        spec = L.Bf16PagedBatchDecodeSpec(b, x["pool"], hq, hkv, **form)
        append = L.RopeProvider.load(0).plan_bf16_paged_append(
            L.Bf16RopePagedKvAppendSpec(b, x["pool"], hq, hkv, **form))
        return _Step(case, x, spec, append)
    p = _Program(case, x)
    qr, o, lse = _empty(n, hq)
    table = [x["indptr"], x["indices"], x["last"]]
    if op == "append":
        p.out = {"q": qr, "k_pages": x["kp"], "v_pages": x["vp"]}
        p.plan = L.RopeProvider.load(0).plan_bf16_paged_append_tokens(
            L.Bf16RopePagedKvAppendTokensSpec.extended(n, b, x["pool"], hq, hkv, **form))
        writes = [qr, x["kp"], x["vp"]]
        if fp8:  # FP8 pages: the caller's own validation workspace, zeroed once
            writes.append(torch.zeros(p.plan.workspace_bytes, dtype=torch.uint8, device="cuda"))
        return p.open([x["q"], x["nk"], x["nv"], x["req"], x["pos"], *table, *scales], writes,
                      lambda r, w, rw: L.Bf16RopePagedKvAppendTokensArgs(
                          *r[:8], *w[:3], *(w[3:] + r[8:] if fp8 else [])))
    p.out = {"out": o, "lse": lse}
    if op == "prefill":
        p.plan = L.PrefillProvider.load(0).plan_bf16_paged(
            L.Bf16PagedPrefillSpec(b, n, x["pool"], hq, hkv, **form))
        return p.open([x["q"], x["kp"], x["vp"], x["qo"], *table, *scales], [o, lse],
                      lambda r, w, rw: L.Bf16PagedPrefillArgs(*r[:7], *w, *r[7:]))
    p.plan = L.DecodeProvider.load(0).plan_bf16_paged_batch(
        L.Bf16PagedBatchDecodeSpec(b, x["pool"], hq, hkv, **form))
    writes = [o, lse]
    if fp8:  # the extended operands: a workspace and the scales
        writes.append(torch.empty(p.plan.workspace_bytes, dtype=torch.uint8, device="cuda"))
    return p.open([x["q"], x["kp"], x["vp"], *table, *scales], writes,
                  lambda r, w, rw: L.Bf16PagedBatchDecodeArgs(*r[:6], *w, *r[6:]))


def run(state):
    return state()


# ---- what a pass cannot do without ----------------------------------------------
def _visible(lens, rows):
    """Visible tokens summed over the query rows (bottom-right causal mask)."""
    return sum(r * (n - r) + r * (r + 1) // 2 for n, r in zip(lens, rows))


def work(case):
    hq, hkv = case["hq"], case["hkv"]
    op = case["op"]
    if op in ("single", "split_k"):
        return {"bytes": case["kv"] * hkv * D * 4 + hq * (D * 4 + 4), "flops": 4 * D * hq * case["kv"]}
    lens, rows = _lengths(case)
    n, tokens = sum(rows), sum(lens)
    elem = 1 if case.get("dtype") == "fp8_e4m3" else 2
    heads = n * hq * (D * 4 + 4)  # Q read, O and LSE written
    if op == "ragged":
        return {"bytes": tokens * hkv * D * 4 + heads, "flops": 4 * D * hq * _visible(lens, rows)}
    table = 4 * (2 * len(lens) + 1 + sum(-(-t // case["page"]) for t in lens))
    new = n * (hq * D * 4 + hkv * D * 2 * (2 + elem))  # Q in and out, K/V rows in and to pages
    if op == "append":
        return {"bytes": new + table + 8 * n, "flops": 3 * n * (hq + hkv) * D}
    attend = {"bytes": 2 * tokens * hkv * D * elem + heads + table,
              "flops": 4 * D * hq * _visible(lens, rows)}
    if op == "step":
        return {"bytes": attend["bytes"] + new, "flops": attend["flops"] + 3 * n * (hq + hkv) * D}
    return attend


def tolerance(case):
    """Outputs are rounded to BF16 (about 1.7e-3 of the result by itself), and
    the attention weights may be on their way (about 1.1e-3 more); two correct
    results differ by up to 2.5e-3.  FP8 pages an append writes are bytes in
    which a rounding tie of the rotation may move."""
    if case["op"] == "append" and case["dtype"] != "bf16":
        return {"rel": 8e-3, "max": 4e-2, "differ": 1e-3}
    return {"rel": 8e-3, "max": 4e-2}


# ---- the same in 64 bits ----------------------------------------------------------
def _attend(q, k, v, out, lse):
    """Bottom-right causal attention of one request: q [R, Hq, D] over k, v
    [N, Hkv, D], written to out and lse (log2), rows in blocks."""
    R, hq, N = q.shape[0], q.shape[1], k.shape[0]
    group = hq // k.shape[1]
    t = torch.arange(N, device=q.device)
    for h in range(k.shape[1]):
        kt, vh = k[:, h].double().t().contiguous(), v[:, h].double()
        step = max(1, (1 << 27) // (N * group))
        for a in range(0, R, step):
            z = min(R, a + step)
            heads = slice(h * group, (h + 1) * group)
            rows = q[a:z, heads].double().reshape(-1, D)
            s = rows.matmul(kt).mul_(D ** -0.5)
            if R > 1:
                end = N - R + torch.arange(a, z, device=q.device).repeat_interleave(group)
                s.masked_fill_(t[None, :] > end[:, None], -math.inf)
            m = s.amax(1, keepdim=True)
            s.sub_(m).exp_()
            l = s.sum(1, keepdim=True)
            out[a:z, heads] = (s.matmul(vh) / l).reshape(z - a, group, D)
            lse[a:z, heads] = ((m + l.log()) / math.log(2)).reshape(z - a, group)


def _rope(x, pos):
    """NeoX rotation of x [T, H, D] at positions pos, theta 10000."""
    inv = 10000.0 ** (-torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D)
    a = pos.double()[:, None] * inv
    c, s = a.cos()[:, None], a.sin()[:, None]
    x1, x2 = x.double()[..., : D // 2], x.double()[..., D // 2:]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], -1)


def _gather(case, pages, x, r, n, scale=1.0):
    """Request r's n rows [n, Hkv, D] out of its pages."""
    ip = x["indptr"].tolist()
    p = pages[x["indices"][ip[r]:ip[r + 1]].long()]
    if case["dtype"] != "bf16" and p.dtype == torch.uint8:
        p = p.view(torch.float8_e4m3fn).float().double() * scale
    if case["layout"] == "HND":
        p = p.transpose(1, 2)
    return p.reshape(-1, case["hkv"], D)[:n]


def _scatter(case, pages, x, req, pos, rows):
    P, ip = case["page"], x["indptr"].long()
    page = x["indices"].long()[ip[req.long()] + pos.long() // P]
    slot = pos.long() % P
    if case["layout"] == "HND":
        pages[page, :, slot] = rows
    else:
        pages[page, slot] = rows


def exact(case, seed):
    x = _inputs(case, seed)
    op, hq = case["op"], case["hq"]
    n = x["q"].shape[0]
    out = torch.zeros(n if op not in ("single", "split_k") else 1, hq, D, device="cuda",
                      dtype=torch.float64)
    lse = out.new_zeros(out.shape[0], hq)
    if op in ("single", "split_k"):
        _attend(x["q"][None], x["k"], x["v"], out, lse)
        return {"out": out, "lse": lse}
    lens, rows = _lengths(case)
    qs = _starts(rows).tolist()
    if op == "ragged":
        ks = _starts(lens).tolist()
        for r in range(len(lens)):
            _attend(x["q"][qs[r]:qs[r + 1]], x["k"][ks[r]:ks[r + 1]], x["v"][ks[r]:ks[r + 1]],
                    out[qs[r]:qs[r + 1]], lse[qs[r]:qs[r + 1]])
        return {"out": out, "lse": lse}
    got, q, kp, vp = {"out": out, "lse": lse}, x["q"], x["kp"], x["vp"]
    if op in ("append", "step"):
        req = x["req"] if op == "append" else torch.arange(n, device="cuda")
        pos = x["pos"] if op == "append" else torch.tensor(lens, device="cuda") - 1
        q = _rope(q, pos)
        if case["dtype"] == "bf16":
            kp, vp = kp.double(), vp.double()
            _scatter(case, kp, x, req, pos, _rope(x["nk"], pos))
            _scatter(case, vp, x, req, pos, x["nv"].double())
            pages = {"q": q, "k_pages": kp, "v_pages": vp}
        else:  # bytes: no value in 64 bits
            pages = {"q": q, "k_pages": None, "v_pages": None}
        if op == "append":
            return pages
        got.update(pages)
    for r, t in enumerate(lens):
        _attend(q[qs[r]:qs[r + 1]], _gather(case, kp, x, r, t, K_SCALE),
                _gather(case, vp, x, r, t, V_SCALE), out[qs[r]:qs[r + 1]], lse[qs[r]:qs[r + 1]])
    return got
