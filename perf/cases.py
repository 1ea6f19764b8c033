"""Performance cases of moba_hip: the calls a user's program makes, over the
range of sizes, head shapes, data types and options it makes them with.

Kinds of case (``case["kind"]``):

* ``train``    prefill forward and backward through ``run_impl("opt_hip")``;
* ``prefill``  the forward alone, as inference runs it (no graph is recorded);
* ``decode``   one route + attention call of a prepared decode batch at the
               positions its cache holds;
* ``serve``    a batch of requests from empty cache slots to its last token:
               prompts appended, a prepared decode lease, ``steps`` tokens;
* ``merge``    the standalone global-softmax merge of (o, lse) partials.

``lengths`` holds the sequence (or prompt, or context) lengths of the batch as
text, comma-separated.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PACKAGE = os.path.join(_ROOT, "moba-merge-cuda_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import moba_hip  # noqa: E402

_DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_EPS = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11, "fp32": 2.0 ** -24}


def listed():
    return [
        # Long-context training step, multi-head attention at 32K tokens with
        # 4K chunks: the largest and most compute-bound call.
        dict(name="train_mha_32k", kind="train", lengths="32768", hq=32, hkv=32, d=128,
             chunk=4096, topk=3, dtype="bf16", precision="upstream", scale=128 ** -0.5),
        # Training step of a Qwen2-0.5B attention layer (14 q / 2 kv heads).
        dict(name="train_gqa_16k", kind="train", lengths="16384", hq=14, hkv=2, d=64,
             chunk=2048, topk=3, dtype="bf16", precision="upstream", scale=1.0),
        # Many short chunks: 64 chunks of 512 keys, top-4, where routing and
        # short remote loops weigh more.
        dict(name="train_chunk512_32k", kind="train", lengths="32768", hq=8, hkv=8, d=128,
             chunk=512, topk=4, dtype="bf16", precision="upstream", scale=1.0),
        # A packed batch of documents of ragged lengths, fp16, fp32 routing.
        dict(name="train_ragged_fp16", kind="train", lengths="5003,311,4097,1,2049,777", hq=28,
             hkv=4, d=64, chunk=512, topk=3, dtype="fp16", precision="fp32", scale=1.0),
        # Wide heads (head dim 256, the largest supported).
        dict(name="train_d256_8k", kind="train", lengths="8192", hq=16, hkv=4, d=256,
             chunk=1024, topk=3, dtype="bf16", precision="upstream", scale=1.0),
        # Prompt prefill of a Qwen2-1.5B attention layer in inference.
        dict(name="prefill_8k", kind="prefill", lengths="8192", hq=12, hkv=2, d=128,
             chunk=512, topk=4, dtype="bf16", precision="upstream", scale=1.0),
        # A short prompt pair: launches and host work decide.
        dict(name="prefill_small", kind="prefill", lengths="180,120", hq=4, hkv=2, d=64,
             chunk=64, topk=3, dtype="bf16", precision="upstream", scale=1.0),
        # Batch-8 decode, Qwen2-1.5B shape, pages of 48 tokens (not a divisor
        # of the chunk), contexts uniform in [2048, 16384].
        dict(name="decode_b8", kind="decode",
             lengths="15883,8359,14466,8938,2711,6290,10424,10009", hq=12, hkv=2, d=128,
             chunk=512, topk=4, page=48, extra=264, dtype="bf16", graph=False),
        # Batch-32 MQA decode in fp16 from a captured hipGraph, contexts
        # uniform in [1024, 32768].
        dict(name="decode_mqa_b32_graph", kind="decode",
             lengths="32351,29306,32082,28845,2877,4025,3805,12855,28401,6564,25140,27532,22969,"
                     "29002,11121,9267,20879,7977,20907,2194,20068,23347,6213,15136,21945,13919,"
                     "27358,24715,29212,17705,32133,13215", hq=16, hkv=1, d=96,
             chunk=1024, topk=8, page=64, extra=264, dtype="fp16", graph=True),
        # Batch-16 decode at 32K with short chunks: 256 candidate chunks a row.
        dict(name="decode_b16_chunk128", kind="decode", lengths=",".join(["32768"] * 16), hq=32,
             hkv=8, d=128, chunk=128, topk=4, page=16, extra=264, dtype="bf16", graph=False),
        # Four requests served from prompt to 32nd token on one cache.
        dict(name="serve_b4", kind="serve", lengths="2048,517,4099,1290", hq=32, hkv=8, d=64,
             chunk=128, topk=4, page=16, steps=32, dtype="bf16"),
        # Partials of two remote branches merged into the self branch.
        dict(name="merge_16k", kind="merge", tokens=16384, hq=14, d=64, kmax=2, dtype="bf16"),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["train", "train", "train", "prefill", "prefill", "decode", "decode",
                       "decode", "serve", "merge"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind in ("train", "prefill"):
        hq, hkv = rng.choice([(8, 8), (32, 32), (16, 16), (14, 2), (12, 2), (28, 4), (32, 8),
                              (16, 4), (8, 1), (6, 3)])
        d = rng.choice([64, 64, 96, 128, 128, 128, 192, 256, 40])
        chunk = rng.choice([64, 128, 256, 512, 1024, 2048, 4096, 300])
        topk = rng.choice([1, 2, 3, 3, 4, 4, 8])
        while True:
            tokens = log(256, 32768)
            cuts = sorted(rng.sample(range(1, tokens), rng.choice([0, 0, 1, 3, 6])))
            lengths = [b - a for a, b in zip([0] + cuts, cuts + [tokens])]
            case = dict(kind=kind, lengths=",".join(map(str, lengths)), hq=hq, hkv=hkv, d=d,
                        chunk=chunk, topk=topk, dtype=dtype,
                        precision=rng.choice(["upstream", "upstream", "fp32"]), scale=1.0)
            # within the largest listed case: operations (wide heads run at a
            # lower rate), and chunks per token for the routing
            if (work(case)["flops"] <= (4e12 if d <= 128 else 1e12)
                    and tokens // chunk <= 256 and tokens * hq <= 1 << 20):
                return case
    if kind == "merge":
        return dict(kind=kind, tokens=log(64, 32768), hq=rng.choice([1, 4, 8, 14, 28]),
                    d=rng.choice([40, 64, 96, 128, 256]), kmax=rng.choice([1, 2, 3, 7]),
                    dtype=rng.choice(["bf16", "fp16", "fp32"]))
    hq, hkv = rng.choice([(12, 2), (14, 2), (28, 4), (32, 8), (16, 1), (32, 1), (8, 8), (16, 4)])
    d = rng.choice([64, 80, 96, 128, 128, 256])
    case = dict(kind=kind, hq=hq, hkv=hkv, d=d, chunk=rng.choice([128, 256, 512, 1024, 2048]),
                topk=rng.choice([2, 4, 4, 8]), page=rng.choice([16, 32, 48, 64]), dtype=dtype)
    if kind == "serve":
        case["lengths"] = ",".join(str(log(64, 4096)) for _ in range(rng.randint(1, 6)))
        case["steps"] = rng.randint(8, 40)
    else:
        batch = log(1, 32)
        case["lengths"] = ",".join(str(log(256, 32768)) for _ in range(batch))
        case["extra"] = 264
        case["graph"] = rng.random() < 0.4
    return case


def _lengths(case):
    return [int(x) for x in case["lengths"].split(",")]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


# ------------------------------------------------------------------- inputs

def _prefill_inputs(case, seed):
    g = _generator(seed)
    T, dtype = sum(_lengths(case)), _DTYPE[case["dtype"]]

    def rnd(heads):
        return (torch.randn((T, heads, case["d"]), generator=g, device="cuda")
                * case["scale"]).to(dtype)
    return rnd(case["hq"]), rnd(case["hkv"]), rnd(case["hkv"]), rnd(case["hq"])


def _decode_inputs(case, seed):
    """Per sequence the K and V it holds, then the query rows and one new
    token's K and V for each sequence."""
    g = _generator(seed)
    dtype, hkv, d = _DTYPE[case["dtype"]], case["hkv"], case["d"]

    def rnd(n, heads):
        return torch.randn((n, heads, d), generator=g, device="cuda", dtype=dtype)
    lengths = _lengths(case)
    kv = [(rnd(n, hkv), rnd(n, hkv)) for n in lengths]
    n = len(lengths)
    return kv, rnd(n, case["hq"]), rnd(n, hkv), rnd(n, hkv)


def _merge_inputs(case, seed):
    g = _generator(seed)
    T, H, D, dtype = case["tokens"], case["hq"], case["d"], _DTYPE[case["dtype"]]
    # each row holds up to kmax remote partials (three in four are there),
    # in the arbitrary order an expert-major branch leaves them
    present = torch.rand((T * H, case["kmax"]), generator=g, device="cuda") < 0.75
    present[0, 0] = True
    rows = present.nonzero()[:, 0]
    mapping = rows[torch.randperm(rows.numel(), generator=g, device="cuda")].to(torch.int32)
    M = mapping.numel()

    def rnd(*shape):
        return torch.randn(shape, generator=g, device="cuda")
    return (rnd(T, H, D).to(dtype), rnd(T, H) + 6.0, rnd(M, D).to(dtype), rnd(M) + 6.0, mapping)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "prefill"):
        q, k, v, dout = _prefill_inputs(case, seed)
        if kind == "train":
            for t in (q, k, v):
                t.requires_grad_(True)
        lengths = _lengths(case)
        cu = [0]
        for n in lengths:
            cu.append(cu[-1] + n)
        return dict(case=case, q=q, k=k, v=v, dout=dout, longest=max(lengths),
                    cu=torch.tensor(cu, device="cuda", dtype=torch.int32),
                    config=dict(chunk_size=case["chunk"], topk=case["topk"],
                                route_precision=case["precision"]))
    if kind == "merge":
        return dict(case=case, args=_merge_inputs(case, seed))
    kv, q, kn, vn = _decode_inputs(case, seed)
    lengths = _lengths(case)
    rows = list(range(len(lengths)))
    cache = moba_hip.PagedKVCache(
        len(rows), max(lengths) + (case["steps"] if kind == "serve" else case["extra"]),
        case["hkv"], case["d"], page_size=case["page"], chunk_size=case["chunk"],
        dtype=_DTYPE[case["dtype"]])
    if kind == "serve":
        cu = [0]
        for n in lengths:
            cu.append(cu[-1] + n)
        return dict(case=case, cache=cache, rows=rows, cu=cu, q=q, kn=kn, vn=vn,
                    k=torch.cat([a for a, _ in kv]), v=torch.cat([b for _, b in kv]))
    # sequences grow in turns, so that their pages lie among each other's
    for lo in range(0, max(lengths), 2048):
        for sid in rows:
            if lo < lengths[sid]:
                k, v = (x[lo:lo + 2048] for x in kv[sid])
                cache.append(k, v, sequence_ids=[sid], cu_seqlens=[0, k.shape[0]])
    plan = cache.prepare_decode(rows, case["hq"], topk=case["topk"], check_finite=False)
    plan.q.copy_(q)  # the bound buffer: the projection before it writes there
    if case["graph"]:
        plan.capture("attend")
    return dict(case=case, cache=cache, plan=plan)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        q, k, v = state["q"], state["k"], state["v"]
        out = moba_hip.run_impl("opt_hip", q, k, v, state["cu"], state["longest"],
                                state["config"])
        return (out, *torch.autograd.grad(out, (q, k, v), grad_outputs=state["dout"]))
    if kind == "prefill":
        with torch.no_grad():
            return moba_hip.run_impl("opt_hip", state["q"], state["k"], state["v"], state["cu"],
                                     state["longest"], state["config"])
    if kind == "merge":
        return moba_hip.merge_forward(*state["args"], kmax=case["kmax"])
    if kind == "decode":
        plan = state["plan"]
        res = plan.attend(plan.q, use_graph=case["graph"])
        return res.output, res.lse, res.selected_blocks
    cache = state["cache"]
    outs = torch.empty((case["steps"], *state["q"].shape), device="cuda",
                       dtype=state["q"].dtype)
    cache.reset()
    cache.append(state["k"], state["v"], sequence_ids=state["rows"], cu_seqlens=state["cu"])
    with cache.prepare_decode(state["rows"], case["hq"], topk=case["topk"],
                              check_finite=False) as plan:
        plan.q.copy_(state["q"])
        plan.k.copy_(state["kn"])
        plan.v.copy_(state["vn"])
        for out in outs:
            res = plan.step(plan.q, plan.k, plan.v)
            out.copy_(res.output)  # what the rest of the model takes from the step
    return outs, res.lse, res.selected_blocks


# --------------------------------------------------------------- work, bounds

def _pairs(case):
    """Attended (query head, key) pairs of a prefill: the causal triangle of
    every chunk plus min(topk - 1, candidates) whole chunks per row."""
    chunk, total, lengths = case["chunk"], 0, _lengths(case)
    candidates = sum(-(-n // chunk) - 1 for n in lengths)
    remote = min(case["topk"] - 1, candidates)
    for n in lengths:
        if remote == 0:
            total += n * (n + 1) // 2
            continue
        for i, lo in enumerate(range(0, n, chunk)):
            m = min(chunk, n - lo)
            total += m * (m + 1) // 2 + m * min(remote, i) * chunk
    return total * case["hq"]


def _decode_work(case, positions):
    """Bytes and operations of one decode step at ``positions``: the current
    chunk and the expected union, over a kv head's q heads, of the closed
    chunks they choose; the closed chunks' means; query, output and LSE."""
    hq, hkv, d, chunk = case["hq"], case["hkv"], case["d"], case["chunk"]
    group, nbytes, flops = hq // hkv, 0, 0
    for pos in positions:
        closed = pos // chunk
        own = pos - closed * chunk + 1
        picks = min(case["topk"] - 1, closed)
        union = closed * (1 - (1 - picks / closed) ** group) if closed else 0
        nbytes += hkv * d * 2 * (2 * (own + union * chunk) + closed)
        nbytes += hq * d * 2 * 2 + hq * 4 + hq * 4 * case["topk"]
        flops += hq * (4 * d * (own + picks * chunk) + 2 * d * closed)
    return nbytes, flops


def work(case):
    kind, d = case["kind"], case["d"]
    if kind in ("train", "prefill"):
        T, hq, hkv = sum(_lengths(case)), case["hq"], case["hkv"]
        qo, kv = T * hq * d * 2, T * hkv * d * 2
        train = kind == "train"
        # forward: q, k, v in, out; backward: dout in, dq, dk, dv out
        return dict(bytes=2 * qo + 2 * kv + (2 * qo + 2 * kv if train else 0),
                    flops=_pairs(case) * d * (14 if train else 4))
    if kind == "merge":
        rows, size = case["tokens"] * case["hq"], 4 if case["dtype"] == "fp32" else 2
        remote = 0.75 * case["kmax"] * rows
        return dict(bytes=int((2 * rows + remote) * d * size + 8 * rows + 8 * remote),
                    flops=int(2 * (rows + remote) * d))
    lengths = _lengths(case)
    if kind == "decode":
        nbytes, flops = _decode_work(case, [n - 1 for n in lengths])
        return dict(bytes=int(nbytes), flops=int(flops))
    nbytes, flops = 8 * sum(lengths) * case["hkv"] * d, 0  # prompt K/V in and into the pages
    for i in range(case["steps"]):
        b, f = _decode_work(case, [n + i for n in lengths])
        nbytes, flops = nbytes + b, flops + f
    return dict(bytes=int(nbytes), flops=int(flops))


def tolerance(case):
    # Outputs and gradients are stored in the input type, and probabilities
    # (and dS) enter the second product in it: a few half-ulps, as measured
    # against exact().
    if case["kind"] == "merge":
        return {"rel": 2 * _EPS[case["dtype"]], "max": 4 * _EPS[case["dtype"]]}
    return {"rel": 3 * _EPS[case["dtype"]], "max": 32 * _EPS[case["dtype"]]}


# --------------------------------------------------------------------- exact

def _choose(scores, legal, remote):
    """Boolean choice of the ``remote`` best legal chunks (last dimension)."""
    masked = scores.masked_fill(~legal, -math.inf)
    idx = masked.topk(min(remote, scores.shape[-1]), dim=-1).indices
    return torch.zeros_like(masked, dtype=torch.bool).scatter_(-1, idx, True) & legal


def _round(x, dtype):
    return x.to(_DTYPE[dtype]).double()


def _exact_prefill(case, seed):
    q, k, v, dout = (t.double() for t in _prefill_inputs(case, seed))
    lengths, chunk, hq, hkv = _lengths(case), case["chunk"], case["hq"], case["hkv"]
    group, scale = hq // hkv, case["d"] ** -0.5
    remote = min(case["topk"] - 1, sum(-(-n // chunk) - 1 for n in lengths))
    # per chunk: first key, last key, and the rows of each head beyond it
    chunks, at = [], 0
    for n in lengths:
        step = chunk if remote else n
        starts = list(range(at, at + n, step))
        chosen = None
        if remote and len(starts) > 1:
            means = torch.stack([k[s:s + chunk].mean(0) for s in starts[:-1]])  # [F, hkv, d]
            if case["precision"] == "upstream":
                means = _round(means, case["dtype"])
            own = torch.arange(n, device="cuda") // chunk
            legal = torch.arange(len(starts) - 1, device="cuda")[None] < own[:, None]
            scores = torch.einsum("tghd,fgd->tghf",
                                  q[at:at + n].view(n, hkv, group, -1), means)
            chosen = _choose(scores, legal[:, None, None].expand_as(scores), remote)
            chosen = chosen.reshape(n, hq, -1)
        for i, s in enumerate(starts):
            e = min(s + step, at + n)
            picked = [None] * hq
            if chosen is not None and i + 1 < len(starts):
                picked = [chosen[:, h, i].nonzero()[:, 0] + at for h in range(hq)]
            chunks.append((s, e, picked))
        at += n

    def blocks():
        """(head, kv head, query rows, first key, last key, causal mask)."""
        for s, e, picked in chunks:
            for h in range(hq):
                for lo in range(s, e, 4096):  # the chunk's own rows, causal
                    hi = min(lo + 4096, e)
                    rows = torch.arange(lo, hi, device="cuda")
                    keys = torch.arange(s, hi, device="cuda")
                    yield h, h // group, rows, s, hi, keys[None] > rows[:, None]
                if picked[h] is not None and picked[h].numel():
                    yield h, h // group, picked[h], s, e, None

    def scores(h, kh, rows, s, e, mask):
        x = (q[rows, h] @ k[s:e, kh].t()) * scale
        return x if mask is None else x.masked_fill_(mask, -math.inf)

    lse = torch.full(q.shape[:2], -math.inf, device="cuda", dtype=torch.float64)
    out = torch.zeros_like(q)
    for h, kh, rows, s, e, mask in blocks():
        x = scores(h, kh, rows, s, e, mask)
        part = torch.logsumexp(x, 1)
        new = torch.logaddexp(lse[rows, h], part)
        o = x.sub_(new[:, None]).exp_() @ v[s:e, kh]
        out[rows, h] = out[rows, h] * (lse[rows, h] - new).exp()[:, None] + o
        lse[rows, h] = new
    if case["kind"] == "prefill":
        return out
    delta = (out * dout).sum(-1)
    dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for h, kh, rows, s, e, mask in blocks():
        p = scores(h, kh, rows, s, e, mask).sub_(lse[rows, h][:, None]).exp_()
        g = dout[rows, h]
        dv[s:e, kh] += p.t() @ g
        ds = p.mul_((g @ v[s:e, kh].t()).sub_(delta[rows, h][:, None])).mul_(scale)
        dq[rows, h] += ds @ k[s:e, kh]
        dk[s:e, kh] += ds.t() @ q[rows, h]
    return out, dq, dk, dv


def _exact_decode(case, seed):
    kv, q, kn, vn = _decode_inputs(case, seed)
    hq, hkv, chunk = case["hq"], case["hkv"], case["chunk"]
    group, scale = hq // hkv, case["d"] ** -0.5
    steps = case.get("steps", 0)

    def attend(qb, k, v):
        """Output and LSE of one query row at the last of the keys given."""
        n = k.shape[0]
        closed = (n - 1) // chunk
        attended = torch.zeros((hkv, group, n), dtype=torch.bool, device="cuda")
        attended[..., closed * chunk:] = True
        if closed and case["topk"] > 1:
            means = _round(k[:closed * chunk].view(closed, chunk, hkv, -1).mean(1), case["dtype"])
            score = torch.einsum("hgd,fhd->hgf", qb, means)
            chosen = _choose(score, torch.ones_like(score, dtype=torch.bool), case["topk"] - 1)
            attended[..., :closed * chunk] = chosen.repeat_interleave(chunk, dim=-1)
        x = torch.einsum("hgd,nhd->hgn", qb, k) * scale
        x = x.masked_fill(~attended, -math.inf)
        return (torch.einsum("hgn,nhd->hgd", x.softmax(-1), v).reshape(hq, -1),
                torch.logsumexp(x, -1).view(hq))

    rows = []
    for b, (k, v) in enumerate(kv):
        k = torch.cat([k, kn[b:b + 1].expand(steps, -1, -1)]).double()
        v = torch.cat([v, vn[b:b + 1].expand(steps, -1, -1)]).double()
        qb = q[b].double().view(hkv, group, -1)
        ends = [k.shape[0] - steps + i + 1 for i in range(steps)] or [k.shape[0]]
        rows.append([attend(qb, k[:n], v[:n]) for n in ends])
    out = torch.stack([torch.stack([o for o, _ in row]) for row in rows], 1)
    lse = torch.stack([row[-1][1] for row in rows])
    return out if steps else out[0], lse, None


def _exact_merge(case, seed):
    so, sl, ro, rl, mapping = _merge_inputs(case, seed)
    T, H, D = so.shape
    so, sl, ro, rl = so.double().view(T * H, D), sl.double().view(-1), ro.double(), rl.double()
    rows = mapping.long()
    top = sl.scatter_reduce(0, rows, rl, "amax")
    weight = (rl - top[rows]).exp()
    own = (sl - top).exp()
    total = own.index_add(0, rows, weight)
    out = (so * own[:, None]).index_add(0, rows, ro * weight[:, None]) / total[:, None]
    return out.view(T, H, D), (top + total.log()).view(T, H)


def exact(case, seed):
    if case["kind"] in ("train", "prefill"):
        return _exact_prefill(case, seed)
    if case["kind"] == "merge":
        return _exact_merge(case, seed)
    return _exact_decode(case, seed)
