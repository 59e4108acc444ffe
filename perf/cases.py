"""The work that the framework is measured on: what a serving program has it
do for one request, through the public entry points (`prismkv_amd.Native8B`
and `prismkv_amd.core`).

* decode      the routed decode step of a stack of layers, each with its own
              tables and K/V (a model never decodes one layer twice in a row,
              so no table is cache-resident): `Native8B.__call__`, either
              eagerly or replayed from a HIP graph that the program captured
              once (the tail then stays as long as it was); with the strict
              unique cap, and with the q_activation router;
* two_call    the reference's two-call API: `route` and then `attention`;
* append      one update block of the interval policy, `Native8B.append`;
* build       the prefill index of one layer, `Native8B.from_keys`;
* replay      the per-group fp32 surface, `core.select_buckets` + `core.attend`.

Geometry: 8 KV groups x 4 query heads, head_dim 128, 3000 buckets, Top-16.
Keys, values and queries are N(0, 1) (or, for the stress configuration, keys
of a 64-component mixture, sigma 0.3), and the tables of a case that decodes
hold each key in the buckets of its 8 largest activations of a random
encoder, made here with torch: such a case measures the decode alone.
"""
import math

import torch

G, HQ, D, F, TOP = 8, 4, 128, 3000, 16
CHUNK, CHUNKS = 32, 94
KEY_MEAN = 8  # memberships per key


def listed():
    return [
        # the smallest request: one short prompt's layer, called eagerly; launch and host latency count
        dict(name="decode_short", kind="decode", layers=1, history=600, tail=32, graph=False),
        # a chat-sized context of no round size, one eager call per layer
        dict(name="decode_8k", kind="decode", layers=8, history=8009, tail=131, graph=False),
        # the kernel-check geometry (64K history, 256-row tail) as the captured decode step replays it
        dict(name="decode_64k", kind="decode", layers=8, history=65536, tail=256, graph=True),
        # the long-history geometry just before an update (131K history, 4096-row tail), captured
        dict(name="decode_131k", kind="decode", layers=6, history=131072, tail=4096, graph=True),
        # the stress geometry: 262K mixture keys under a strict budget of 1/16 of the history, captured
        dict(name="capped_262k", kind="decode", layers=4, history=262144, tail=256, graph=True, cap=0.0625,
             mixture=True),
        # a history past what one launch serves: the selection and the attention run apart
        dict(name="decode_700k", kind="decode", layers=1, history=700001, tail=1000, graph=False),
        # the other router: the queries' own activations choose up to 64 buckets
        dict(name="qact_32k", kind="decode", layers=4, history=32768, tail=512, graph=False, router="q_activation"),
        # a caller of the reference's two-call API, ragged
        dict(name="two_call_20k", kind="two_call", layers=4, history=20011, tail=777),
        # the update of the long-history configuration: 1024 tokens onto 131072
        dict(name="append_1024", kind="append", history=131072, block=1024),
        # the default update interval's block at a ragged history
        dict(name="append_4096", kind="append", history=33001, block=4096),
        # the prefill index of a 64K prompt's layer
        dict(name="build_64k", kind="build", history=65536),
        # the replay configuration: 8 groups one by one, fp32, 1024 history and 32 tail tokens
        dict(name="replay_fp32", kind="replay", history=1024, tail=32),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "capped", "qact", "two_call", "append", "append", "build", "build",
                       "replay", "long"])
    if kind in ("decode", "capped", "qact", "two_call"):
        history, tail = _between(rng, 600, 200000), _between(rng, 1, 4096)
        layers = rng.randint(1, 8 if history < 70000 else 4)
        if kind == "two_call":
            return dict(kind="two_call", layers=layers, history=history, tail=tail)
        case = dict(kind="decode", layers=layers, history=history, tail=tail, graph=rng.random() < 0.5)
        if kind == "capped":
            case.update(cap=rng.choice([0.03125, 0.0625, 0.125]), mixture=rng.random() < 0.5)
        if kind == "qact":
            case.update(router="q_activation", graph=False)
        return case
    if kind == "long":
        return dict(kind="decode", layers=1, history=_between(rng, 530000, 700000), tail=_between(rng, 1, 4096),
                    graph=False)
    if kind == "append":
        return dict(kind="append", history=_between(rng, 4000, 131072), block=_between(rng, 64, 4096))
    if kind == "build":
        return dict(kind="build", history=_between(rng, 6000, 65536))
    return dict(kind="replay", history=_between(rng, 300, 8000), tail=_between(rng, 1, 512))


# ------------------------------------------------------------------ inputs (plain torch)

def _generator(seed, layer=0):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + layer)


def _rows(n, gen):
    """bf16 N(0, 1) rows [8, n, 128], one group at a time."""
    x = torch.empty(G, n, D, dtype=torch.bfloat16, device="cuda")
    for g in range(G):
        x[g] = torch.randn(n, D, generator=gen, device="cuda")
    return x


def _mixture_rows(n, gen):
    x = torch.empty(G, n, D, dtype=torch.bfloat16, device="cuda")
    for g in range(G):
        centers = torch.randn(64, D, generator=gen, device="cuda")
        comp = torch.randint(0, 64, (n,), generator=gen, device="cuda")
        x[g] = centers[comp] + 0.3 * torch.randn(n, D, generator=gen, device="cuda")
    return x


def _encoders(gen):
    W = torch.randn(G, F, D, generator=gen, device="cuda") / D ** 0.5
    b = 0.05 * torch.randn(G, F, generator=gen, device="cuda")
    return W, b


def _memberships(keys, W):
    """(bucket, token) pairs, bucket-major and token-ascending, of each key's 8
    largest positive activations."""
    feats, toks = [], []
    for lo in range(0, len(keys), 32768):
        val, idx = (keys[lo:lo + 32768].float() @ W.T).topk(KEY_MEAN, dim=1)
        keep = val > 0
        feats.append(idx[keep])
        toks.append(torch.arange(lo, lo + len(val), device="cuda")[:, None].expand_as(idx)[keep])
    order = (torch.cat(feats) * len(keys) + torch.cat(toks)).sort().values
    return order // len(keys), order % len(keys)


def _moments(keys, feat, tok, dtype=torch.float32):
    """Counts, means and population variances of the buckets; sums in 64 bits,
    so that the order of the additions does not show."""
    n = torch.bincount(feat, minlength=F)
    den = n.clamp_min(1)[:, None].double()
    step = 1 << 20
    total = torch.zeros(F, D, dtype=torch.float64, device="cuda")
    for i in range(0, len(tok), step):
        total.index_add_(0, feat[i:i + step], keys[tok[i:i + step]].double())
    mean = (total / den).to(dtype)
    total.zero_()
    for i in range(0, len(tok), step):
        f = feat[i:i + step]
        total.index_add_(0, f, (keys[tok[i:i + step]].double() - mean[f].double()).square())
    return n, mean, (total / den).to(dtype)


def _tables(k, history, W, groups=G):
    """Per group: counts, mean, variance and the bucket lists as (bucket, token) pairs."""
    counts, mean, var, pairs = [], [], [], []
    for g in range(groups):
        keys = k[g, :history]
        pairs.append(_memberships(keys, W[g]))
        n, m, v = _moments(keys, *pairs[-1])
        counts.append(n)
        mean.append(m)
        var.append(v)
    return torch.stack(counts), torch.stack(mean), torch.stack(var), pairs


def _layer(case, seed, layer):
    """One layer's K, V, queries, encoders and tables."""
    gen = _generator(seed, layer)
    n = case["history"] + case["tail"]
    k = _mixture_rows(n, gen) if case.get("mixture") else _rows(n, gen)
    v = _rows(n, gen)
    q = torch.randn(G, HQ, D, generator=gen, device="cuda").to(torch.bfloat16)
    W, b = _encoders(gen)
    return k, v, q, W, b, _tables(k, case["history"], W)


QUERY_SCALE = 1.25


def _operator(case, parts):
    from prismkv_amd import Native8B
    k, v, q, W, b, (counts, mean, var, pairs) = parts
    width = max(len(t) for _, t in pairs)
    csr = torch.stack([torch.nn.functional.pad(t.int(), (0, width - len(t))) for _, t in pairs])
    offsets = torch.cat((torch.zeros(G, 1, dtype=torch.int64, device="cuda"), counts.cumsum(1)), dim=1)
    op = Native8B.from_tables(case["history"], counts, mean, var, csr, offsets, unique_cap=case.get("cap"))
    if case.get("router") == "q_activation":
        op.set_query_encoders(W, b, torch.full((G,), QUERY_SCALE))
        op.router = "q_activation"
    return op


def _append_inputs(case, seed):
    gen = _generator(seed)
    k = _rows(case["history"] + case["block"], gen)
    W, b = _encoders(gen)
    center = torch.stack([k[g, :case["history"]].double().mean(0).float() for g in range(G)])
    scale = 1.0 + 0.5 * torch.rand(G, generator=gen, device="cuda")
    return k, W, b, center, scale


def _replay_inputs(case, seed):
    gen = _generator(seed)
    n = case["history"] + case["tail"]
    k, v = (torch.randn(G, n, D, generator=gen, device="cuda") for _ in range(2))
    q = torch.randn(G, HQ, D, generator=gen, device="cuda")
    W, _ = _encoders(gen)
    return k, v, q, _tables(k, case["history"], W)


# ------------------------------------------------------------------ the cases

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "two_call"):
        state = dict(kind=kind, layers=[])
        for i in range(case["layers"]):
            parts = _layer(case, seed, i)
            state["layers"].append((_operator(case, parts), parts[2], parts[0], parts[1]))
        if case.get("graph"):
            # the captured decode step: warmed up once on a side stream, then captured
            def step():
                for op, q, k, v in state["layers"]:
                    op(q, k, v)
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                step()
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"]):
                step()
        return state
    if kind == "append":
        k, W, b, center, scale = _append_inputs(case, seed)
        tables = _tables(k, case["history"], W)
        from prismkv_amd import Native8B
        counts, mean, var, pairs = tables
        width = max(len(t) for _, t in pairs)
        csr = torch.stack([torch.nn.functional.pad(t.int(), (0, width - len(t))) for _, t in pairs])
        offsets = torch.cat((torch.zeros(G, 1, dtype=torch.int64, device="cuda"), counts.cumsum(1)), dim=1)
        op = Native8B.from_tables(case["history"], counts, mean, var, csr, offsets, center=center,
                                  capacity=case["history"] + case["block"])
        op.set_encoder_tables(W, b, scale, KEY_MEAN)
        first = case["history"] // 32
        return dict(kind=kind, op=op, k=k, block=case["block"], history=case["history"], first=first,
                    n=op.n.clone(), moments=op.moments.clone(), bits=op.bits[:, :, first:].clone())
    if kind == "build":
        gen = _generator(seed)
        k = _rows(case["history"], gen)
        W, b = _encoders(gen)
        scale = 1.0 + 0.5 * torch.rand(G, generator=gen, device="cuda")
        return dict(kind=kind, k=k, W=W, b=b, scale=scale, history=case["history"])
    from prismkv_amd.core import FeatureIndex
    k, v, q, (counts, mean, var, pairs) = _replay_inputs(case, seed)
    indices = []
    for g in range(G):
        lists = list(torch.split(pairs[g][1], counts[g].tolist()))
        indices.append(FeatureIndex(case["history"], k[g, :case["history"]].mean(0), counts[g], mean[g], var[g], lists))
    return dict(kind=kind, k=k, v=v, q=q, indices=indices, history=case["history"])


def run(state):
    kind = state["kind"]
    if kind == "decode":
        if "graph" in state:
            state["graph"].replay()
        else:
            for op, q, k, v in state["layers"]:
                op(q, k, v)
        return [_selection(op) for op, _, _, _ in state["layers"]]
    if kind == "two_call":
        for op, q, k, v in state["layers"]:
            op.route(q)
            op.attention(q, k, v)
        return [_selection(op) for op, _, _, _ in state["layers"]]
    if kind == "append":
        # several continuations of one shared prefix: the prefix's tables are put
        # back, then this continuation's block is indexed
        op = state["op"]
        op.n.copy_(state["n"])
        op.moments.copy_(state["moments"])
        op.bits[:, :, state["first"]:] = state["bits"]
        op.history = state["history"]
        op.append(state["k"], state["block"])
        return dict(counts=op.n, moments=op.moments, bits=op.bits, activations=op.update_activations(state["block"]))
    if kind == "build":
        from prismkv_amd import Native8B
        op = Native8B.from_keys(state["k"], state["history"], state["W"], state["b"], state["scale"], KEY_MEAN)
        return dict(counts=op.n, moments=op.moments, bits=op.bits, center=op.center)
    from prismkv_amd import core
    out = []
    for g, index in enumerate(state["indices"]):
        ids, meta = core.select_buckets(state["q"][g], index)
        # (the ids' number differs from input to input: `out` is the attention over all of them)
        out.append(dict(scores=meta["scores"], raw=meta["raw"], unique=meta["unique"],
                        out=core.attend(state["q"][g], state["k"][g], state["v"][g], ids, state["history"])))
    return out


def _selection(op):
    return dict(out=op.out, ids=op.ids, count=op.count, features=op.features, valid=op.valid, raw=op.raw)


def work(case):
    H = case["history"]
    tables = G * F * (2 * D * 4 + 4)  # moments and sizes
    if case["kind"] in ("decode", "two_call"):
        T, L = case["tail"], case["layers"]
        # distinct ids of the 16 best (up to 64) buckets, as these workloads have them
        unique = (0.19 if case.get("mixture") else 0.13) * H * (2.0 if case.get("router") else 1.0)
        if case.get("cap"):
            unique = min(unique, case["cap"] * H)
        selected = 60 if case.get("router") else TOP
        rows = G * (unique * (2 * D * 2 + 4) + T * 2 * D * 2 + selected * H / 8)
        first = G * F * (D * 4 + 8) if case.get("router") else tables
        return dict(bytes=L * (first + rows + 2 * G * HQ * D * 2),
                    flops=L * G * HQ * (2 * (F * (D if case.get("router") else 2 * D)) + 4 * D * (unique + T)))
    if case["kind"] == "append":
        N = case["block"]
        return dict(bytes=G * (N * D * 2 + F * D * 4 + N * F * 4 + F * N / 8) + 2 * tables, flops=G * 2.0 * N * F * D)
    if case["kind"] == "build":
        return dict(bytes=G * (H * D * 2 + F * D * 4 + F * H / 8) + tables, flops=G * 2.0 * H * F * D)
    T = case["tail"]
    return dict(bytes=tables + G * (0.13 * H * (2 * D * 4 + 8) + T * 2 * D * 4 + TOP * H / 8),
                flops=G * HQ * (2.0 * F * 2 * D + 4 * D * (0.13 * H + T)))


def tolerance(case):
    if case["kind"] in ("decode", "two_call"):
        # bf16 outputs of an exact softmax: two roundings of 2^-9 apart at most,
        # rms about 1.7e-3 against 64 bits; the selection is whole numbers and the same
        return dict(rel=5e-3, max=0.05)
    if case["kind"] in ("append", "build"):
        # a few memberships sit at the budget's edge within the rounding of the 128-term
        # fp32 sums (of 4.2 million in a 64K build, 2-3 differ between two fp32 orders and
        # 4 from 64 bits); each takes its bucket's size, mean and variance with it: rel
        # 4.5e-4, max 0.23 and 3.3e-4 of the sizes measured.  The activations themselves
        # differ by 2e-7, which `exact` holds them to.
        return dict(rel=2e-3, max=0.9, differ=1.5e-3)
    return dict(rel=1e-5, max=1e-3)


# ------------------------------------------------------------------ 64 bits

def _ranked(q, counts, mean, var):
    """Scores and the 16 best live buckets of one group, in 64 bits."""
    q = q.double()
    logits = counts.clamp_min(1).double().log() + (q @ mean.double().T) / math.sqrt(D)
    logits = logits + (q * q) @ var.double().T / (2 * D)
    logits = logits.masked_fill(counts == 0, -math.inf)
    scores = torch.softmax(logits, dim=-1).mean(0)
    order = torch.argsort(scores, descending=True, stable=True)
    return scores, order[counts[order] > 0][:TOP]


def _ranked_by_activation(q, counts, W, b):
    act = torch.relu((q.double() / QUERY_SCALE) @ W.double().T + b.double())
    scores = torch.zeros(F, dtype=torch.float64, device="cuda")
    for a in act:
        best = torch.argsort(a, descending=True, stable=True)[:TOP]
        scores[best] += a[best] / a[best].sum().clamp_min(1e-20) / HQ
    order = torch.argsort(scores, descending=True, stable=True)
    return order[(scores[order] > 0) & (counts[order] > 0)]


def _attend(q, k, v, order, pair, history, cap):
    """The union of the ranked buckets (skipping one that would overflow the
    budget) and the exact attention over it and the tail, in 64 bits."""
    limit = history if cap is None else math.floor(history * cap)
    taken = torch.zeros(history, dtype=torch.bool, device="cuda")
    size = 0
    for bucket in order.tolist():
        members = pair[1][pair[0] == bucket]
        fresh = int((~taken[members]).sum())
        if size + fresh <= limit:
            taken[members] = True
            size += fresh
    rows = torch.cat((taken.nonzero().flatten(), torch.arange(history, len(k), device="cuda")))
    p = torch.softmax(q.double() @ k[rows].double().T / math.sqrt(D), dim=-1)
    return p @ v[rows].double()


def exact(case, seed):
    kind, none = case["kind"], dict(ids=None, count=None, features=None, valid=None, raw=None)
    if kind in ("decode", "two_call"):
        out = []
        for i in range(case["layers"]):
            k, v, q, W, b, (counts, mean, var, pairs) = _layer(case, seed, i)
            heads = []
            for g in range(G):
                order = _ranked_by_activation(q[g], counts[g], W[g], b[g]) if case.get("router") else \
                    _ranked(q[g], counts[g], mean[g], var[g])[1]
                heads.append(_attend(q[g], k[g], v[g], order, pairs[g], case["history"], case.get("cap")))
            out.append(dict(none, out=torch.stack(heads)))
        return out
    if kind == "append":
        # the tables follow from which memberships the budget's edge takes, which
        # rounding decides: 64 bits have no say in them, only in the activations
        k, W, b, center, scale = _append_inputs(case, seed)
        x = (k[:, case["history"]:].double() - center.double()[:, None]) / scale.double()[:, None, None]
        act = torch.stack([torch.relu(x[g] @ W[g].double().T + b[g].double()) for g in range(G)])
        return dict(counts=None, moments=None, bits=None, activations=act)
    if kind == "build":
        k = _rows(case["history"], _generator(seed))
        return dict(counts=None, moments=None, bits=None,
                    center=torch.stack([k[g].double().mean(0) for g in range(G)]))
    k, v, q, (counts, mean, var, pairs) = _replay_inputs(case, seed)
    out = []
    for g in range(G):
        scores, order = _ranked(q[g], counts[g], mean[g], var[g])
        out.append(dict(raw=None, unique=None, scores=scores,
                        out=_attend(q[g], k[g], v[g], order, pairs[g], case["history"], None)))
    return out
