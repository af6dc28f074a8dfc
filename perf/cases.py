"""The attention work of a voice assistant on one MI355X, as cases to time.

A case is one pass of what an application does around this library: a token
step through a model's layers, a prompt or a conversation turn through one
layer or a few, an encoder layer. Shapes are the ones the tests, the benchmark
and the layer stack of this repository use (a Llama chat model of 32 query and
8 KV heads, a translator of 40 and 40, a Whisper of 20 heads of 64), with
lengths that are not round. Token steps, and a turn over a few layers, are
captured in a HIP graph once and replayed, as the benchmark runs them; prompts
and the encoder are called eagerly, since each has a length of its own.

Kinds (the `kind` of a case):

  short_prompt   rows appended to an f32 cache, then causal attention over it
                 (Whisper's prompt, the f32 MHA prefill): one layer, eager
  whisper_step   one token of the Whisper decoder: K and V rows into the f32
                 self cache, self-attention, cross-attention over the encoder's
                 f16 K/V, in every layer
  encoder        the Whisper encoder's self-attention off its stacked q/k/v rows
  step           one token of a Llama: q rotated, k rotated and stored with v,
                 attention over the f16 cache (reference layout with the int8
                 twin of the context; tiled layout with or without it), for `rows` sequences
                 in every layer
  turn           a conversation turn (or a prompt, past = 0): q and k rotated,
                 K and V appended, causal attention over past and new
                 positions; `graph` captures `layers` of it
  q8_step        one token of `nseq` sequences over a Q8_0 cache: rotate,
                 quantise and store per sequence (`store`), then the batched
                 attention, in every layer
  q8_fill        a prompt's keys rotated and quantised with its values into a
                 Q8_0 cache slot
"""
import math

import torch

from ttsxabe_amd.gpu import DecodeScratch, Gpu, KvCacheQ8, TiledCache16

THETA = 500000.0


def listed():
    return [
        # The smallest call: a 100-odd row prompt through one f32 layer (8 heads of 64). Latency and launches.
        dict(name="short_prompt_f32", kind="short_prompt", heads=8, kv=8, hd=64, n=127, past=0, cap=448),
        # Speech recognition, one decoded token: 16 layers, 113 positions said, a 1500-frame window.
        dict(name="whisper_step", kind="whisper_step", layers=16, heads=20, hd=64, tk=113, cap=448, t=1500),
        # Speech recognition, one encoder layer over a 30 s window.
        dict(name="whisper_encoder", kind="encoder", heads=20, hd=64, t=1500),
        # Chat, one token early in a conversation, the drop-in cache layout and the int8 twin the o-projection reads.
        dict(name="chat_step_short", kind="step", layers=32, heads=32, kv=8, hd=128, tk=211, cap=256, rows=1,
             tiled=False, twin=True, scaled=True),
        # Chat, one token in a long conversation, the tiled cache: the benchmark's shape at a length that is not round.
        dict(name="chat_step_4k", kind="step", layers=32, heads=32, kv=8, hd=128, tk=4001, cap=4096, rows=1,
             tiled=True, twin=False, scaled=True),
        # Translation, two sentences decoded side by side, multi-head attention in the drop-in layout with the twin.
        dict(name="translator_step", kind="step", layers=40, heads=40, kv=40, hd=128, tk=739, cap=1024, rows=2,
             tiled=False, twin=True, scaled=False),
        # Serving, one token of eight sequences over Q8_0 caches, stores included.
        dict(name="q8_step_8", kind="q8_step", layers=8, heads=32, kv=8, hd=128, nseq=8, low=256, high=4096, cap=4096,
             store=True),
        # Serving, the batched Q8_0 attention alone at 32 long sequences: the most bytes a decode reads.
        dict(name="q8_decode_32", kind="q8_step", layers=4, heads=32, kv=8, hd=128, nseq=32, low=256, high=8192,
             cap=8192, store=False),
        # Chat, a user's next turn after three thousand positions, four layers, the drop-in layout.
        dict(name="chat_turn", kind="turn", layers=4, heads=32, kv=8, hd=128, n=173, past=3011, cap=4096,
             tiled=False, graph=True, scaled=True),
        # Chat, a document as first prompt, one layer, the drop-in layout.
        dict(name="chat_prompt_2k", kind="turn", layers=1, heads=32, kv=8, hd=128, n=1999, past=0, cap=2048,
             tiled=False, graph=False, scaled=True),
        # Chat, the largest prompt, one layer, the tiled layout: matrix work.
        dict(name="chat_prompt_8k", kind="turn", layers=1, heads=32, kv=8, hd=128, n=8192, past=0, cap=8192,
             tiled=True, graph=False, scaled=False),
        # Serving, a prompt into a Q8_0 slot.
        dict(name="q8_fill_3k", kind="q8_fill", heads=32, kv=8, hd=128, n=3001, past=0, cap=8192, slots=4),
    ]


def _log(rng, low, high):
    """A whole number between low and high, spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _room(need):
    """Positions a cache holds for `need`: the layer stack's powers of two from 256."""
    return max(256, 1 << (need - 1).bit_length())


def draw(rng):
    kind = rng.choice(["short_prompt", "whisper_step", "encoder", "step", "step", "turn", "turn", "prompt", "prompt",
                       "q8_step", "q8_fill"])
    if kind == "short_prompt":
        heads = rng.choice([6, 8, 12, 16, 20])
        n = _log(rng, 3, 224)
        return dict(kind=kind, heads=heads, kv=heads, hd=64, n=n, past=rng.randint(0, 448 - n), cap=448)
    if kind == "whisper_step":
        return dict(kind=kind, layers=16, heads=rng.choice([6, 8, 12, 16, 20]), hd=64, tk=rng.randint(1, 448),
                    cap=448, t=_log(rng, 100, 1500))
    if kind == "encoder":
        return dict(kind=kind, heads=rng.choice([6, 8, 12, 16, 20]), hd=64, t=_log(rng, 75, 1500))
    heads, kv, hd = rng.choice([(32, 8, 128), (32, 8, 128), (40, 40, 128), (32, 8, 64), (8, 2, 128), (16, 8, 128)])
    tiled, scaled = rng.random() < 0.5, rng.random() < 0.5
    if kind == "step":
        tk = _log(rng, 5, 8000 if kv <= 8 else 4000)
        rows = rng.randint(1, 4) if tk < 1500 else 1
        return dict(kind=kind, layers=rng.choice([8, 16]), heads=heads, kv=kv, hd=hd, tk=tk, cap=_room(tk), rows=rows,
                    tiled=tiled, twin=not tiled or rng.random() < 0.5, scaled=scaled)
    if kind == "turn":
        n, past = _log(rng, 6, 500), _log(rng, 100, 7600 if kv <= 8 else 3500)
        return dict(kind=kind, layers=4, heads=heads, kv=kv, hd=hd, n=n, past=past, cap=_room(n + past), tiled=tiled,
                    graph=True, scaled=scaled)
    if kind == "prompt":
        n = _log(rng, 300, 7900 if kv <= 8 else 3968)
        return dict(kind="turn", layers=1, heads=heads, kv=kv, hd=hd, n=n, past=0, cap=_room(n), tiled=tiled,
                    graph=False, scaled=scaled)
    heads, kv, hd = rng.choice([(32, 8, 128), (32, 8, 128), (32, 8, 64), (16, 4, 128)])
    if kind == "q8_step":
        nseq, high = _log(rng, 2, 32), _log(rng, 500, 8000)
        store = rng.random() < 0.5
        return dict(kind=kind, layers=4, heads=heads, kv=kv, hd=hd, nseq=nseq, low=rng.randint(20, high // 2),
                    high=high, cap=_room(high), store=store)
    n = _log(rng, 100, 7900)
    past = rng.randint(0, 8192 - n)
    return dict(kind=kind, heads=heads, kv=kv, hd=hd, n=n, past=past, cap=8192, slots=4)


# ------------------------------------------------------------------- inputs


def _gen(seed, what=0):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + what) % (1 << 62))


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _freq_div(c):
    """Per-frequency divisors of a long-context Llama: 1 for the fast pairs, 8 for the slow ones, a ramp between."""
    if not c.get("scaled"):
        return None
    j = torch.arange(c["hd"] // 2, device="cuda", dtype=torch.float32)
    return 1.0 + 7.0 * ((j / (c["hd"] // 2) - 0.4) / 0.3).clamp(0.0, 1.0)


def _lengths(c):
    """The live positions of the sequences: part of the case, so that a pass is the same work whatever the seed."""
    g = torch.Generator().manual_seed(1000 * c["nseq"] + c["low"] + c["high"])
    return [int(x) for x in torch.randint(c["low"], c["high"] + 1, (c["nseq"],), generator=g)]


def _step_inputs(c, seed):
    """q, k, v of one token [layers, rows, heads * hd], and the f16 caches as they lie before it:
    K [layers, rows, kv, cap, hd], V [layers, rows, kv, hd, cap], zero from position tk - 1 on."""
    L, R, H, KV, D, cap = c["layers"], c["rows"], c["heads"], c["kv"], c["hd"], c["cap"]
    g = _gen(seed)
    q, k, v = _normal(g, L, R, H * D), _normal(g, L, R, KV * D), _normal(g, L, R, KV * D)
    kc = torch.empty(L, R, KV, cap, D, dtype=torch.float16, device="cuda").normal_(generator=g)
    vc = torch.empty(L, R, KV, D, cap, dtype=torch.float16, device="cuda").normal_(generator=g)
    kc[:, :, :, c["tk"] - 1:] = 0
    vc[..., c["tk"] - 1:] = 0
    return q, k, v, kc, vc


def _turn_inputs(c, seed):
    """As _step_inputs, for n rows [layers, n, heads * hd] at positions past.. and caches [layers, kv, ...]."""
    L, N, H, KV, D, cap = c["layers"], c["n"], c["heads"], c["kv"], c["hd"], c["cap"]
    g = _gen(seed)
    q, k, v = _normal(g, L, N, H * D), _normal(g, L, N, KV * D), _normal(g, L, N, KV * D)
    kc = torch.zeros(L, KV, cap, D, dtype=torch.float16, device="cuda")
    vc = torch.zeros(L, KV, D, cap, dtype=torch.float16, device="cuda")
    if c["past"]:
        kc[:, :, :c["past"]] = _normal(g, L, KV, c["past"], D)
        vc[..., :c["past"]] = _normal(g, L, KV, D, c["past"])
    return q, k, v, kc, vc


def _short_inputs(c, seed):
    H, D, N, cap = c["heads"], c["hd"], c["n"], c["cap"]
    g = _gen(seed)
    q, k, v = _normal(g, N, H * D), _normal(g, N, H * D), _normal(g, N, H * D)
    kc, vc = _normal(g, H, cap, D), _normal(g, H, D, cap)
    kc[:, c["past"]:] = 0
    vc[..., c["past"]:] = 0
    return q, k, v, kc, vc


def _whisper_inputs(c, seed):
    L, H, D, cap, t = c["layers"], c["heads"], c["hd"], c["cap"], c["t"]
    g = _gen(seed)
    q, k, v, qx = (_normal(g, L, H * D) for _ in range(4))
    kc, vc = _normal(g, L, H, cap, D), _normal(g, L, H, D, cap)
    kc[:, :, c["tk"] - 1:] = 0
    vc[..., c["tk"] - 1:] = 0
    xk = torch.empty(L, H, t, D, dtype=torch.float16, device="cuda").normal_(generator=g)
    xv = torch.empty(L, H, D, -(-t // 4) * 4, dtype=torch.float16, device="cuda").normal_(generator=g)
    return q, k, v, qx, kc, vc, xk, xv


def _q8_rows(c, seed, layer, s, n):
    """The K and V rows [n, kv * hd] that sequence s holds in a layer."""
    g = _gen(seed, 1 + layer * 64 + s)
    return _normal(g, n, c["kv"] * c["hd"]), _normal(g, n, c["kv"] * c["hd"])


def _q8_token(c, seed):
    L, S, H, KV, D = c["layers"], c["nseq"], c["heads"], c["kv"], c["hd"]
    g = _gen(seed)
    return _normal(g, L, S, H * D), _normal(g, L, S, KV * D), _normal(g, L, S, KV * D)


def _q8_slots(c):
    """Sequence s sits in this slot: not in order, as sequences come and go."""
    return [(5 * s + 3) % c["nseq"] if c["nseq"] % 5 else c["nseq"] - 1 - s for s in range(c["nseq"])]


# ------------------------------------------------------------------ prepare


def _captured(step):
    """One eager call of the step (the scratch takes its size), then the step in a HIP graph."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = step()
    torch.cuda.current_stream().wait_stream(s)
    return graph, out


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    """One pass: the captured graph, or the calls themselves."""
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["step"]()


def _prepare_short(c, seed):
    g = Gpu(0)
    q, k, v, kc, vc = _short_inputs(c, seed)
    q, k, v, kc, vc = (x.view(-1) for x in (q, k, v, kc, vc))
    H, D, N, P, cap, scale = c["heads"], c["hd"], c["n"], c["past"], c["cap"], c["hd"] ** -0.5

    def step():
        g.cache_append(k, 0, kc, N, H, D, cap, P, False)
        g.cache_append(v, 0, vc, N, H, D, cap, P, True)
        return {"ctx": g.flash_attn(q, kc, vc, N, P, H, H, D, cap, scale, True), "k": kc, "v": vc}

    return {"step": step}


def _prepare_whisper(c, seed):
    g, scratch = Gpu(0), DecodeScratch()
    q, k, v, qx, kc, vc, xk, xv = _whisper_inputs(c, seed)
    L, H, D, tk, cap, t, scale = c["layers"], c["heads"], c["hd"], c["tk"], c["cap"], c["t"], c["hd"] ** -0.5
    # The cross cache's capacity is its frame count, rounded up to the four halves a V row is read by.
    tc = -(-t // 4) * 4
    xk = torch.cat([xk, torch.zeros(L, H, tc - t, D, dtype=torch.float16, device="cuda")], 2)

    def step():
        self_ctx, cross_ctx = [], []
        for i in range(L):
            g.cache_append(k[i], 0, kc[i].view(-1), 1, H, D, cap, tk - 1, False)
            g.cache_append(v[i], 0, vc[i].view(-1), 1, H, D, cap, tk - 1, True)
            self_ctx.append(g.attn_decode(q[i], kc[i].view(-1), vc[i].view(-1), H, H, D, tk, cap, scale, True,
                                          scratch))
            cross_ctx.append(g.attn_decode_f16(qx[i], xk[i].view(-1), xv[i].view(-1), H, H, D, t, tc, scale, True,
                                               scratch))
        return {"self": self_ctx, "cross": cross_ctx, "k": kc, "v": vc}

    graph, out = _captured(step)
    return {"graph": graph, "out": out, "scratch": scratch, "inputs": (q, k, v, qx, kc, vc, xk, xv)}


def _prepare_encoder(c, seed):
    g = Gpu(0)
    qkv = _normal(_gen(seed), c["t"] * 3 * c["heads"] * c["hd"])
    return {"step": lambda: {"ctx": g.flash_attn_rows(qkv, c["t"], c["heads"], c["hd"], c["hd"] ** -0.5)}}


def _prepare_step(c, seed):
    g, scratch = Gpu(0), DecodeScratch()
    fresh, k, v, kc, vc = _step_inputs(c, seed)
    q, fd = fresh.clone(), _freq_div(c)
    L, R, H, KV, D, tk, cap, scale = (c["layers"], c["rows"], c["heads"], c["kv"], c["hd"], c["tk"], c["cap"],
                                      c["hd"] ** -0.5)
    n = H * D
    ctx = torch.zeros(L, R, n, device="cuda")
    twins = [g.q8_zeros(R, n) for _ in range(L)] if c["twin"] else [None] * L
    if c["tiled"]:
        caches = []
        for i in range(L):
            for r in range(R):
                caches.append(TiledCache16(KV, D, cap))
                g.t16_from_ref(kc[i, r].view(-1), vc[i, r].view(-1), caches[-1], max(tk - 1, 1))
        stack = torch.stack([t.data for t in caches])  # one allocation for every layer
        for t, data in zip(caches, stack):
            t.data = data
        kc = vc = None

    def step():
        for i in range(L):
            qi, ki, vi, oi = q[i].view(-1), k[i].view(-1), v[i].view(-1), ctx[i].view(-1)
            for r in range(R):
                if c["tiled"]:
                    t = caches[i * R + r]
                    g.t16_rope_cache(qi, r * n, ki, r * KV * D, vi, r * KV * D, fd, H, THETA, tk - 1, t)
                    if c["twin"] or R > 1:
                        g.attn_decode_t16_q_row(qi, r * n, t, H, tk, scale, False, scratch, oi, twins[i], r)
                    else:
                        g.attn_decode_t16(qi, t, H, tk, scale, False, scratch, out=oi)
                    continue
                kr, vr = kc[i, r].view(-1), vc[i, r].view(-1)
                g.rope_cache_f16(qi, r * n, ki, r * KV * D, vi, r * KV * D, fd, H, KV, D, THETA, tk - 1, kr, vr, cap)
                g.attn_decode_f16_q_row(qi, r * n, kr, vr, H, KV, D, tk, cap, scale, False, scratch, oi, twins[i], r)
        return {"ctx": ctx, "q": q}

    graph, out = _captured(step)
    q.copy_(fresh)  # the eager call rotated it
    if c["twin"]:
        out["codes"] = [t.buf[: t.scale_offset()] for t in twins[:30]]
        out["scales"] = [t.buf[t.scale_offset():].view(torch.float32) for t in twins[:30]]
    if c["tiled"]:
        out["cache"] = stack
    else:
        out["k"], out["v"] = kc, vc
    return {"graph": graph, "out": out, "scratch": scratch, "inputs": (q, k, v, fd, kc, vc),
            "tiled": caches if c["tiled"] else None}


def _prepare_turn(c, seed):
    g = Gpu(0)
    q, k, v, kc, vc = _turn_inputs(c, seed)
    fd = _freq_div(c)
    L, N, P, H, KV, D, cap, scale = (c["layers"], c["n"], c["past"], c["heads"], c["kv"], c["hd"], c["cap"],
                                     c["hd"] ** -0.5)
    caches = []
    if c["tiled"]:
        for i in range(L):
            caches.append(TiledCache16(KV, D, cap))
            if P:
                g.t16_from_ref(kc[i].view(-1), vc[i].view(-1), caches[i], P)
        kc = vc = None

    def layer(i):
        qi, ki, vi = q[i].view(-1), k[i].view(-1), v[i].view(-1)
        g.rope_scaled(qi, 0, fd, N, H, D, THETA, P)
        g.rope_scaled(ki, 0, fd, N, KV, D, THETA, P)
        if c["tiled"]:
            t = caches[i]
            g.t16_append(ki, 0, t, N, P, False)
            g.t16_append(vi, 0, t, N, P, True)
            return g.flash_attn_t16(qi, t, N, P, H, scale, True)
        kl, vl = kc[i].view(-1), vc[i].view(-1)
        g.cache_append_f16(ki, 0, kl, N, KV, D, cap, P, False)
        g.cache_append_f16(vi, 0, vl, N, KV, D, cap, P, True)
        return g.flash_attn_f16(qi, kl, vl, N, P, H, KV, D, cap, scale, True)

    def step():
        ctx = [layer(i) for i in range(L)]
        return {"ctx": ctx, "q": q, "krot": k, "k": [t.data for t in caches] if c["tiled"] else kc, "v": vc}

    if not c["graph"]:
        return {"step": step}
    fresh = q.clone(), k.clone()
    graph, out = _captured(step)
    q.copy_(fresh[0])  # the eager call rotated them
    k.copy_(fresh[1])
    return {"graph": graph, "out": out, "inputs": (q, k, v, fd, kc, vc), "tiled": caches}


def _prepare_q8(c, seed):
    g, scratch = Gpu(0), DecodeScratch()
    fresh, k, v = _q8_token(c, seed)
    q = fresh.clone()
    L, S, H, KV, D, cap, scale = c["layers"], c["nseq"], c["heads"], c["kv"], c["hd"], c["cap"], c["hd"] ** -0.5
    lens, slots = _lengths(c), _q8_slots(c)
    n, m = H * D, KV * D
    caches = []
    for i in range(L):
        caches.append(KvCacheQ8(S, KV, D, cap))
        for s in range(S):
            kr, vr = _q8_rows(c, seed, i, s, lens[s])
            g.kv_q8_append(kr.view(-1), 0, vr.view(-1), 0, caches[i], slots[s], lens[s], 0)
    tk_dev = torch.tensor(lens, dtype=torch.int32, device="cuda")
    slot_dev = torch.tensor(slots, dtype=torch.int32, device="cuda")
    ctx = torch.zeros(L, S * n, device="cuda")

    def step():
        for i in range(L):
            qi = q[i].view(-1)
            if c["store"]:
                ki, vi = k[i].view(-1), v[i].view(-1)
                for s in range(S):
                    g.rope_cache_q8(qi, s * n, ki, s * m, vi, s * m, None, H, THETA, lens[s] - 1, caches[i], slots[s])
            g.attn_decode_q8_batch(qi, caches[i], tk_dev, slot_dev, c["high"], H, scale, False, scratch, out=ctx[i])
        return {"ctx": ctx, "q": q, "cache": [t.data for t in caches] if c["store"] else None}

    graph, out = _captured(step)
    q.copy_(fresh)  # the eager call rotated it
    return {"graph": graph, "out": out, "scratch": scratch, "inputs": (q, k, v, tk_dev, slot_dev), "caches": caches}


def _prepare_q8_fill(c, seed):
    g = Gpu(0)
    k, v = _q8_rows(c, seed, 0, 0, c["n"])
    k, v = k.view(-1), v.view(-1)
    cache = KvCacheQ8(c["slots"], c["kv"], c["hd"], c["cap"])

    def step():
        g.rope(k, 0, c["n"], c["kv"], c["hd"], THETA, c["past"])
        g.kv_q8_append(k, 0, v, 0, cache, 1, c["n"], c["past"])
        return {"k": k, "cache": cache.data}

    return {"step": step}


_PREPARE = {"short_prompt": _prepare_short, "whisper_step": _prepare_whisper, "encoder": _prepare_encoder,
            "step": _prepare_step, "turn": _prepare_turn, "q8_step": _prepare_q8, "q8_fill": _prepare_q8_fill}


# --------------------------------------------------------- work, tolerance


def _pairs(n, past):
    return n * past + n * (n + 1) // 2


def work(case):
    """Each input read once, each output written once: projections, the live K/V, the context, what is stored."""
    c, k = case, case["kind"]
    H, D = c["heads"], c["hd"]
    KV = c.get("kv", H)
    if k == "short_prompt":
        rows, live = c["n"] * H * D * 4, (c["past"] + c["n"]) * H * D * 4
        return {"bytes": 4 * rows + 2 * live, "flops": 4 * D * H * _pairs(c["n"], c["past"])}
    if k == "whisper_step":
        per = 6 * H * D * 4 + 2 * c["tk"] * H * D * 4 + 2 * c["t"] * H * D * 2
        return {"bytes": c["layers"] * per, "flops": c["layers"] * 4 * D * H * (c["tk"] + c["t"])}
    if k == "encoder":
        return {"bytes": c["t"] * H * D * (3 * 4 + 2), "flops": 4 * D * H * c["t"] * c["t"]}
    if k == "step":
        row = (3 * H + 2 * KV) * D * 4 + 2 * c["tk"] * KV * D * 2 + (H * D * 9 // 8 if c["twin"] else 0)
        return {"bytes": c["layers"] * c["rows"] * row, "flops": c["layers"] * c["rows"] * 4 * D * H * c["tk"]}
    if k == "turn":
        # q in, rotated q out, context out; k in, rotated k out, v in; both caches' new rows out, past rows in.
        rows = c["n"] * (3 * H + 3 * KV) * D * 4 + 2 * (c["n"] + c["past"]) * KV * D * 2
        return {"bytes": c["layers"] * rows, "flops": c["layers"] * 4 * D * H * _pairs(c["n"], c["past"])}
    if k == "q8_step":
        keys = sum(_lengths(c))
        per = 2 * KV * (D + D // 16) * keys + c["nseq"] * (2 * H + (H + 2 * KV if c["store"] else 0)) * D * 4
        return {"bytes": c["layers"] * per, "flops": c["layers"] * 4 * D * H * keys}
    return {"bytes": c["n"] * KV * D * (3 * 4 + 2) + c["n"] * KV * D // 8, "flops": 0}


def tolerance(case):
    """About four times what was measured between the path and its sums in 64 bits.

    f16 attention (probabilities rounded to f16): 2.3e-4 to 4.7e-4. f32 decode: 2e-7, and behind a rotation what the
    f32 angle is off at position p, about 1e-8 p (4.3e-5 at 4000). An element that a rotation moves over a rounding
    boundary is one f16 step (1e-3 of its value) or one code off where it is stored."""
    c, k = case, case["kind"]
    if k == "short_prompt":
        return {"rel": 1.5e-3, "max": 2e-2}
    if k == "whisper_step":
        return {"rel": 2e-6, "max": 2e-5}
    if k == "encoder":
        return {"rel": 2e-3, "max": 2e-2}
    if k == "step":
        return {"rel": 1e-5 + 4e-8 * c["tk"], "max": 4e-3, "differ": 1e-3}
    if k == "turn":
        return {"rel": 1.3e-3, "max": 2e-2}
    if k == "q8_step":
        return {"rel": 1e-3, "max": 1e-2, "differ": 1e-6}
    return {"rel": 1e-5 + 2e-8 * (c["n"] + c["past"]), "max": 4e-3, "differ": 1e-3}


# -------------------------------------------------------------------- exact


def _half(x):
    """A value as an f16 cache holds it."""
    return x.float().half().double()


def _rotated(x, c, pos):
    """x [n, heads * hd] rotated at positions pos [n] in 64 bits, halves paired."""
    n, D = x.shape[0], c["hd"]
    inv = THETA ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    fd = _freq_div(c)
    if fd is not None:
        inv = inv / fd.double()
    a = pos.double().view(-1, 1, 1) * inv
    x = x.double().view(n, -1, D)
    lo, hi = x[..., : D // 2], x[..., D // 2:]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1).reshape(n, -1)


def _attend(q, K, V, scale, past=None):
    """q [n, H, D], K and V [kv, keys, D], all 64-bit; causal from `past` where it is given. [n, H * D]."""
    n, H, D = q.shape
    KV, keys = K.shape[0], K.shape[1]
    out = torch.empty(n, H, D, dtype=torch.float64, device="cuda")
    dead = None
    if past is not None and n > 1:
        dead = torch.arange(keys, device="cuda").view(1, -1) > torch.arange(n, device="cuda").view(-1, 1) + past
    for h in range(H):
        kv = h // (H // KV)
        s = q[:, h].contiguous() @ K[kv].t().contiguous()
        s *= scale
        if dead is not None:
            s.masked_fill_(dead, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ V[kv].contiguous()
    return out.reshape(n, H * D)


def _steps(q, K, V, scale):
    """One query [H, D] over K, V [kv, keys, D]: [H * D]."""
    H, D = q.shape
    s = torch.matmul(K, q.view(K.shape[0], -1, D).transpose(1, 2).contiguous()) * scale
    p = torch.softmax(s, 1).transpose(1, 2).contiguous()
    return torch.matmul(p, V).reshape(H * D)


def _quantised(x):
    """Q8_0 of x [n, kv * hd] in blocks of 32, as it reads back, in 64 bits."""
    b = x.double().view(x.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    code = torch.where(d > 0, b / d, torch.zeros_like(b))
    code = torch.sign(code) * torch.floor(code.abs() + 0.5)
    return (code * _half(d)).view(x.shape[0], -1)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _exact_short(c, seed):
    q, k, v, kc, vc = _short_inputs(c, seed)
    H, D, N, P = c["heads"], c["hd"], c["n"], c["past"]
    kc[:, P:P + N] = k.view(N, H, D).transpose(0, 1)
    vc[..., P:P + N] = v.view(N, H, D).permute(1, 2, 0)
    K, V = kc[:, : P + N].double(), vc[..., : P + N].transpose(1, 2).double()
    return {"ctx": _attend(q.view(N, H, D).double(), K, V, D ** -0.5, P).view(-1), "k": kc.double().view(-1),
            "v": vc.double().view(-1)}


def _exact_whisper(c, seed):
    q, k, v, qx, kc, vc, xk, xv = _whisper_inputs(c, seed)
    L, H, D, tk, t = c["layers"], c["heads"], c["hd"], c["tk"], c["t"]
    a, x = [], []
    for i in range(L):
        kc[i, :, tk - 1] = k[i].view(H, D)
        vc[i, :, :, tk - 1] = v[i].view(H, D)
        a.append(_steps(q[i].view(H, D).double(), kc[i, :, :tk].double(),
                        vc[i, :, :, :tk].transpose(1, 2).double().contiguous(), D ** -0.5))
        x.append(_steps(qx[i].view(H, D).double(), xk[i].double(),
                        xv[i, :, :, :t].transpose(1, 2).double().contiguous(), D ** -0.5))
    return {"self": a, "cross": x, "k": kc.double(), "v": vc.double()}


def _exact_encoder(c, seed):
    T, H, D = c["t"], c["heads"], c["hd"]
    x = _normal(_gen(seed), T * 3 * H * D).view(T, 3, H, D).double()
    return {"ctx": _attend(x[:, 0], x[:, 1].transpose(0, 1), x[:, 2].transpose(0, 1), D ** -0.5).view(-1)}


def _exact_step(c, seed):
    q, k, v, kc, vc = _step_inputs(c, seed)
    L, R, H, KV, D, tk = c["layers"], c["rows"], c["heads"], c["kv"], c["hd"], c["tk"]
    pos = torch.full((R,), tk - 1, device="cuda")
    ctx, rot = [], []
    for i in range(L):
        qr, kr = _rotated(q[i], c, pos), _rotated(k[i], c, pos)
        kc[i, :, :, tk - 1] = kr.view(R, KV, D).float().half()
        vc[i, :, :, :, tk - 1] = v[i].view(R, KV, D).half()
        rot.append(qr)
        ctx.append(torch.stack([_steps(qr[r].view(H, D), kc[i, r, :, :tk].double(),
                                       vc[i, r, :, :, :tk].transpose(1, 2).double().contiguous(), D ** -0.5)
                                for r in range(R)]))
    out = {"ctx": torch.stack(ctx), "q": torch.stack(rot)}
    if c["twin"]:
        out["codes"] = [None] * min(L, 30)
        out["scales"] = [(x.view(-1, 32).abs().amax(-1) / 127) for x in ctx[:30]]
    if c["tiled"]:
        out["cache"] = None
    else:
        out["k"], out["v"] = kc.double(), vc.double()
    return out


def _exact_turn(c, seed):
    q, k, v, kc, vc = _turn_inputs(c, seed)
    L, N, P, H, KV, D = c["layers"], c["n"], c["past"], c["heads"], c["kv"], c["hd"]
    pos = torch.arange(P, P + N, device="cuda")
    ctx, qs, ks = [], [], []
    for i in range(L):
        qr, kr = _rotated(q[i], c, pos), _rotated(k[i], c, pos)
        kc[i, :, P:P + N] = kr.view(N, KV, D).transpose(0, 1).float().half()
        vc[i, :, :, P:P + N] = v[i].view(N, KV, D).permute(1, 2, 0).half()
        K, V = kc[i, :, : P + N].double(), vc[i, :, :, : P + N].transpose(1, 2).double()
        ctx.append(_attend(qr.view(N, H, D), K, V, D ** -0.5, P).view(-1))
        qs.append(qr)
        ks.append(kr)
    return {"ctx": ctx, "q": torch.stack(qs), "krot": torch.stack(ks),
            "k": [None] * L if c["tiled"] else kc.double(), "v": None if c["tiled"] else vc.double()}


def _exact_q8(c, seed):
    q, k, v = _q8_token(c, seed)
    L, S, H, KV, D = c["layers"], c["nseq"], c["heads"], c["kv"], c["hd"]
    lens = _lengths(c)
    pos = torch.tensor([n - 1 for n in lens], device="cuda")
    ctx, qs = [], []
    for i in range(L):
        qr, kr = q[i].double(), k[i].double()
        if c["store"]:
            qr, kr = _rotated(q[i], c, pos), _rotated(k[i], c, pos)
        rows = []
        for s in range(S):
            K, V = _q8_rows(c, seed, i, s, lens[s])
            K, V = _quantised(K), _quantised(V)
            if c["store"]:
                K[-1], V[-1] = _quantised(kr[s: s + 1])[0], _quantised(v[i, s: s + 1])[0]
            K, V = (x.view(-1, KV, D).transpose(0, 1).contiguous() for x in (K, V))
            rows.append(_steps(qr[s].view(H, D), K, V, D ** -0.5))
        ctx.append(torch.cat(rows))
        qs.append(qr)
    return {"ctx": torch.stack(ctx), "q": torch.stack(qs), "cache": [None] * L if c["store"] else None}


def _exact_q8_fill(c, seed):
    k, _ = _q8_rows(c, seed, 0, 0, c["n"])
    return {"k": _rotated(k, c, torch.arange(c["past"], c["past"] + c["n"], device="cuda")).view(-1), "cache": None}


_EXACT = {"short_prompt": _exact_short, "whisper_step": _exact_whisper, "encoder": _exact_encoder,
          "step": _exact_step, "turn": _exact_turn, "q8_step": _exact_q8, "q8_fill": _exact_q8_fill}
