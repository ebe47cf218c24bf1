"""The work whose speed this framework is judged by, as a program that uses it has it done.

Each case is one call (or one captured layer loop) of a public entry point on synthetic tensors of
the sizes the framework serves: Qwen3-shaped heads (16 or 32 query heads over 8 KV heads, head
dimension 128), K and V from N(0, 1) with four outlier channels scaled by 8, queries from N(0, 1).

Kinds, by ``case["kind"]``:

* ``decode``  -- ``int4.SparseDecodeStep`` on an ``Int4KCache``: int4 scoring, block top-k and
  sparse attention, ``layers`` layers with their own caches captured in one HIP graph, as a serving
  loop captures the layers of a model.
* ``mode``    -- a decode step for a mode string (``SparseDecodeStep.for_mode``): the new token is
  quantized into the cache (``int4_pack_k``, ``build_slab`` over one token), the history is
  selected from and the protected tokens are attended as well.
* ``build``   -- the int4 structures of a prefilled cache: pack, channel choice, slab.
* ``prefill`` -- ``prefill.select_blocks``: a query chunk against all cached keys.
* ``reuse``, ``attn``, ``blocks`` -- one layer step of the exact fp32 modes with candidate reuse
  (``ReuseDecodeStep``), candidate attention (``QabsCandidateAttentionStep``) and block bounds
  (``BlockSelectDecodeStep``), captured like ``decode``.
* ``dropin``  -- the reference-signature functions of ``qabs_cuda_kernels`` on head-expanded K/V,
  called one after the other as a program written for that module calls them.
"""

from __future__ import annotations

import math

import torch

from kv_cache_amd import blocksel, int4, modes, prefill, qabs_cuda_kernels, reuse

DEV = "cuda"
D = 128
SCALING = D ** -0.5
TOP_FRACTION = 0.02      # the reuse and block modes keep this share of the history
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # One sequence of a small model at a short context: the smallest decode step, latency only.
        dict(name="decode_b1_t4096", kind="decode", batch=1, q_heads=16, kv_heads=8, tokens=4096, group=32,
             selected=32, block=1, topk=256, layers=4, dtype="bf16"),
        # A small model serving eight sequences, block selection: the ordinary decode step.
        dict(name="decode_b8_t32768", kind="decode", batch=8, q_heads=16, kv_heads=8, tokens=32768, group=32,
             selected=32, block=16, topk=128, layers=2, dtype="bf16"),
        # A larger model at full batch and context: the largest decode step, bound by memory.
        dict(name="decode_b32_t32768", kind="decode", batch=32, q_heads=32, kv_heads=8, tokens=32768, group=128,
             selected=64, block=16, topk=256, layers=1, dtype="bf16"),
        # One long document, single tokens selected from 131072.
        dict(name="decode_b1_t131072", kind="decode", batch=1, q_heads=32, kv_heads=8, tokens=131072, group=128,
             selected=64, block=1, topk=1024, layers=2, dtype="bf16"),
        # A token-selecting mode string at an odd length in fp16, the new token appended, with sink,
        # recent and current tokens kept: what an integration runs for each layer and token.
        dict(name="mode_b4_t20011", kind="mode", mode="qabs32cand5attn", batch=4, q_heads=32, kv_heads=8,
             tokens=20011, group=32, sink=4, recent=64, layers=2, dtype="fp16"),
        # The int4 structures of two freshly prefilled sequences.
        dict(name="build_b2_t32768", kind="build", batch=2, kv_heads=8, tokens=32768, group=128, selected=64,
             dtype="bf16"),
        # The last chunk of a long prefill.
        dict(name="prefill_2048x65536", kind="prefill", batch=1, q_heads=32, kv_heads=8, queries=2048, tokens=65536,
             topk=64, dtype="bf16"),
        # A ragged chunk in the middle of two shorter prefills, two query heads per KV head, fp16.
        dict(name="prefill_509x12345", kind="prefill", batch=2, q_heads=16, kv_heads=8, queries=509, tokens=12345,
             topk=32, dtype="fp16"),
        # The exact candidate-reuse step of one sequence.
        dict(name="reuse_b1_t32768", kind="reuse", mode="qabs8cand5reuse", batch=1, q_heads=32, kv_heads=8,
             tokens=32768, sink=4, recent=16, layers=4, dtype="bf16"),
        # Exact candidate attention for a small batch at an odd length.
        dict(name="attn_b4_t16411", kind="attn", mode="qabs8cand3attn", batch=4, q_heads=32, kv_heads=8,
             tokens=16411, sink=4, recent=16, layers=2, dtype="bf16"),
        # The block-bound selector of one sequence.
        dict(name="blocks_b1_t32768", kind="blocks", mode="qbb64q8s3cand3", batch=1, q_heads=32, kv_heads=8,
             tokens=32768, sink=4, recent=16, layers=4, dtype="bf16"),
        # The reference-signature functions on head-expanded K/V.
        dict(name="dropin_b1_t8191", kind="dropin", batch=1, heads=32, tokens=8191, dims=16, cand=0.1, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges; its bytes stay at or below the largest listed decode step's."""
    kind = rng.choice(["decode", "decode", "decode", "mode", "build", "prefill", "reuse", "attn", "blocks", "dropin"])
    q_heads = rng.choice([16, 32])
    half = rng.choice(["bf16", "bf16", "fp16"])
    if kind in ("decode", "mode"):
        tokens = _log(rng, 1024, 131072)
        if rng.random() < 0.25:
            tokens = max(1024, tokens // 4096 * 4096)
        batch = _log(rng, 1, max(1, min(32, (1 << 20) // tokens)))
        layers = 2 if batch * tokens <= 1 << 17 else 1
        group = rng.choice([32, 64, 128])
        if kind == "mode":
            mode = "qabs%dcand%dattn" % (rng.choice([16, 32, 64]), rng.choice([3, 5, 10]))
            return dict(kind=kind, mode=mode, batch=batch, q_heads=q_heads, kv_heads=8, tokens=tokens, group=group,
                        sink=rng.choice([0, 4]), recent=rng.choice([0, 16, 64]), layers=layers, dtype=half)
        block = rng.choice([1, 16, 16, 32])
        keep = max(16, min(8192, int(tokens * math.exp(rng.uniform(math.log(1 / 128), math.log(1 / 8))))))
        return dict(kind=kind, batch=batch, q_heads=q_heads, kv_heads=8, tokens=tokens, group=group,
                    selected=rng.choice([16, 32, 64]), block=block, topk=max(1, keep // block), layers=layers,
                    dtype=half)
    if kind == "build":
        tokens = _log(rng, 512, 131072)
        return dict(kind=kind, batch=_log(rng, 1, max(1, min(16, (1 << 18) // tokens))), kv_heads=8, tokens=tokens,
                    group=rng.choice([32, 64, 128]), selected=rng.choice([16, 32, 64]), dtype=half)
    if kind == "prefill":
        tokens = _log(rng, 2048, 65536)
        queries = min(_log(rng, 64, 2048), tokens)
        return dict(kind=kind, batch=1, q_heads=q_heads, kv_heads=8, queries=queries, tokens=tokens,
                    topk=rng.choice([16, 32, 64]), dtype=half)
    if kind == "dropin":
        return dict(kind=kind, batch=_log(rng, 1, 2), heads=q_heads, tokens=_log(rng, 1000, 16384),
                    dims=rng.choice([8, 16, 32]), cand=rng.choice([0.05, 0.1]),
                    dtype=rng.choice(["bf16", "fp16", "fp32"]))
    tokens = _log(rng, 2048, 36000)
    batch = _log(rng, 1, max(1, min(8, (1 << 17) // tokens)))
    mode = {"reuse": rng.choice(["qabs8cand5reuse", "qabs16cand10reusefinal", "qabs8cand5reuse2set"]),
            "attn": rng.choice(["qabs8cand3attn", "qabs16cand10attn"]),
            "blocks": rng.choice(["qbb64q8s3cand3", "qbb16q8s12cand4"])}[kind]
    return dict(kind=kind, mode=mode, batch=batch, q_heads=q_heads, kv_heads=8, tokens=tokens, sink=4,
                recent=rng.choice([0, 16]), layers=2, dtype=half)


# -- inputs ---------------------------------------------------------------------


def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 64 + salt)


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32)


def _outliers(gen, x):
    """Four channels of x scaled by 8, the same for every head and token."""
    x[..., torch.randperm(D, generator=gen, device=DEV)[:4]] *= 8.0
    return x


def _kv(gen, batch, heads, tokens, dtype):
    return tuple(_outliers(gen, _randn(gen, batch, heads, tokens, D)).to(dtype) for _ in range(2))


def _layer(case, seed, layer, queries=1):
    """q [B, Hq, D] for each of ``queries`` consecutive tokens, K and V of one layer."""
    gen = _gen(seed, layer)
    dtype = DTYPES[case["dtype"]]
    k, v = _kv(gen, case["batch"], case["kv_heads"], case["tokens"], dtype)
    qs = [_randn(gen, case["batch"], case["q_heads"], D)]
    for _ in range(queries - 1):   # consecutive tokens' queries resemble each other
        qs.append(0.9 * qs[-1] + math.sqrt(1 - 0.81) * _randn(gen, case["batch"], case["q_heads"], D))
    return [q.to(dtype) for q in qs], k, v


def _captured(run):
    """``run`` warmed up and captured in a graph; returns the replay."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    return graph


def _prepare_decode(case, seed):
    layers = []
    for l in range(case["layers"]):
        (q,), k, v = _layer(case, seed, l)
        cache = int4.Int4KCache.from_prefill(k, case["group"], case["selected"])
        step = int4.SparseDecodeStep(case["batch"], case["q_heads"], case["kv_heads"], D, case["tokens"],
                                     case["block"], case["topk"], DEV, dtype=q.dtype)
        layers.append((step, q, cache, k, v))

    def run():
        for step, q, cache, k, v in layers:
            step(q, cache, k, v, SCALING)

    return {"layers": layers, "graph": _captured(run), "out": [(s[0].out, s[0].sel) for s in layers]}


def _prepare_mode(case, seed):
    layers = []
    t = case["tokens"]
    plan = modes.decode_plan(case["mode"], t, D)
    for l in range(case["layers"]):
        (q,), k, v = _layer(case, seed, l)
        cap = int4.round_capacity(t)
        packed, scales = int4.int4_pack_k(k, case["group"], capacity=cap, t_end=t - 1)
        chan, _ = int4.select_channels(packed, scales, t - 1, case["group"], plan.selected)
        slab, slab_scales = int4.build_slab(k, chan, capacity=cap, t_end=t - 1)
        cache = int4.Int4KCache(packed, scales, chan, slab, slab_scales, t, case["group"])
        step = int4.SparseDecodeStep.for_mode(case["mode"], case["batch"], case["q_heads"], case["kv_heads"], D, t,
                                              DEV, protect_sink=case["sink"], protect_recent=case["recent"],
                                              dtype=q.dtype)
        layers.append((step, q, cache, k, v))

    def run():
        for step, q, c, k, v in layers:
            int4.int4_pack_k(k, case["group"], packed=c.packed, scales=c.scales, t_begin=t - 1, t_end=t)
            int4.build_slab(k, c.chan_idx, slab=c.slab, slab_scales=c.slab_scales, t_begin=t - 1, t_end=t)
            step(q, c, k, v, SCALING)

    return {"layers": layers, "graph": _captured(run),
            "out": [(s.out, s.sel, c.packed[:, :, t - 1], c.scales[:, :, t - 1], c.slab_scales[:, :, t - 1])
                    for s, _, c, _, _ in layers]}


def _prepare_build(case, seed):
    k = _outliers(g := _gen(seed, 0), _randn(g, case["batch"], case["kv_heads"], case["tokens"], D))
    k = k.to(DTYPES[case["dtype"]])
    b, h, t, cap = case["batch"], case["kv_heads"], case["tokens"], int4.round_capacity(case["tokens"])
    # the cache's buffers, zero past the last token
    return {"case": case, "k": k,
            "packed": torch.zeros((b, h, cap, D // 2), dtype=torch.uint8, device=DEV),
            "scales": torch.zeros((b, h, cap, D // case["group"]), dtype=torch.float16, device=DEV),
            "slab": torch.zeros((b, h, cap, case["selected"] // 2), dtype=torch.uint8, device=DEV),
            "slab_scales": torch.zeros((b, h, cap), dtype=torch.float16, device=DEV)}


def _run_build(s):
    case = s["case"]
    int4.int4_pack_k(s["k"], case["group"], packed=s["packed"], scales=s["scales"])
    chan, stats = int4.select_channels(s["packed"], s["scales"], case["tokens"], case["group"], case["selected"])
    int4.build_slab(s["k"], chan, slab=s["slab"], slab_scales=s["slab_scales"])
    return s["packed"], s["scales"], chan, stats, s["slab"], s["slab_scales"]


def _prefill_inputs(case, seed):
    gen = _gen(seed, 0)
    dtype = DTYPES[case["dtype"]]
    k = _outliers(gen, _randn(gen, case["batch"], case["kv_heads"], case["tokens"], D)).to(dtype)
    q = _outliers(gen, _randn(gen, case["batch"], case["q_heads"], case["queries"], D)).to(dtype)
    return q, k


def _prepare_prefill(case, seed):
    q, k = _prefill_inputs(case, seed)
    packed, scales = int4.int4_pack_k(k, D)
    return {"case": case, "q": q, "packed": packed, "scales": scales}


def _run_prefill(s):
    case = s["case"]
    return prefill.select_blocks(s["q"], s["packed"], s["scales"], case["tokens"],
                                 case["tokens"] - case["queries"], case["topk"])


def _prepare_reuse(case, seed):
    layers = []
    t = case["tokens"]
    for l in range(case["layers"]):
        (q0, q1), k, v = _layer(case, seed, l, queries=2)
        step = reuse.ReuseDecodeStep(case["mode"], case["batch"], case["q_heads"], case["kv_heads"], D, t,
                                     top_fraction=TOP_FRACTION, protect_sink=case["sink"],
                                     protect_recent=case["recent"], device=DEV, dtype=q0.dtype)
        step.prefill(k)
        step(q0, k[:, :, : t - 1], v[:, :, : t - 1], SCALING)   # the token before
        previous, final = step.cand[1 - step.flip].clone(), step.fin.clone()
        layers.append((step, q1, k, v, step.cand[step.flip], previous if step.use_prev_candidate else None,
                       final if step.use_prev_final else None))

    def run():
        for step, q, k, v, current, previous, final in layers:
            step.launch(q, k, v, SCALING, current, previous, final)

    return {"layers": layers, "graph": _captured(run), "out": [(x[0].out, x[4], x[0].fin) for x in layers]}


def _prepare_attn(case, seed):
    layers = []
    for l in range(case["layers"]):
        (q,), k, v = _layer(case, seed, l)
        step = reuse.QabsCandidateAttentionStep(case["mode"], case["batch"], case["q_heads"], case["kv_heads"], D,
                                                case["tokens"], protect_sink=case["sink"],
                                                protect_recent=case["recent"], device=DEV, dtype=q.dtype)
        step.prefill(k)
        layers.append((step, q, k, v))

    def run():
        for step, q, k, v in layers:
            step.launch(q, k, v, SCALING)

    return {"layers": layers, "graph": _captured(run), "out": [(x[0].out, x[0].hf) for x in layers]}


def _prepare_blocks(case, seed):
    layers = []
    for l in range(case["layers"]):
        (q,), k, v = _layer(case, seed, l)
        step = blocksel.BlockSelectDecodeStep(case["mode"], case["batch"], case["q_heads"], case["kv_heads"], D,
                                              case["tokens"], top_fraction=TOP_FRACTION, protect_sink=case["sink"],
                                              protect_recent=case["recent"], device=DEV, dtype=q.dtype)
        step(q, k, v, SCALING)   # brings the block bounds and the dim-major copy up to the history
        layers.append((step, q, k, v))

    def run():
        for step, q, k, v in layers:
            step.launch(q, k, v, SCALING)

    return {"layers": layers, "graph": _captured(run), "out": [(x[0].out, x[0].keep) for x in layers]}


def _dropin_inputs(case, seed):
    gen = _gen(seed, 0)
    dtype = DTYPES[case["dtype"]]
    b, h, t = case["batch"], case["heads"], case["tokens"]
    k, v = _kv(gen, b, h, t, dtype)
    q = _randn(gen, b, h, D).to(dtype)
    dims = q.float().abs().topk(case["dims"], dim=-1).indices
    masks = [torch.rand((b, h, t - 1), generator=gen, device=DEV) < share for share in (case["cand"],) * 2 + (TOP_FRACTION,)]
    return q, k, v, dims, masks


def _prepare_dropin(case, seed):
    q, k, v, dims, masks = _dropin_inputs(case, seed)
    return {"case": case, "q": q, "k": k, "v": v, "dims": dims, "masks": masks,
            "history": k[:, :, :-1], "kdm": k[:, :, :-1].transpose(2, 3).contiguous()}


def _run_dropin(s):
    ref, q, (cur, prev, final) = qabs_cuda_kernels, s["q"], s["masks"]
    partial = ref.partial_scores(q, s["history"], s["case"]["dims"])
    dim_major = ref.partial_scores_dim_major(q, s["kdm"], s["dims"])
    full = ref.candidate_full_scores(q, s["history"], cur, prev, final, 4, 16, SCALING)
    indices, valid, kept = ref.reuse_select(q, s["k"], cur, prev, final, 4, 16, TOP_FRACTION, True, SCALING)
    out = ref.final_attention(q, s["k"], s["v"], indices, valid, SCALING)
    return partial, dim_major, full, indices, valid, kept, out


_PREPARE = {"decode": _prepare_decode, "mode": _prepare_mode, "build": _prepare_build, "prefill": _prepare_prefill,
            "reuse": _prepare_reuse, "attn": _prepare_attn, "blocks": _prepare_blocks, "dropin": _prepare_dropin}
_RUN = {"build": _run_build, "prefill": _run_prefill, "dropin": _run_dropin}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    state["kind"] = case["kind"]
    return state


def run(state):
    eager = _RUN.get(state["kind"])
    if eager is not None:
        return eager(state)
    state["graph"].replay()
    return state["out"]


# -- what a pass cannot do without ------------------------------------------------


def work(case):
    kind, size = case["kind"], 4 if case["dtype"] == "fp32" else 2
    row = D * size
    if kind == "build":
        n = case["batch"] * case["kv_heads"] * case["tokens"]
        return {"bytes": n * (row + D // 2 + 2 * D // case["group"] + case["selected"] // 2 + 2), "flops": 2 * n * D}
    if kind == "prefill":
        t, nq = case["tokens"], case["queries"]
        rows, nb = case["batch"] * case["q_heads"] * nq, -(-t // 64)
        seen = nq * (t - nq) + nq * (nq + 1) // 2
        return {"bytes": rows * (row + 4 * nb + 4 * case["topk"]) + case["batch"] * case["kv_heads"] * t * (D // 2 + 2),
                "flops": 2 * D * case["batch"] * case["q_heads"] * seen}
    if kind == "dropin":
        n = case["batch"] * case["heads"] * case["tokens"]
        union = 1 - (1 - case["cand"]) ** 2 * (1 - TOP_FRACTION)
        kept = TOP_FRACTION
        # partial scores from whole rows (token-major) and from S runs (dim-major), the union's rows
        # scored twice, the kept rows attended; three fp32 results, masks in and out
        return {"bytes": n * (row + case["dims"] * size + union * row + kept * 2 * row + 12 + 4 + 9 * kept),
                "flops": n * (4 * case["dims"] + 4 * D * union + 4 * D * kept)}
    b, hq, hkv, t, layers = (case[x] for x in ("batch", "q_heads", "kv_heads", "tokens", "layers"))
    if kind in ("decode", "mode"):
        if kind == "mode":
            plan = modes.decode_plan(case["mode"], t, D)
            selected, kept, n_sel = plan.selected, plan.topk + case["sink"] + case["recent"] + 1, plan.topk
        else:
            selected, kept, n_sel = case["selected"], case["topk"] * case["block"], case["topk"]
        kept = min(kept, t)
        rows = b * hkv
        return {"bytes": layers * (rows * (t * (selected // 2 + 2) + kept * 2 * row + 4 * n_sel) + 2 * b * hq * row),
                "flops": layers * (rows * 2 * selected * t + b * hq * 4 * D * kept)}
    rows = b * hq
    if kind == "reuse":
        dims, cand = reuse.parse_reuse_mode(case["mode"])[:2]
        reads, scored, kept = t * dims * size, 1.2 * cand * t, TOP_FRACTION * t
    elif kind == "attn":
        dims, cand = reuse.parse_qabs_attn_mode(case["mode"])[:2]
        reads, scored, kept = t * dims * size, 0, cand * t
    else:
        _, block, _, dims, scan, cand = blocksel.parse_block_mode(case["mode"])
        reads, scored, kept = (t / block + scan * t) * dims * size, cand * t, TOP_FRACTION * t
    # each query head's own channels of K, the rows it scores in full, the rows it attends over
    return {"bytes": layers * rows * (reads + (scored + 2 * kept) * row + t / 4),
            "flops": layers * rows * (2 * dims * t + 2 * D * scored + 4 * D * kept)}


def tolerance(case):
    if case["kind"] in ("build", "prefill"):
        return "exact"      # codes, scales, statistics and the products scale * integer are defined bit by bit
    if case["kind"] == "dropin" and case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    # attention outputs rounded to 16 bits after probabilities rounded to 16 bits
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3, "max": 8e-2 if case["dtype"] == "bf16" else 1e-2}


# -- the same results in plain torch, 64 bits ---------------------------------------


def _fp16_scale(amax, steps):
    """fp16(amax / steps), the quotient rounded to fp32 first, +inf saturated."""
    return (amax.double() / steps).float().to(torch.float16).clamp(max=65504.0)


def _codes(x, scale):
    """clamp(rint(fp32(x / scale)), -8, 7), 0 where the scale is 0."""
    s = scale.double()
    r = torch.where(s == 0, torch.zeros_like(s), x.double() / torch.where(s == 0, torch.ones_like(s), s))
    return r.float().round().clamp(-8, 7)


def _pack(k, group):
    """codes [..., D] and fp16 scales [..., D / group] of K rows."""
    x = k.float().unflatten(-1, (D // group, group))
    scale = _fp16_scale(x.abs().amax(-1), 7.0)
    return _codes(x, scale[..., None]).flatten(-2), scale


def _subset(codes, scale, group, selected):
    """Channel ids [..., S] of the largest sum |code| * scale, lower channel first on ties."""
    stat = (codes.abs().double().unflatten(-1, (D // group, group)) * (scale.double() * 2.0 ** 24)[..., None])
    stat = stat.flatten(-2).to(torch.int64).sum(-2)
    order = torch.sort(stat, dim=-1, descending=True, stable=True).indices
    return order[..., :selected].sort(-1).values


def _slab(k, chan):
    x = torch.gather(k.float(), -1, chan[..., None, :].expand(*k.shape[:-1], chan.size(-1)))
    scale = _fp16_scale(x.abs().amax(-1), 7.0)
    return _codes(x, scale[..., None]), scale


def _int8_query(x):
    """(int8 values, as float64) of fp32 rows: rint(x / (amax / 127)), divisions rounded to fp32."""
    qs = (x.abs().amax(-1, keepdim=True).double() / 127.0).float()
    safe = torch.where(qs == 0, torch.ones_like(qs), qs)
    return torch.where(qs == 0, torch.zeros_like(x), (x.double() / safe.double()).float().round().clamp(-127, 127)).double()


def _first_largest(x, k):
    """Mask of the k largest of each row, lower index first on ties."""
    order = torch.sort(x, dim=-1, descending=True, stable=True).indices[..., :k]
    return torch.zeros_like(x, dtype=torch.bool).scatter_(-1, order, True)


def _attend(q, k, v, mask):
    """q [G, D] over the rows of k, v [T, D] that mask [T] (or [G, T]) keeps, in float64."""
    if mask.dim() == 1:
        keep = mask.nonzero()[:, 0]
        k, v, mask = k[keep], v[keep], None
    s = (q.double() @ k.double().T) * SCALING
    if mask is not None:
        s = s.masked_fill(~mask, -math.inf)
    return torch.softmax(s, dim=-1) @ v.double()


def _protect(mask, case, history):
    mask[..., : case["sink"]] = True
    if case["recent"]:
        mask[..., max(0, history - case["recent"]):] = True


def _exact_decode(case, seed):
    outs = []
    g = case["q_heads"] // case["kv_heads"]
    mode = case["kind"] == "mode"
    plan = modes.decode_plan(case["mode"], case["tokens"], D) if mode else None
    selected, block, topk = (plan.selected, plan.block, plan.topk) if mode else (case["selected"], case["block"], case["topk"])
    t = case["tokens"]
    n = t - 1 if mode else t
    for l in range(case["layers"]):
        (q,), k, v = _layer(case, seed, l)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        tail = []
        for b in range(case["batch"]):
            codes, scale = _pack(k[b], case["group"])
            chan = _subset(codes[:, :n], scale[:, :n], case["group"], selected)
            tail.append((scale[:, t - 1],))
            slab, slab_scale = _slab(k[b], chan)
            tail[-1] += (slab_scale[:, t - 1],)
            for h in range(case["kv_heads"]):
                qh = q[b, h * g:(h + 1) * g]
                total = qh[0, chan[h]].float()
                for i in range(1, g):
                    total = total + qh[i, chan[h]].float()
                ints = slab[h, :n].double() @ _int8_query(total)
                key = (slab_scale[h, :n].double() * ints).float()
                nb = -(-n // block)
                best = torch.full((nb * block,), -math.inf, device=DEV)
                best[:n] = key
                keep = _first_largest(best.view(nb, block).amax(-1), min(topk, nb))
                mask = torch.zeros(t, dtype=torch.bool, device=DEV)
                mask[:n] = keep.repeat_interleave(block)[:n]
                if mode:
                    _protect(mask[:n], case, n)
                    mask[n] = True
                out[b, h * g:(h + 1) * g] = _attend(qh, k[b, h], v[b, h], mask)
        outs.append((out, None, None, torch.stack([x[0] for x in tail]).double(),
                     torch.stack([x[1] for x in tail]).double()) if mode else (out, None))
    return outs


def _exact_build(case, seed):
    k = _outliers(g := _gen(seed, 0), _randn(g, case["batch"], case["kv_heads"], case["tokens"], D))
    k = k.to(DTYPES[case["dtype"]])
    codes, scale = _pack(k, case["group"])
    chan = _subset(codes, scale, case["group"], case["selected"])
    _, slab_scale = _slab(k, chan)
    pad = int4.round_capacity(case["tokens"]) - case["tokens"]
    return (None, torch.nn.functional.pad(scale.double(), (0, 0, 0, pad)), None, None, None,
            torch.nn.functional.pad(slab_scale.double(), (0, pad)))


def _exact_prefill(case, seed):
    q, k = _prefill_inputs(case, seed)
    t, nq = case["tokens"], case["queries"]
    g, nb = case["q_heads"] // case["kv_heads"], -(-t // 64)
    out = torch.empty((case["batch"], case["q_heads"], nq, nb), dtype=torch.float64, device=DEV)
    pos = torch.arange(t, device=DEV)
    for b in range(case["batch"]):
        for h in range(case["kv_heads"]):
            codes, scale = _pack(k[b, h], D)
            codes, scale = codes.double().T.contiguous(), scale[:, 0].double()
            for i in range(h * g, (h + 1) * g):
                for r in range(0, nq, 256):
                    rows = _int8_query(q[b, i, r:r + 256].float())
                    key = (rows @ codes) * scale
                    last = t - nq + r + torch.arange(rows.size(0), device=DEV)
                    key.masked_fill_(pos[None, :] > last[:, None], -math.inf)
                    key = torch.nn.functional.pad(key, (0, nb * 64 - t), value=-math.inf)
                    out[b, i, r:r + 256] = key.view(-1, nb, 64).amax(-1)
    return None, out


def _ordered_dot(q, k, dims):
    """sum_s q[dims_s] * k[:, dims_s] in fp32, product and sum rounded one by one in this order (the
    scores that selections rank are defined so); q [D], k [T, D]."""
    q, k = q.float(), k.float()
    total = torch.zeros(k.size(0), device=k.device)
    for d in dims:
        total = total + q[d] * k[:, d]
    return total


def _top_dims(q, count):
    return torch.sort(q.float().abs(), descending=True, stable=True).indices[:count].tolist()


def _reuse_row(case, q, k, history, previous, final):
    """One query head's candidate and final masks over k[:history]."""
    dims, cand, use_prev, use_final, _ = reuse.parse_reuse_mode(case["mode"])
    partial = _ordered_dot(q, k[:history], _top_dims(q, dims))
    count = min(history, max(1, math.ceil(cand * history)))
    current = partial >= partial.topk(count).values[-1]
    union = current.clone()
    for m in ([previous] if use_prev else []) + ([final] if use_final else []):
        if m is not None:
            union[: m.numel()] |= m
    score = _ordered_dot(q, k[:history], range(D)) * torch.tensor(SCALING, dtype=torch.float32)
    score = score.masked_fill(~union, -math.inf)
    keep = _first_largest(score, min(history, max(1, math.ceil(TOP_FRACTION * history)))) & union
    _protect(keep, case, history)
    return current, keep


def _exact_rows(case, seed, queries, select):
    """Attention of each query head over the history mask ``select`` gives and its own token."""
    g = case["q_heads"] // case["kv_heads"]
    outs = []
    for l in range(case["layers"]):
        qs, k, v = _layer(case, seed, l, queries=queries)
        out = torch.empty(qs[-1].shape, dtype=torch.float64, device=DEV)
        for b in range(case["batch"]):
            for h in range(case["q_heads"]):
                kh, vh = k[b, h // g], v[b, h // g]
                mask = torch.cat([select([q[b, h] for q in qs], kh), torch.ones(1, dtype=torch.bool, device=DEV)])
                out[b, h] = _attend(qs[-1][b, h][None], kh, vh, mask)[0]
        outs.append(out)
    return outs


def _exact_reuse(case, seed):
    history = case["tokens"] - 1

    def select(qs, k):
        previous, final = _reuse_row(case, qs[0], k, history - 1, None, None)
        return _reuse_row(case, qs[1], k, history, previous, final)[1]

    return [(o, None, None) for o in _exact_rows(case, seed, 2, select)]


def _exact_attn(case, seed):
    history = case["tokens"] - 1
    dims, cand = reuse.parse_qabs_attn_mode(case["mode"])[:2]

    def select(qs, k):
        partial = _ordered_dot(qs[0], k[:history], _top_dims(qs[0], dims))
        keep = _first_largest(partial, min(history, max(1, math.ceil(cand * history))))
        _protect(keep, case, history)
        return keep

    return [(o, None) for o in _exact_rows(case, seed, 1, select)]


def _exact_blocks(case, seed):
    history = case["tokens"] - 1
    _, block, _, dims, scan, cand = blocksel.parse_block_mode(case["mode"])
    nb = -(-history // block)
    n_scan = min(nb, max(1, math.ceil(scan * history / block)))

    def select(qs, k):
        q, x = qs[0], k[:history]
        order = _top_dims(q, dims)
        pad = nb * block - history
        low = torch.nn.functional.pad(x.float(), (0, 0, 0, pad), value=math.inf).view(nb, block, D).amin(1)
        high = torch.nn.functional.pad(x.float(), (0, 0, 0, pad), value=-math.inf).view(nb, block, D).amax(1)
        bound = _ordered_dot(q, torch.where(q.float() >= 0, high, low), order)
        scanned = _first_largest(bound, n_scan).repeat_interleave(block)[:history]
        partial = _ordered_dot(q, x, order).masked_fill(~scanned, -math.inf)
        n_cand = min(n_scan * block, max(1, math.ceil(cand * history)))
        chosen = _first_largest(partial, min(n_cand, history)) & scanned
        score = _ordered_dot(q, x, range(D)) * torch.tensor(SCALING, dtype=torch.float32)
        n_keep = min(n_cand, max(1, math.ceil(TOP_FRACTION * history)))
        keep = _first_largest(score.masked_fill(~chosen, -math.inf), n_keep) & chosen
        _protect(keep, case, history)
        return keep

    return [(o, None) for o in _exact_rows(case, seed, 1, select)]


def _exact_dropin(case, seed):
    q, k, v, dims, masks = _dropin_inputs(case, seed)
    history = case["tokens"] - 1
    partial = torch.empty((case["batch"], case["heads"], history), dtype=torch.float64, device=DEV)
    dim_major, full = torch.empty_like(partial), torch.empty_like(partial)
    out = torch.empty((case["batch"], 1, case["heads"], D), dtype=torch.float64, device=DEV)
    protect = dict(sink=4, recent=16)
    for b in range(case["batch"]):
        for h in range(case["heads"]):
            qh, kh = q[b, h].double(), k[b, h].double()
            top = torch.tensor(_top_dims(q[b, h], case["dims"]), device=DEV)
            partial[b, h] = kh[:history, top] @ qh[top]
            dim_major[b, h] = kh[:history, dims[b, h]] @ qh[dims[b, h]]
            union = masks[0][b, h] | masks[1][b, h] | masks[2][b, h]   # what is ranked
            scored = union.clone()                                      # what candidate_full_scores fills
            _protect(scored, protect, history)
            full[b, h] = ((kh[:history] @ qh) * SCALING).masked_fill(~scored, -math.inf)
            score = _ordered_dot(q[b, h], k[b, h, :history], range(D)) * torch.tensor(SCALING, dtype=torch.float32)
            score = score.masked_fill(~union, -math.inf)
            keep = _first_largest(score, max(1, math.ceil(TOP_FRACTION * history))) & union
            _protect(keep, protect, history)
            mask = torch.cat([keep, torch.ones(1, dtype=torch.bool, device=DEV)])
            out[b, 0, h] = _attend(q[b, h][None], k[b, h], v[b, h], mask)[0]
    return partial, dim_major, full, None, None, None, out


_EXACT = {"decode": _exact_decode, "mode": _exact_decode, "build": _exact_build, "prefill": _exact_prefill,
          "reuse": _exact_reuse, "attn": _exact_attn, "blocks": _exact_blocks, "dropin": _exact_dropin}


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)
