"""The calls this framework spends a user's time in, as cases that can be timed.

A case is a dict of plain values.  Six kinds of call, each through the
package's own entry points:

  decode     one layer's decode step on a filled cold store:
             ColdKVStore.retrieve_attend, with the step's new hot row written
             by the call (as the attention wrapper calls it);
  retrieve   ColdKVStore.retrieve_top_kv alone: the selected K and V rows
             (callers that attend by themselves; fp32 models);
  query      a query of many positions over [retrieved ; hot]: retrieve_top_kv
             with that query, then attention.prefill_attention (a follow-up
             prompt on a filled cache);
  prefill    attention.prefill_attention of one prefill chunk;
  evict      rows leaving the hot window in bulk (what a prefill chunk or the
             end of a prefill does), then the pages' summaries and rows read
             back (what saving a cache reads);
  model      a small random-init decoder through KIVMiddleware: chunked
             prefill, then decode steps with retrieval; returns logits.

Shapes are those of kiv_amd/synthetic.py and bench.py, the tests, or generic.
Cold keys are either clustered by segment (kiv_amd/synthetic.py's generator)
or plain normal draws, which no page bound can prune.
"""

from __future__ import annotations

import math

import torch

from kiv_amd import ColdKVStore, KIVConfig, KIVMiddleware, ModelTopology
from kiv_amd.attention import prefill_attention

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SEGMENT = 1024  # tokens that share a centroid in clustered keys
MASK_KINDS = ("bool", "float", "causal")


def listed() -> list[dict]:
    return [
        # A first follow-up on a short chat: every default of KIVConfig (host
        # tier, no pruning), a cold tier of a few pages and a ragged rest.
        # The call is all launches and latency.
        dict(name="decode_short_default", kind="decode", batch=1, hq=32, hkv=4, dim=64, dtype="fp16", cold=1000,
             hot=300, top_pages=32, top_p=256, page=128, tier="host", prune=False, clustered=True, mask=False),
        # The default options on a long document: the host link carries the
        # K of every union page.
        dict(name="decode_host_default", kind="decode", batch=1, hq=28, hkv=4, dim=128, dtype="bf16", cold=70003,
             hot=2048, top_pages=32, top_p=256, page=128, tier="host", prune=False, clustered=True, mask=False),
        # The repository's headline: a million cold tokens in host memory,
        # exact page pruning.
        dict(name="decode_host_pruned_1m", kind="decode", batch=1, hq=28, hkv=4, dim=128, dtype="bf16", cold=1048576,
             hot=2048, top_pages=32, top_p=256, page=128, tier="host", prune=True, clustered=True, mask=False),
        # The same context held in HBM.
        dict(name="decode_hbm_1m", kind="decode", batch=1, hq=28, hkv=4, dim=128, dtype="bf16", cold=1048576,
             hot=2048, top_pages=32, top_p=256, page=128, tier="hbm", prune=False, clustered=True, mask=False),
        # K in HBM, V in host memory; keys that do not cluster, so the union
        # is wide (the layer of the whole-model run).
        dict(name="decode_split_wide_union", kind="decode", batch=1, hq=12, hkv=2, dim=128, dtype="bf16",
             cold=1046531, hot=2048, top_pages=32, top_p=256, page=128, tier="split", prune=False, clustered=False,
             mask=False),
        # Two sequences of different length served together (a padding mask),
        # multi-head attention, wide selections, a cold length off the page.
        dict(name="decode_batch2_mha_mask", kind="decode", batch=2, hq=32, hkv=32, dim=96, dtype="fp16", cold=32847,
             hot=1531, top_pages=64, top_p=512, page=128, tier="hbm", prune=False, clustered=True, mask=True),
        # fp32 rows returned to a caller that attends by itself.
        dict(name="retrieve_fp32", kind="retrieve", batch=1, hq=16, hkv=4, dim=128, dtype="fp32", cold=100100,
             hot=0, top_pages=32, top_p=256, page=128, tier="hbm", prune=False, clustered=False, mask=False),
        # A follow-up prompt of a couple of hundred tokens on a 128k context.
        dict(name="query_200_over_131k", kind="query", batch=1, hq=28, hkv=4, dim=128, dtype="bf16", cold=131072 + 57,
             hot=2048, top_pages=32, top_p=256, page=128, tier="hbm", prune=False, clustered=False, qlen=200),
        # One chunk of a long prefill: 4096 positions over the 4096-token cap
        # plus the chunk, under the boolean mask the model builds.
        dict(name="prefill_chunk_4096", kind="prefill", batch=1, hq=12, hkv=2, dim=128, dtype="bf16", qlen=4096,
             keys=8192, mask_kind="bool"),
        # A short batch of prompts, off every tile size.
        dict(name="prefill_batch2_ragged", kind="prefill", batch=2, hq=32, hkv=8, dim=64, dtype="fp16", qlen=777,
             keys=1531, mask_kind="causal"),
        # The eviction after a prefill chunk: 4096 rows in two ragged pieces.
        dict(name="evict_chunk_4096", kind="evict", batch=1, hq=28, hkv=4, dim=128, dtype="bf16", tokens=4096,
             first=1000, page=128, tier="hbm"),
        # A whole call: four layers of a 1.5B-shaped decoder, a 12k-token
        # prompt in 4096-token chunks, then four decode steps.
        dict(name="model_prefill_decode", kind="model", layers=4, hidden=1536, inter=8960, vocab=8192, hq=12, hkv=2,
             dtype="bf16", tokens=12000, chunk=4096, cap=4096, hot=2048, steps=4, top_pages=32, top_p=256,
             tier="hbm"),
    ]


# ------------------------------------------------------------------ drawing
_HEADS = ((32, 4, 64), (28, 4, 128), (12, 2, 128), (32, 32, 96), (8, 1, 256), (14, 2, 64), (16, 4, 128), (32, 8, 128))


def _log(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _cold(rng, batch: int, hkv: int, dim: int, esize: int) -> int:
    """Cold tokens, log-uniform; K and V within 2 GiB."""
    most = min(1 << 20, (1 << 31) // (2 * batch * hkv * dim * esize))
    return _log(rng, 200, most)


def draw(rng) -> dict:
    kind = rng.choice(("decode", "decode", "decode", "decode", "retrieve", "query", "prefill", "prefill", "evict"))
    hq, hkv, dim = rng.choice(_HEADS)
    if kind in ("decode", "retrieve"):
        dtype = rng.choice(("bf16", "bf16", "fp16", "fp32"))
        batch = rng.choice((1, 1, 1, 2, 3))
        page = rng.choice((128, 128, 128, 64, 256))
        cold = _cold(rng, batch, hkv, dim, 4 if dtype == "fp32" else 2)
        top_pages = rng.choice((8, 16, 32, 64))
        top_p = min(_log(rng, 32, 1024), page * min(top_pages, max(1, cold // page)))
        return dict(kind=kind, batch=batch, hq=hq, hkv=hkv, dim=dim, dtype=dtype, cold=cold,
                    hot=_log(rng, 1, 4096) if kind == "decode" else 0, top_pages=top_pages, top_p=top_p, page=page,
                    tier=rng.choice(("host", "hbm", "split")), prune=rng.random() < 0.4,
                    clustered=rng.random() < 0.5, mask=kind == "decode" and rng.random() < 0.3)
    if kind == "query":
        cold = _cold(rng, 1, hkv, dim, 2) // 4 + 200
        top_pages = rng.choice((16, 32))
        return dict(kind=kind, batch=1, hq=hq, hkv=hkv, dim=dim, dtype=rng.choice(("bf16", "fp16")), cold=cold,
                    hot=_log(rng, 256, 4096), top_pages=top_pages,
                    top_p=min(_log(rng, 32, 512), 128 * min(top_pages, max(1, cold // 128))), page=128,
                    tier=rng.choice(("host", "hbm", "split")), prune=rng.random() < 0.4,
                    clustered=rng.random() < 0.5, qlen=_log(rng, 2, 256))
    if kind == "prefill":
        batch = rng.choice((1, 1, 2))
        qlen = _log(rng, 16, 4096 // batch)
        return dict(kind=kind, batch=batch, hq=hq, hkv=hkv, dim=dim, dtype=rng.choice(("bf16", "bf16", "fp16")),
                    qlen=qlen, keys=qlen + _log(rng, 1, 4096), mask_kind=rng.choice(MASK_KINDS))
    tokens = _log(rng, 128, 8192)
    return dict(kind="evict", batch=1, hq=hq, hkv=hkv, dim=dim, dtype=rng.choice(("bf16", "fp16", "fp32")),
                tokens=tokens, first=rng.randrange(1, tokens), page=rng.choice((128, 128, 64, 256)),
                tier=rng.choice(("host", "hbm", "split")))


# ------------------------------------------------------------------- inputs
def _gen(seed: int, salt: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(1_000_003 * seed + salt)


def _randn(gen, *shape) -> torch.Tensor:
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)


def _keys(case, seed: int):
    """(cold K, cold V, hot K, hot V, query) in the case's dtype."""
    B, hq, hkv, D = case["batch"], case["hq"], case["hkv"], case["dim"]
    cold, hot, Q, dt = case["cold"], case["hot"], case.get("qlen", 1), DTYPES[case["dtype"]]
    gen = _gen(seed, 11)
    total = cold + hot
    k = torch.empty(B, hkv, total, D, dtype=dt, device="cuda")
    v = torch.empty_like(k)
    cent = None
    if case["clustered"]:
        cent = _randn(gen, B, hkv, -(-total // SEGMENT), D)
    step = 65536
    for t0 in range(0, total, step):
        n = min(step, total - t0)
        x = _randn(gen, B, hkv, n, D)
        if cent is not None:
            seg = torch.arange(t0, t0 + n, device="cuda") // SEGMENT
            x = cent[:, :, seg] + 0.3 * x
        k[:, :, t0:t0 + n] = x.to(dt)
        v[:, :, t0:t0 + n] = _randn(gen, B, hkv, n, D).to(dt)
    if cent is not None:
        # Every head asks for one old segment of its sequence.
        target = torch.randint(0, max(1, cold // SEGMENT), (B,), generator=gen, device="cuda")
        rows = torch.arange(hq, device="cuda") // (hq // hkv)
        q = cent[torch.arange(B, device="cuda")[:, None], rows[None, :], target[:, None]][:, :, None, :]
        q = q + 0.1 * _randn(gen, B, hq, Q, D)
    else:
        q = _randn(gen, B, hq, Q, D)
    return k[:, :, :cold], v[:, :, :cold], k[:, :, cold:], v[:, :, cold:], q.to(dt)


def _config(case) -> KIVConfig:
    return KIVConfig(hot_budget=max(1, case.get("hot", 1)), top_p=case.get("top_p", 256), page_size=case["page"],
                     top_pages=case.get("top_pages", 32), cold_tier=case["tier"],
                     score_rounding="fp32" if case["dtype"] == "fp32" else "activation",
                     reserve_tokens=case.get("cold", 0), fine_pruning=bool(case.get("prune", False)))


def _store(case, cfg) -> ColdKVStore:
    topo = ModelTopology.manual(global_layer_indices=(0,), num_query_heads=case["hq"], num_kv_heads=case["hkv"],
                                head_dim=case["dim"], num_hidden_layers=1)
    return ColdKVStore(cfg, topo, torch.device("cuda", 0))


def _hot_mask(case, seed: int) -> torch.Tensor | None:
    """Padding mask of a decode batch: the sequences start at different
    columns of the hot window (True: attend)."""
    if not case.get("mask"):
        return None
    B, T = case["batch"], case["hot"]
    start = torch.randint(0, max(1, T // 2), (B, 1), generator=_gen(seed, 13), device="cuda")
    return (torch.arange(T, device="cuda")[None, :] >= start)[:, None, None, :]


def _chunk_mask(kind: str, Q: int, T: int, dt: torch.dtype) -> torch.Tensor | None:
    """The chunk's causal rule as the tensor a model builds ([1, 1, Q, T])."""
    if kind == "causal":
        return None
    vis = torch.arange(T, device="cuda")[None, :] <= torch.arange(Q, device="cuda")[:, None] + (T - Q)
    if kind == "bool":
        return vis[None, None]
    return torch.zeros(1, 1, Q, T, dtype=dt, device="cuda").masked_fill(~vis, float("-inf"))


# ------------------------------------------------------------------ running
def prepare(case, seed: int) -> dict:
    kind = case["kind"]
    if kind in ("decode", "retrieve", "query"):
        ck, cv, hk, hv, q = _keys(case, seed)
        cfg = _config(case)
        store = _store(case, cfg)
        store.evict_from_hot(ck, cv)
        st = dict(case=case, store=store, cfg=cfg, q=q, scaling=case["dim"] ** -0.5)
        if kind == "decode":
            # The step's new row, not yet in the window.
            st.update(hk=hk.contiguous(), hv=hv.contiguous(), mask=_hot_mask(case, seed))
            st.update(new_k=st["hk"][:, :, -1:].clone(), new_v=st["hv"][:, :, -1:].clone())
            st["hk"][:, :, -1:].zero_()
            st["hv"][:, :, -1:].zero_()
        elif kind == "query":
            st.update(hk=hk.contiguous(), hv=hv.contiguous(),
                      mask=_chunk_mask("bool", case["qlen"], case["hot"], q.dtype) if case["qlen"] <= case["hot"]
                      else None)
        return st
    if kind == "prefill":
        B, hq, hkv, D, Q, T = (case[k] for k in ("batch", "hq", "hkv", "dim", "qlen", "keys"))
        dt, gen = DTYPES[case["dtype"]], _gen(seed, 17)
        return dict(case=case, q=_randn(gen, B, hq, Q, D).to(dt), k=_randn(gen, B, hkv, T, D).to(dt),
                    v=_randn(gen, B, hkv, T, D).to(dt), mask=_chunk_mask(case["mask_kind"], Q, T, dt),
                    scaling=D ** -0.5)
    if kind == "evict":
        k, v = _evicted(case, seed)
        cfg = _config(case)
        return dict(case=case, store=_store(case, cfg), k=k, v=v)
    return _prepare_model(case, seed)


def _evicted(case, seed: int):
    gen, dt = _gen(seed, 19), DTYPES[case["dtype"]]
    shape = (case["batch"], case["hkv"], case["tokens"], case["dim"])
    return (_randn(gen, *shape).to(dt), _randn(gen, *shape).to(dt))


def run(st: dict):
    kind = st["case"]["kind"]
    if kind == "decode":
        # The output, and the window's row that the call writes.
        hk, hv = st["hk"], st["hv"]
        row_k, row_v = hk[:, :, -1:], hv[:, :, -1:]
        out = st["store"].retrieve_attend(st["q"], st["scaling"], st["cfg"], hk, hv, st["mask"],
                                          hot_rows=(st["new_k"], st["new_v"], row_k, row_v))
        return out, row_k, row_v
    if kind == "retrieve":
        return st["store"].retrieve_top_kv(st["q"], st["scaling"], st["cfg"])
    if kind == "query":
        k, v = st["store"].retrieve_top_kv(st["q"], st["scaling"], st["cfg"])
        return prefill_attention(st["q"], k, v, st["hk"], st["hv"], st["mask"], st["scaling"])
    if kind == "prefill":
        return prefill_attention(st["q"], None, None, st["k"], st["v"], st["mask"], st["scaling"],
                                 causal=st["mask"] is None)
    if kind == "evict":
        # A new conversation's rows each time: the store is emptied, its
        # memory is kept.
        store, n = st["store"], st["case"]["first"]
        store.reset()
        store.evict_from_hot(st["k"][:, :, :n], st["v"][:, :, :n])
        store.evict_from_hot(st["k"][:, :, n:], st["v"][:, :, n:])
        return (*store.read_summaries(), *store.read_tokens())
    return _run_model(st)


def _prepare_model(case, seed: int) -> dict:
    from transformers import Qwen2Config, Qwen2ForCausalLM

    cfg = Qwen2Config(vocab_size=case["vocab"], hidden_size=case["hidden"], intermediate_size=case["inter"],
                      num_hidden_layers=case["layers"], num_attention_heads=case["hq"],
                      num_key_value_heads=case["hkv"], max_position_embeddings=case["tokens"] + 8192, rope_theta=1e6,
                      tie_word_embeddings=True)
    cfg._attn_implementation = "sdpa"
    torch.manual_seed(seed)
    with torch.device("cuda"):
        model = Qwen2ForCausalLM(cfg)
    model = model.to(DTYPES[case["dtype"]]).eval()
    kcfg = KIVConfig(hot_budget=case["hot"], top_p=case["top_p"], page_size=128, top_pages=case["top_pages"],
                     cold_tier=case["tier"])
    mw = KIVMiddleware(model, kcfg)
    mw.install()
    ids = torch.randint(0, case["vocab"], (1, case["tokens"] + case["steps"]), generator=_gen(seed, 23),
                        device="cuda")
    return dict(case=case, mw=mw, model=model, ids=ids, cache=mw.create_cache())


@torch.no_grad()
def _run_model(st: dict):
    case, ids, cache = st["case"], st["ids"], st["cache"]
    T = case["tokens"]
    cache.reset()
    out = [st["mw"].chunked_prefill(ids[:, :T], cache, chunk_size=case["chunk"], prefill_hot_cap=case["cap"])]
    for i in range(case["steps"]):
        step = st["model"](input_ids=ids[:, T + i:T + i + 1], past_key_values=cache, use_cache=True)
        out.append(step.logits[:, -1, :])
    return out


# ------------------------------------------------------------ what it needs
def _esize(case) -> int:
    return 4 if case["dtype"] == "fp32" else 2


def work(case) -> dict:
    """Bytes read or written once and operations no implementation avoids.

    A retrieval must read every page summary, the K rows of its candidates
    and the selected V; the union is at least one query row's top pages, and
    that smallest union is what is counted (the real one is wider)."""
    kind, b = case["kind"], _esize(case)
    if kind == "model":
        T, d, f, L = case["tokens"] + case["steps"], case["hidden"], case["inter"], case["layers"]
        hd = d // case["hq"]
        weights = L * (2 * d * d + 2 * d * case["hkv"] * hd + 3 * d * f)
        attn = 0
        for s in range(0, case["tokens"], case["chunk"]):
            q = min(case["chunk"], case["tokens"] - s)
            attn += 4 * d * (q * min(s, case["cap"]) + q * (q + 1) // 2) * L
        return {"bytes": 2 * (weights + case["vocab"] * d) * (1 + case["steps"]) + 4 * case["tokens"] * d,
                "flops": 2 * weights * T + attn + 2 * case["vocab"] * d * (1 + case["steps"])}
    B, hq, hkv, D = case["batch"], case["hq"], case["hkv"], case["dim"]
    row = B * hkv * D * b  # one token's K or V, every kv head
    if kind == "prefill":
        Q, T = case["qlen"], case["keys"]
        pairs = Q * (T - Q) + Q * (Q + 1) // 2
        mask = 0 if case["mask_kind"] == "causal" else Q * T * (1 if case["mask_kind"] == "bool" else b)
        return {"bytes": 2 * B * hq * Q * D * b + 2 * T * row + mask, "flops": 4 * B * hq * D * pairs}
    if kind == "evict":
        T, pages = case["tokens"], case["tokens"] // case["page"]
        # in, into the store, out of it again; two summaries per page row
        return {"bytes": 3 * 2 * T * row + 2 * pages * B * hkv * D * (b + 4), "flops": T * B * hkv * D}
    Q, N = case.get("qlen", 1), case["cold"] // case["page"]
    P = min(case["top_p"], case["cold"])
    cand = min(case["top_pages"], N) * case["page"] + case["cold"] % case["page"]
    read = N * row + cand * row + P * row
    flops = 2 * B * hq * Q * D * (N + cand)
    if kind == "retrieve":
        return {"bytes": B * hq * Q * D * b + read + 2 * P * row, "flops": flops}
    T = case["hot"]
    pairs = Q * (P + T) if kind == "decode" or Q > T else Q * (P + T - Q) + Q * (Q + 1) // 2
    return {"bytes": 2 * B * hq * Q * D * b + read + P * row + 2 * T * row, "flops": flops + 4 * B * hq * D * pairs}


# ---------------------------------------------------------- checking values
def tolerance(case) -> dict:
    """About four times the distance between the outputs and exact() below:
    attention in bf16 0.0016 to 0.0024, fp16 0.0002 to 0.0003, fp32 4e-7; the
    fp32 page means 5e-9.  Retrieved rows are copies (a token ranked
    differently shows as a whole row).  The model's logits pass through its
    bf16 layers (0.005 to 0.03 between two attention paths)."""
    kind = case["kind"]
    if kind == "model":
        return {"rel": 5e-2}
    if kind == "evict":
        return {"rel": 1e-5}
    if kind == "retrieve":
        return {"rel": 1e-2}
    return {"rel": {"bf16": 1e-2, "fp16": 1.2e-3, "fp32": 1e-5}[case["dtype"]]}


def _round(x: torch.Tensor, case) -> torch.Tensor:
    """x through the precision that scores are ranked in."""
    return x.to(DTYPES[case["dtype"]]).double()


def _scores(case, q, rows):
    """Ranked scores [hq, Q, n] of one sequence's query rows: the dot product,
    then the scaling, each rounded to the activation dtype."""
    g = case["hq"] // case["hkv"]
    out = []
    for h in range(case["hkv"]):
        dot = q[h * g:(h + 1) * g].reshape(-1, case["dim"]) @ rows[h].T
        if case["dtype"] == "fp32":
            s = dot * case["dim"] ** -0.5
        else:
            s = _round(_round(dot, case) * case["dim"] ** -0.5, case)
        out.append(s.reshape(g, -1, rows.shape[1]))
    return torch.cat(out)


def _summaries(case, k):
    """Page means of one sequence's cold K, rounded to fp32, then to the dtype."""
    N, ps = k.shape[1] // case["page"], case["page"]
    out = torch.empty(k.shape[0], N, k.shape[2], dtype=torch.float64, device=k.device)
    for p0 in range(0, N, 512):
        n = min(512, N - p0)
        pages = k[:, p0 * ps:(p0 + n) * ps].double().view(k.shape[0], n, ps, -1)
        out[:, p0:p0 + n] = pages.mean(2).float().to(DTYPES[case["dtype"]]).double()
    return out


def _select(case, q, k):
    """Ids of the top P cold tokens of one sequence, best first."""
    N, ps, cold = k.shape[1] // case["page"], case["page"], k.shape[1]
    union = torch.empty(0, dtype=torch.long, device=k.device)
    if N:
        s = _scores(case, q, _summaries(case, k)).reshape(-1, N)
        union = torch.sort(s, dim=1, descending=True, stable=True)[1][:, :case["top_pages"]].unique()
    return union, N * ps, cold


def _top(case, q, k, union, first_partial):
    ps, cold = case["page"], k.shape[1]
    ids = torch.cat([(union[:, None] * ps + torch.arange(ps, device=k.device)).reshape(-1),
                     torch.arange(first_partial, cold, device=k.device)])
    best = torch.cat([_scores(case, q, k[:, part].double()).amax((0, 1)) for part in ids.split(16384)])
    order = torch.sort(best, descending=True, stable=True)[1]
    return ids[order[:min(case["top_p"], ids.numel())]]


def _attend(case, q, keys, vals, bias):
    """softmax(q k * scaling + bias) v of one sequence -> [Q, hq, D]."""
    g = case["hq"] // case["hkv"]
    out = torch.empty(q.shape[1], case["hq"], case["dim"], dtype=torch.float64, device=q.device)
    for h in range(case["hq"]):
        kh, vh = keys[h // g], vals[h // g]
        for r in range(0, q.shape[1], 512):
            s = q[h, r:r + 512] @ kh.T * case["dim"] ** -0.5
            if bias is not None:
                s = s + (bias[r:r + 512] if bias.shape[0] > 1 else bias)
            out[r:r + 512, h] = torch.softmax(s, dim=-1) @ vh
    return out


def exact(case, seed: int):
    kind = case["kind"]
    if kind == "model":
        return None  # a chain of 16-bit layers and discrete choices has no 64-bit value of its own
    if kind == "prefill":
        st = prepare(case, seed)
        Q, T = case["qlen"], case["keys"]
        vis = torch.arange(T, device="cuda")[None, :] <= torch.arange(Q, device="cuda")[:, None] + (T - Q)
        bias = torch.zeros(Q, T, dtype=torch.float64, device="cuda").masked_fill(~vis, float("-inf"))
        return torch.stack([_attend(case, st["q"][i].double(), st["k"][i].double(), st["v"][i].double(), bias)
                            for i in range(case["batch"])])
    if kind == "evict":
        k, v = _evicted(case, seed)
        one = torch.stack([_summaries(case, k[i]) for i in range(case["batch"])])  # [B, hkv, N, D]
        N, ps = case["tokens"] // case["page"], case["page"]
        mean = k[:, :, :N * ps].double().view(*k.shape[:2], N, ps, -1).mean(3)
        return one.permute(2, 0, 1, 3).contiguous(), mean.permute(2, 0, 1, 3).contiguous(), k.double(), v.double()
    ck, cv, hk, hv, q = _keys(case, seed)
    # The union is over the whole batch, as are the candidates.
    parts = [_select(case, q[i].double(), ck[i]) for i in range(case["batch"])]
    union = torch.cat([p[0] for p in parts]).unique()
    mask = _hot_mask(case, seed) if kind == "decode" else None
    outs, ks, vs = [], [], []
    for i in range(case["batch"]):
        top = _top(case, q[i].double(), ck[i], union, parts[i][1])
        ks.append(ck[i][:, top].double())
        vs.append(cv[i][:, top].double())
        if kind == "retrieve":
            continue
        Q, T = q.shape[2], case["hot"]
        bias = torch.zeros(Q, top.numel() + T, dtype=torch.float64, device="cuda")
        if kind == "query" and Q <= T:
            hidden = torch.arange(T, device="cuda")[None, :] > torch.arange(Q, device="cuda")[:, None] + (T - Q)
            bias[:, top.numel():].masked_fill_(hidden, float("-inf"))
        if mask is not None:
            bias[:, top.numel():].masked_fill_(~mask[i, 0], float("-inf"))
        outs.append(_attend(case, q[i].double(), torch.cat([ks[-1], hk[i].double()], 1),
                            torch.cat([vs[-1], hv[i].double()], 1), bias))
    if kind == "retrieve":
        return torch.stack(ks), torch.stack(vs)
    if kind == "decode":
        return torch.stack(outs), hk[:, :, -1:].double(), hv[:, :, -1:].double()
    return torch.stack(outs)
