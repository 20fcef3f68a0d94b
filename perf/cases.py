"""The work that this framework is measured on, through its public entry points.

Five kinds of case, each with what it stands for:

  pass      one pass of a decoder model over tokens that follow a filled cache (model_runner.DecoderModel
            .forward): a draft's single-token pass, the verify pass over the last token and k proposals, and
            verify passes of a running batch with contexts of many lengths, in bf16 and with fp8 weights
  prompt    admission of one prompt or of several prompts of different lengths to an engine
            (spec_decode SpecEngine.add_request / add_requests), the draft's prefill included where there is one
  text      a text through a layer-list model (seq_engine.SeqEngine.step): the last token's logits (a prompt) or
            every token's (scoring), in bf16 or float32
  turn      short requests through a layer-list model from their prompts to their last decoded token
  accept    the sampling end of a speculative step at temperature > 0: softmax of the target's and the draft's
            logits, the bonus token's draw and the rejection sampler

Weights, tokens, caches and uniforms are seeded random; sizes are the presets' of config.py and those of the
layer-list models of bench.py."""
import math

import torch

from vllm_omni_draft_amd import config, ops, weights
from vllm_omni_draft_amd.engine import EngineConfig, SpecEngine
from vllm_omni_draft_amd.kv_cache import PAGE, PagedKVCache
from vllm_omni_draft_amd.model_runner import DecoderModel
from vllm_omni_draft_amd.seq_engine import SeqEngine, SeqEngineConfig

DEV = "cuda"
F64 = torch.float64
# Layer-list models: head size, vocabulary, window, pool and rank of bench.py's, and its sizes by width.
HEAD, SEQ_VOCAB, WINDOW, POOL, RANK = 128, 32000, 1024, 16, 64
PUGUZEN = {1024: dict(heads=8, kv=2, ff=4096), 2048: dict(heads=16, kv=4, ff=8192)}
NABURAX = {1024: dict(heads=8, kv=2, q_rank=384, s_heads=16, experts=8, eff=1024),
           2048: dict(heads=16, kv=4, q_rank=768, s_heads=32, experts=16, eff=2048)}
KV_RANK, ROT, STATE, SVDIM, KEEP, TOP = 512, 64, 128, 64, 4, 2
BUCKETS, MUL_PREV, MUL_CUR = 65521, 31, 17
SCALING = {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}
EPS = 1e-5


def listed():
    return [
        # one proposal of the small draft model: the smallest and most frequent call of speculative decoding
        dict(name="draft_token", kind="pass", model="llama-3.2-1b", layers=16, fp8=False, seqs=1, rows=1, ctx_min=1000, ctx_max=1000),
        # the target's verify pass of one user's request, k = 5
        dict(name="verify_one", kind="pass", model="llama-3-8b", layers=32, fp8=False, seqs=1, rows=6, ctx_min=1024, ctx_max=1024),
        # a few users on an 8B target whose weights are held in fp8
        dict(name="verify_few_fp8", kind="pass", model="llama-3-8b", layers=32, fp8=True, seqs=4, rows=4, ctx_min=300, ctx_max=2000),
        # a full serving batch, contexts of many lengths (eight of the model's layers: the cache of 32 sequences)
        dict(name="verify_batch", kind="pass", model="qwen2.5-7b", layers=8, fp8=False, seqs=32, rows=6, ctx_min=64, ctx_max=1024),
        # a request of ordinary length is admitted: target and draft prefill
        dict(name="prompt", kind="prompt", model="llama-3-8b", layers=32, draft="llama-3.2-1b", seqs=1, len_min=1024, len_max=1024),
        # a long document, plain decoding
        dict(name="prompt_long", kind="prompt", model="llama-3-8b", layers=32, draft="", seqs=1, len_min=4096, len_max=4096),
        # several requests of different lengths are admitted together
        dict(name="prompts_ragged", kind="prompt", model="qwen2.5-7b", layers=28, draft="", seqs=8, len_min=64, len_max=1000),
        # a prompt through a recurrent / windowed model
        dict(name="puguzen_prompt", kind="text", family="puguzen", width=2048, dtype="bfloat16", tokens=2048, score=False),
        # a text scored in float32 (logits of every token), as a trace is replayed in it
        dict(name="puguzen_score_f32", kind="text", family="puguzen", width=1024, dtype="float32", tokens=777, score=True),
        # a text scored by a model with latent attention, a state-space recurrence and routed experts
        dict(name="naburax_score", kind="text", family="naburax", width=2048, dtype="bfloat16", tokens=1024, score=True),
        # four short requests of such a model, from admission to the last token
        dict(name="naburax_turn", kind="turn", family="naburax", width=2048, seqs=4, tokens=100, steps=24),
        # the sampling end of a step of eight users at temperature 0.8
        dict(name="accept_sampled", kind="accept", vocab=128256, seqs=8, k=5),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["pass", "pass", "prompt", "prompt", "text", "text", "turn", "accept"])
    if kind == "pass":
        model = rng.choice(["llama-3.2-1b", "qwen2.5-0.5b", "llama-3-8b", "qwen2.5-7b"])
        fp8 = rng.random() < 0.3
        rows = rng.randint(1, 6)
        seqs = _log(rng, 1, 32)
        deep = config.PRESETS[model]["n_layers"]
        hi = _log(rng, 64, 4096 if seqs <= 4 else 1024)
        return dict(kind=kind, model=model, layers=rng.randint(6, deep) if seqs <= 4 else rng.randint(4, 8), fp8=fp8, seqs=seqs, rows=rows,
                    ctx_min=_log(rng, 16, hi), ctx_max=hi)
    if kind == "prompt":
        model = rng.choice(["llama-3.2-1b", "qwen2.5-0.5b", "llama-3-8b", "qwen2.5-7b"])
        seqs = rng.choice([1, 1, 2, 3, 5, 8])
        hi = _log(rng, 24, 4000 if seqs == 1 else 1000 if seqs < 5 else 500)
        draft = {"llama-3-8b": "llama-3.2-1b"}.get(model, "") if rng.random() < 0.5 else ""
        return dict(kind=kind, model=model, layers=rng.randint(8, config.PRESETS[model]["n_layers"]), draft=draft, seqs=seqs,
                    len_min=hi if seqs == 1 else _log(rng, 17, hi), len_max=hi)
    if kind == "text":
        family = rng.choice(["puguzen", "naburax"])
        f32 = rng.random() < 0.3
        return dict(kind=kind, family=family, width=1024 if f32 else rng.choice([1024, 2048]), dtype="float32" if f32 else "bfloat16",
                    tokens=_log(rng, 17, 800 if f32 else 2048), score=rng.random() < 0.5)
    if kind == "turn":
        return dict(kind=kind, family=rng.choice(["puguzen", "naburax"]), width=rng.choice([1024, 2048]), seqs=rng.randint(1, 8),
                    tokens=_log(rng, 5, 300), steps=rng.randint(8, 32))
    return dict(kind=kind, vocab=rng.choice([32000, 50272, 128256, 152064]), seqs=_log(rng, 1, 32), k=rng.randint(1, 7))


# ------------------------------------------------------------------------------------ inputs
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(seed * 1009 + salt)


def _spread(lo, hi, n):
    """n lengths from lo to hi, spread evenly over their logarithm, the longest not last."""
    if n == 1:
        return [hi]
    ls = [int(round(lo * (hi / lo) ** (i / (n - 1)))) for i in range(n)]
    return ls[1::2] + ls[0::2]


def _model_cfg(name, layers, max_pos=8192):
    return config.preset(name, n_layers=layers, max_pos=max_pos)


def _decoder_state(cfg, gen):
    """Tensors under a checkpoint's names, scaled as weights.random_init scales them."""
    H, F, D = cfg.hidden, cfg.ffn, cfg.head_dim

    def rn(*shape, s=0.02, mean=0.0):
        return torch.randn(*shape, generator=gen, device=DEV, dtype=torch.bfloat16).mul_(s).add_(mean)

    st = {"model.embed_tokens.weight": rn(cfg.vocab, H, s=1.0), "model.norm.weight": rn(H, s=0.05, mean=1.0)}
    if not cfg.tie_embeddings:
        st["lm_head.weight"] = rn(cfg.vocab, H)
    for i in range(cfg.n_layers):
        p = f"model.layers.{i}."
        for nm, rows in (("q", cfg.n_heads * D), ("k", cfg.n_kv_heads * D), ("v", cfg.n_kv_heads * D)):
            st[p + f"self_attn.{nm}_proj.weight"] = rn(rows, H)
            if cfg.qkv_bias:
                st[p + f"self_attn.{nm}_proj.bias"] = rn(rows)
        st[p + "self_attn.o_proj.weight"] = rn(H, cfg.n_heads * D)
        st[p + "mlp.gate_proj.weight"], st[p + "mlp.up_proj.weight"] = rn(F, H), rn(F, H)
        st[p + "mlp.down_proj.weight"] = rn(H, F)
        st[p + "input_layernorm.weight"] = rn(H, s=0.05, mean=1.0)
        st[p + "post_attention_layernorm.weight"] = rn(H, s=0.05, mean=1.0)
    return st


def _pass_inputs(case, seed):
    """Contexts, tokens and the cache's keys and values [layers, page, kv head, 16 * dim] of a pass."""
    cfg = _model_cfg(case["model"], case["layers"])
    B, q = case["seqs"], case["rows"]
    ctx = _spread(case["ctx_min"], case["ctx_max"], B)
    g = _gen(seed, 1)
    max_ctx = max(ctx) + q
    toks = torch.randint(0, cfg.vocab, (B, q), generator=g, device=DEV, dtype=torch.int32)
    kv = PagedKVCache(cfg, PagedKVCache.pages_for(cfg, B, max_ctx), B, max_ctx, DEV)
    for b in range(B):
        kv.ensure_capacity(b, ctx[b] + q)
    kv.k.normal_(generator=g)
    kv.v.normal_(generator=g)
    return cfg, ctx, toks, kv, max_ctx


def _prompts(case, seed, vocab):
    ls = _spread(case["len_min"], case["len_max"], case["seqs"])
    t = torch.randint(0, vocab, (sum(ls),), generator=_gen(seed, 2), device=DEV).tolist()
    out = []
    for n in ls:
        out.append(t[:n])
        t = t[n:]
    return out


def _seq_cfg(family, width):
    M, L, S = config.MixerSpec, config.SeqLayerSpec, config.SeqModelConfig
    if family == "puguzen":
        z = PUGUZEN[width]
        H = z["heads"]
        rot = dict(rot_dims=HEAD, rot_base=1e6)
        ret = M("retention", H, HEAD, HEAD, decay=tuple(_decay(i, H) for i in range(H)), **rot)
        att = M("attention", H, HEAD, HEAD, kv_heads=z["kv"], rot_layout="interleaved", scale=HEAD ** -0.5, window=WINDOW, pool=POOL, **rot)
        gla = M("gla", H, HEAD, HEAD, tau=16.0, rank=RANK)
        cfg = S("puguzen", width, SEQ_VOCAB, [L(m, z["ff"]) for m in (ret, att, gla, att)], norm_eps=EPS)
    else:
        z = NABURAX[width]
        H = z["heads"]
        lat = M("latent_attention", H, HEAD, HEAD, q_rank=z["q_rank"], kv_rank=KV_RANK, rot_dim=ROT, rot_dims=ROT, rot_base=1e6,
                rot_layout="interleaved", rot_scaling=dict(SCALING), scale=(HEAD + ROT) ** -0.5, window=WINDOW)
        par = M("parallel", H, HEAD, HEAD, kv_heads=z["kv"], scale=HEAD ** -0.5, window=WINDOW, keep_first=KEEP,
                ssd=config.SsdSpec(heads=z["s_heads"], vdim=SVDIM, state=STATE, groups=1, taps=4, norm_groups=1), left_scale=0.5,
                right_scale=0.5)
        ex = config.ExpertsSpec(z["experts"], TOP, z["eff"])
        cfg = S("naburax", width, SEQ_VOCAB, [L(m, 0, ex) for m in (lat, par, lat, par)], block="postnorm", embed_scale=1.0,
                bigram={"buckets": BUCKETS, "mul_prev": MUL_PREV, "mul_cur": MUL_CUR}, tied_head=False, logit_scale=1.0, norm_eps=EPS)
    cfg.validate()
    return cfg


def _decay(i, heads):
    return 1 - 2.0 ** (-5 - 3 * i / heads)


def _seq_state(family, width, dtype, gen):
    """Tensors under a checkpoint's names, scaled as weights.seq_random_state scales them."""
    W, D = width, HEAD

    def rn(*shape, s, mean=0.0):
        return torch.randn(*shape, generator=gen, device=DEV, dtype=dtype).mul_(s).add_(mean)

    st = {"embed": rn(SEQ_VOCAB, W, s=1.0)}
    if family == "puguzen":
        z = PUGUZEN[width]
        H, G, F = z["heads"], z["kv"], z["ff"]
        st["final.norm"] = rn(W, s=0.1)
        for i, kind in enumerate(("retention", "attention", "gla", "attention")):
            p, kvh = f"l{i}.", G if kind == "attention" else H
            st[p + "norm1"] = rn(W, s=0.1)
            for nm, rows in (("q", H * D), ("k", kvh * D), ("v", kvh * D), ("g", H * D)):
                st[p + "mix." + nm] = rn(rows, W, s=W ** -0.5)
            st[p + "mix.o"] = rn(W, H * D, s=(H * D) ** -0.5)
            if kind == "attention":
                st[p + "mix.pb"] = rn(H, s=1.0, mean=-4.0)
            if kind == "gla":
                st[p + "mix.norm"], st[p + "mix.a1"] = rn(D, s=0.1, mean=1.0), rn(RANK, W, s=W ** -0.5)
                st[p + "mix.a2"], st[p + "mix.a2.b"] = rn(H * D, RANK, s=RANK ** -0.5), rn(H * D, s=1.0, mean=3.0)
            st[p + "rg1"], st[p + "rg1.b"] = rn(W, W, s=W ** -0.5), rn(W, s=0.5)
            st[p + "mlp.gate"], st[p + "mlp.up"] = rn(F, W, s=W ** -0.5), rn(F, W, s=W ** -0.5)
            st[p + "mlp.down"] = rn(W, F, s=F ** -0.5)
            st[p + "rg2"], st[p + "rg2.b"] = rn(W, W, s=W ** -0.5), rn(W, s=0.5)
        return st
    z = NABURAX[width]
    H, G, Hs, F, E = z["heads"], z["kv"], z["s_heads"], z["eff"], z["experts"]
    # Routers as training leaves them: a token's embedding points to two experts by a margin (a router whose rows
    # know nothing of the tokens ties all the time, and rounding then decides which experts run).
    dirs = rn(E, W, s=W ** -0.5)
    at = torch.rand(SEQ_VOCAB, E, generator=gen, device=DEV).topk(TOP, -1).indices
    st["embed"] += 20.0 * dirs[at].sum(1)
    st["final.norm"], st["head"], st["bigram"] = rn(W, s=0.1, mean=1.0), rn(SEQ_VOCAB, W, s=W ** -0.5), rn(BUCKETS + 1, W, s=0.5)
    for i in range(4):
        p = f"l{i}."
        st[p + "norm1"], st[p + "norm2"] = rn(W, s=0.1, mean=1.0), rn(W, s=0.1, mean=1.0)
        if i % 2 == 0:
            qr = z["q_rank"]
            st[p + "mix.dq"], st[p + "mix.dq.norm"] = rn(qr, W, s=W ** -0.5), rn(qr, s=0.1, mean=1.0)
            st[p + "mix.uq"] = rn(H * (D + ROT), qr, s=qr ** -0.5)
            st[p + "mix.dkv"], st[p + "mix.dkv.norm"] = rn(KV_RANK + ROT, W, s=W ** -0.5), rn(KV_RANK, s=0.1, mean=1.0)
            st[p + "mix.uk"], st[p + "mix.uv"] = rn(H * D, KV_RANK, s=KV_RANK ** -0.5), rn(H * D, KV_RANK, s=KV_RANK ** -0.5)
            st[p + "mix.o"] = rn(W, H * D, s=(H * D) ** -0.5)
        else:
            for nm, rows in (("q", H * D), ("k", G * D), ("v", G * D)):
                st[p + "mix.left." + nm] = rn(rows, W, s=W ** -0.5)
            st[p + "mix.left.q.norm"], st[p + "mix.left.k.norm"] = rn(H * D, s=0.1, mean=1.0), rn(G * D, s=0.1, mean=1.0)
            st[p + "mix.left.o"] = rn(W, H * D, s=(H * D) ** -0.5)
            inner = Hs * SVDIM
            st[p + "mix.right.in"] = rn(2 * inner + 2 * STATE + Hs, W, s=W ** -0.5)
            st[p + "mix.right.conv"], st[p + "mix.right.conv.b"] = rn(inner + 2 * STATE, 4, s=0.5), rn(inner + 2 * STATE, s=0.1)
            st[p + "mix.right.dt_bias"], st[p + "mix.right.A_log"] = rn(Hs, s=0.5, mean=-1.0), rn(Hs, s=0.5, mean=-1.0)
            st[p + "mix.right.D"], st[p + "mix.right.norm"] = rn(Hs, s=0.2, mean=1.0), rn(inner, s=0.1, mean=1.0)
            st[p + "mix.right.o"] = rn(W, inner, s=inner ** -0.5)
        st[p + "mlp.router"] = 0.2 * dirs.roll(i, 0)
        for e in range(E):
            st[p + f"mlp.e{e}.gate"], st[p + f"mlp.e{e}.up"] = rn(F, W, s=W ** -0.5), rn(F, W, s=W ** -0.5)
            st[p + f"mlp.e{e}.down"] = rn(W, F, s=F ** -0.5)
    return st


def _tokens(seed, n, vocab):
    return torch.randint(0, vocab, (n,), generator=_gen(seed, 3), device=DEV).tolist()


def _accept_inputs(case, seed):
    """The draft's logits, the target's (the draft's and a difference: the two agree often), proposals drawn
    from the draft's distribution, uniforms and temperatures."""
    g, B, k, V = _gen(seed, 4), case["seqs"], case["k"], case["vocab"]
    d = torch.randn(B * k, V, generator=g, device=DEV) * 2.0
    t = torch.randn(B, k + 1, V, generator=g, device=DEV) * 2.0
    t[:, :k] = t[:, :k] * 0.25 + d.view(B, k, V)
    temps = torch.full((B,), 0.8, device=DEV)
    ids = torch.multinomial(torch.softmax(d / 0.8, -1), 1, generator=g).view(B, k)
    u = torch.rand(B, 2 * k + 2, generator=g, device=DEV)
    return t.view(B * (k + 1), V), d, temps, ids, u[:, :k].contiguous(), u[:, k:2 * k + 1].contiguous(), u[:, 2 * k + 1].contiguous()


# ------------------------------------------------------------------------------------ the calls
def prepare(case, seed):
    kind = case["kind"]
    st = {"case": dict(case)}
    if kind == "pass":
        cfg, ctx, toks, kv, max_ctx = _pass_inputs(case, seed)
        w = weights.from_state_dict(cfg, _decoder_state(cfg, _gen(seed)), DEV, fp8=case["fp8"])
        rows = case["seqs"] * case["rows"]
        st.update(kv=kv, toks=toks, lens=torch.tensor(ctx, dtype=torch.int32, device=DEV), max_ctx=max_ctx,
                  model=DecoderModel(w, max_ctx, wide=rows > 16), logits=torch.empty(rows, cfg.vocab, device=DEV))
    elif kind == "prompt":
        cfg = _model_cfg(case["model"], case["layers"])
        w = weights.from_state_dict(cfg, _decoder_state(cfg, _gen(seed)), DEV)
        dw = None
        if case["draft"]:
            dc = config.preset(case["draft"])
            dw = weights.from_state_dict(dc, _decoder_state(dc, _gen(seed, 5)), DEV)
        st["prompts"] = _prompts(case, seed, cfg.vocab)
        st["engine"] = SpecEngine(w, dw, EngineConfig(k=5 if dw else 0, max_batch=case["seqs"], max_seq_len=case["len_max"] + 256))
    elif kind in ("text", "turn"):
        dtype = torch.float32 if case.get("dtype") == "float32" else torch.bfloat16
        cfg = _seq_cfg(case["family"], case["width"])
        w = weights.seq_from_state_dict(cfg, _seq_state(case["family"], case["width"], dtype, _gen(seed)), DEV, dtype)
        n, B = case["tokens"] + case.get("steps", 0), case.get("seqs", 1)
        t = _tokens(seed, n * B, SEQ_VOCAB)
        st["texts"] = [t[b * n:(b + 1) * n] for b in range(B)]
        st["engine"] = SeqEngine(w, SeqEngineConfig(max_seqs=B, max_tokens=B * (n + PAGE), max_seq_len=n + PAGE))
    else:
        st["in"] = _accept_inputs(case, seed)
        st["scratch"] = ops.sampling_scratch(case["seqs"] * (case["k"] + 1), DEV)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "pass":
        st["model"].forward(st["kv"], st["toks"], case["rows"], 0, st["lens"], 0, case["seqs"], case["rows"], st["logits"],
                            st["max_ctx"])
        return st["logits"]
    if kind == "prompt":
        eng, ps = st["engine"], st["prompts"]
        eng.reset()
        eng.add_request(0, ps[0]) if len(ps) == 1 else eng.add_requests(ps)   # (the first tokens: the logits' arg-max)
        with torch.cuda.stream(eng.stream):   # the prompts' whole pages of keys and values, as a cache is handed on
            pages = torch.cat([eng.t_kv.block_tables[b, :len(p) // PAGE] for b, p in enumerate(ps)])
            return {"logits": eng.t_logits[:len(ps)], "k": eng.t_kv.k[:, pages], "v": eng.t_kv.v[:, pages]}
    if kind == "text":
        t = st["texts"][0]
        out = st["engine"].step([("text", t, range(len(t)) if case["score"] else [len(t) - 1])])
        st["engine"].finish("text")
        return out
    if kind == "turn":
        eng, n = st["engine"], case["tokens"]
        out = [eng.step([(f"r{b}", t[:n], [n - 1]) for b, t in enumerate(st["texts"])])]
        for i in range(case["steps"]):
            out.append(eng.step([(f"r{b}", [t[n + i]], [0]) for b, t in enumerate(st["texts"])]))
        for b in range(case["seqs"]):
            eng.finish(f"r{b}")
        return out
    t, d, temps, ids, u_accept, u_recover, u_bonus = st["in"]
    B, k, V = case["seqs"], case["k"], case["vocab"]
    t_probs = ops.softmax_rows(t, temps, rows_per_seq=k + 1, scratch=st["scratch"])
    d_probs = ops.softmax_rows(d, temps, rows_per_seq=k, scratch=st["scratch"])
    bonus = ops.sample_rows(t_probs, u_bonus, row_offset=k, row_step=k + 1, scratch=st["scratch"])
    out = ops.rejection_sample(t_probs.view(B, k + 1, V), bonus, d_probs.view(B, k, V), ids, u_accept, u_recover, scratch=st["scratch"])
    return {"target": t_probs, "draft": d_probs, "bonus": bonus, "out": out}


# ------------------------------------------------------------------------------------ what a pass cannot do without
def _decoder_work(cfg, tokens, keys, logit_rows, weight_bytes):
    """tokens: rows of the pass; keys: for each cached or new key read once the sum over sequences; pairs are
    counted by the caller in keys_pairs."""
    per_layer = cfg.qkv_rows * cfg.hidden + cfg.hidden * cfg.n_heads * cfg.head_dim + 3 * cfg.ffn * cfg.hidden
    kv = 2 * cfg.n_layers * cfg.n_kv_heads * cfg.head_dim * 2
    nbytes = weight_bytes * (cfg.n_layers * per_layer + cfg.vocab * cfg.hidden) + kv * keys + 4 * logit_rows * cfg.vocab
    return nbytes, 2.0 * cfg.n_layers * per_layer * tokens + 2.0 * cfg.vocab * cfg.hidden * logit_rows


def work(case):
    kind = case["kind"]
    if kind == "pass":
        cfg = _model_cfg(case["model"], case["layers"])
        ctx, q = _spread(case["ctx_min"], case["ctx_max"], case["seqs"]), case["rows"]
        nbytes, flops = _decoder_work(cfg, case["seqs"] * q, sum(ctx) + case["seqs"] * q, case["seqs"] * q, 1 if case["fp8"] else 2)
        flops += sum(4.0 * q * (c + q / 2) for c in ctx) * cfg.n_heads * cfg.head_dim * cfg.n_layers
        return {"bytes": nbytes, "flops": flops}
    if kind == "prompt":
        ls = _spread(case["len_min"], case["len_max"], case["seqs"])
        nbytes = flops = 0
        for name, layers in ((case["model"], case["layers"]), (case["draft"], None)):
            if not name:
                continue
            cfg = _model_cfg(name, layers or config.PRESETS[name]["n_layers"])
            b, f = _decoder_work(cfg, sum(ls), sum(ls), case["seqs"] if layers else 0, 2)
            nbytes += b
            flops += f + sum(2.0 * n * n for n in ls) * cfg.n_heads * cfg.head_dim * cfg.n_layers
        return {"bytes": nbytes, "flops": flops}
    if kind == "accept":
        R = case["seqs"] * (2 * case["k"] + 1)
        # logits read, probabilities written, and at least one target and one draft row read by the draws
        return {"bytes": 4.0 * case["vocab"] * (2 * R + 2 * case["seqs"]), "flops": 5.0 * R * case["vocab"]}
    W, n, B, steps = case["width"], case["tokens"], case.get("seqs", 1), case.get("steps", 0)
    el = 4 if case.get("dtype") == "float32" else 2
    rows = n * B
    out_rows = (n if case.get("score") else 1) * B
    nbytes = flops = 0.0
    for r, ctx, outs, times in ((rows, n, out_rows, 1), (B, n, B, steps)):   # the prompts, then the single tokens
        pairs = r * min(ctx, WINDOW) / (2.0 if times == 1 and ctx <= WINDOW else 1.0)
        if case["family"] == "puguzen":
            z = PUGUZEN[W]
            H, G, F = z["heads"], z["kv"], z["ff"]
            mats = 4 * (2 * W * W + 3 * W * F + 2 * W * H * HEAD) + 2 * W * (2 * H + 2 * G) * HEAD + 2 * RANK * W
            act, held = mats, mats
            attn = 2 * 4.0 * pairs * H * HEAD
            rec = 2 * 4.0 * r * H * HEAD * HEAD
        else:
            z = NABURAX[W]
            H, G, E, F = z["heads"], z["kv"], z["experts"], z["eff"]
            inner = z["s_heads"] * SVDIM
            lat = W * (z["q_rank"] + KV_RANK + ROT) + z["q_rank"] * H * (HEAD + ROT) + 2 * H * HEAD * KV_RANK + W * H * HEAD
            par = W * (H + 2 * G) * HEAD + W * (2 * inner + 2 * STATE + z["s_heads"]) + W * H * HEAD + W * inner
            act = 2 * lat + 2 * par + 4 * TOP * 3 * W * F
            held = 2 * lat + 2 * par + 4 * min(E, r * TOP) * 3 * W * F
            attn = 2 * 2.0 * pairs * H * (2 * HEAD + ROT) + 2 * 4.0 * pairs * H * HEAD
            rec = 2 * 4.0 * r * inner * STATE
        nbytes += times * (el * (held + SEQ_VOCAB * W) + 4.0 * outs * SEQ_VOCAB + el * r * W)
        flops += times * (2.0 * act * r + 2.0 * SEQ_VOCAB * W * outs + attn + rec)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "accept":
        # f32 sums of a row's exponentials; a draw may fall on the neighbour where two sums differ in the last bits
        return {"rel": 1e-5, "differ": 0.02}
    if case.get("dtype") == "float32":
        return {"rel": 1e-5}
    if kind in ("text", "turn"):
        return {"rel": 2e-2}   # bf16 operands, f32 residual
    # bf16 rows and residual between the layers: 0.02 off 64 bits at 8 layers, 0.04 at 32
    return {"rel": 8e-2}


# ------------------------------------------------------------------------------------ in 64 bits
def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _angles(cfg, pos):
    d = cfg.head_dim
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, d, 2, dtype=F64, device=DEV) / d))
    sc = cfg.rope_scaling
    if sc:   # long wavelengths stretched by `factor`, a ramp between the two
        old = sc["original_max_position_embeddings"]
        wl = 2 * math.pi / inv
        ramp = ((old / wl - sc["low_freq_factor"]) / (sc["high_freq_factor"] - sc["low_freq_factor"])).clamp(0, 1)
        inv = (1 - ramp) * inv / sc["factor"] + ramp * inv
    return pos.to(F64)[:, None] * inv[None, :]


def _turn_halves(x, a):
    u, v = x.chunk(2, -1)
    c, s = a.cos()[:, None, :], a.sin()[:, None, :]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _fp8(w):
    s = (w.float().abs().amax(1, keepdim=True).clamp_min(1e-12) / 448.0)
    return (w.float() / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).to(F64) * s.to(F64)


def _softmax_rows_over(q, k, v, mask, scale, block=512):
    """q [T, H, dk], k [n, G, dk], v [n, G, dv], mask [T, n]."""
    T, H, _ = q.shape
    n, G, _ = k.shape
    out = torch.empty(T, H, v.shape[2], dtype=F64, device=DEV)
    for g in range(G):
        hs = slice(g * (H // G), (g + 1) * (H // G))
        for t in range(0, T, block):
            s = torch.matmul(q[t:t + block, hs].transpose(0, 1), k[:, g].T.contiguous()) * scale
            s.masked_fill_(~mask[t:t + block], float("-inf"))
            out[t:t + block, hs] = torch.matmul(torch.softmax(s, -1), v[:, g]).transpose(0, 1)
    return out


def _decoder_exact(cfg, st, tokens, starts, ends, past, fp8, last_only):
    """tokens: flat rows; sequence b is rows starts[b]..ends[b]-1 behind past(layer, b) -> (k, v, n) or nothing.
    Returns (logits, per layer the new keys and values)."""
    wt = _fp8 if fp8 else lambda w: w.to(F64)
    D, Hq, G = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads
    x = st["model.embed_tokens.weight"][tokens].to(F64)
    new = []
    for i in range(cfg.n_layers):
        p = f"model.layers.{i}."
        h = _rms(x, st[p + "input_layernorm.weight"].to(F64), cfg.norm_eps)
        qkv = []
        for nm in "qkv":
            y = h @ wt(st[p + f"self_attn.{nm}_proj.weight"]).T
            b = st.get(p + f"self_attn.{nm}_proj.bias")
            qkv.append((y if b is None else y + b.to(F64)).view(x.shape[0], -1, D))
        o = torch.empty(x.shape[0], Hq * D, dtype=F64, device=DEV)
        kept = []
        for b, (lo, hi) in enumerate(zip(starts, ends)):
            pk, pv, n0 = past(i, b)
            pos = torch.arange(n0, n0 + hi - lo, device=DEV)
            a = _angles(cfg, pos)
            q, k, v = _turn_halves(qkv[0][lo:hi], a), _turn_halves(qkv[1][lo:hi], a), qkv[2][lo:hi]
            kept.append((k, v))
            if n0:
                k, v = torch.cat([pk, k]), torch.cat([pv, v])
            mask = torch.arange(k.shape[0], device=DEV)[None, :] <= pos[:, None]
            o[lo:hi] = _softmax_rows_over(q, k, v, mask, D ** -0.5).reshape(hi - lo, Hq * D)
        new.append(kept)
        x = x + o @ wt(st[p + "self_attn.o_proj.weight"]).T
        h = _rms(x, st[p + "post_attention_layernorm.weight"].to(F64), cfg.norm_eps)
        gate = h @ wt(st[p + "mlp.gate_proj.weight"]).T
        x = x + (gate * torch.sigmoid(gate) * (h @ wt(st[p + "mlp.up_proj.weight"]).T)) @ wt(st[p + "mlp.down_proj.weight"]).T
    if last_only:
        x = x[torch.tensor(ends, device=DEV) - 1]
    head = st.get("lm_head.weight", st["model.embed_tokens.weight"])
    return _rms(x, st["model.norm.weight"].to(F64), cfg.norm_eps) @ wt(head).T, new


_SLOT = [(t & 3) | ((t >> 3) & 1) << 2 | ((t >> 2) & 1) << 3 for t in range(PAGE)]   # token t's column of a value page


def _from_pages(k, v, D):
    """Pages [pages, G, 16 * D] -> keys and values [tokens, G, D]."""
    n, G, _ = k.shape
    kk = k.view(n, G, D // 8, PAGE, 8).permute(0, 3, 1, 2, 4).reshape(n * PAGE, G, D)
    vv = v.view(n, G, D, PAGE)[..., _SLOT].permute(0, 3, 1, 2).reshape(n * PAGE, G, D)
    return kk, vv


def _to_pages(k, v):
    T, G, D = k.shape
    n = T // PAGE
    k, v = k[:n * PAGE].view(n, PAGE, G, D), v[:n * PAGE].view(n, PAGE, G, D)
    kp = k.permute(0, 2, 3, 1).reshape(n, G, D // 8, 8, PAGE).transpose(3, 4).reshape(n, G, D * PAGE)
    vp = torch.empty(n, G, D, PAGE, dtype=v.dtype, device=v.device)
    vp[..., _SLOT] = v.permute(0, 2, 3, 1)
    return kp, vp.reshape(n, G, D * PAGE)


def _pass_exact(case, seed):
    cfg, ctx, toks, kv, _ = _pass_inputs(case, seed)
    q = case["rows"]

    def past(layer, b):
        pages = torch.tensor(kv.pages_of(b), device=DEV)
        k, v = _from_pages(kv.k[layer, pages], kv.v[layer, pages], cfg.head_dim)
        return k[:ctx[b]].to(F64), v[:ctx[b]].to(F64), ctx[b]

    starts = [b * q for b in range(case["seqs"])]
    return _decoder_exact(cfg, _decoder_state(cfg, _gen(seed)), toks.view(-1).long(), starts, [s + q for s in starts], past,
                          case["fp8"], False)[0]


def _prompt_exact(case, seed):
    cfg = _model_cfg(case["model"], case["layers"])
    st = _decoder_state(cfg, _gen(seed))
    ps = _prompts(case, seed, cfg.vocab)
    ends = [sum(len(p) for p in ps[:i + 1]) for i in range(len(ps))]
    starts = [0] + ends[:-1]
    tokens = torch.tensor([t for p in ps for t in p], device=DEV)
    logits, new = _decoder_exact(cfg, st, tokens, starts, ends, lambda layer, b: (None, None, 0), False, True)
    k, v = [], []
    for kept in new:
        pages = [_to_pages(*kv) for kv in kept]
        k.append(torch.cat([a for a, _ in pages]).float())
        v.append(torch.cat([b for _, b in pages]).float())
    return {"logits": logits, "k": torch.stack(k), "v": torch.stack(v)}


def _turn_pairs(x, pos, freq, mag=1.0):
    a = pos.to(F64)[:, None] * freq[None, :]
    c, s = a.cos()[:, None, :] * mag, a.sin()[:, None, :] * mag
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)


def _scan(q, k, v, decay):
    """S <- decay S + k v^T, o = S^T q: q, k, decay [T, H, dk], v [T, H, dv]."""
    T, H, dk = q.shape
    S = torch.zeros(H, dk, v.shape[2], dtype=F64, device=DEV)
    out = torch.empty(T, H, v.shape[2], dtype=F64, device=DEV)
    for t in range(T):
        S.mul_(decay[t][:, :, None]).addcmul_(k[t][:, :, None], v[t][:, None, :])
        out[t] = (S * q[t][:, :, None]).sum(1)
    return out


def _unit(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _puguzen_exact(width, st, tokens):
    z = PUGUZEN[width]
    H, G, D = z["heads"], z["kv"], HEAD
    T = len(tokens)
    pos = torch.arange(T, device=DEV)
    freq = 1e6 ** (-2.0 * torch.arange(D // 2, dtype=F64, device=DEV) / D)
    x = st["embed"][tokens]
    for i, kind in enumerate(("retention", "attention", "gla", "attention")):
        w = {n[len(f"l{i}."):]: t for n, t in st.items() if n.startswith(f"l{i}.")}
        h = _unit(x) * (1 + w["norm1"])
        q, k, v = (h @ w["mix." + n].T for n in "qkv")
        q, k, v = q.view(T, H, D), k.view(T, -1, D), v.view(T, -1, D)
        g = h @ w["mix.g"].T
        if kind == "attention":
            q, k = _unit(_turn_pairs(q, pos, freq)), _unit(_turn_pairs(k, pos, freq))
            nb = T // POOL   # whole blocks; a block is seen once it lies wholly before the window
            kb, vb = (t[:nb * POOL].view(nb, POOL, G, D).mean(1) for t in (k, v))
            kk, vv = torch.cat([k, kb]), torch.cat([v, vb])
            last = torch.arange(nb, device=DEV) * POOL + POOL - 1
            d = pos[:, None] - pos[None, :]
            mask = torch.cat([(d >= 0) & (d < WINDOW), last[None, :] <= pos[:, None] - WINDOW], 1)
            o = torch.empty(T, H, D, dtype=F64, device=DEV)
            for hd in range(H):
                s = torch.sigmoid(q[:, hd] @ kk[:, hd // (H // G)].T * D ** -0.5 + w["mix.pb"][hd])
                o[:, hd] = (s * mask) @ vv[:, hd // (H // G)]
            y = (o.reshape(T, H * D) * torch.sigmoid(g)) @ w["mix.o"].T
        else:
            if kind == "retention":
                a = pos.to(F64)[:, None] * freq[None, :]
                q, k = _turn_halves(q, a), _turn_halves(k, a) * D ** -0.5
                decay = torch.tensor([_decay(j, H) for j in range(H)], dtype=F64, device=DEV)[None, :, None].expand(T, H, D)
                o = _unit(_scan(q, k, v, decay))
            else:
                decay = torch.sigmoid((h @ w["mix.a1"].T) @ w["mix.a2"].T + w["mix.a2.b"]).pow(1 / 16.0).view(T, H, D)
                o = _unit(_scan(q * D ** -0.5, k, v, decay)) * w["mix.norm"]
            y = (o.reshape(T, H * D) * g * torch.sigmoid(g)) @ w["mix.o"].T
        ff = (torch.relu(h @ w["mlp.gate"].T) * (h @ w["mlp.up"].T)) @ w["mlp.down"].T
        x = x + torch.sigmoid(h @ w["rg1"].T + w["rg1.b"]) * y + torch.sigmoid(h @ w["rg2"].T + w["rg2.b"]) * ff
    return _unit(x) * (1 + st["final.norm"]), st["embed"]


def _stretched(dims, base, sc):
    """Rotary frequencies of a stretched context: slow pairs divided by `factor`, a ramp over the pairs between."""
    i = torch.arange(dims // 2, dtype=F64, device=DEV)
    f = base ** (-2.0 * i / dims)
    at = lambda turns: dims * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
    lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


def _naburax_exact(width, st, tokens):
    z = NABURAX[width]
    H, G, D, Hs, E = z["heads"], z["kv"], HEAD, z["s_heads"], z["experts"]
    T = len(tokens)
    inner = Hs * SVDIM
    pos = torch.arange(T, device=DEV)
    d = pos[:, None] - pos[None, :]
    seen = (d >= 0) & (d < WINDOW)
    tk = torch.tensor(tokens, device=DEV)
    pair = torch.cat([torch.tensor([BUCKETS], device=DEV), (tk[:-1] * MUL_PREV + tk[1:] * MUL_CUR) % BUCKETS])
    x = st["embed"][tokens] + st["bigram"][pair]
    for i in range(4):
        w = {n[len(f"l{i}."):]: t for n, t in st.items() if n.startswith(f"l{i}.")}
        if i % 2 == 0:
            freq, mag = _stretched(ROT, 1e6, SCALING)
            q = (_rms(x @ w["mix.dq"].T, w["mix.dq.norm"], EPS) @ w["mix.uq"].T).view(T, H, D + ROT)
            kv = x @ w["mix.dkv"].T
            c = _rms(kv[:, :KV_RANK], w["mix.dkv.norm"], EPS)
            kr = _turn_pairs(kv[:, None, KV_RANK:], pos, freq, mag).expand(T, H, ROT)
            q = torch.cat([q[..., :D], _turn_pairs(q[..., D:], pos, freq, mag)], -1)
            k = torch.cat([(c @ w["mix.uk"].T).view(T, H, D), kr], -1)
            o = _softmax_rows_over(q, k, (c @ w["mix.uv"].T).view(T, H, D), seen, (D + ROT) ** -0.5)
            a = o.reshape(T, H * D) @ w["mix.o"].T
        else:
            q = _rms(x @ w["mix.left.q"].T, w["mix.left.q.norm"], EPS).view(T, H, D)
            k = _rms(x @ w["mix.left.k"].T, w["mix.left.k.norm"], EPS).view(T, G, D)
            v = (x @ w["mix.left.v"].T).view(T, G, D)
            kept = seen | ((d >= 0) & (pos[None, :] < KEEP))
            left = _softmax_rows_over(q, k, v, kept, D ** -0.5).reshape(T, H * D) @ w["mix.left.o"].T
            u = x @ w["mix.right.in"].T
            zg, xbc, dt = u[:, :inner], u[:, inner:2 * inner + 2 * STATE], u[:, 2 * inner + 2 * STATE:]
            full = torch.cat([torch.zeros(3, xbc.shape[1], dtype=F64, device=DEV), xbc])
            conv = sum(full[j:j + T] * w["mix.right.conv"][:, j] for j in range(4)) + w["mix.right.conv.b"]
            conv = conv * torch.sigmoid(conv)
            xs = conv[:, :inner].view(T, Hs, SVDIM)
            bs, cs = conv[:, inner:inner + STATE], conv[:, inner + STATE:]
            dt = torch.nn.functional.softplus(dt + w["mix.right.dt_bias"])
            decay = torch.exp(-torch.exp(w["mix.right.A_log"]) * dt)
            wide = lambda t: t[:, None, :].expand(T, Hs, STATE)
            y = _scan(wide(cs), wide(bs), xs * dt[..., None], decay[..., None].expand(T, Hs, STATE)) + w["mix.right.D"][:, None] * xs
            y = _unit(y.reshape(T, inner) * zg * torch.sigmoid(zg)) * w["mix.right.norm"]
            a = 0.5 * left + 0.5 * (y @ w["mix.right.o"].T)
        x = x + _rms(a, w["norm1"], EPS)
        score, at = torch.sigmoid(x @ w["mlp.router"].T).topk(TOP, -1)
        ff = torch.zeros_like(x)
        for e in range(E):
            rows, col = (at == e).nonzero(as_tuple=True)
            h = x[rows] * score[rows, col][:, None]
            gate = h @ w[f"mlp.e{e}.gate"].T
            ff.index_add_(0, rows, (gate * torch.sigmoid(gate) * (h @ w[f"mlp.e{e}.up"].T)) @ w[f"mlp.e{e}.down"].T)
        x = x + _rms(ff, w["norm2"], EPS)
    return _rms(x, st["final.norm"], EPS), st["head"]


def exact(case, seed):
    kind = case["kind"]
    if kind == "pass":
        return _pass_exact(case, seed)
    if kind == "prompt":
        return _prompt_exact(case, seed)
    if kind == "accept":
        t, d, temps, *_ = _accept_inputs(case, seed)
        soft = lambda x: torch.softmax(x.to(F64) / temps[0].to(F64), -1)
        return {"target": soft(t), "draft": soft(d), "bonus": None, "out": None}
    dtype = torch.float32 if case.get("dtype") == "float32" else torch.bfloat16
    st = {n: t.to(F64) for n, t in _seq_state(case["family"], case["width"], dtype, _gen(seed)).items()}
    model = _puguzen_exact if case["family"] == "puguzen" else _naburax_exact
    n, B, steps = case["tokens"], case.get("seqs", 1), case.get("steps", 0)
    t = _tokens(seed, (n + steps) * B, SEQ_VOCAB)
    first = 0 if case.get("score") else n - 1
    rows = []
    for b in range(B):
        x, head = model(case["width"], st, t[b * (n + steps):(b + 1) * (n + steps)])
        rows.append(x[first:] @ head.T)
    return rows[0] if kind == "text" else [torch.stack([r[i] for r in rows]) for i in range(steps + 1)]
