"""The Naburax decoder family on the GPU against the plain CPU restatement in oracle/naburax.py:
every mechanism alone through its entry point, then whole models through the engine (prompts
whole, token by token, in portions, in mixed batches, over reused slots and pages) and through
the worker and scheduler.  Small random models of several shapes; where random weights would hide
a fault (one far key among many, a kept first token, a window's edge) the inputs are made so
that it shows."""
import pytest
import torch

from oracle import naburax as N

pytestmark = pytest.mark.gpu

DEV = "cuda"
PAGE = 16


def dev(t, dtype=None):
    return t.to(dtype or t.dtype).contiguous().to(DEV)


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def rel(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return ((a - b).pow(2).mean().sqrt() / b.pow(2).mean().sqrt().clamp_min(1e-30)).item()


# ------------------------------------------------------------------ model shapes
def latent(heads=2, dim=8, rot_dim=8, vdim=8, q_rank=12, kv_rank=16, window=9, scale=0.3, rot_dims=None,
           base=10000.0, scaling="default", mlp="default"):
    if scaling == "default":
        scaling = {"factor": 4.0, "original": 64, "fast": 8.0, "slow": 1.0}
    m = dict(heads=heads, dim=dim, rot_dim=rot_dim, vdim=vdim, q_rank=q_rank, kv_rank=kv_rank, scale=scale,
             mask={"size": window}, rot={"dims": rot_dim if rot_dims is None else rot_dims, "base": base})
    if scaling:
        m["rot"]["scaling"] = scaling
    return {"type": "latent_attention", "mixer": m, "mlp": experts() if mlp == "default" else mlp}


def parallel(heads=4, kv_heads=2, dim=8, vdim=8, window=7, keep_first=2, scale=0.3, s_heads=2, s_vdim=8, state=8,
             groups=1, taps=4, norm_groups=1, left_scale=0.7, right_scale=0.4, mlp="default"):
    m = dict(left=dict(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, scale=scale,
                       mask={"size": window, "keep_first": keep_first}),
             right=dict(heads=s_heads, vdim=s_vdim, state=state, groups=groups, conv=taps, norm_groups=norm_groups),
             left_scale=left_scale, right_scale=right_scale)
    return {"type": "parallel", "mixer": m, "mlp": experts() if mlp == "default" else mlp}


def experts(n=4, top=2, ff=24):
    return {"kind": "moe", "expert": {"ff": ff}, "router": {"experts": n, "top": top}}


def model_cfg(layers, width=32, vocab=80, eps=1e-5, scale=3.0, logit_scale=0.7, bigram="default"):
    if bigram == "default":
        bigram = {"buckets": 53, "mul_prev": 31, "mul_cur": 7}
    emb = {"scale": scale}
    if bigram:
        emb["bigram"] = bigram
    return {"architecture": "Naburax", "width": width, "vocab": vocab, "norm": {"eps": eps}, "embedding": emb,
            "logit_scale": logit_scale, "layers": layers}


SHAPES = {
    "two_kinds": model_cfg([latent(), parallel(), latent(window=5)]),
    # sizes that divide nothing; every pair of sizes that may coincide made different; three experts of
    # five; a recurrence first; several groups and norm groups; a window shorter than the kept tokens
    "odd": model_cfg([parallel(heads=6, kv_heads=3, dim=12, vdim=20, window=3, keep_first=5, s_heads=6, s_vdim=10,
                               state=12, groups=3, taps=3, norm_groups=2, mlp=experts(5, 3, 20)),
                      latent(heads=3, dim=12, rot_dim=6, vdim=10, q_rank=9, kv_rank=21, window=11, rot_dims=4,
                             mlp=None),
                      parallel(heads=2, kv_heads=2, dim=20, vdim=4, window=9, keep_first=0, s_heads=1, s_vdim=24,
                               state=20, taps=2, mlp=experts(3, 1, 10))],
                     width=40, vocab=131, eps=1e-6, bigram={"buckets": 17, "mul_prev": 1000003, "mul_cur": 999983}),
    # window 1, one head, one tap, one expert, no rotation scaling, no bigram table, scales of one
    "ones": model_cfg([latent(heads=1, dim=4, rot_dim=2, vdim=6, q_rank=5, kv_rank=8, window=1, scaling=None,
                              mlp=experts(1, 1, 8)),
                       parallel(heads=1, kv_heads=1, dim=8, vdim=12, window=1, keep_first=1, s_heads=1, s_vdim=4,
                                state=4, taps=1, left_scale=1.0, right_scale=1.0, mlp=None),
                       latent(heads=2, dim=4, rot_dim=0, vdim=6, q_rank=5, kv_rank=8, window=40)],
                      width=24, vocab=50, scale=1.0, logit_scale=1.0, bigram=None),
    # widths that are multiples of 32: bfloat16 serving takes the tiled linear kernels
    "aligned": model_cfg([latent(heads=4, dim=16, rot_dim=16, vdim=8, q_rank=32, kv_rank=64, window=20,
                                 mlp=experts(8, 2, 32)),
                          parallel(heads=4, kv_heads=1, dim=16, vdim=16, window=12, keep_first=3, s_heads=4,
                                   s_vdim=16, state=16, groups=2, norm_groups=4, mlp=experts(8, 2, 32))],
                         width=64, vocab=178),
    # heads wider than a lane group, a latent wider than two tiles of value columns, a wide state
    "wide": model_cfg([latent(heads=2, dim=24, rot_dim=8, vdim=40, q_rank=20, kv_rank=136, window=33),
                       parallel(heads=2, kv_heads=1, dim=72, vdim=136, window=33, keep_first=1, s_heads=2, s_vdim=72,
                                state=40, taps=5)], width=48, vocab=64),
}


def build(cfg, dtype=torch.float32, seed=0, tiled=True, **eng_kw):
    from vllm_omni_draft_amd import config, weights
    from vllm_omni_draft_amd.seq_engine import SeqEngine, SeqEngineConfig
    st = N.random_tensors(cfg, seed)
    mc = config.naburax_config(cfg, {k: tuple(v.shape) for k, v in st.items()})
    w = weights.seq_from_state_dict(mc, st, DEV, dtype, tiled=tiled)
    kw = dict(max_seqs=4, max_tokens=1024)
    kw.update(eng_kw)
    return st, SeqEngine(w, SeqEngineConfig(**kw))


def prompt(cfg, n, seed=0):
    g = torch.Generator().manual_seed(1000 + seed)
    return torch.randint(0, cfg["vocab"], (n,), generator=g).tolist()


def f64(st):
    return {k: v.double() for k, v in st.items()}


def oracle_logits(cfg, st, toks, layer_out=None):
    return N.forward(cfg, f64(st), toks, N.Sequence(len(cfg["layers"])), layer_out)


# ------------------------------------------------------------------ mechanisms alone
def test_embed_hashed():
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(0)
    V, W, buckets = 70, 36, 13
    table, bg = torch.randn(V, W, generator=g), torch.randn(buckets + 1, W, generator=g)
    toks = torch.randint(0, V, (9,), generator=g).tolist()
    cfg = {"embedding": {"scale": 2.5, "bigram": {"buckets": buckets, "mul_prev": 2000003, "mul_cur": 1999993}}}
    seq = N.Sequence(0)
    want = N.embed(cfg, {"embed": table.double(), "bigram": bg.double()}, toks, seq)
    x = ops.embed_hashed(i32(toks), dev(table), 2.5, i32([-1] + toks[:-1]), dev(bg), 2000003, 1999993)
    assert rel(x, want) < 1e-6
    # a sequence that goes on: the first row pairs with the token before
    want2 = N.embed(cfg, {"embed": table.double(), "bigram": bg.double()}, toks[:3], seq)
    x2 = ops.embed_hashed(i32(toks[:3]), dev(table), 2.5, i32([toks[-1]] + toks[:2]), dev(bg), 2000003, 1999993)
    assert rel(x2, want2) < 1e-6
    x3 = ops.embed_hashed(i32(toks), dev(table), 0.5)
    assert rel(x3, table.double()[toks] * 0.5) < 1e-6


@pytest.mark.parametrize("width,parts", [(5, 1), (72, 3), (1000, 2), (64, 64)])
def test_rmsnorm_parts(width, parts):
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(width)
    x, w, z = torch.randn(6, width, generator=g) * 3, torch.randn(width, generator=g), torch.randn(6, width, generator=g)
    out = ops.rmsnorm_parts(dev(x), dev(w), 1e-5, parts)
    want = N.rms_norm(x.double().view(6, parts, -1), None, 1e-5).reshape(6, width) * w.double()
    assert rel(out, want) < 1e-6
    out, out_b = ops.rmsnorm_parts(dev(x), dev(w), 1e-3, parts, gate=dev(z), bf16_copy=True)
    y = x.double() * N.silu(z.double())
    assert rel(out, N.rms_norm(y.view(6, parts, -1), None, 1e-3).reshape(6, width) * w.double()) < 1e-6
    assert torch.equal(out_b, out.to(torch.bfloat16))


@pytest.mark.parametrize("dims,n,scaling", [(8, 8, None), (6, 10, {"factor": 8.0, "original": 128, "fast": 16.0, "slow": 2.0}),
                                            (32, 32, {"factor": 40.0, "original": 4096, "fast": 32.0, "slow": 1.0})])
def test_rope_rows_with_blended_frequencies(dims, n, scaling):
    from vllm_omni_draft_amd import config, ops
    g = torch.Generator().manual_seed(dims)
    H, off = 3, 5
    x = torch.randn(7, H * (off + n), generator=g)
    pos = torch.tensor([0, 1, 2, 63, 64, 5000, 100000])
    f, mag = config.rotary_frequencies(dims, 50000.0, scaling)
    f_ref, mag_ref = N.yarn_frequencies(dims, 50000.0, scaling)
    assert abs(mag - mag_ref) < 1e-12 and torch.allclose(f, f_ref, rtol=1e-12, atol=0)
    if scaling:   # the ends of the ramp: fast pairs keep their frequency, slow ones are divided by the factor
        plain = N.yarn_frequencies(dims, 50000.0, None)[0]
        assert f_ref[0] == plain[0] and abs(f_ref[-1] / plain[-1] - 1 / scaling["factor"]) < 1e-9
    xd = dev(x)
    ops.rope_rows(xd, i32(pos.tolist()), H, off + n, off, dims, dev(f), mag)
    v = x.double().view(7, H, off + n)
    want = torch.cat([v[..., :off], N.rotate_pairs(v[..., off:], pos, dims, f_ref, mag_ref)], -1).reshape(7, -1)
    assert (xd.cpu().double() - want).abs().max() < 2e-6


def fill_cache(k, v, pages_of, G):
    """k [n, G*dk], v [n, G*dv] or None for one sequence in slot 0 -> caches, block table."""
    from vllm_omni_draft_amd import ops
    n = k.shape[0]
    dk = k.shape[1] // G
    n_pages = max(pages_of) + 1
    kc = torch.zeros(n_pages, G, PAGE, dk, dtype=k.dtype, device=DEV)
    vc = None
    if v is not None:
        vc = torch.zeros(n_pages, G, PAGE, v.shape[1] // G, dtype=k.dtype, device=DEV)
    bt = torch.zeros(2, len(pages_of), dtype=torch.int32, device=DEV)
    bt[0] = i32(pages_of)
    bt[1] = 0
    ops.cache_append(dev(k.float()), dev(v.float()) if v is not None else None, kc, vc, i32(list(range(n))),
                     i32([0] * n), bt, G, dk, v.shape[1] // G if v is not None else 0)
    return kc, vc, bt


@pytest.mark.parametrize("H,G,dk,dv,window,keep", [(4, 2, 16, 16, 6, 2), (3, 1, 12, 20, 50, 0), (2, 2, 72, 136, 1, 3),
                                                   (9, 1, 8, 8, 17, 40), (16, 2, 8, 300, 5, 1)])
@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
def test_window_softmax_attention_random(H, G, dk, dv, window, keep, cdt):
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(H * 100 + dk)
    n = 45
    q = torch.randn(n, H * dk, generator=g)
    k, v = torch.randn(n, G * dk, generator=g).to(cdt), torch.randn(n, G * dv, generator=g).to(cdt)
    pages = [5, 1, 3]                                  # pages out of order
    kc, vc, bt = fill_cache(k, v, pages, G)
    rows = [0, 1, 2, window - 1, window, window + 1, 16, 31, 32, 44]
    rows = sorted({r for r in rows if 0 <= r < n})
    out = ops.window_softmax_attention(dev(q[rows]), kc, vc, i32(rows), i32([0] * len(rows)), bt, H, G, dk, dv,
                                       window, keep, 0.2)
    want = N.masked_softmax_attention(q.double()[rows].view(-1, H, dk), k.double().view(n, G, dk),
                                      v.double().view(n, G, dv), torch.tensor(rows), 0.2, window, keep)
    assert rel(out, want.reshape(len(rows), -1)) < 3e-6


def test_window_softmax_attention_values_inside_key_rows():
    """Latent attention: the value of a token is the first dv channels of its cached key row."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(3)
    n, H, dk, dv = 40, 5, 24, 16
    q, k = torch.randn(n, H * dk, generator=g), torch.randn(n, dk, generator=g)
    kc, _, bt = fill_cache(k, None, [2, 0, 1], 1)
    rows = list(range(n))
    out = ops.window_softmax_attention(dev(q), kc, None, i32(rows), i32([0] * n), bt, H, 1, dk, dv, 11, 0, 0.3)
    want = N.masked_softmax_attention(q.double().view(n, H, dk), k.double().view(n, 1, dk),
                                      k.double()[:, :dv].reshape(n, 1, dv), torch.tensor(rows), 0.3, 11, 0)
    assert rel(out, want.reshape(n, -1)) < 3e-6


@pytest.mark.parametrize("window,keep", [(1, 0), (1, 2), (5, 0), (5, 3), (16, 1), (17, 16), (33, 4), (300, 2), (3, 7)])
@pytest.mark.parametrize("decode", [False, True])
def test_window_softmax_attention_sees_exactly_its_keys(window, keep, decode):
    """Key j carries a score far above all others only for the query that looks for j, and value
    one-hot(j): the output of query (i, target j) is one-hot(j) if i sees j, else has no weight
    on j.  Every (position, target) pair near a border: the window's edge, the kept tokens' edge,
    page borders, the sequence's first tokens."""
    from vllm_omni_draft_amd import ops
    n, dk = 70, 8
    dv = n
    # key j = a random unit vector; the query that looks for j is 60 times that vector
    gen = torch.Generator().manual_seed(window * 7 + keep)
    code = torch.randn(n, dk, generator=gen)
    code = code / code.norm(dim=1, keepdim=True)
    k, v = code.clone(), torch.eye(n)
    kc, vc, bt = fill_cache(k, v, [4, 0, 2, 3, 1], 1)
    targets = lambda i: sorted({j for j in (0, 1, keep - 1, keep, keep + 1, i - window - 1, i - window, i - window + 1,
                                            i - window + 2, i - 1, i, 15, 16, 17, 31, 32) if 0 <= j <= i})
    pairs = [(i, j) for i in range(n) for j in targets(i)]
    if decode:      # one launch per query row, as single decoded tokens come
        pairs = [p for p in pairs if p[0] in (0, 1, keep, window - 1, window, window + 1, 16, 33, n - 1) and p[0] < n]
        outs = [ops.window_softmax_attention(dev(code[j:j + 1] * 60), kc, vc, i32([i]), i32([0]), bt, 1, 1, dk, dv,
                                             window, keep, 1.0) for i, j in pairs]
        out = torch.cat(outs).cpu()
    else:
        q = torch.stack([code[j] * 60 for _, j in pairs])
        out = ops.window_softmax_attention(dev(q), kc, vc, i32([i for i, _ in pairs]), i32([0] * len(pairs)), bt, 1,
                                           1, dk, dv, window, keep, 1.0).cpu()
    for r, (i, j) in enumerate(pairs):
        sees = N.visible(i, j, window, keep)
        assert abs(out[r].sum().item() - 1) < 1e-4                  # a softmax: the weights sum to one
        assert torch.all(out[r, i + 1:] == 0), (i, j)               # nothing from the future
        if sees:
            assert out[r, j] > 0.5, (i, j, out[r, j].item())
        else:
            assert out[r, j] == 0, (i, j, out[r, j].item())


@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
def test_window_softmax_attention_many_keys(cdt):
    """More keys than two tiles, a far key that stands out in the first tile, kept tokens ahead."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(9)
    n, H, G, dk, dv, window, keep = 700, 2, 1, 16, 24, 640, 3
    q = torch.randn(4, H * dk, generator=g)
    k, v = torch.randn(n, dk, generator=g).to(cdt), torch.randn(n, dv, generator=g).to(cdt)
    k[70] = (q[0, :dk] * 3).to(cdt)                    # row 699 of head 0 finds key 70, just inside its window
    pages = torch.randperm(44, generator=g).tolist()
    kc, vc, bt = fill_cache(k, v, pages, G)
    rows = [699, 698, 650, 300]
    out = ops.window_softmax_attention(dev(q), kc, vc, i32(rows), i32([0] * 4), bt, H, G, dk, dv, window, keep, 0.5)
    want = N.masked_softmax_attention(q.double().view(4, H, dk), k.double().view(n, G, dk), v.double().view(n, G, dv),
                                      torch.tensor(rows), 0.5, window, keep)
    assert rel(out, want.reshape(4, -1)) < 3e-6
    assert rel(out[0, :dv], v[70].double()) < 1e-3     # that key takes all the weight
    # few rows have their keys cut over workgroups and merged; many rows, or no scratch, take them in one sweep
    whole = ops.window_softmax_attention(dev(q), kc, vc, i32(rows), i32([0] * 4), bt, H, G, dk, dv, window, keep, 0.5,
                                         split=False)
    assert rel(whole, want.reshape(4, -1)) < 3e-6 and rel(whole, out) < 2e-6
    many = list(range(600, 700))
    q2 = torch.randn(100, H * dk, generator=g)
    out2 = ops.window_softmax_attention(dev(q2), kc, vc, i32(many), i32([0] * 100), bt, H, G, dk, dv, window, keep, 0.5)
    one = ops.window_softmax_attention(dev(q2[37:38]), kc, vc, i32(many[37:38]), i32([0]), bt, H, G, dk, dv, window,
                                       keep, 0.5)
    assert rel(one[0], out2[37]) < 2e-6


@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
def test_fused_preparation_equals_its_pieces(cdt):
    """The one-launch preparations of both attention kinds give the values of norm, rotation and
    append run one after the other, in the residual buffers and in the cache."""
    from vllm_omni_draft_amd import config, ops
    g = torch.Generator().manual_seed(5)
    n, qr, rk, dr, dims = 21, 20, 24, 10, 6
    pos, slot = i32(list(range(40, 40 + n))), i32([1] * n)
    bt = torch.zeros(2, 4, dtype=torch.int32, device=DEV)
    bt[1] = i32([3, 0, 2, 1])
    ql, kv = torch.randn(n, qr, generator=g), torch.randn(n, rk + dr, generator=g)
    qw, kw = torch.randn(qr, generator=g).to(cdt), torch.randn(rk, generator=g).to(cdt)
    f, mag = config.rotary_frequencies(dims, 1e4, {"factor": 4.0, "original": 32, "fast": 8.0, "slow": 1.0})
    rnd = cdt == torch.bfloat16
    # pieces
    q1 = ops.rmsnorm_parts(dev(ql), dev(qw), 1e-5, round_bf16=rnd)
    kv1 = dev(kv)
    kv1[:, :rk] = ops.rmsnorm_parts(dev(kv[:, :rk]), dev(kw), 1e-5, round_bf16=rnd)
    ops.rope_rows(kv1, pos, 1, 0, rk, dims, dev(f), mag)
    c1 = torch.zeros(4, 1, PAGE, rk + dr, dtype=cdt, device=DEV)
    ops.cache_append(kv1, None, c1, None, pos, slot, bt, 1, rk + dr, 0)
    # one launch
    q2, kv2, c2 = dev(ql), dev(kv), torch.zeros_like(c1)
    ops.latent_prep(q2, dev(qw), kv2, dev(kw), rk, dr, 1e-5, dims, dev(f), mag, c2, pos, slot, bt)
    assert torch.equal(q1, q2) and torch.equal(kv1, kv2) and torch.equal(c1, c2)
    # q and k normed over the whole projection, k and v appended
    H, G, dk, dv = 6, 3, 12, 20
    q, k, v = torch.randn(n, H * dk, generator=g), torch.randn(n, G * dk, generator=g), torch.randn(n, G * dv, generator=g)
    qnw, knw = torch.randn(H * dk, generator=g).to(cdt), torch.randn(G * dk, generator=g).to(cdt)
    qa, ka = ops.rmsnorm_parts(dev(q), dev(qnw), 1e-5), ops.rmsnorm_parts(dev(k), dev(knw), 1e-5)
    kc1, vc1 = torch.zeros(4, G, PAGE, dk, dtype=cdt, device=DEV), torch.zeros(4, G, PAGE, dv, dtype=cdt, device=DEV)
    ops.cache_append(ka, dev(v), kc1, vc1, pos, slot, bt, G, dk, dv)
    qb, kb, kc2, vc2 = dev(q), dev(k), torch.zeros_like(kc1), torch.zeros_like(vc1)
    ops.qk_norm_append(qb, dev(qnw), kb, dev(knw), dev(v), G, dk, dv, 1e-5, kc2, vc2, pos, slot, bt)
    assert torch.equal(qa, qb) and torch.equal(ka, kb) and torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
    assert rel(qb, N.rms_norm(q.double(), qnw.double(), 1e-5)) < 1e-6


@pytest.mark.parametrize("M,B,N_,K", [(1, 3, 7, 5), (5, 2, 130, 24), (40, 6, 16, 136)])
@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16])
def test_matmul_rows_batched(M, B, N_, K, wdt):
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(M + K)
    x, w = torch.randn(M, B, K, generator=g), torch.randn(B, N_, K, generator=g).to(wdt)
    xr = x.to(torch.bfloat16).double() if wdt == torch.bfloat16 else x.double()
    y = ops.matmul_rows_batched(dev(x), dev(w))
    assert rel(y, torch.einsum("mbk,bnk->mbn", xr, w.double())) < 2e-6


@pytest.mark.parametrize("C,taps", [(5, 4), (300, 3), (64, 1), (7, 7)])
def test_causal_conv_rows_in_portions(C, taps):
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(C)
    n = 23
    x, w, b = torch.randn(n, C, generator=g), torch.randn(C, taps, generator=g), torch.randn(C, generator=g)
    want = N.silu(N.short_conv(x.double(), w.double(), b.double(), {}))
    state = torch.full((3, max(taps - 1, 1), C), 7.0, device=DEV)        # stale: a new sequence must not read it
    cuts = [0, 1, 3, 4, 10, 12, n]                                        # portions of 1, 2, 1, 6, 2, 11 tokens
    outs = []
    for lo, hi in zip(cuts, cuts[1:]):
        # the sequence sits in slot 2, behind another entry's rows in slot 0 that must not leak in
        other = torch.randn(2, C, generator=g)
        xx = torch.cat([other, x[lo:hi]])
        rows = hi - lo
        o = ops.causal_conv_rows(dev(xx), dev(w), dev(b), state, i32([0, 1] + list(range(lo, hi))),
                                 i32([0, 0] + [2] * rows), i32([[0, 0, 2, 0], [2, 2, rows, lo]]))
        outs.append(o[2:])
    assert rel(torch.cat(outs), want) < 1e-6


@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C,H,taps", [(5, 3, 4), (256, 300, 1), (300, 8, 2), (1000, 32, 7), (513, 16, 8), (40, 4, 9)])
def test_convolution_and_steps_of_decoded_tokens_in_one_launch(C, H, taps, wdt):
    """A row an entry, contexts shorter and longer than the taps, beside others' rows in a stack with the step sizes' columns:
    outputs, moved tails, step sizes and decays are the bits of the launches apart (nine taps still take those); no argument of
    theirs may be missing."""
    import ctypes as Ct
    from tests.gpu_util import internal
    from vllm_omni_draft_amd import ops
    vp, i32_, i64_ = Ct.c_void_p, Ct.c_int, Ct.c_int64
    f = internal("sd_conv_steps_", i32_, vp, i64_, vp, vp, i32_, vp, vp, vp, vp, i32_, vp, i64_, i32_, i32_, i32_, i32_, vp, vp, vp, vp, vp,
                 i32_, vp)
    g = torch.Generator().manual_seed(C + taps)
    pos = [0, 1, taps - 1, taps, 50]
    R, ld = len(pos), C + H + 3
    stack = dev(torch.randn(R, ld, generator=g))
    w, b, dt_bias, a_log = (dev(torch.randn(*s, generator=g).to(wdt)) for s in ((C, taps), (C,), (H,), (H,)))
    tails = dev(torch.randn(R + 2, max(taps - 1, 1), C, generator=g))
    slots, entries = i32([4, 0, 6, 2, 3]), i32([[s, r, 1, p] for r, (s, p) in enumerate(zip([4, 0, 6, 2, 3], pos))])
    p = lambda t: None if t is None else t.data_ptr()
    for bias in (b, None):
        tail, out = tails.clone(), torch.empty(R, C, device=DEV)
        step, decay = torch.empty(R, H, device=DEV), torch.empty(R, H, device=DEV)
        args = [p(stack), ld, p(w), p(bias), int(wdt == torch.float32), p(tail), None, p(slots), p(entries), R, p(out), C, R, C, taps, 1,
                p(stack) + 4 * C, p(dt_bias), p(a_log), p(step), p(decay), H, ops._stream()]
        rows = i32(pos)
        args[6] = p(rows)
        assert f(*args) == 0
        tail2 = tails.clone()
        out2 = ops.causal_conv_rows(stack[:, :C].contiguous(), w, bias, tail2, i32(pos), slots, entries)
        step2, decay2 = ops.ssd_steps(stack[:, C:C + H].contiguous(), dt_bias, a_log)
        for got, want in ((out, out2), (tail, tail2), (step, step2), (decay, decay2)):
            assert torch.equal(got, want)
    for at in (0, 2, 5, 6, 7, 8, 10, 16, 17, 18, 19, 20):
        assert f(*[None if i == at else v for i, v in enumerate(args)]) == -1, at


def ssd_reference(x, B, C, dt, a_log, dt_bias, D, S):
    """x [T, H, P], B, C [T, G, N], dt [T, H]; S [H, N, P] changed in place."""
    T, H, P = x.shape
    G = B.shape[1]
    step = N.softplus(dt + dt_bias)
    y = torch.empty_like(x)
    for t in range(T):
        for h in range(H):
            g = h // (H // G)
            S[h] = torch.exp(-torch.exp(a_log[h]) * step[t, h]) * S[h] + step[t, h] * torch.outer(B[t, g], x[t, h])
            y[t, h] = S[h].T @ C[t, g] + D[h] * x[t, h]
    return y


@pytest.mark.parametrize("H,G,N_,P", [(2, 1, 8, 8), (6, 3, 20, 12), (4, 4, 48, 72), (1, 1, 130, 5)])
def test_ssd_steps_and_scan(H, G, N_, P):
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(H * 10 + N_)
    T = 37
    x, B, C = torch.randn(T, H * P, generator=g), torch.randn(T, G * N_, generator=g), torch.randn(T, G * N_, generator=g)
    dt = torch.randn(T, H, generator=g) * 2
    dt[3] = 40.0                                       # a large step: softplus is the identity there, no clamp
    a_log, dt_bias, D = torch.randn(H, generator=g), torch.randn(H, generator=g), torch.randn(H, generator=g)
    S = torch.zeros(H, N_, P, dtype=torch.float64)
    want = ssd_reference(x.double().view(T, H, P), B.double().view(T, G, N_), C.double().view(T, G, N_), dt.double(),
                         a_log.double(), dt_bias.double(), D.double(), S)
    step, decay = ops.ssd_steps(dev(dt), dev(dt_bias), dev(a_log))
    assert rel(step, N.softplus(dt.double() + dt_bias.double())) < 1e-6
    state = torch.full((3, H, N_, P), 5.0, device=DEV)  # stale
    outs = []
    cuts = [0, 2, 3, 20, T]
    for lo, hi in zip(cuts, cuts[1:]):
        outs.append(ops.decay_scan_rows(dev(C[lo:hi]), dev(B[lo:hi]), dev(x[lo:hi]), decay[lo:hi].contiguous(),
                                        step[lo:hi].contiguous(), dev(D), state, i32([[1, 0, hi - lo, lo]]), H, G,
                                        N_, P))
    assert rel(torch.cat(outs), want.reshape(T, -1)) < 2e-6
    assert rel(state[1], S) < 2e-6


@pytest.mark.parametrize("E,top,F,W,rows", [(4, 2, 24, 32, 9), (5, 3, 20, 40, 70), (1, 1, 8, 24, 3), (16, 1, 64, 48, 150),
                                            (7, 7, 10, 20, 5),
                                            # widths that are multiples of 32: bfloat16 takes the matrix-core kernels
                                            (8, 2, 96, 64, 100), (3, 1, 32, 32, 33), (6, 3, 160, 1056, 5),
                                            # many rows per expert: the matrix-core kernels take tiles of 128 rows
                                            (4, 2, 64, 160, 301), (2, 1, 32, 64, 700)])
@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16])
def test_routed_experts(E, top, F, W, rows, wdt):
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(E * 10 + top)
    x = torch.randn(rows, W, generator=g)
    if wdt == torch.bfloat16:
        x = x.to(wdt).float()
    Wt = {"router": (torch.randn(E, W, generator=g) * W ** -0.5).to(wdt)}    # (logits of order one: no tied scores)
    for e in range(E):
        Wt[f"e{e}.gate"], Wt[f"e{e}.up"] = (torch.randn(F, W, generator=g) * W ** -0.5).to(wdt), \
            (torch.randn(F, W, generator=g) * W ** -0.5).to(wdt)
        Wt[f"e{e}.down"] = (torch.randn(W, F, generator=g) * F ** -0.5).to(wdt)
    mlp = {"router": {"experts": E, "top": top}}
    want = N.routed_experts(x.double(), {k: v.double() for k, v in Wt.items()}, mlp)
    logits = ops.matmul_rows(dev(x), dev(Wt["router"]))
    sel_e, sel_w = ops.moe_route(logits, top)
    s = torch.sigmoid(x.double() @ Wt["router"].double().T)
    assert torch.equal(sel_e.cpu().long().sort(1).values, torch.topk(s, top).indices.sort(1).values)
    gu = torch.stack([torch.cat([Wt[f"e{e}.gate"], Wt[f"e{e}.up"]]) for e in range(E)])
    dn = torch.stack([Wt[f"e{e}.down"] for e in range(E)])
    out = ops.moe_experts(dev(x), sel_e, sel_w, dev(gu), dev(dn))
    assert rel(out.sum(1), want) < (2e-6 if wdt == torch.float32 else 1e-2)
    # a row's results do not depend on the rows around it
    one = ops.moe_experts(dev(x[:1]), sel_e[:1].contiguous(), sel_w[:1].contiguous(), dev(gu), dev(dn))
    if wdt == torch.float32:
        assert torch.equal(one[0], out[0])
    else:       # (a few assignments run as matrix-vector products, many as tiles: bfloat16 rounding apart)
        assert rel(one[0], out[0]) < 1e-2


@pytest.mark.parametrize("E,K,top,wdt", [(5, 40, 3, torch.float32), (16, 1000, 2, torch.bfloat16), (130, 64, 7, torch.float32)])
def test_router_product_and_choice_in_one_launch(E, K, top, wdt):
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(E)
    x, w = torch.randn(9, K, generator=g), (torch.randn(E, K, generator=g) * K ** -0.5).to(wdt)
    xr = x.to(torch.bfloat16).double() if wdt == torch.bfloat16 else x.double()
    e, sw, logits = ops.moe_route_rows(dev(x), dev(w), top)
    want = xr @ w.double().T
    assert rel(logits, want) < 2e-6
    tk = torch.topk(torch.sigmoid(want), top)
    assert torch.equal(e.cpu().long(), tk.indices) and rel(sw, tk.values) < 1e-6
    e1, sw1, l1 = ops.moe_route_rows(dev(x[4:5]), dev(w), top)          # a row alone: the same bits
    assert torch.equal(l1[0], logits[4]) and torch.equal(e1[0], e[4]) and torch.equal(sw1[0], sw[4])


def test_router_other_scores():
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(1)
    z = torch.randn(6, 11, generator=g)
    z[2, 4] = z[2, 9] = 3.0                            # equals: the lower index goes first
    e, w = ops.moe_route(dev(z), 3, "softmax", True)
    p = torch.softmax(z.double(), 1)
    top = torch.topk(p, 3)
    assert rel(w, top.values / top.values.sum(1, keepdim=True)) < 1e-6
    assert e[2].tolist()[:2] == [4, 9]


def test_postnorm_residual():
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(2)
    x, a, b, w = (torch.randn(5, 70, generator=g), torch.randn(15, 70, generator=g), torch.randn(5, 70, generator=g),
                  torch.randn(70, generator=g))
    xd = dev(x)
    ops.postnorm_residual(xd, dev(a), dev(w), 1e-5, n_a=3, sa=0.6, b=dev(b), sb=0.5)
    y = 0.6 * a.double().view(5, 3, 70).sum(1) + 0.5 * b.double()
    assert rel(xd, x.double() + N.rms_norm(y, w.double(), 1e-5)) < 1e-6


@pytest.mark.parametrize("W", [255, 257, 512, 513, 1024, 1025, 2047, 2048, 2049, 4100])
@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16])
def test_rows_of_more_columns_than_a_thread_holds(W, wdt):
    """Residual update, embedding and the norms of both preparations at the edges of one, two, four and eight columns a thread (256 a
    workgroup), and beyond, where a second batch of columns is read and the norms read them twice; a float32 sum of 4100 products in strands
    of 17 is within 1e-6 of a float64 one."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(W)
    rn = lambda *shape: torch.randn(*shape, generator=g)
    n, rnd = 3, wdt == torch.bfloat16
    x, a, b, w = rn(n, W), rn(2 * n, W), rn(n, W), rn(W).to(wdt)
    xd = dev(x)
    ops.postnorm_residual(xd, dev(a), dev(w), 1e-5, n_a=2, sa=0.6, b=dev(b), sb=0.5)
    y = 0.6 * a.double().view(n, 2, W).sum(1) + 0.5 * b.double()
    assert rel(xd, x.double() + N.rms_norm(y, w.double(), 1e-5)) < 1e-6
    table, bg, toks = rn(20, W).to(wdt), rn(8, W).to(wdt), [3, 19, 0]
    e, e_b = ops.embed_hashed(i32(toks), dev(table), 2.5, i32([-1] + toks[:-1]), dev(bg), 31, 7, bf16_copy=True)
    rows = [7] + [(p * 31 + t * 7) % 7 for p, t in zip(toks, toks[1:])]
    assert rel(e, table.double()[toks] * 2.5 + bg.double()[rows]) < 1e-6 and torch.equal(e_b, e.to(torch.bfloat16))
    pos, slot, bt = i32([14, 15, 16]), i32([0] * n), i32([[1, 0]])
    kv, dr = rn(n, W + 8), 8
    f = torch.zeros(dr // 2, dtype=torch.float64)       # (no rotation)
    kvd, xq, cache = dev(kv), dev(x), torch.zeros(2, 1, PAGE, W + dr, dtype=wdt, device=DEV)
    ops.latent_prep(xq, dev(w), kvd, dev(w), W, dr, 1e-5, dr, dev(f), 1.0, cache, pos, slot, bt)
    assert torch.equal(xq, ops.rmsnorm_parts(dev(x), dev(w), 1e-5, round_bf16=rnd))
    assert torch.equal(kvd[:, :W], ops.rmsnorm_parts(dev(kv[:, :W]), dev(w), 1e-5, round_bf16=rnd))
    assert torch.equal(kvd[:, W:].cpu(), kv[:, W:]) and torch.equal(cache[[1, 1, 0], 0, [14, 15, 0]], kvd.to(wdt))
    q, k, v = dev(x), dev(b), dev(a[:n])
    kc, vc = (torch.zeros(2, 1, PAGE, W, dtype=wdt, device=DEV) for _ in range(2))
    ops.qk_norm_append(q, dev(w), k, dev(w), v, 1, W, W, 1e-5, kc, vc, pos, slot, bt)
    assert rel(q, N.rms_norm(x.double(), w.double(), 1e-5)) < 1e-6 and rel(k, N.rms_norm(b.double(), w.double(), 1e-5)) < 1e-6
    assert torch.equal(kc[[1, 1, 0], 0, [14, 15, 0]], k.to(wdt)) and torch.equal(vc[[1, 1, 0], 0, [14, 15, 0]], v.to(wdt))


# ------------------------------------------------------------------ whole models
@pytest.mark.parametrize("shape", list(SHAPES))
def test_prompt_logits_match_the_plain_model(shape):
    cfg = SHAPES[shape]
    st, eng = build(cfg)
    toks = prompt(cfg, 61)
    lo = []
    want = oracle_logits(cfg, st, toks, lo)
    got, trace = eng.step([("a", toks, list(range(len(toks))))], layer_out=True)
    for i, x in enumerate(lo):
        assert rel(trace[i], x) < 3e-6, f"residual after layer {i}"
    assert rel(got, want) < 3e-6


@pytest.mark.parametrize("shape,tiled", [("two_kinds", False), ("odd", False), ("aligned", True), ("aligned", False),
                                         ("wide", False)])
def test_bfloat16_serving_stays_close(shape, tiled):
    cfg = SHAPES[shape]
    st, eng = build(cfg, torch.bfloat16, tiled=tiled)
    toks = prompt(cfg, 50, 1)
    want = oracle_logits(cfg, st, toks)
    got = eng.step([("a", toks, list(range(len(toks))))])
    # (a token whose router scores lie within bfloat16 rounding of each other may take another
    # expert than the plain model, and the tokens behind it feel that: most rows are close)
    rows = sorted(rel(got[r], want[r]) for r in range(len(toks)))
    assert rows[len(rows) // 2] < 2e-2 and rows[int(len(rows) * 0.9)] < 6e-2, rows[-5:]


@pytest.mark.parametrize("shape,dtype,tiled", [("two_kinds", torch.float32, True), ("odd", torch.float32, True),
                                               ("ones", torch.float32, True), ("wide", torch.float32, True),
                                               ("odd", torch.bfloat16, False), ("aligned", torch.bfloat16, True)])
def test_cut_anywhere_batched_anyhow(shape, dtype, tiled):
    """The logits of a position are the same however its prompt was cut into steps (down to two
    tokens and to single decoded tokens), whatever else shares the batch and whichever slot and
    pages the request got."""
    cfg = SHAPES[shape]
    st, eng = build(cfg, dtype, tiled=tiled)
    pa, pb, pc = prompt(cfg, 57, 1), prompt(cfg, 34, 2), prompt(cfg, 9, 3)
    whole = {}
    for name, p in (("a", pa), ("b", pb), ("c", pc)):
        whole[name] = eng.step([(name, p, list(range(len(p))))])
        eng.finish(name)
    exact = dtype == torch.float32 or not tiled

    def same(x, y, what):
        if exact:
            assert torch.equal(x, y), what
        else:
            assert rel(x, y) < 1e-2, what
    # token by token
    eng.step([("pad", prompt(cfg, 20, 9), [])])       # another slot and other pages than before
    got = torch.cat([eng.step([("a", [t], [0])]) for t in pa])
    same(got, whole["a"], "token by token")
    eng.finish("a")
    # portions of changing size, down to two tokens, beside other requests' portions and single tokens
    cuts_a = [0, 2, 4, 17, 19, 32, 33, 48, 57]
    cuts_b = [0, 16, 17, 18, 20, 34]
    got_a, got_b, got_c = [], [], []
    ia = ib = ic = 0
    while ia < len(cuts_a) - 1 or ib < len(cuts_b) - 1 or ic < len(pc):
        entries, kinds = [], []
        if ia < len(cuts_a) - 1:
            lo, hi = cuts_a[ia], cuts_a[ia + 1]
            entries.append(("a", pa[lo:hi], list(range(hi - lo))))
            kinds.append(got_a)
            ia += 1
        if ic < len(pc):
            entries.append(("c", pc[ic:ic + 1], [0]))
            kinds.append(got_c)
            ic += 1
        if ib < len(cuts_b) - 1:
            lo, hi = cuts_b[ib], cuts_b[ib + 1]
            entries.append(("b", pb[lo:hi], list(range(hi - lo))))
            kinds.append(got_b)
            ib += 1
        out = eng.step(entries)
        at = 0
        for (_, t, _), dst in zip(entries, kinds):
            dst.append(out[at:at + len(t)])
            at += len(t)
    same(torch.cat(got_a), whole["a"], "portions of a")
    same(torch.cat(got_b), whole["b"], "portions of b")
    same(torch.cat(got_c), whole["c"], "single tokens of c")


def test_slots_and_pages_are_used_again():
    cfg = SHAPES["two_kinds"]
    st, eng = build(cfg, max_seqs=3, max_tokens=12 * PAGE, max_seq_len=6 * PAGE)
    ref = {}
    for r in range(10):
        p = prompt(cfg, 20 + 7 * (r % 5), r)
        ref[r] = (p, oracle_logits(cfg, st, p)[-1])
    live, nxt, done = {}, 0, 0
    while done < 10:
        while len(live) < 3 and nxt < 10:
            live[nxt] = 0
            nxt += 1
        entries = []
        for r in list(live):
            p = ref[r][0]
            n = min(len(p) - live[r], 13 if r % 2 else 1000)
            entries.append((str(r), p[live[r]:live[r] + n], [n - 1] if live[r] + n == len(p) else []))
            live[r] += n
        out = eng.step(entries)
        at = 0
        for rid, _, want in entries:
            if want:
                assert rel(out[at], ref[int(rid)][1]) < 3e-6, rid
                at += 1
                eng.finish(rid)
                del live[int(rid)]
                done += 1
    assert eng.free_slots == 3 and eng.cache.allocator.num_free == 12


def test_a_step_larger_than_a_pass():
    cfg = SHAPES["two_kinds"]
    st, eng = build(cfg, max_rows=16)
    pa, pb = prompt(cfg, 45, 4), prompt(cfg, 21, 5)
    out = eng.step([("a", pa, [0, 15, 16, 44]), ("b", pb, [20])])
    assert eng.passes == 5
    wa, wb = oracle_logits(cfg, st, pa), oracle_logits(cfg, st, pb)
    assert rel(out[:4], wa[[0, 15, 16, 44]]) < 3e-6 and rel(out[4], wb[20]) < 3e-6


def test_page_tables_are_there_for_any_stream_after_a_refused_step():
    """A step refused at its second entry, under a stream that is busy: the first entry's pages are in the table for a step under another
    stream; and so are those that SeqCache.ensure_capacity took."""
    from vllm_omni_draft_amd.kv_cache import OutOfPages
    cfg = SHAPES[sorted(SHAPES)[0]]
    toks = prompt(cfg, 200)
    want = build(cfg)[1].step([("a", toks, range(200))])
    _, eng = build(cfg)
    eng.step([("pad", prompt(cfg, 40, 9), [])])        # (the pages of "a" are not the table's zeros)
    busy = torch.cuda.Stream()
    with torch.cuda.stream(busy):
        torch.cuda._sleep(50_000_000)
        with pytest.raises(OutOfPages):
            eng.step([("a", toks, range(200)), ("b", [1] * 5000, [])])
    assert busy.query()
    assert torch.equal(eng.step([("a", toks, range(200))]), want)
    slot = eng.seqs["a"].slot
    with torch.cuda.stream(busy):
        torch.cuda._sleep(50_000_000)
        eng.cache.ensure_capacity(slot, 500)
    assert eng.cache.block_tables[slot, :32].tolist() == eng.cache.pages_of(slot)


@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_norm_and_router_in_one_launch_have_the_bits_of_two(shape):
    """More than 256 rows (the norm, then the router) against pieces of 1, 64, 255 and 256 rows (one launch)."""
    cfg = SHAPES[shape]
    st, eng = build(cfg, torch.float32)
    toks = prompt(cfg, 577)
    want = eng.step([("a", toks, range(577))])
    eng.finish("a")
    at, got = 0, []
    for n in (1, 64, 1, 255, 256):
        got.append(eng.step([("b", toks[at:at + n], range(n))]))
        at += n
    assert at == 577 and torch.equal(torch.cat(got), want)


@pytest.mark.parametrize("width,n", [(2047, 17), (2048, 16), (2049, 33), (2112, 5), (4100, 17)])
@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16])
def test_norm_and_router_of_wide_rows_in_one_launch_have_the_bits_of_two(width, n, wdt):
    """Rows of one load ahead and of more (2048 columns), a wave's second and third expert, weights of both types: twelve prompts of 24
    tokens in one pass (288 rows: two launches) against six at a time (144 rows: one)."""
    cfg = model_cfg([latent(mlp=experts(n, 3, 8)), parallel(mlp=experts(n, 2, 8))], width=width)
    _, eng = build(cfg, wdt, max_seqs=12)
    step = lambda ids: eng.step([(f"r{i}", prompt(cfg, 24, i), range(24)) for i in ids])
    want = step(range(12))
    for i in range(12):
        eng.finish(f"r{i}")
    assert torch.equal(torch.cat([step(range(6)), step(range(6, 12))]), want)


def test_a_far_token_through_the_recurrence_and_a_kept_first_token():
    """The recurrence's decay made (almost) one, so that a token 150 positions back still carries
    weight; and a kept first token whose key every later query finds."""
    cfg = model_cfg([parallel(window=4, keep_first=1, mlp=None)], bigram=None)
    st = N.random_tensors(cfg, 5)
    st["l0.mix.right.A_log"] = torch.full_like(st["l0.mix.right.A_log"], -9.0)
    st["l0.mix.left.q.norm"] *= 4
    from vllm_omni_draft_amd import config, weights
    from vllm_omni_draft_amd.seq_engine import SeqEngine, SeqEngineConfig
    mc = config.naburax_config(cfg)
    eng = SeqEngine(weights.seq_from_state_dict(mc, st, DEV, torch.float32), SeqEngineConfig(max_seqs=2, max_tokens=512))
    base, other = prompt(cfg, 160, 6), prompt(cfg, 160, 6)
    other[0] = (base[0] + 1) % cfg["vocab"]           # only the first token differs
    wa, wb = oracle_logits(cfg, st, base), oracle_logits(cfg, st, other)
    assert rel(wa[-1], wb[-1]) > 1e-3                  # ... and the last position still feels it
    ga = eng.step([("a", base[:100], [])])
    ga = torch.cat([eng.step([("a", [t], [0])]) for t in base[100:]])
    gb = eng.step([("b", other, [159])])
    assert rel(ga[-1], wa[-1]) < 3e-6 and rel(gb[0], wb[-1]) < 3e-6


def test_long_decoding():
    cfg = SHAPES["odd"]
    st, eng = build(cfg)
    toks = prompt(cfg, 230, 7)
    want = oracle_logits(cfg, st, toks)
    eng.step([("a", toks[:10], [])])
    got = torch.cat([eng.step([("a", [t], [0])]) for t in toks[10:]])
    assert rel(got, want[10:]) < 5e-6
    assert rel(got[-1], want[-1]) < 5e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decode_steps_replayed_as_graphs(dtype):
    cfg = SHAPES["aligned"]
    st, plain = build(cfg, dtype, use_graph=False)
    _, graphed = build(cfg, dtype, use_graph=True)
    ps = [prompt(cfg, n, i) for i, n in enumerate((7, 19, 3))]
    for eng in (plain, graphed):
        eng.step([(str(i), p[:-1], []) for i, p in enumerate(ps)])
    nxt = [p[-1] for p in ps]
    for step in range(12):
        a = plain.step([(str(i), [t], [0]) for i, t in enumerate(nxt)])
        b = graphed.step([(str(i), [t], [0]) for i, t in enumerate(nxt)])
        assert torch.equal(a, b), step
        nxt = a.argmax(1).tolist()
    assert graphed.graph_replays >= 10


def test_greedy_generation_through_worker_and_scheduler():
    from vllm_omni_draft_amd import config, weights
    from vllm_omni_draft_amd.scheduler import SpecDecodeScheduler
    from vllm_omni_draft_amd.seq_engine import SeqWorker, SeqWorkerConfig
    cfg = SHAPES["two_kinds"]
    st = N.random_tensors(cfg, 3)
    mc = config.naburax_config(cfg, {k: tuple(v.shape) for k, v in st.items()})
    worker = SeqWorker(SeqWorkerConfig(weights.seq_from_state_dict(mc, st, DEV, torch.float32), max_num_seqs=3,
                                       max_model_len=128))
    worker.init_device()
    worker.load_model()
    sched = SpecDecodeScheduler.for_worker(worker)
    prompts = [prompt(cfg, n, i) for i, n in enumerate((5, 33, 1, 18, 64, 9, 2))]   # more requests than slots
    reqs = sched.generate(prompts, max_tokens=10)
    assert worker.engine.free_slots == 3
    t64 = f64(st)
    for p, r in zip(prompts, reqs):
        assert len(r.output_token_ids) == 10 and r.finish_reason == "length"
        seq = N.Sequence(len(cfg["layers"]))
        logits = N.forward(cfg, t64, p, seq)[-1]
        for tok in r.output_token_ids:
            best = int(logits.argmax())
            if tok != best:                      # legitimate only at a near-tie of the plain model
                top = torch.topk(logits, 2).values
                assert (top[0] - top[1]) / logits.std() < 1e-4
                break
            logits = N.forward(cfg, t64, [tok], seq)[-1]


@pytest.mark.parametrize("H,G,dk,dv", [(4, 1, 128, 128), (6, 2, 128, 128), (16, 1, 576, 512), (5, 1, 576, 512)])
@pytest.mark.parametrize("window,keep", [(5000, 0), (100, 0), (70, 3), (33, 70), (1, 1)])
def test_rows_softmax_attention_against_float64(H, G, dk, dv, window, keep):
    """Portions that start anywhere, lengths at the edges of a workgroup's tokens and of stages of 64 keys, kept tokens
    before and inside the window, rows of caches whose pages lie anywhere and hold NaN behind the portion: against
    float64, with the bound of the kernel on the vector pipe (sums of f32 products)."""
    from vllm_omni_draft_amd import ops
    latent = dv == 512
    g = torch.Generator(device="cuda").manual_seed(H + window)
    runs = [(0, 1), (0, 65), (130, 64), (63, 2), (15, 17)]
    lens = [p + n for p, n in runs]
    pages = (max(lens) + 15) // 16
    perm = torch.randperm(len(runs) * pages, generator=g, device="cuda").to(torch.int32)
    bt = perm.view(len(runs), pages)
    kc = torch.randn(len(runs) * pages, G, 16, dk, generator=g, device="cuda").to(torch.bfloat16)
    vc = None if latent else torch.randn(len(runs) * pages, G, 16, dv, generator=g, device="cuda").to(torch.bfloat16)
    rows = sum(n for _, n in runs)
    q = torch.randn(rows, H * dk, generator=g, device="cuda") * 2
    ents, row, want = [], 0, []
    for s, (p0, n) in enumerate(runs):
        ents.append([s, row, n, p0])
        m = p0 + n
        for c in (kc,) if latent else (kc, vc):
            c[bt[s, m // 16:].long()[1:] if m % 16 else bt[s, m // 16:].long()] = float("nan")
            if m % 16:
                c[bt[s, m // 16].long(), :, m % 16:] = float("nan")
        k = kc[bt[s].long()].transpose(1, 2).reshape(-1, G, dk)[:m].double()
        v = k[..., :dv] if latent else vc[bt[s].long()].transpose(1, 2).reshape(-1, G, dv)[:m].double()
        qq = q[row:row + n].double().view(n, H, dk)
        i = torch.arange(p0, m, device="cuda")[:, None]
        j = torch.arange(m, device="cuda")[None, :]
        seen = (j <= i) & ((i - j < window) | (j < keep))
        for t in range(0, n, 64):
            o = []
            for h in range(H):
                sc = qq[t:t + 64, h] @ k[:, h // (H // G)].T * dk ** -0.5
                sc = sc.masked_fill(~seen[t:t + 64], float("-inf"))
                o.append(torch.softmax(sc, -1) @ v[:, h // (H // G)])
            want.append(torch.cat(o, 1))
        row += n
    got = ops.rows_softmax_attention(q, kc, vc, bt.contiguous(), i32(ents), H, G, dk, dv, window, keep, dk ** -0.5)
    off = ((got.double() - torch.cat(want)).norm() / torch.cat(want).norm()).item()
    assert off < 3e-6, off


@pytest.mark.parametrize("F,W", [(8, 8), (40, 504), (2040, 512), (24, 2048), (2056, 2064), (13 * 8, 4104)])
@pytest.mark.parametrize("act", ["silu", "relu2"])
def test_moe_experts_of_a_few_assignments(F, W, act):
    """Rows and matrices of less than 512 columns, at the edges of the 2048 whose weights and values are asked for ahead, and of more; column
    counts that leave waves without work; an index of no expert among the chosen (its row is left as it was)."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator(device="cuda").manual_seed(F * W)
    n, E, top, mats = 5, 3, 2, 1 if act == "relu2" else 2
    x = torch.randn(n, W, generator=g, device="cuda")
    gu = (torch.randn(E, mats * F, W, generator=g, device="cuda") * W ** -0.5).to(torch.bfloat16)
    dn = (torch.randn(E, W, F, generator=g, device="cuda") * F ** -0.5).to(torch.bfloat16)
    sel = torch.tensor([[0, 1], [2, 0], [1, 2], [2, 1], [0, E]], dtype=torch.int32, device="cuda")
    w = torch.rand(n, top, generator=g, device="cuda") + 0.5
    out = ops.moe_experts(x, sel, w, gu, dn, True, act)
    for r in range(n):
        for t in range(top):
            e = int(sel[r, t])
            if e >= E:
                continue
            h = (gu[e].double() @ x[r].to(torch.bfloat16).double()) * w[r, t].double()
            a = torch.relu(h) ** 2 if mats == 1 else torch.nn.functional.silu(h[:F]) * h[F:]
            # (an activation beside a rounding edge of bf16 may round the other way: 2^-8 of it at most)
            assert rel(out[r, t], dn[e].double() @ a.to(torch.bfloat16).double()) < 2 ** -8, (r, t)


@pytest.mark.parametrize("E,n", [(1, 9), (3, 512), (3, 513), (1024, 700), (1025, 700), (2050, 1300)])
def test_assignments_grouped_by_expert(E, n):
    """One expert, groups at the edges of the 1024 assignments that a trip takes and of the 1024 experts counted at a time, experts that
    nobody chose, and indices of no expert (their rows are left): rows grouped with others against eight rows at a time, whose
    assignments are not grouped."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator(device="cuda").manual_seed(E + n)
    F = W = 16
    x = torch.randn(n, W, generator=g, device="cuda")
    gu, dn = (torch.randn(E, r, W, generator=g, device="cuda") for r in (2 * F, W))
    sel = torch.randint(0, E + 1, (n, 2), generator=g, device="cuda").to(torch.int32)
    sel[n // 2:, 0] = E - 1
    w = torch.rand(n, 2, generator=g, device="cuda")
    out = ops.moe_experts(x, sel, w, gu, dn)
    few = torch.cat([ops.moe_experts(x[i:i + 8], sel[i:i + 8], w[i:i + 8], gu, dn) for i in range(0, n, 8)])
    assert torch.equal(out[sel < E], few[sel < E])


@pytest.mark.parametrize("n,E,K", [(769, 5, 70), (770, 16, 2048), (771, 24, 513), (772, 2048, 64), (770, 2049, 64), (1537, 5, 70), (513, 17, 130),
                                   (771, 9, 2048)])
@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16])
def test_router_of_four_rows_a_workgroup_has_the_bits_of_one(n, E, K, wdt):
    """Row counts that leave one to four rows to the last workgroup, fewer and more experts than waves, the most and one more than that
    share a workgroup's LDS; gates, a bias, a correction, both scores: against the same rows 250 at a time, one a workgroup."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator(device="cuda").manual_seed(n + E)
    x = torch.randn(n, K, generator=g, device="cuda")
    w, wg = (torch.randn(r, K, generator=g, device="cuda").to(wdt) for r in (E, 3))
    c = torch.randn(E, generator=g, device="cuda")
    calls = [lambda t: ops.moe_route_rows_gated(t, w, 2, "softmax", True, 1e-3, 1.5, wg), lambda t: ops.moe_route_rows_biased(t, w, c, 3),
             lambda t: ops.moe_route_rows_corrected(t, w, c, 2, "sigmoid")]
    for f in calls:
        for got, few in zip(f(x), zip(*[f(x[i:i + 250]) for i in range(0, n, 250)])):
            assert torch.equal(got, torch.cat(few))


@pytest.mark.parametrize("lens,C", [([1, 2, 3, 5, 100, 4, 13], 300), ([127, 1], 257), ([126, 3], 64), ([1] * 130, 40)])
@pytest.mark.parametrize("wdt,bias", [(torch.float32, True), (torch.bfloat16, False)])
def test_four_rows_a_thread_of_a_convolution_have_the_bits_of_one(lens, C, wdt, bias):
    """128 rows and more (four taps): portions that begin and end inside a thread's four rows, shorter than the taps, alone in it, with the
    inputs kept before them and without, and a last thread of one to four rows; against every portion by itself, outputs and kept inputs."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + C)
    n, E = sum(lens), len(lens)
    x, w = torch.randn(n, C, generator=g, device="cuda"), torch.randn(C, 4, generator=g, device="cuda").to(wdt)
    b = torch.randn(C, generator=g, device="cuda").to(wdt) if bias else None
    start = [(0, 7, 1, 2)[e % 4] for e in range(E)]
    kept = torch.randn(E, 3, C, generator=g, device="cuda")
    pos = [start[e] + i for e in range(E) for i in range(lens[e])]
    slot = [e for e in range(E) for _ in range(lens[e])]
    rows = [sum(lens[:e]) for e in range(E)]
    one, all_ = kept.clone(), kept.clone()
    got = ops.causal_conv_rows(x, w, b, all_, i32(pos), i32(slot), i32([[e, rows[e], lens[e], start[e]] for e in range(E)]))
    for e in range(E):
        s = slice(rows[e], rows[e] + lens[e])
        alone = ops.causal_conv_rows(x[s].contiguous(), w, b, one, i32(pos[s]), i32(slot[s]), i32([[e, 0, lens[e], start[e]]]))
        assert torch.equal(got[s], alone), e
    assert torch.equal(all_, one)


@pytest.mark.parametrize("E,F,W,n", [(4, 96, 160, 100), (3, 64, 128, 63), (2, 160, 96, 300), (5, 320, 64, 200)])
@pytest.mark.parametrize("act,scale_input", [("silu", True), ("silu", False), ("relu2", False)])
def test_moe_experts_of_many_rows_have_the_bits_of_few(E, F, W, n, act, scale_input):
    """Groups at the edges of the tiles of 64 rows, an expert that nobody chose and one that most did, columns and k that
    end inside a tile: the products through LDS against those of the kernel that converts f32 rows itself, bit for bit."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator(device="cuda").manual_seed(E * n)
    x = torch.randn(n, W, generator=g, device="cuda")
    mats = 1 if act == "relu2" else 2
    gu = (torch.randn(E, mats * F, W, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
    dn = (torch.randn(E, W, F, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
    sel_w = torch.rand(n, 2, generator=g, device="cuda")
    for full in (n, 64, 65, 1):   # rows whose first choice is expert 0; the last expert is never chosen
        sel = torch.randint(1, max(E - 1, 2), (n, 2), generator=g, device="cuda", dtype=torch.int32)
        sel[:full, 0] = 0
        a = ops.moe_experts(x, sel, sel_w, gu, dn, scale_input, act, bf16_copy=True)
        assert torch.equal(a, ops.moe_experts(x, sel, sel_w, gu, dn, scale_input, act)), full


@pytest.mark.parametrize("act", ["silu", "relu2"])
def test_moe_experts_in_tiles_of_192_rows_have_the_bits_of_few(act):
    """112 and more assignments an expert over 384 and more blocks: groups at the edges of the tiles of 192 rows and of their
    pairs of 16, columns and k that end inside a tile."""
    from vllm_omni_draft_amd import ops
    E, F, W, n = 4, 12320, 96, 300
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn(n, W, generator=g, device="cuda")
    gu = (torch.randn(E, (1 if act == "relu2" else 2) * F, W, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
    dn = (torch.randn(E, W, F, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
    sel_w = torch.rand(n, 2, generator=g, device="cuda")
    for full in (n, 192, 193, 32, 17):   # assignments of expert 0; the last expert is never chosen
        sel = torch.randint(1, E - 1, (n, 2), generator=g, device="cuda", dtype=torch.int32)
        sel[:full, 0] = 0
        a = ops.moe_experts(x, sel, sel_w, gu, dn, True, act, bf16_copy=True)
        assert torch.equal(a, ops.moe_experts(x, sel, sel_w, gu, dn, True, act)), full


@pytest.mark.parametrize("act", ["silu", "relu2"])
def test_moe_experts_in_tall_tiles_of_many_experts(act):
    """The same where the rule takes tall tiles: 128 assignments an expert over 64 experts, columns and k that end inside a
    tile of either product, groups of one to six tall tiles."""
    import ctypes as C
    from tests.gpu_util import internal
    from vllm_omni_draft_amd import ops
    E, F, W, n = 64, 552, 416, 4096
    tall = internal("sd_moe_tall_", C.c_bool, *[C.c_int] * 5)
    assert tall(2 * n, E, F, W, 0 if act == "silu" else 1)
    g = torch.Generator(device="cuda").manual_seed(8)
    x = torch.randn(n, W, generator=g, device="cuda")
    gu = (torch.randn(E, (1 if act == "relu2" else 2) * F, W, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
    dn = (torch.randn(E, W, F, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
    sel_w = torch.rand(n, 2, generator=g, device="cuda")
    for full in (1000, 193, 192, 17):   # assignments of expert 0; the last expert is never chosen
        sel = torch.randint(1, E - 1, (n, 2), generator=g, device="cuda", dtype=torch.int32)
        sel[:full, 0] = 0
        a = ops.moe_experts(x, sel, sel_w, gu, dn, True, act, bf16_copy=True)
        assert torch.equal(a, ops.moe_experts(x, sel, sel_w, gu, dn, True, act)), full


@pytest.mark.parametrize("H,G,dk,dv,maps", [(16, 1, 576, 512, 1), (8, 1, 584, 8, 1), (6, 2, 128, 128, 1), (12, 2, 256, 40, 2)])
@pytest.mark.parametrize("extras", [False, True])
def test_decode_attention_from_lds_against_float64(H, G, dk, dv, maps, extras):
    """The cut launch of a bf16 cache whose tiles lie in LDS: contexts at the edges of tiles of 64 keys, groups of four heads
    that are not full, values that are part of the key rows (G = 1), kept tokens behind a window; sinks, capped scores and
    chunks.  f32 sums of up to 1024 products against float64."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(H + dk)
    pos = [0, 63, 64, 150, 199]
    R, nb = len(pos), 13
    kc = torch.randn(R * nb, G * maps, 16, dk, generator=g).to(torch.bfloat16)
    vc = None if G == 1 else torch.randn(R * nb, G, 16, dv, generator=g).to(torch.bfloat16)
    bt = torch.randperm(R * nb, generator=g).view(R, nb)
    q = torch.randn(R, H * maps * dk, generator=g)
    window, keep, chunk, cap = (100, 3, 0, 0.0) if not extras else (0, 0, 160, 5.0)
    sinks = torch.randn(H * maps, generator=g) if extras else None
    if maps > 1:
        got = ops.multimap_softmax_attention(dev(q), kc.cuda(), vc.cuda(), i32(pos), i32(list(range(R))), bt.int().cuda(), H, G, maps, dk,
                                             dv, dk ** -0.5, window, keep, chunk, cap, None if sinks is None else dev(sinks))
    else:
        got = ops.masked_softmax_attention(dev(q), kc.cuda(), None if vc is None else vc.cuda(), i32(pos), i32(list(range(R))),
                                           bt.int().cuda(), H, G, dk, dv, dk ** -0.5, window, keep, chunk, cap,
                                           None if sinks is None else dev(sinks))
    want = torch.zeros(R, H, maps, dv, dtype=torch.float64)
    for r, i in enumerate(pos):
        lo = max(i - window + 1, 0) if window else 0
        lo = max(lo, i - i % chunk) if chunk else lo
        js = torch.tensor(sorted(set(range(min(keep, lo))) | set(range(lo, i + 1))))
        for h in range(H):
            for m in range(maps):
                gr = h // (H // G)
                k = kc[bt[r][js // 16], gr * maps + m, js % 16].double()
                v = k[:, :dv] if vc is None else vc[bt[r][js // 16], gr, js % 16].double()
                s = k @ q[r].view(H, maps, dk)[h, m].double() * dk ** -0.5
                s = cap * torch.tanh(s / cap) if cap else s
                if sinks is not None:
                    s = torch.cat([s, sinks.view(H, maps)[h, m].double().view(1)])
                    v = torch.cat([v, torch.zeros(1, dv, dtype=torch.float64)])
                want[r, h, m] = torch.softmax(s, 0) @ v
    off = ((got.cpu().double() - want.view(R, -1)).norm() / want.norm()).item()
    assert off < 3e-6, off


@pytest.mark.parametrize("H,G,dk,dv,maps", [(16, 1, 576, 512, 1), (7, 1, 576, 512, 1), (6, 2, 128, 128, 1), (4, 2, 256, 256, 1), (8, 2, 32, 256, 1),
                                           (12, 2, 256, 40, 2)])
def test_decode_attention_from_lds_sums_in_the_order_of_the_general_kernel(H, G, dk, dv, maps):
    """The same bits as over an f32 cache of the same values, which the general kernel takes: parts of the channels and shares of
    a tile's keys are added in one order in both.  Key rows of whole pieces of 32 channels are cut alike in either type; an
    infinite key and one that is no number are among them; scores that lose with distance, and gated heads."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator().manual_seed(H + dk)
    pos = [0, 2, 63, 64, 150, 199]
    R, nb = len(pos), 13
    kc = torch.randn(R * nb, G * maps, 16, dk, generator=g).to(torch.bfloat16)
    vc = None if G == 1 else torch.randn(R * nb, G, 16, dv, generator=g).to(torch.bfloat16)
    bt = torch.randperm(R * nb, generator=g).view(R, nb)
    kc[bt[4, 3], 0, 5, 1], kc[bt[5, 8], 0, 0, 7] = float("inf"), float("nan")
    q, sinks = torch.randn(R, H * maps * dk, generator=g), torch.randn(H * maps, generator=g)
    for window, keep, chunk, cap, sk in ((100, 3, 0, 0.0, None), (0, 0, 160, 5.0, sinks)):
        def run(cast):
            k, v = cast(kc).cuda(), None if vc is None else cast(vc).cuda()
            at = (dev(q), k, v, i32(pos), i32(list(range(R))), bt.int().cuda(), H, G)
            rest = (dk, dv, dk ** -0.5, window, keep, chunk, cap, None if sk is None else dev(sk))
            return (ops.multimap_softmax_attention(*at, maps, *rest) if maps > 1 else ops.masked_softmax_attention(*at, *rest)).cpu()
        torch.testing.assert_close(run(lambda t: t), run(lambda t: t.float()), rtol=0, atol=0, equal_nan=True)
    if maps > 1:
        return
    d1, d2, gates = (dev(torch.rand(*n, generator=g)) for n in ((H,), (H,), (R, H)))
    for f, kw in ((ops.distance_softmax_attention, dict(dist1=d1, dist2=d2)), (ops.gated_softmax_attention, dict(gates=gates, sinks=dev(sinks)))):
        def run(cast):
            k, v = cast(kc).cuda(), None if vc is None else cast(vc).cuda()
            return f(dev(q), k, v, i32(pos), i32(list(range(R))), bt.int().cuda(), H, G, dk, dv, dk ** -0.5, 120, softcap=4.0, **kw).cpu()
        torch.testing.assert_close(run(lambda t: t), run(lambda t: t.float()), rtol=0, atol=0, equal_nan=True)


def same_where_finite(got, want, tol=1e-5):
    """The same entries are finite in both, and those agree."""
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    ok = torch.isfinite(want)
    assert (got - want)[ok].abs().max() <= tol * want[ok].abs().max()


@pytest.mark.parametrize("H,G,dk,dv,window,keep", [(4, 2, 128, 128, 5000, 0), (6, 1, 128, 128, 40, 3), (3, 1, 576, 512, 5000, 0)])
def test_rows_softmax_attention_of_scores_that_are_no_numbers(H, G, dk, dv, window, keep):
    """Queries and keys with infinities and NaN (keys before the portion, so that every row or none sees them): the rows
    that come out finite are those of the kernel on the vector pipe, an infinite score of the right sign is a weight of 0
    (queries of few bits too, whose lower parts are 0), and nothing not a number is left out of a sum."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator(device="cuda").manual_seed(dk + window)
    p0, n = 100, 70
    pages = (p0 + n + 15) // 16
    bt = torch.randperm(pages, generator=g, device="cuda").to(torch.int32).view(1, pages)
    kc = torch.randn(pages, G, 16, dk, generator=g, device="cuda").to(torch.bfloat16)
    vc = None if dv == 512 else torch.randn(pages, G, 16, dv, generator=g, device="cuda").to(torch.bfloat16)
    q = torch.randn(n, H * dk, generator=g, device="cuda")
    q[::2] = q[::2].to(torch.bfloat16).float()
    q[5, 3], q[9, dk + 7], q[12, 1] = float("nan"), float("inf"), float("-inf")
    at = lambda p: (bt[0, p // 16].long(), 0, p % 16)
    if vc is not None:      # (a latent row's channels are values too)
        kc[at(70)][4] = float("-inf")
        if window > p0:
            kc[at(20)][9] = float("inf")
    pos, slot = i32(range(p0, p0 + n)), i32([0] * n)
    want = ops.window_softmax_attention(q, kc, vc, pos, slot, bt, H, G, dk, dv, window, keep, 0.0625)
    got = ops.rows_softmax_attention(q, kc, vc, bt, i32([[0, 0, n, p0]]), H, G, dk, dv, window, keep, 0.0625)
    assert not torch.isfinite(want).all()
    same_where_finite(got, want)


@pytest.mark.parametrize("H,G,dk,dv", [(4, 2, 128, 128), (16, 1, 128, 128), (3, 1, 576, 512)])
@pytest.mark.parametrize("window,keep", [(5000, 0), (40, 0), (70, 33), (1, 1)])
def test_rows_softmax_attention_of_values_that_are_no_numbers(H, G, dk, dv, window, keep):
    """Infinite and NaN keys and values before, inside and at the end of a portion: they reach the rows that see their
    token, in the channels that they are in, and no other row or channel: as on the vector pipe, which reads the keys that a
    row sees and no others."""
    from vllm_omni_draft_amd import ops
    g = torch.Generator(device="cuda").manual_seed(dk + window + H)
    p0, n = 37, 150
    pages = (p0 + n + 15) // 16
    bt = torch.randperm(pages, generator=g, device="cuda").to(torch.int32).view(1, pages)
    kc = torch.randn(pages, G, 16, dk, generator=g, device="cuda").to(torch.bfloat16)
    vc = None if dv == 512 else torch.randn(pages, G, 16, dv, generator=g, device="cuda").to(torch.bfloat16)
    q = torch.randn(n, H * dk, generator=g, device="cuda")
    pos, slot, ents = i32(range(p0, p0 + n)), i32([0] * n), i32([[0, 0, n, p0]])
    run = lambda: (ops.window_softmax_attention(q, kc, vc, pos, slot, bt, H, G, dk, dv, window, keep, dk ** -0.5),
                   ops.rows_softmax_attention(q, kc, vc, bt, ents, H, G, dk, dv, window, keep, dk ** -0.5))
    clean = run()[1]
    inf, nan = float("inf"), float("nan")
    for p, c, x in ((p0 + 99, 7, inf), (p0 + 100, 120, -inf), (p0 + 130, slice(None), nan), (p0 + n - 1, 0, nan), (36, 5, nan), (2, 9, inf)):
        if p < p0 and window > p0:
            continue              # (every row would see it)
        if vc is not None:
            vc[bt[0, p // 16].long(), 0, p % 16, c] = x
        else:
            kc[bt[0, p // 16].long(), 0, p % 16, slice(None)] = nan
        want, got = run()
        if window > 1 or p >= p0 or p < keep:
            assert not torch.isfinite(want).all()
        same_where_finite(got, want)
        touched = ~torch.isfinite(want)
        assert torch.equal(got[~touched], clean[~touched])       # (and the rest has its bits)
    kc[bt[0, (p0 + 60) // 16].long(), 0, (p0 + 60) % 16] = nan
    want, got = run()
    same_where_finite(got, want)


def test_a_portions_bits_do_not_depend_on_what_shares_its_pass():
    """The state-space recurrence on either side of the line between the scan and chunks (64 rows): the same bits alone
    and beside a long prompt and seventy decoded tokens."""
    from tests.test_gpu_puguzen import beside_others
    cfg = model_cfg([parallel(s_heads=16, s_vdim=32, state=64, window=20) for _ in range(3)], width=128)
    st, toks, alone, beside = beside_others(build, cfg, [400, 64, 20, 65])
    for t, a, b in zip(toks, alone, beside):
        assert torch.equal(a, b), len(t)
        want = oracle_logits(cfg, st, t)
        assert sorted(rel(b[r], want[r]) for r in range(len(t)))[len(t) // 2] < 2e-2   # (see test_bfloat16_serving_stays_close)


def test_attention_of_a_portion_does_not_depend_on_what_shares_its_pass():
    """The same with heads whose long portions attend on the matrix cores (grouped heads of 128 channels with kept tokens,
    latent rows of 512 + 64), short portions and decoded tokens beside them on the vector pipe; and a prompt in one pass
    and cut against the plain model."""
    from tests.test_gpu_puguzen import beside_others
    attn = dict(heads=4, kv_heads=2, dim=128, vdim=128, scale=128 ** -0.5)
    lat = dict(heads=2, dim=32, rot_dim=64, vdim=32, q_rank=32, kv_rank=512, scale=0.1)
    cfg = model_cfg([latent(window=60, **lat), parallel(window=50, keep_first=3, s_heads=4, s_vdim=32, state=32, **attn)], width=128)
    mid = lambda x, y: sorted(rel(x[r], y[r]) for r in range(len(y)))[len(y) // 2]   # (see test_bfloat16_serving_stays_close)
    st, toks, alone, beside = beside_others(build, cfg, [150, 64, 20, 65])
    for t, a, b in zip(toks, alone, beside):
        assert torch.equal(a, b), len(t)
        assert mid(b, oracle_logits(cfg, st, t)) < 2e-2
    cfg = model_cfg([latent(window=1000, **lat), parallel(window=200, keep_first=3, s_heads=4, s_vdim=32, state=32, **attn)], width=128)
    st, eng = build(cfg, torch.bfloat16)
    t = prompt(cfg, 400, 1)
    want = oracle_logits(cfg, st, t)
    for cuts in ([400], [100, 300], [70, 1, 200, 17, 112]):
        at, got = 0, []
        for c in cuts:
            got.append(eng.step([("c", t[at:at + c], list(range(c)))]))
            at += c
        eng.finish("c")
        assert mid(torch.cat(got), want) < 2e-2, cuts
