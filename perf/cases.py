"""Timed cases of the MI355X Qwen3-30B-A3B FP8 library: what its users' programs run, through the
package's public entry points.

Kinds of case (a case is a dict of plain values):

- moe      one MoE block of `tokens` rows (omega_gpu_moe_batch_dev), as a decode or serving layer
           runs it: norm, router, top-8 of 128 experts, FP8 gate|up / SwiGLU / down, residual.
- paged    decode attention of `seqs` sequences over a bf16 page pool
           (omega_gpu_paged_attention_batch_dev), contexts log-uniform in [lo, hi], seeded.
- token    one greedy token of the whole 48-layer model at batch 1 (DecodeGraph).
- serve    one greedy step of `seqs` sequences of the whole 48-layer model (BatchDecode).
- prompt   one layer of a whole prompt of `m` tokens through the prefill driver
           (WholePromptPrefill: embedding rows in, host routing plan, the last token's row out).
           One layer, because a rounding that moves an e4m3 code of one layer's activations moves
           the routing of the next: two correct implementations differ by several percent after
           a few.
- proj     a prefill projection of `m` rows: activation quantiser and W8A8 GEMM.
- experts  the routed experts of a prefill layer: quantiser, grouped gate|up GEMM with SwiGLU,
           quantiser, grouped down GEMM, weighted combine (the plan is the caller's).
- attn     the prefill attention of `m` tokens behind `pos0` cached positions.

The whole-model kinds use weights that the library synthesises on the device; all other inputs
are made here with torch from the seed.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "aien-sovereign-core-mv_amd"))
import omega_amd as om  # noqa: E402
from omega_amd import prefill as pf  # noqa: E402

H, E, TOP, INTER, VOCAB, LAYERS = 2048, 128, 8, 768, 151936, 48
QH, KVH, HD, QKV, OUT = 32, 4, 128, 5120, 4096
EPS, THETA = 1e-6, 1e6
KV_TOKEN = 2 * KVH * HD * 2                       # K and V bytes of one position in one layer
EXPERT = 2 * INTER * H + H * INTER                # e4m3 bytes of one expert
LAYER_DENSE = QKV * H + H * OUT + E * H * 2       # q|k|v, o (e4m3) and the router rows (bf16)


def listed():
    return [
        # one decoded token's expert block: the smallest call, bound by launches and latency
        dict(name="moe_1", kind="moe", tokens=1),
        # a few conversations decoding together, an odd number of them
        dict(name="moe_7", kind="moe", tokens=7),
        # a full serving batch
        dict(name="moe_32", kind="moe", tokens=32),
        # one conversation's attention at an ordinary context, not a whole number of pages
        dict(name="paged_1", kind="paged", seqs=1, lo=1999, hi=1999),
        # a serving batch's attention, ragged contexts up to 32k
        dict(name="paged_32", kind="paged", seqs=32, lo=1024, hi=32768),
        # the headline workload: batch-1 greedy decode behind a 512-token prompt
        dict(name="token", kind="token", context=545),
        # the batched serving step, 32 sequences with ragged contexts
        dict(name="serve_32", kind="serve", seqs=32, lo=256, hi=8192),
        # a layer of a chat prompt: driver, host plan and kernels of the time to first token
        dict(name="prompt_517", kind="prompt", m=517),
        # the q|k|v projection of a chat prompt
        dict(name="proj_512", kind="proj", m=512, n=QKV, k=H),
        # the routed experts of a long prompt, a ragged number of tokens
        dict(name="experts_2000", kind="experts", m=2000),
        # the attention of a long prompt
        dict(name="attn_2048", kind="attn", m=2048, pos0=0),
        # the next chunk of a conversation behind a cached history
        dict(name="attn_chunk", kind="attn", m=333, pos0=3700),
    ]


def _log(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["moe", "paged", "proj", "experts", "attn", "prompt"])
    if kind == "moe":
        return dict(kind=kind, tokens=rng.randint(1, 64))
    if kind == "paged":
        lo = _log(rng, 64, 8192)
        return dict(kind=kind, seqs=_log(rng, 1, 32), lo=lo, hi=lo * rng.choice([1, 2, 4]) + rng.randint(0, 15))
    if kind == "proj":
        n, k = rng.choice([(QKV, H), (H, OUT)])
        return dict(kind=kind, m=_log(rng, 16, 4096), n=n, k=k)
    if kind == "experts":
        return dict(kind=kind, m=_log(rng, 16, 3000))
    if kind == "attn":
        return dict(kind=kind, m=_log(rng, 16, 2500), pos0=rng.choice([0, _log(rng, 16, 6000)]))
    return dict(kind=kind, m=_log(rng, 32, 1500))


# ------------------------------------------------------------------ inputs
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + salt)
    return g


def _normal(seed, salt, *shape):
    return torch.randn(*shape, generator=_gen(seed, salt), device="cuda")


def _fp8_weights(seed, salt, experts, n, k):
    """W ~ N(0, 0.02) as a checkpoint holds it: e4m3 codes and one bf16 scale per 128 x 128 block."""
    codes = torch.empty(experts, n, k, dtype=torch.uint8, device="cuda")
    scales = torch.empty(experts, n // 128, k // 128, dtype=torch.bfloat16, device="cuda")
    g = _gen(seed, salt)
    for e0 in range(0, experts, 16):
        e1 = min(experts, e0 + 16)
        w = torch.randn(e1 - e0, n, k, generator=g, device="cuda") * 0.02
        b = w.view(e1 - e0, n // 128, 128, k // 128, 128)
        s = (b.abs().amax(dim=(2, 4)) / 448.0).to(torch.bfloat16)
        q = (b / s.float()[:, :, None, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
        codes[e0:e1] = q.reshape(e1 - e0, n, k).view(torch.uint8)
        scales[e0:e1] = s
    return codes, scales


def _upload(w):
    codes, scales = w
    e, n, k = codes.shape
    return om.Fp8Tensor.upload(e, n, k, codes.cpu().numpy(), scales.view(torch.uint16).cpu().numpy())


def _dequant(w, e):
    codes, scales = w
    v = codes[e].view(torch.float8_e4m3fn).double()
    s = scales[e].double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    return v * s


def _moe_inputs(seed):
    gate = (_normal(seed, 1, E, H) * 0.02).to(torch.bfloat16)
    norm = 1.0 + 0.1 * _normal(seed, 2, H)
    return gate, norm, _fp8_weights(seed, 3, E, 2 * INTER, H), _fp8_weights(seed, 4, E, H, INTER)


def _contexts(case, seed):
    rng = np.random.default_rng(seed)
    v = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"] + 1), case["seqs"]))
    return np.clip(v.astype(np.int64), case["lo"], case["hi"]).astype(np.int32)


def _plan(seed, m):
    """The routing of m tokens: top-8 of noisy logits with a mild preference per expert, grouped by
    expert in token order."""
    logits = _normal(seed, 11, m, E) + 0.5 * _normal(seed, 12, E)
    top, ids = logits.topk(TOP, dim=1)
    wts = torch.softmax(top, 1)
    flat = ids.reshape(-1).cpu()
    order = torch.argsort(flat, stable=True)
    a2g = torch.empty_like(order)
    a2g[order] = torch.arange(order.numel())
    counts = torch.bincount(flat, minlength=E)
    return dict(counts=counts, token=(order // TOP), a2g=a2g, wts=wts)


class _State:
    pass


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _tiles(tensors, counts):
    """`tensors`: (weight, scale) device addresses per expert; the GEMM's tile table over `counts` rows per expert, on the device"""
    tab = pf.build_tiles(pf.qgemm_bm(), [v[0] for v in tensors], [v[1] for v in tensors], counts)
    return _dev(tab.view(np.uint8)), len(tab)


def prepare(case, seed):
    s = _State()
    s.case = dict(case)
    getattr(sys.modules[__name__], "_prepare_" + case["kind"])(s, case, seed)
    om.sync()
    torch.cuda.synchronize()
    return s


def _prepare_moe(s, case, seed):
    t = case["tokens"]
    gate, norm, gu, dn = _moe_inputs(seed)
    s.router = om.Router(1)
    s.router.set_layer(0, gate.view(torch.uint16).cpu().numpy(), norm.cpu().numpy())
    s.router.set_directory(0, np.zeros(2 * E, np.uint64), np.zeros(2 * E, np.uint64))
    s.gu, s.dn = _upload(gu), _upload(dn)
    s.h = _normal(seed, 5, t, H)
    s.ids = torch.zeros(t, TOP, dtype=torch.int32, device="cuda")
    s.wts = torch.zeros(t, TOP, device="cuda")
    s.out = torch.zeros(t, H, device="cuda")
    if t >= 16:  # a serving program's tensors have their matrix-core layout from the first step on
        torch.cuda.synchronize()
        _run_moe(s)


def _run_moe(s):
    L = om.lib()
    rc = L.omega_gpu_moe_batch_dev(s.router.as_raw(), 0, s.gu.as_raw(), s.dn.as_raw(), s.case["tokens"],
                                   s.h.data_ptr(), EPS, 1, s.h.data_ptr(), s.ids.data_ptr(), s.wts.data_ptr(),
                                   s.out.data_ptr())
    om._check(rc, "fp8gemm")
    return {"out": s.out, "ids": s.ids, "weights": s.wts}


def _prepare_paged(s, case, seed):
    ctx = _contexts(case, seed)
    pages = (ctx + 15) // 16
    total, s.blocks = int(pages.sum()), int(pages.max())
    s.layout = om.kv_layout(total, 16, 2, KVH, HD)  # the second of two layers is read
    s.pool = torch.empty(s.layout.pool_bytes // 2, dtype=torch.bfloat16, device="cuda")
    s.pool.normal_(generator=_gen(seed, 1))
    perm = np.random.default_rng(seed + 1).permutation(total).astype(np.int32)
    tab = np.full((case["seqs"], s.blocks), -1, np.int32)
    at = 0
    for i, p in enumerate(pages):
        tab[i, :p] = perm[at:at + p]
        at += p
    s.ctx, s.tab = _dev(ctx), _dev(tab)
    s.max_ctx = int(ctx.max())
    s.q = _normal(seed, 2, case["seqs"], QH, HD)
    s.out = torch.zeros(case["seqs"], QH, HD, device="cuda")


def _run_paged(s):
    rc = om.lib().omega_gpu_paged_attention_batch_dev(
        s.q.data_ptr(), s.pool.data_ptr(), C.byref(s.layout), s.tab.data_ptr(), s.ctx.data_ptr(), s.blocks,
        s.case["seqs"], s.max_ctx, 1, QH, KVH, HD, s.out.data_ptr())
    om._check(rc, "attention")
    return {"out": s.out}


def _prepare_token(s, case, seed):
    ctx = case["context"]
    s.model = om.SynthDecodeModel(seed % (1 << 30) + 1, om.round_max_pos(ctx + 64))
    payload = torch.randn(s.model.cache.payload_len(ctx) // 2, generator=_gen(seed, 1), device="cuda")
    payload = payload.to(torch.bfloat16).view(-1, LAYERS, 2, 16, KVH * HD)
    if ctx % 16:
        payload[-1, :, :, ctx % 16:] = 0
    s.model.cache.import_kv(0, ctx, payload.view(torch.uint16).cpu().numpy().reshape(-1).view(np.uint8))
    s.tok = int(torch.randint(VOCAB, (1,), generator=_gen(seed, 2), device="cuda"))


def _run_token(s):
    s.next, _ = s.model.graph.token_id(s.tok, s.case["context"])
    _, _, logits = s.model.graph.read(logits=True)
    return {"logits": logits}  # the greedy token is their argmax


def _prepare_serve(s, case, seed):
    n = case["seqs"]
    ctx = _contexts(case, seed)
    pages = ctx // 16 + 1
    total, blocks = int(pages.sum()), int(pages.max())
    s.layout = om.kv_layout(total, 16, LAYERS, KVH, HD)
    s.pool = torch.empty(s.layout.pool_bytes // 2, dtype=torch.bfloat16, device="cuda")
    s.pool.normal_(generator=_gen(seed, 1))
    perm = np.random.default_rng(seed + 1).permutation(total).astype(np.int32)
    tab = np.full((n, blocks), -1, np.int32)
    at = 0
    for i, p in enumerate(pages):
        tab[i, :p] = perm[at:at + p]
        at += p
    torch.cuda.synchronize()
    wseed = seed % (1 << 30) + 1
    ones, one_hd = np.ones(H, np.float32), np.ones(HD, np.float32)
    s.router = om.Router(LAYERS)
    s.layers = []
    for l in range(LAYERS):
        tid = [om.synth_tensor_id(l, k) for k in (0, 1, 2, 3, 8)]
        s.layers.append((om.Fp8Tensor.synth(1, QKV, H, wseed, tid[0]), om.Fp8Tensor.synth(1, H, OUT, wseed, tid[1]),
                         om.Fp8Tensor.synth(E, 2 * INTER, H, wseed, tid[2]),
                         om.Fp8Tensor.synth(E, H, INTER, wseed, tid[3])))
        s.router.set_layer(l, om.synth_bf16_host(wseed, tid[4], (E, H), 0.02), ones)
        s.router.set_directory(l, np.zeros(2 * E, np.uint64), np.zeros(2 * E, np.uint64))
    s.lm = om.Bf16Tensor.synth(VOCAB, H, wseed, 2, 0.02)
    s.embed = om.Bf16Tensor.synth(VOCAB, H, wseed, 1, 0.02)
    s.bd = om.BatchDecode(LAYERS, VOCAB, n, blocks, blocks * 16, EPS, THETA, s.router, s.lm, s.embed,
                          s.pool.data_ptr(), s.layout)
    for l, ts in enumerate(s.layers):
        s.bd.set_layer(l, *ts, ones, one_hd, one_hd)
    s.bd.set_final_norm(ones)
    s.bd.set_tables(tab)
    s.bd.set_keep_logits(True)
    s.tok = torch.randint(VOCAB, (n,), generator=_gen(seed, 2), device="cuda").cpu().numpy().astype(np.uint32)
    s.pos = ctx.astype(np.uint32)
    _run_serve(s)  # the step graph of this batch size, as a running server holds it


def _run_serve(s):
    s.next = s.bd.step(s.tok, s.pos)
    _, _, logits, _ = s.bd.read(s.case["seqs"], logits=True)
    return {"logits": logits}  # the greedy tokens are their argmax


def _prompt_inputs(seed, m):
    """the embedding rows, the norms and the dense projections of the layer (its experts and router
    are _moe_inputs)"""
    x = (_normal(seed, 21, m, H) * 0.02).to(torch.bfloat16).float()
    norms = [1.0 + 0.1 * _normal(seed, 22 + i, n) for i, n in enumerate((H, H, HD, HD))]
    return x, norms, _fp8_weights(seed, 26, 1, QKV, H), _fp8_weights(seed, 27, 1, H, OUT)


def _prepare_prompt(s, case, seed):
    m = case["m"]
    x, (inorm, fnorm, qn, kn), qkv, o = _prompt_inputs(seed, m)
    gate, post, gu, dn = _moe_inputs(seed)
    s.cache = om.DecodeAttnCache(1, om.round_max_pos(m), THETA)
    s.cache.set_norms(0, qn.cpu().numpy(), kn.cpu().numpy())
    s.weights = dict(qkv=_upload(qkv), o=_upload(o), gate_up=_upload(gu), down=_upload(dn),
                     input_norm=inorm.cpu().numpy(), post_norm=post.cpu().numpy(), router=gate.float().cpu().numpy())
    rows = x.cpu().numpy()
    s.tokens = list(range(m))
    s.wp = pf.WholePromptPrefill([s.weights], fnorm.cpu().numpy(), lambda t: rows[t], s.cache, EPS)


def _run_prompt(s):
    return {"hidden": s.wp.run(s.tokens, 0)}


def _prepare_proj(s, case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    s.w = _upload(_fp8_weights(seed, 1, 1, n, k))
    s.x = _normal(seed, 2, m, k)
    bm = pf.qgemm_bm()
    s.q = torch.zeros(m + bm, k, dtype=torch.uint8, device="cuda")
    s.s = torch.zeros(m + bm, k // 128, device="cuda")
    s.y = torch.zeros(m, n, device="cuda")
    s.tiles, s.nt = _tiles([s.w.entry(0)], [m])


def _run_proj(s):
    m, n, k = s.case["m"], s.case["n"], s.case["k"]
    pf.quant(k, pf.IN_F32, m, s.x.data_ptr(), s.q.data_ptr(), s.s.data_ptr())
    pf.qgemm(n, k, pf.PLAIN, s.tiles.data_ptr(), s.nt, 0, s.q.data_ptr(), s.s.data_ptr(), s.y.data_ptr())
    return {"y": s.y}


def _prepare_experts(s, case, seed):
    m = case["m"]
    g, bm = m * TOP, pf.qgemm_bm()
    s.gu, s.dn = _upload(_fp8_weights(seed, 3, E, 2 * INTER, H)), _upload(_fp8_weights(seed, 4, E, H, INTER))
    p = _plan(seed, m)
    counts = p["counts"].tolist()
    s.tgu, s.ngu = _tiles([s.gu.entry(e) for e in range(E)], counts)
    s.tdn, s.ndn = _tiles([s.dn.entry(e) for e in range(E)], counts)
    s.rowidx = _dev(np.concatenate([p["token"].numpy(), np.zeros(bm)]).astype(np.int32))
    s.inv = _dev(p["a2g"].numpy().astype(np.int32))
    s.wts = p["wts"].contiguous()
    s.x = _normal(seed, 5, m, H)
    s.xq = torch.zeros(m + bm, H, dtype=torch.uint8, device="cuda")
    s.xs = torch.zeros(m + bm, H // 128, device="cuda")
    s.act = torch.zeros(g, INTER, dtype=torch.bfloat16, device="cuda")
    s.aq = torch.zeros(g + bm, INTER, dtype=torch.uint8, device="cuda")
    s.as_ = torch.zeros(g + bm, INTER // 128, device="cuda")
    s.down = torch.zeros(g, H, device="cuda")
    s.out = torch.zeros(m, H, device="cuda")


def _run_experts(s):
    m = s.case["m"]
    g = m * TOP
    pf.quant(H, pf.IN_F32, m, s.x.data_ptr(), s.xq.data_ptr(), s.xs.data_ptr())
    pf.qgemm(2 * INTER, H, pf.SWIGLU_NAT, s.tgu.data_ptr(), s.ngu, s.rowidx.data_ptr(), s.xq.data_ptr(),
             s.xs.data_ptr(), s.act.data_ptr())
    pf.quant(INTER, pf.IN_BF16, g, s.act.data_ptr(), s.aq.data_ptr(), s.as_.data_ptr())
    pf.qgemm(H, INTER, pf.PLAIN, s.tdn.data_ptr(), s.ndn, 0, s.aq.data_ptr(), s.as_.data_ptr(), s.down.data_ptr())
    pf.moe_combine(H, TOP, m, s.down.data_ptr(), s.inv.data_ptr(), s.wts.data_ptr(), s.out.data_ptr())
    return {"out": s.out, "act": s.act}


def _prepare_attn(s, case, seed):
    m, pos0 = case["m"], case["pos0"]
    s.cache = om.DecodeAttnCache(1, om.round_max_pos(pos0 + m), THETA)
    qn, kn = (1.0 + 0.1 * _normal(seed, k, HD) for k in (1, 2))
    s.cache.set_norms(0, qn.cpu().numpy(), kn.cpu().numpy())
    for h in range(KVH if pos0 else 0):
        k, v = _history(seed, pos0, h)
        s.cache.write_rows(0, h, 0, k.view(torch.uint16).cpu().numpy(), v.view(torch.uint16).cpu().numpy())
    s.qkv = _normal(seed, 3, m, QKV)
    s.out = torch.zeros(m, OUT, device="cuda")
    s.attn = pf.PrefillAttention(s.cache)


def _history(seed, pos0, h):
    return tuple(_normal(seed, 10 + 2 * h + i, pos0, HD).to(torch.bfloat16) for i in (0, 1))


def _run_attn(s):
    s.attn.attend_dev(0, s.case["pos0"], s.case["m"], s.qkv.data_ptr(), EPS, 1.0, s.out.data_ptr())
    return {"out": s.out}


def run(state):
    return _RUN[state.case["kind"]](state)


_RUN = dict(moe=_run_moe, paged=_run_paged, token=_run_token, serve=_run_serve, prompt=_run_prompt, proj=_run_proj,
            experts=_run_experts, attn=_run_attn)


# ------------------------------------------------------------------ what a pass cannot do without
def _distinct(t):
    """expected number of distinct experts of t tokens' uniform top-8"""
    return E * (1.0 - (1.0 - TOP / E) ** t)


def _mean_ctx(case):
    lo, hi = case["lo"], case["hi"] + 1
    return (hi - lo) / math.log(hi / lo)


def work(case):
    k = case["kind"]
    if k == "moe":
        t = case["tokens"]
        return dict(bytes=_distinct(t) * EXPERT + E * H * 2 + 3 * t * H * 4,
                    flops=2.0 * t * (TOP * EXPERT + E * H))
    if k == "paged":
        n = case["seqs"] * _mean_ctx(case)
        return dict(bytes=n * KV_TOKEN + 2 * case["seqs"] * OUT * 4, flops=4.0 * n * QH * HD)
    if k == "token":
        w = LAYERS * (LAYER_DENSE + TOP * EXPERT) + 2 * VOCAB * H
        return dict(bytes=w + LAYERS * KV_TOKEN * case["context"] + 4 * VOCAB,
                    flops=2.0 * (w - VOCAB * H) + 4.0 * LAYERS * case["context"] * QH * HD)
    if k == "serve":
        n = case["seqs"] * _mean_ctx(case)
        w = LAYERS * (LAYER_DENSE + _distinct(case["seqs"]) * EXPERT) + 2 * VOCAB * H
        return dict(bytes=w + LAYERS * KV_TOKEN * n + 4 * VOCAB * case["seqs"],
                    flops=2.0 * case["seqs"] * (LAYERS * (LAYER_DENSE + TOP * EXPERT) + VOCAB * H) +
                    4.0 * LAYERS * n * QH * HD)
    if k == "prompt":
        m = case["m"]
        return dict(bytes=LAYER_DENSE + _distinct(m) * EXPERT + m * KV_TOKEN + 4 * m * H,
                    flops=2.0 * m * (LAYER_DENSE + TOP * EXPERT) + 2.0 * m * m * QH * HD)
    if k == "proj":
        m, n, kk = case["m"], case["n"], case["k"]
        return dict(bytes=n * kk + 4.0 * m * (n + kk), flops=2.0 * m * n * kk)
    if k == "experts":
        m = case["m"]
        return dict(bytes=_distinct(m) * EXPERT + 8.0 * m * H + 2.0 * m * TOP * INTER, flops=2.0 * m * TOP * EXPERT)
    m, p = case["m"], case["pos0"]
    return dict(bytes=4.0 * m * (QKV + OUT) + KV_TOKEN * (p + 2.0 * m), flops=4.0 * QH * HD * (m * p + m * (m + 1) / 2))


def tolerance(case):
    """About four times the difference measured against exact(), or, for the whole-model kinds,
    between two summation orders of the attention."""
    return dict(
        moe=dict(rel=2e-5, differ=0.005),   # f32 rows as four e4m3 terms: 4e-6
        paged=dict(rel=2e-5),               # f32 queries and probabilities as bf16 pairs: 3e-6
        token=dict(rel=3e-4),               # K and V rounded to bf16 in 48 layers: 4e-5
        # 6e-5 a row, and 0.1 in a row where a near-tie of the top-8 goes the other way: about
        # one such row in a step of 32 rows and 48 layers, 0.017 of the whole
        serve=dict(rel=3e-2, max=0.99),
        prompt=dict(rel=3e-2, max=0.5),     # moved e4m3 codes of the activation rows: 1e-2
        proj=dict(rel=6e-5),                # e4m3 products in f32 sums: 1.5e-5
        experts=dict(rel=4e-3, max=0.5),    # a bf16 rounding moves an e4m3 code: 1.1e-3
        attn=dict(rel=6e-5),                # f32 queries and probabilities as bf16 pairs: 1.4e-5
    )[case["kind"]]


# ------------------------------------------------------------------ plain torch in 64 bits
def _quantised(x):
    """e4m3 rounding of each 128-value block at a power-of-two scale: the largest value above
    1.75 x 2^e is scaled by 2^(e - 7), else by 2^(e - 8)"""
    b = x.float().view(*x.shape[:-1], -1, 128)
    m = b.abs().amax(-1, keepdim=True).clamp_min(2.0 ** -100)
    frac, exp = torch.frexp(m)                      # m = frac 2^exp, frac in [0.5, 1)
    e = exp - 1 - 8 + (frac > 0.875).to(exp.dtype)
    scale = torch.ldexp(torch.ones_like(m), e)
    q = (b / scale).clamp(-448, 448).to(torch.float8_e4m3fn).double() * scale.double()
    return q.view(x.shape)


def _rms(x, w):
    x = x.double()
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos):
    inv = 1.0 / THETA ** (torch.arange(0, HD, 2, dtype=torch.float64, device="cuda") / HD)
    a = pos.double()[:, None] * inv
    c, s = a.cos().float().double()[:, None], a.sin().float().double()[:, None]
    x0, x1 = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], -1)


def _exact_moe(case, seed):
    gate, norm, gu, dn = _moe_inputs(seed)
    h = _normal(seed, 5, case["tokens"], H)
    x = _rms(h, norm)
    top, ids = (x @ gate.double().T).topk(TOP, dim=1)
    wts = torch.softmax(top, 1)
    out = h.double().clone()
    for e in ids.unique().tolist():
        r, slot = (ids == e).nonzero(as_tuple=True)
        y = x[r] @ _dequant(gu, e).T
        a = torch.nn.functional.silu(y[:, :INTER]) * y[:, INTER:]
        out[r] += wts[r, slot, None] * (a @ _dequant(dn, e).T)
    return {"out": out, "ids": None, "weights": wts}


def _exact_paged(case, seed):
    s = _State()
    s.case = case
    _prepare_paged(s, case, seed)
    kv = s.pool.view(-1, 2, 2, 16, KVH, HD)[:, 1]
    outs = []
    for i, n in enumerate(s.ctx.tolist()):
        p = kv[s.tab[i, :(n + 15) // 16].long()].transpose(0, 1).reshape(2, -1, KVH, HD)[:, :n].double()
        k, v = p[0].permute(1, 0, 2), p[1].permute(1, 0, 2)
        q = s.q[i].double().view(KVH, QH // KVH, HD)
        w = torch.softmax(q.matmul(k.transpose(1, 2).contiguous()) / math.sqrt(HD), -1)
        outs.append(w.matmul(v.contiguous()).reshape(QH, HD))
    return {"out": torch.stack(outs)}


def _exact_proj(case, seed):
    x = _normal(seed, 2, case["m"], case["k"])
    return {"y": _quantised(x) @ _dequant(_fp8_weights(seed, 1, 1, case["n"], case["k"]), 0).T}


def _exact_experts(case, seed):
    m = case["m"]
    gu, dn = _fp8_weights(seed, 3, E, 2 * INTER, H), _fp8_weights(seed, 4, E, H, INTER)
    p = _plan(seed, m)
    x = _quantised(_normal(seed, 5, m, H))
    token = p["token"].cuda()
    act = torch.empty(m * TOP, INTER, dtype=torch.bfloat16, device="cuda")
    down = torch.empty(m * TOP, H, dtype=torch.float64, device="cuda")
    at = 0
    for e, n in enumerate(p["counts"].tolist()):
        y = x[token[at:at + n]] @ _dequant(gu, e).T
        a = (torch.nn.functional.silu(y[:, :INTER]) * y[:, INTER:]).to(torch.bfloat16)
        act[at:at + n] = a
        if n:
            down[at:at + n] = _quantised(a) @ _dequant(dn, e).T
        at += n
    rows = down[p["a2g"].cuda()].view(m, TOP, H)
    return {"out": (p["wts"].double()[:, :, None] * rows).sum(1), "act": act.double()}


def _exact_attn(case, seed):
    m, pos0 = case["m"], case["pos0"]
    qn, kn = (1.0 + 0.1 * _normal(seed, k, HD) for k in (1, 2))
    qkv = _normal(seed, 3, m, QKV)
    pos = torch.arange(pos0, pos0 + m, device="cuda")
    q = _rope(_rms(qkv[:, :OUT].view(m, QH, HD), qn), pos)
    k = _rope(_rms(qkv[:, OUT:OUT + KVH * HD].view(m, KVH, HD), kn), pos).float().to(torch.bfloat16)
    v = qkv[:, OUT + KVH * HD:].reshape(m, KVH, HD).to(torch.bfloat16)
    out = torch.empty(m, KVH, QH // KVH, HD, dtype=torch.float64, device="cuda")
    for h in range(KVH):
        old = _history(seed, pos0, h)
        kk = torch.cat([old[0], k[:, h]]).double()
        vv = torch.cat([old[1], v[:, h]]).double()
        for t0 in range(0, m, 256):
            t1 = min(m, t0 + 256)
            qq = q[t0:t1].view(t1 - t0, KVH, QH // KVH, HD)[:, h].reshape(-1, HD)
            sc = (qq @ kk.T / math.sqrt(HD)).view(t1 - t0, QH // KVH, -1)
            seen = torch.arange(pos0 + m, device="cuda")[None] <= pos[t0:t1, None]
            w = torch.softmax(sc.masked_fill(~seen[:, None], -math.inf), -1).view(-1, pos0 + m)
            out[t0:t1, h] = (w @ vv).view(t1 - t0, QH // KVH, HD)
    return {"out": out.view(m, OUT)}


def exact(case, seed):
    """None for token and serve, whose weights exist on the device only (30 G of them made again and
    multiplied in 64 bits takes longer than a comparison may), and for prompt: an error of 1e-5 in
    one of its products moves e4m3 codes of the next one's rows, so its row is 1 to 3 percent from
    any other computation's, a 64-bit one's too, and says nothing of its precision. Its products
    and its attention are the proj, experts and attn cases."""
    f = getattr(sys.modules[__name__], "_exact_" + case["kind"], None)
    return f(case, seed) if f else None
