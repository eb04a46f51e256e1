"""The work whose speed is measured: what a decode engine has this library do, through its public
entry points (vib3_amd.moe, vib3_amd.mxfp4, vib3_amd.kernels), over the range of shapes, types and
options it serves.

Kinds of work (``case["kind"]``):

* ``int4_layer``   a whole INT4 MoE sublayer of one token: router, top-k, page-table lookup, gate/up,
                   SwiGLU, down, weighted sum; with ``norm`` also the RMSNorm of the f32 residual
                   stream, the shared experts' sigmoid gates and the residual add
* ``int4_expert``  one INT4 expert page by page through the launcher API (partial_swiglu per up/gate
                   page, partial_matmul per down page, weighted accumulate)
* ``nvfp4_layer``  an NVFP4 MoE sublayer: fused RMSNorm + FP4 quantizer, router top-k, the fused experts
* ``nvfp4_pages``  NVFP4 experts over the converter's pages, one launch per page
* ``nvfp4_encode`` an f16 weight matrix to tiled NVFP4 (what a loader does per matrix)
* ``mxfp4_batch``  a batch of tokens through MXFP4 experts (grouping, grouped GEMM, combine)
"""
import math

import torch

from vib3_amd import kernels, moe, mxfp4
from vib3_amd._lib import DT_BF16, DT_F16, ROUTER_SIGMOID, ROUTER_SOFTMAX

DEV = "cuda"
_DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_SDT = {"f16": DT_F16, "bf16": DT_BF16}
_POOL_LIMIT = 10e9  # bytes of resident experts of one case


# ------------------------------------------------------------------------------- the cases


def listed():
    return [
        # Kimi-K2.5 MoE layer, batch 1: the decode hot path (8 routed of 384 + 1 shared expert)
        dict(name="int4_layer_kimi", kind="int4_layer", hidden=7168, inter=2048, experts=384, top_k=8, shared=1,
             group=32, scales="bf16", x="bf16", scoring="sigmoid", tile=0, norm=False, f32_mid=False),
        # the same block as the engine runs it: f32 residual stream in and out, pre-norm, gated shared
        # expert, weights in 64-row pages scattered over a page pool
        dict(name="int4_sublayer_kimi_paged", kind="int4_layer", hidden=7168, inter=2048, experts=384, top_k=8,
             shared=1, group=32, scales="bf16", x="f32", scoring="sigmoid", tile=64, norm=True, f32_mid=False),
        # Mixtral-8x7B MoE layer, batch 1: few, wide experts
        dict(name="int4_layer_mixtral", kind="int4_layer", hidden=4096, inter=14336, experts=8, top_k=2, shared=0,
             group=128, scales="f16", x="f16", scoring="softmax", tile=0, norm=False, f32_mid=False),
        # a small model's layer: everything fits in a few microseconds, so the fixed costs show
        dict(name="int4_layer_small", kind="int4_layer", hidden=1024, inter=512, experts=64, top_k=4, shared=1,
             group=64, scales="f16", x="f16", scoring="softmax", tile=0, norm=False, f32_mid=False),
        # one Mixtral expert through the per-page launchers, one page per matrix
        dict(name="int4_expert_mixtral", kind="int4_expert", hidden=4096, inter=14336, group=128, scales="f16",
             x="f16", rows=0),
        # an expert whose sizes are no multiple of anything, over 520-row pages, f32 activations
        dict(name="int4_expert_ragged", kind="int4_expert", hidden=1000, inter=1364, group=32, scales="bf16",
             x="f32", rows=520),
        # NVFP4 MoE sublayer at the Kimi shape: norm + quantize, router, 8 experts in two launches
        dict(name="nvfp4_layer_kimi", kind="nvfp4_layer", hidden=7168, inter=2048, experts=384, top_k=8),
        # eight NVFP4 experts whose matrices span pages of 520 / 1820 rows (the converter's 2 MiB pages)
        dict(name="nvfp4_pages_kimi", kind="nvfp4_pages", hidden=7168, inter=2048, active=8, rows=520,
             rows_down=1820, path="preq"),
        # a loader converting one large f16 projection to tiled NVFP4
        dict(name="nvfp4_encode", kind="nvfp4_encode", rows=8192, cols=7168),
        # batched decode at the Kimi shape: a few requests, an ordinary batch, the largest batch
        dict(name="mxfp4_batch_4", kind="mxfp4_batch", hidden=7168, inter=2048, experts=384, top_k=8, tokens=4,
             skew=1.1),
        dict(name="mxfp4_batch_64", kind="mxfp4_batch", hidden=7168, inter=2048, experts=384, top_k=8, tokens=64,
             skew=1.1),
        dict(name="mxfp4_batch_512", kind="mxfp4_batch", hidden=7168, inter=2048, experts=384, top_k=8, tokens=512,
             skew=1.1),
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["int4_layer", "int4_layer", "int4_expert", "nvfp4_layer", "nvfp4_pages", "nvfp4_encode",
                       "mxfp4_batch", "mxfp4_batch"])
    if kind == "int4_layer":
        hidden = 32 * _log_int(rng, 16, 224)
        inter = 32 * _log_int(rng, 8, 448)
        # wide experts come with few active ones (as the layer's LDS staging of h also asks for)
        most = 10 if inter <= 2048 else 7 if inter <= 4096 else 3 if inter <= 8192 else 2
        shared = rng.randint(0, 2 if most > 3 else 0)
        top_k = rng.randint(1, min(8, most - shared))
        fit = int(_POOL_LIMIT / (3 * hidden * inter * 0.5626)) - shared
        experts = _log_int(rng, max(8, top_k), max(8, min(384, fit)))
        norm = rng.random() < 0.4
        return dict(kind=kind, hidden=hidden, inter=inter, experts=experts, top_k=top_k, shared=shared,
                    group=rng.choice([32, 64, 128]), scales=rng.choice(["bf16", "f16"]),
                    x="f32" if norm else rng.choice(["bf16", "f16", "f32"]),
                    scoring=rng.choice(["sigmoid", "softmax"]), tile=rng.choice([0, 0, 64, 96, 200]), norm=norm,
                    f32_mid=inter <= 2048 and rng.random() < 0.15)
    if kind == "int4_expert":
        ragged = rng.random() < 0.5
        step = 1 if ragged else 32
        return dict(kind=kind, hidden=step * _log_int(rng, 256 // step, 7168 // step),
                    inter=step * _log_int(rng, 256 // step, (4096 if ragged else 14336) // step),
                    group=rng.choice([32, 64, 128]), scales=rng.choice(["bf16", "f16"]),
                    x=rng.choice(["f32", "f16", "bf16"]), rows=rng.choice([0, 0, 520, 1820]))
    if kind == "nvfp4_layer":
        hidden = 128 * _log_int(rng, 8, 56)
        top_k = rng.randint(1, 8)
        inter = 128 * _log_int(rng, 2, 22)
        fit = int(_POOL_LIMIT / (3 * hidden * inter * 0.5626))
        return dict(kind=kind, hidden=hidden, inter=inter, experts=_log_int(rng, 8, min(384, fit)), top_k=top_k)
    if kind == "nvfp4_pages":
        return dict(kind=kind, hidden=64 * _log_int(rng, 8, 112), inter=64 * _log_int(rng, 4, 64),
                    active=rng.randint(1, 8), rows=rng.choice([260, 520, 4096]),
                    rows_down=rng.choice([455, 1820, 7168]), path=rng.choice(["preq", "preq", "f32", "scalar"]))
    if kind == "nvfp4_encode":
        return dict(kind=kind, rows=16 * _log_int(rng, 8, 512), cols=64 * _log_int(rng, 8, 112))
    hidden, inter = 256 * rng.randint(4, 28), 256 * rng.randint(2, 16)
    top_k = rng.randint(1, 8)
    fit = min(384, int(_POOL_LIMIT / (3 * hidden * inter * 0.5314)))
    return dict(kind="mxfp4_batch", hidden=hidden, inter=inter, experts=_log_int(rng, 8, fit), top_k=top_k,
                tokens=_log_int(rng, 1, 512), skew=rng.choice([0.0, 0.8, 1.1]))


# ------------------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, sigma=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=DEV) * sigma).to(dtype)


def _spans(rows, per_page):
    """(first row, rows) of each page of a matrix; per_page 0: one page."""
    per_page = per_page or rows
    return [(r, min(per_page, rows - r)) for r in range(0, rows, per_page)]


def _prepare_int4_layer(c, seed):
    shape = moe.BankShape(hidden=c["hidden"], inter=c["inter"], group_size=c["group"], scale_dtype=_SDT[c["scales"]],
                          scale_sigma=0.01, num_experts=c["experts"], num_shared=c["shared"])
    bank = moe.Int4ExpertBank(shape, seed=seed, layout="paged" if c["tile"] else "contiguous",
                              tile_rows=c["tile"] or 64, device=DEV)
    g = _gen(seed)
    H = c["hidden"]
    w = _randn(g, c["experts"], H, sigma=0.8 / math.sqrt(H))
    sigmoid = c["scoring"] == "sigmoid"
    bias = _randn(g, c["experts"], sigma=0.1) if sigmoid else None
    extra = {}
    if c["norm"]:
        extra["norm_weight"] = (1 + 0.1 * _randn(g, H)).half()
        if c["shared"]:
            extra["shared_gate"] = _randn(g, c["shared"], H, sigma=0.02, dtype=torch.float16)
    layer = moe.MoeInt4Layer(bank, w, bias, top_k=c["top_k"],
                             scoring_mode=ROUTER_SIGMOID if sigmoid else ROUTER_SOFTMAX,
                             scaling_factor=2.827 if sigmoid else 1.0, normalize=True,
                             flags=1 if c["f32_mid"] else 0, **extra)  # 1: VIB3_MOE_F32_INTERMEDIATE
    x = _randn(g, H, sigma=20.0 if c["norm"] else 1.0, dtype=_DT[c["x"]])
    return dict(layer=layer, bank=bank, w=w, bias=bias, x=x, **extra)


def _int4_pages(g, rows, k, group, scales, per_page):
    """One INT4 matrix as pages: [rows x ceil(k/2)] nibbles, then [rows x ceil(k/group)] scales."""
    pages = []
    for r0, n in _spans(rows, per_page):
        pk, ng = (k + 1) // 2, (k + group - 1) // group
        codes = torch.randint(0, 256, (n * pk,), dtype=torch.uint8, generator=g, device=DEV)
        sc = ((_randn(g, n * ng).abs() + 0.1) * 0.01).to(_DT[scales])
        pages.append((r0, n, torch.cat([codes, sc.view(torch.uint8)])))
    return pages


def _prepare_int4_expert(c, seed):
    g = _gen(seed)
    H, I = c["hidden"], c["inter"]
    s = dict(up=_int4_pages(g, I, H, c["group"], c["scales"], c["rows"]),
             gate=_int4_pages(g, I, H, c["group"], c["scales"], c["rows"]),
             down=_int4_pages(g, H, I, c["group"], c["scales"], c["rows"]),
             x=_randn(g, H, dtype=_DT[c["x"]]), weight=0.37,
             h=torch.zeros(I, dtype=torch.float16, device=DEV), d=torch.zeros(H, dtype=torch.float16, device=DEV),
             out=torch.zeros(H, dtype=torch.float32, device=DEV))
    return s


def _nvfp4_scales(words, g, mantissa):
    """In place: bf16 block scales 2^-10 .. 2^-6 (with a random mantissa where the path reads it)."""
    e = torch.randint(117, 122, words.shape, dtype=torch.int16, generator=g, device=DEV)
    words.copy_((e << 7) | (words & 0x7F if mantissa else 0))


def _prepare_nvfp4_layer(c, seed):
    g = _gen(seed)
    H, I, E, K = c["hidden"], c["inter"], c["experts"], c["top_k"]
    sizes = [I * H // 2 + I * (H // 32) * 2] * 2 + [H * I // 2 + H * (I // 32) * 2]
    pool = torch.empty(E, sum(sizes), dtype=torch.uint8, device=DEV)
    pool.view(-1).view(torch.int64).random_(-2**63, None, generator=g)
    table = torch.empty(1, E, 3, dtype=torch.int64)
    off = 0
    for s in range(3):
        rows, k = (I, H) if s < 2 else (H, I)
        table[0, :, s] = pool.data_ptr() + off + torch.arange(E, dtype=torch.int64) * sum(sizes)
        _nvfp4_scales(pool[:, off + rows * k // 2: off + sizes[s]].view(torch.int16), g, False)
        off += sizes[s]
    kernels.moe_prewarm_gpu_bufs(I, I)
    z = lambda n, dt: torch.zeros(n, dtype=dt, device=DEV)  # noqa: E731
    return dict(pool=pool, table=table.to(DEV), sizes=sizes, x=_randn(g, H, sigma=20.0),
                norm_weight=(1 + 0.1 * _randn(g, H)).half(),
                w=_randn(g, E, H, sigma=0.8 / math.sqrt(H), dtype=torch.float16), bias=_randn(g, E, sigma=0.1),
                scoring=kernels.Sigmoid(2.827, True), ws=kernels.RouterWorkspace(E, DEV), codes=z(H // 2, torch.uint8),
                scales=z(H // 32, torch.uint8), xn=z(H, torch.float16), ids=z(K, torch.int16),
                wts=z(K, torch.float32), out=z(H, torch.float32))


def _nvfp4_pages(g, rows, k, per_page, mantissa):
    """One NVFP4 matrix as pages: [rows x k/2] code bytes, then [rows x k/32] bf16 scale words."""
    pages = []
    for r0, n in _spans(rows, per_page):
        page = torch.randint(0, 256, (n * k // 2 + n * (k // 32) * 2,), dtype=torch.uint8, generator=g, device=DEV)
        _nvfp4_scales(page[n * k // 2:].view(torch.int16), g, mantissa)
        pages.append((r0, n, page))
    return pages


def _prepare_nvfp4_pages(c, seed):
    g = _gen(seed)
    H, I, scalar = c["hidden"], c["inter"], c["path"] == "scalar"
    experts = [dict(up=_nvfp4_pages(g, I, H, c["rows"], scalar), gate=_nvfp4_pages(g, I, H, c["rows"], scalar),
                    down=_nvfp4_pages(g, H, I, c["rows_down"], scalar), weight=0.1 + 0.05 * i)
               for i in range(c["active"])]
    z = lambda n, dt: torch.zeros(n, dtype=dt, device=DEV)  # noqa: E731
    return dict(experts=experts, x=_randn(g, H), codes=z(H // 2, torch.uint8), scales=z(H // 32, torch.uint8),
                h=z(I, torch.float32), hcodes=z(I // 2, torch.uint8), hscales=z(I // 32, torch.uint8),
                d=z(H, torch.float32), out=z(H, torch.float32))


def _prepare_nvfp4_encode(c, seed):
    m, k = c["rows"], c["cols"]
    return dict(w=_randn(_gen(seed), m, k, sigma=0.02, dtype=torch.float16),
                temp=torch.empty(m * k // 2, dtype=torch.uint8, device=DEV))


def _picks(c, seed):
    """top_k distinct experts of every token with P(expert) ~ rank^-skew, the ranks shuffled, and weights
    that sum to 1 per token."""
    g = torch.Generator().manual_seed(seed)
    E, T, K = c["experts"], c["tokens"], c["top_k"]
    logp = -c["skew"] * torch.log(torch.arange(1, E + 1, dtype=torch.float64))[torch.randperm(E, generator=g)]
    gumbel = -torch.log(-torch.log(torch.rand(T, E, dtype=torch.float64, generator=g).clamp_(1e-300, 1 - 1e-16)))
    ids = torch.topk(logp + gumbel, K, dim=1).indices
    w = torch.rand(T, K, generator=g) + 0.05
    return ids, w / w.sum(1, keepdim=True)


def _prepare_mxfp4_batch(c, seed):
    bank = mxfp4.Mxfp4ExpertBank(c["hidden"], c["inter"], c["experts"], seed=seed, device=DEV)
    ids, w = _picks(c, seed)
    return dict(bank=bank, batch=mxfp4.MoeMxfp4Batch(bank, c["tokens"], c["top_k"]),
                x=_randn(_gen(seed), c["tokens"], c["hidden"], dtype=torch.bfloat16),
                ids=ids.to(torch.int16).to(DEV), wts=w.to(DEV))


def prepare(case, seed):
    return dict(globals()["_prepare_" + case["kind"]](case, seed), case=case)


# ------------------------------------------------------------------------------- one pass


def _run_int4_layer(s, c):
    layer = s["layer"]
    out = layer.launch(s["x"], residual=s["x"] if c["norm"] else None)
    return dict(out=out, scores=layer.scores, ids=layer.ids, weights=layer.wts)


def _run_int4_expert(s, c):
    H, I, opt = c["hidden"], c["inter"], dict(group_size=c["group"], scale_dtype=_SDT[c["scales"]])
    for (r0, n, up), (_, _, gate) in zip(s["up"], s["gate"]):
        kernels.partial_swiglu(s["x"], up, gate, s["h"][r0:], H, n, **opt)
    for r0, n, page in s["down"]:
        kernels.partial_matmul(s["h"], page, s["d"][r0:], I, n, **opt)
    s["out"].zero_()
    kernels.weighted_accumulate_f32(s["out"], s["d"], s["weight"], H)
    return dict(h=s["h"], d=s["d"], out=s["out"])


def _run_nvfp4_layer(s, c):
    H, I, E, K = c["hidden"], c["inter"], c["experts"], c["top_k"]
    kernels.fused_rms_norm_quantize_fp4(s["x"], s["norm_weight"], s["codes"], s["scales"], s["xn"], H, 1e-6)
    kernels.run_router_gpu_topk_nosync(s["xn"], s["w"], E, H, K, s["scoring"], s["ids"], s["wts"],
                                       correction_bias=s["bias"], workspace=s["ws"])
    s["out"].zero_()
    kernels.moe_experts_fused_gpu(s["codes"], s["scales"], s["table"], s["ids"], s["wts"], 0, E, K, H, I, H, s["out"])
    return dict(codes=s["codes"], scales=s["scales"], xn=s["xn"], ids=s["ids"], weights=s["wts"], out=s["out"])


def _run_nvfp4_pages(s, c):
    H, I, path = c["hidden"], c["inter"], c["path"]
    swiglu = {"f32": kernels.fused_swiglu_mma_nvfp4, "scalar": kernels.partial_swiglu_f32_f32out}.get(path)
    gemv = {"f32": kernels.gemv_mma_nvfp4, "scalar": kernels.partial_matmul_nvfp4_f32}.get(path)
    if path == "preq":
        kernels.quantize_activation_fp4(s["x"], s["codes"], s["scales"], H)
    s["out"].zero_()
    for e in s["experts"]:
        for (r0, n, up), (_, _, gate) in zip(e["up"], e["gate"]):
            if path == "preq":
                kernels.fused_swiglu_mma_nvfp4_preq(s["codes"], s["scales"], up, gate, s["h"][r0:], H, n)
            else:
                swiglu(s["x"], up, gate, s["h"][r0:], H, n)
        if path == "preq":
            kernels.quantize_activation_fp4(s["h"], s["hcodes"], s["hscales"], I)
        for r0, n, page in e["down"]:
            if path == "preq":
                kernels.gemv_mma_nvfp4_preq(s["hcodes"], s["hscales"], page, s["d"][r0:], I, n)
            else:
                gemv(s["h"], page, s["d"][r0:], I, n)
        kernels.weighted_accumulate_f32(s["out"], s["d"], e["weight"], H)
    return dict(h=s["h"], d=s["d"], out=s["out"])


def _run_nvfp4_encode(s, c):
    data, scales = kernels.fp16_to_nvfp4_weight(s["w"], c["rows"], c["cols"])
    kernels.repack_row_to_tiled(data, s["temp"], c["rows"], c["cols"])
    return dict(data=data, scales=scales)


def _run_mxfp4_batch(s, c):
    return dict(out=s["batch"].launch(s["x"], s["ids"], s["wts"]))


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state, state["case"])


# ------------------------------------------------------------------------------- what a pass needs


def work(case):
    c, kind = case, case["kind"]
    if kind == "nvfp4_encode":
        n = c["rows"] * c["cols"]
        return dict(bytes=2 * n + n // 2 + n // 16, flops=0)
    H, I = c["hidden"], c["inter"]
    mats = [(I, H), (I, H), (H, I)]
    size = {"f32": 4, "f16": 2, "bf16": 2}
    if kind.startswith("int4"):
        one = sum(r * ((k + 1) // 2 + -(-k // c["group"]) * 2) for r, k in mats)
    elif kind.startswith("nvfp4"):
        one = sum(r * (k // 2 + k // 32 * 2) for r, k in mats)
    else:
        one = sum(r * (k // 2 + k // 32) for r, k in mats)
    flops = 6 * H * I
    if kind == "int4_expert":
        return dict(bytes=one + H * size[c["x"]] + 2 * I + 6 * H, flops=flops)
    if kind == "nvfp4_pages":
        return dict(bytes=c["active"] * one + 8 * H, flops=c["active"] * flops)
    if kind == "mxfp4_batch":
        T, K = c["tokens"], c["top_k"]
        touched = int(torch.unique(_picks(c, 0)[0]).numel())
        return dict(bytes=touched * one + T * H * 4 + T * K * 6, flops=T * K * flops)
    n = c["top_k"] + c.get("shared", 0)
    E = c["experts"]
    router = E * H * (4 if kind == "int4_layer" else 2)
    act = H * (size[c["x"]] if kind == "int4_layer" else 4) + 4 * H
    if kind == "nvfp4_layer":
        act += 2 * H + 2 * H + H // 2 + H // 32
    elif c["norm"]:
        act += 2 * H * (1 + c["shared"])
    return dict(bytes=n * one + router + act, flops=n * flops + 2 * E * H)


def tolerance(case):
    """About four times the error against exact() that the sums of this precision show."""
    kind = case["kind"]
    if kind == "nvfp4_encode":
        return "exact"
    if kind == "mxfp4_batch":  # bf16 outputs, f16 intermediates: 1.7e-3 measured
        return dict(rel=7e-3, max=5e-2)
    if kind == "nvfp4_pages" and case["path"] == "scalar":  # f32 throughout: 2.2e-7 measured
        return dict(rel=1e-6, max=2e-5)
    if kind.startswith("nvfp4"):  # 1.7e-7 measured, 2e-4 for the f16 copy; another order of the sums
        return dict(rel=5e-3, max=0.1, differ=2e-3)  # can turn single FP4 codes of h, each about 2e-3
    return dict(rel=1.2e-3, max=2e-2, differ=2e-3)  # f16 intermediates: 3e-4 measured


# ------------------------------------------------------------------------------- in 64 bits


def _e2m1(q):
    lut = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64,
                       device=q.device)
    return lut[q.long()]


def _silu_mul(gate, up):
    return gate / (1 + torch.exp(-gate)) * up


def _int4_matrix(page, rows, k, group, scales):
    """The f64 matrix of one page."""
    pk, ng = (k + 1) // 2, (k + group - 1) // group
    b = page[: rows * pk].view(rows, pk)
    q = torch.stack([b & 15, b >> 4], 2).view(rows, 2 * pk)[:, :k].double() - 8
    raw = page[rows * pk: rows * (pk + 2 * ng)].clone()
    s = raw.view(_DT[scales]).double().view(rows, ng)
    return q * s.repeat_interleave(group, 1)[:, :k]


def _route(logits, bias, top_k, sigmoid):
    key = torch.sigmoid(logits) + bias if sigmoid else logits
    ids = torch.topk(key, top_k).indices
    if not sigmoid:
        return ids, torch.softmax(logits[ids], 0)
    w = torch.sigmoid(logits)[ids]
    return ids, w / w.sum() * 2.827


def _exact_int4_layer(c, s):
    bank, x = s["bank"], s["x"].double()
    H, E = c["hidden"], c["experts"]
    xn = x
    if c["norm"]:
        xn = x / torch.sqrt((x * x).mean() + 1e-6) * s["norm_weight"].double()
    logits = s["w"].double() @ xn
    sigmoid = c["scoring"] == "sigmoid"
    ids, wts = _route(logits, s["bias"].double() if sigmoid else None, c["top_k"], sigmoid)
    use = [(int(i), w) for i, w in zip(ids, wts)]
    for q in range(c["shared"]):
        gate = torch.sigmoid(s["shared_gate"][q].double() @ xn) if c["norm"] else 1.0
        use.append((E + q, gate))
    want, mats = {e for e, _ in use}, {}
    for e, seg, p, r, off in bank.tiles:
        if e in want:
            k = bank.shape.seg_dims(seg)[1]
            mats.setdefault((e, seg), []).append(_int4_matrix(bank.pool[off:], r, k, c["group"], c["scales"]))
    out = x.clone() if c["norm"] else torch.zeros(H, dtype=torch.float64, device=DEV)
    for e, w in use:
        up, gate, down = (torch.cat(mats[(e, seg)]) for seg in range(3))
        out += w * (down @ _silu_mul(gate @ xn, up @ xn))
    return dict(out=out, scores=logits, ids=None, weights=wts)


def _exact_int4_expert(c, s):
    full = lambda name, k: torch.cat([_int4_matrix(p, n, k, c["group"], c["scales"]) for _, n, p in s[name]])  # noqa: E731
    x = s["x"].double()
    h = _silu_mul(full("gate", c["hidden"]) @ x, full("up", c["hidden"]) @ x)
    d = full("down", c["inter"]) @ h
    return dict(h=h, d=d, out=s["weight"] * d)


def _fp4_rounded(v):
    """The values an FP4 activation holds: per 32, E8M0 scale round(log2 amax) - 2 and E2M1 nearest even."""
    b = v.view(-1, 32)
    amax = b.abs().amax(1, keepdim=True)
    scale = torch.exp2((torch.round(torch.log2(amax.clamp_min(1e-300))) - 2).clamp(-127, 127))
    scale = torch.where(amax > 0, scale, torch.ones_like(scale))
    grid = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=v.device)
    r = (b / scale).abs().clamp(max=6)
    lo = (torch.bucketize(r, grid, right=True) - 1).clamp(0, 6)
    a, z = grid[lo], grid[lo + 1]
    up = (r - a > z - r) | ((r - a == z - r) & (lo % 2 == 1))
    return (torch.sign(b) * torch.where(up, z, a) * scale).view(-1)


def _nvfp4_matrix(page, rows, k, layout, mantissa):
    """The f64 matrix of one page: codes split-half ("row": row-major, "tiled": 16 x 64 tiles) or sequential."""
    b = page[: rows * k // 2]
    if layout == "tiled":
        b = b.view(rows // 16, k // 64, 16, 2, 16).permute(0, 2, 1, 3, 4).reshape(rows, k // 32, 16)
    else:
        b = b.view(rows, k // 32, 16)
    lo, hi = _e2m1(b & 15), _e2m1(b >> 4)
    v = torch.stack([lo, hi], 3).view(rows, k // 32, 32) if layout == "seq" else torch.cat([lo, hi], 2)
    w = page[rows * k // 2: rows * k // 2 + rows * (k // 32) * 2].clone().view(torch.int16)
    if not mantissa:
        w = w & 0x7F80
    return (v * w.view(torch.bfloat16).double().view(rows, k // 32, 1)).view(rows, k)


def _exact_nvfp4_layer(c, s):
    H, I = c["hidden"], c["inter"]
    x = s["x"].double()
    xn = x / torch.sqrt((x * x).mean() + 1e-6) * s["norm_weight"].double()
    ids, wts = _route(s["w"].double() @ xn.half().double(), s["bias"].double(), c["top_k"], True)
    a = _fp4_rounded(xn)
    out = torch.zeros(H, dtype=torch.float64, device=DEV)
    for e, w in zip(ids, wts):
        up, gate, down = torch.split(s["pool"][int(e)], s["sizes"])
        h = _silu_mul(_nvfp4_matrix(gate, I, H, "tiled", False) @ a, _nvfp4_matrix(up, I, H, "tiled", False) @ a)
        out += w * (_nvfp4_matrix(down, H, I, "tiled", False) @ _fp4_rounded(h))
    return dict(codes=None, scales=None, xn=xn, ids=None, weights=wts, out=out)


def _exact_nvfp4_pages(c, s):
    H, I, path = c["hidden"], c["inter"], c["path"]
    layout, scalar = "row" if path == "preq" else "seq", path == "scalar"
    rounded = (lambda v: v) if scalar else _fp4_rounded
    full = lambda pages, k: torch.cat([_nvfp4_matrix(p, n, k, layout, scalar) for _, n, p in pages])  # noqa: E731
    a = rounded(s["x"].double())
    out = torch.zeros(H, dtype=torch.float64, device=DEV)
    for e in s["experts"]:
        h = _silu_mul(full(e["gate"], H) @ a, full(e["up"], H) @ a)
        d = full(e["down"], I) @ rounded(h)
        out += e["weight"] * d
    return dict(h=h, d=d, out=out)


def _exact_mxfp4_batch(c, s):
    H, I, T = c["hidden"], c["inter"], c["tokens"]
    bank, x = s["bank"], s["x"].double()
    ids, wts = s["ids"].long(), s["wts"].double()
    base = bank.buf.data_ptr()

    def matrix(e, seg):
        rows, k = bank.dims[seg]
        off = int(bank.table_host[e, seg]) - base
        b = bank.buf[off: off + rows * k // 2].view(rows, k // 2)
        v = torch.stack([_e2m1(b & 15), _e2m1(b >> 4)], 2).view(rows, k // 32, 32)
        sc = bank.buf[off + rows * k // 2: off + rows * k // 2 + rows * (k // 32)].view(rows, k // 32, 1)
        return (v * torch.exp2(sc.double() - 127)).view(rows, k)

    out = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        h = _silu_mul(x[t] @ matrix(e, 1).t(), x[t] @ matrix(e, 0).t())
        out.index_add_(0, t, wts[t, j, None] * (h @ matrix(e, 2).t()))
    return dict(out=out)


def exact(case, seed):
    if case["kind"] == "nvfp4_encode":
        return None  # bytes
    return globals()["_exact_" + case["kind"]](case, prepare(case, seed))
