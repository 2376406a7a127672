"""The work this package does for its callers, as measurable cases: one GPU's expert-parallel
share of an FP8 W8A8 MoE layer (``fp8_w8a8_mega_moe``, eager and as a graph replay) from a
decode batch of a few tokens to the largest prefill, the weight transform of a model load, and
the token cast with the DeepEP-style pre/post-process around an external grouped GEMM.

A layer case has S source tokens with top-k slots. With ``routing`` "softmax" the slots are the
top-k of softmax(N(0,1)) logits over ``global_experts`` and only the first ``experts`` are
local (an EP rank's view: the others' slots are -1); with "zipf" every slot is drawn i.i.d.
from Zipf(1.2) over the local experts with four of them empty.
"""
import math

import torch

from deepgemm_amd import megamoe as mm

E4M3_MAX, AMAX_FLOOR = 448.0, 1.0e-4

# (local experts, hidden, intermediate, top-k, global experts): the repository's main shape and
# the two other expert shapes its tests run (a wide hidden size, a narrow expert)
MAIN = dict(experts=32, hidden=4096, inter=2048, topk=6, global_experts=256)
H7168 = dict(experts=32, hidden=7168, inter=2048, topk=8, global_experts=256)
I1536 = dict(experts=32, hidden=4096, inter=1536, topk=8, global_experts=128)


def _layer(name, tokens, shape, routing="softmax", clamp=0.0, stats=False, bucket=0):
    return dict(name=name, kind="layer", tokens=tokens, routing=routing, clamp=clamp, stats=stats,
                bucket=bucket, **shape)


def listed():
    return [
        # decode, one token on each of 8 ranks: the smallest call a serving loop makes
        _layer("decode_1_per_rank", 8, MAIN),
        # decode as serving engines run it: a captured 256-token bucket, 25 tokens on each rank
        _layer("decode_graph_25_per_rank", 200, MAIN, bucket=256),
        # decode, 128 tokens a rank: the benchmark's headline
        _layer("decode_128_per_rank", 1024, MAIN),
        # decode at a hidden size of 7168 with top-8
        _layer("decode_h7168", 512, H7168),
        # a large decode batch on narrow experts, top-8 of 128
        _layer("decode_i1536", 1024, I1536),
        # EP shares between decode and prefill: chunked prefill mixed with decode
        _layer("mixed_448_per_rank", 3584, MAIN),
        _layer("mixed_1024_per_rank_clamp", 8192, MAIN, clamp=10.0, stats=True),
        # skewed load: the hottest expert holds a third of the rows, four are empty
        _layer("skewed_8192", 8192, MAIN, routing="zipf"),
        # prefill of 4096 and of 32768 tokens a rank
        _layer("prefill_4096_per_rank", 32768, MAIN),
        _layer("prefill_32768_per_rank", 262144, MAIN),
        # model load: one layer's bf16 expert weights into the layout the layer reads
        dict(name="weight_transform", kind="weights", **MAIN),
        # the token path around an external grouped GEMM: cast, preprocess, postprocess
        dict(name="exchange_4000", kind="exchange", tokens=4000, weighted=True, **MAIN),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["layer", "graph", "exchange", "weights"], [0.7, 0.12, 0.13, 0.05])[0]
    shape = dict(rng.choices([MAIN, H7168, I1536], [0.7, 0.15, 0.15])[0])
    if kind == "weights":
        shape["experts"] = rng.randint(4, 32)
        return dict(kind="weights", **shape)
    if kind == "exchange":
        return dict(kind="exchange", tokens=_log_uniform(rng, 16, 40000), weighted=rng.random() < 0.5, **shape)
    clamp = rng.choice([0.0, 0.0, 10.0, 1.0])
    if kind == "graph":
        bucket = _log_uniform(rng, 8, 4096)
        case = _layer("", rng.randint(bucket // 2, bucket), shape, clamp=clamp, bucket=bucket)
    else:
        routing = rng.choices(["softmax", "local", "zipf"], [0.7, 0.15, 0.15])[0]
        # the largest sizes stay within the largest listed case's work (all slots local: 8 times
        # the rows of an EP share)
        most = 262144 if shape == MAIN else 98304
        tokens = _log_uniform(rng, 4, most if routing == "softmax" else 8192)
        if routing == "local":
            shape["global_experts"] = shape["experts"]
        case = _layer("", tokens, shape, routing="zipf" if routing == "zipf" else "softmax",
                      clamp=clamp, stats=rng.random() < 0.3)
    del case["name"]
    return case


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _bf16_weights(case, g):
    e, h, i = case["experts"], case["hidden"], case["inter"]
    w1 = (torch.randn((e, 2 * i, h), generator=g, device="cuda") / math.sqrt(h)).to(torch.bfloat16)
    w2 = (torch.randn((e, h, i), generator=g, device="cuda") / math.sqrt(i)).to(torch.bfloat16)
    return w1, w2


def _tokens(case, g):
    s, e, k, ge = case["tokens"], case["experts"], case["topk"], case["global_experts"]
    x = torch.randn((s, case["hidden"]), generator=g, device="cuda").to(torch.bfloat16)
    if case.get("routing") == "zipf":
        live = torch.randperm(e, generator=g, device="cuda")[4:]
        p = torch.arange(1, live.numel() + 1, device="cuda", dtype=torch.float64) ** -1.2
        draws = torch.multinomial((p / p.sum()).float(), s * k, replacement=True, generator=g)
        idx = live[draws].view(s, k)
        w = torch.rand((s, k), generator=g, device="cuda") + 0.05
    else:
        logits = torch.randn((s, ge), generator=g, device="cuda")
        w, idx = torch.topk(torch.softmax(logits, -1), k, dim=-1)
        idx = torch.where(idx < e, idx, torch.full_like(idx, -1))
    w = (w / w.sum(-1, keepdim=True)).float().contiguous()
    return x, idx.to(torch.int64).contiguous(), w


def _local_slots(t):
    """Local slots of received token t: 1 to 3, 1.4 on average, as top-6 of 256 experts gives."""
    return 1 + (t % 3 == 0) + (t % 16 == 0)


def _received(case, g):
    """Tokens as a dispatch delivers them to a rank: each has a slot on a local expert, the slots
    of other ranks' experts are -1."""
    s, e, k = case["tokens"], case["experts"], case["topk"]
    x = torch.randn((s, case["hidden"]), generator=g, device="cuda").to(torch.bfloat16)
    w, idx = torch.topk(torch.softmax(torch.randn((s, e), generator=g, device="cuda"), -1), k, dim=-1)
    order = torch.rand((s, k), generator=g, device="cuda").argsort(dim=-1)
    idx = torch.where(order < _local_slots(torch.arange(s, device="cuda")).view(-1, 1), idx, -1)
    return x, idx.to(torch.int64).contiguous(), (w / w.sum(-1, keepdim=True)).contiguous()


def _layer_inputs(case, seed):
    """What the layer is given: the tokens' codes, scales and slots, and the packed weights."""
    g = _generator(seed)
    x, idx, w = _tokens(case, g)
    x_fp8, x_sf = mm.cast_to_fp8_channelwise(x)
    w1, w2 = _bf16_weights(case, g)
    l1, l2 = mm.transform_fp8_weights_for_mega_moe(w1, w2)
    return x_fp8, x_sf, idx, w, l1, l2


def prepare(case, seed):
    if case["kind"] == "weights":
        w1, w2 = _bf16_weights(case, _generator(seed))
        return dict(case=case, w1=w1, w2=w2)
    if case["kind"] == "exchange":
        g = _generator(seed)
        x, idx, w = _received(case, g)
        counts = torch.bincount(idx[idx >= 0], minlength=case["experts"]).to(torch.int32)
        rows = int(counts.sum())
        l2_out = torch.randn((rows, case["hidden"]), generator=g, device="cuda").to(torch.bfloat16)
        y = torch.empty((case["tokens"], case["hidden"]), dtype=torch.bfloat16, device="cuda")
        return dict(case=case, x=x, idx=idx, w=w, counts=counts, rows=rows, l2_out=l2_out, y=y)
    x_fp8, x_sf, idx, w, l1, l2 = _layer_inputs(case, seed)
    s, e, h, bucket = case["tokens"], case["experts"], case["hidden"], case["bucket"]
    buf = mm.get_symm_buffer_for_mega_moe(None, e, bucket or s, case["topk"], h, case["inter"])
    buf.x[:s].copy_(x_fp8)
    buf.x_sf[:s].copy_(x_sf)
    buf.topk_idx[:s].copy_(idx)
    buf.topk_weights[:s].copy_(w)
    state = dict(case=case, l1=l1, l2=l2, buf=buf, clamp=case["clamp"] or None,
                 y=torch.zeros((bucket or s, h), dtype=torch.bfloat16, device="cuda"),
                 stats=torch.zeros((e,), dtype=torch.int32, device="cuda") if case["stats"] else None)
    if bucket:
        def call():
            mm.fp8_w8a8_mega_moe(state["y"], l1, l2, buf, activation_clamp=state["clamp"],
                                 big_fused_cuda_graph=True)

        buf.cuda_graph_num_tokens.fill_(s)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            call()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            call()
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "weights":
        return mm.transform_fp8_weights_for_mega_moe(state["w1"], state["w2"])
    if case["kind"] == "exchange":
        x_fp8, x_sf = mm.cast_to_fp8_channelwise(state["x"])
        grouped = mm.deepep_deepgemm_preprocess_channelwise(x_fp8, x_sf, state["idx"], state["w"],
                                                            state["counts"], state["rows"])
        mm.deepep_deepgemm_postprocess_channelwise(state["y"], state["l2_out"], state["idx"], state["w"],
                                                   grouped[4], apply_topk_weights=case["weighted"])
        return (x_fp8, x_sf, *grouped, state["y"])
    if case["bucket"]:
        state["graph"].replay()
        return state["y"][:case["tokens"]]
    mm.fp8_w8a8_mega_moe(state["y"], state["l1"], state["l2"], state["buf"],
                         cumulative_local_expert_recv_stats=state["stats"],
                         activation_clamp=state["clamp"])
    return state["y"] if state["stats"] is None else (state["y"], state["stats"])


def _local_share(case):
    """(expected routed rows, tokens with a local slot, local experts with a row) of a case."""
    s, e, k, ge = case["tokens"], case["experts"], case["topk"], case["global_experts"]
    if case.get("routing") == "zipf":
        p = [r ** -1.2 for r in range(1, e - 4 + 1)]
        hit = sum(1.0 - (1.0 - v / sum(p)) ** (s * k) for v in p)
        return s * k, s, hit
    f = e / ge
    none = 1.0
    for j in range(k):
        none *= max(0.0, (ge - e - j) / (ge - j))
    return s * k * f, s * (1.0 - none), e * (1.0 - (1.0 - k / ge) ** s)


def work(case):
    e, h, i = case["experts"], case["hidden"], case["inter"]
    if case["kind"] == "weights":
        n = 3 * e * h * i
        return dict(bytes=3 * n + 4 * e * (2 * i + h), flops=2 * n)
    s, k = case["tokens"], case["topk"]
    if case["kind"] == "exchange":
        rows = sum(_local_slots(t) for t in range(s))
        cast = s * h * 3 + s * 4
        pre = s * (h + 4) + s * k * 12 + rows * (h + 12) + s * k * 4
        post = rows * h * 2 + s * k * 16 + s * h * 2
        return dict(bytes=cast + pre + post, flops=2 * s * h + rows * h)
    rows, live, hit = _local_share(case)
    weights = hit * (3 * h * i + 4 * (2 * i + h))
    return dict(bytes=weights + live * (h + 4) + s * k * 12 + s * h * 2, flops=6 * rows * h * i)


def tolerance(case):
    if case["kind"] == "weights":
        return "exact"  # codes, and scales that a float division fixes
    if case["kind"] == "exchange":
        return dict(rel=2e-3)  # copies and codes exactly; the bf16 sums up to their rounding
    # the SwiGLU output goes through bf16 and an e4m3 code per row: a rounding that crosses a
    # code's edge moves it by a 16th of its value
    return dict(rel=1e-2)


def _cast64(x):
    amax = x.double().abs().amax(dim=1).clamp(min=AMAX_FLOOR)
    return (x.double() / (amax / E4M3_MAX).view(-1, 1)).to(torch.float8_e4m3fn), amax / E4M3_MAX


def _unpack(w, rows, k):
    """[G, R/16, K*16] blocks of 16 rows by 16 bytes back to [G, R, K]."""
    return (w.view(torch.uint8).view(w.shape[0], rows // 16, k // 16, 16, 16).permute(0, 1, 3, 2, 4)
            .reshape(w.shape[0], rows, k).view(torch.float8_e4m3fn))


def _pack(w):
    g, rows, k = w.shape
    return (w.view(torch.uint8).view(g, rows // 16, 16, k // 16, 16).permute(0, 1, 3, 2, 4)
            .reshape(g, rows // 16, k * 16).view(torch.float8_e4m3fn))


def _exact_weights(case, seed):
    out = []
    for w in _bf16_weights(case, _generator(seed)):
        g, rows, k = w.shape
        codes, scale = torch.empty_like(w, dtype=torch.float8_e4m3fn), torch.empty((g, rows), dtype=torch.float64, device="cuda")
        for e in range(g):
            codes[e], scale[e] = _cast64(w[e])
        out.append((_pack(codes), scale))
    return tuple(out)


def _exact_exchange(case, seed):
    state = prepare(case, seed)
    codes, scale = _cast64(state["x"])
    idx, w, s, k = state["idx"], state["w"], case["tokens"], case["topk"]
    flat = idx.reshape(-1)
    tasks = torch.nonzero(flat >= 0).view(-1)
    tasks = tasks[torch.sort(flat[tasks], stable=True).indices]  # an expert's rows in task order
    out_index = torch.full((s * k,), -1, dtype=torch.int32, device="cuda")
    out_index[tasks] = torch.arange(tasks.numel(), dtype=torch.int32, device="cuda")
    tok = tasks // k
    y = torch.zeros((s, case["hidden"]), dtype=torch.float64, device="cuda")
    rows = state["l2_out"][:tasks.numel()].double()
    y.index_add_(0, tok, rows * w.reshape(-1)[tasks].double().view(-1, 1) if case["weighted"] else rows)
    return (codes, scale, codes.view(torch.uint8)[tok].view(torch.float8_e4m3fn), scale[tok],
            w.reshape(-1)[tasks].double(), flat[tasks].to(torch.int32), out_index.view(s, k), y)


def exact(case, seed):
    if case["kind"] == "weights":
        return _exact_weights(case, seed)
    if case["kind"] == "exchange":
        return _exact_exchange(case, seed)
    x_fp8, x_sf, idx, w, (w1, s1), (w2, s2) = _layer_inputs(case, seed)
    h, i, k = case["hidden"], case["inter"], case["topk"]
    y = torch.zeros((case["tokens"], h), dtype=torch.float64, device="cuda")
    flat, wf = idx.reshape(-1), w.reshape(-1)
    for e in range(case["experts"]):
        tasks = torch.nonzero((flat == e) & (wf != 0)).view(-1)
        if tasks.numel() == 0:
            continue
        # row-major copies, transposed before the product: plain matrices on both sides
        b1 = (_unpack(w1[e:e + 1], 2 * i, h)[0].double() * s1[e].double().view(-1, 1)).t().contiguous()
        b2 = (_unpack(w2[e:e + 1], h, i)[0].double() * s2[e].double().view(-1, 1)).t().contiguous()
        for part in tasks.split(16384):
            tok = part // k
            a = x_fp8.view(torch.uint8)[tok].view(torch.float8_e4m3fn).double() * x_sf[tok].double().view(-1, 1)
            gu = a @ b1
            gate, up = gu[:, :i], gu[:, i:]
            if case["clamp"]:
                gate, up = gate.clamp(max=case["clamp"]), up.clamp(-case["clamp"], case["clamp"])
            act = gate * torch.sigmoid(gate) * up * wf[part].double().view(-1, 1)
            # the activation's e4m3 codes are part of the layer: a code per value, a scale per row
            codes, scale = _cast64(act)
            y.index_add_(0, tok, (codes.double() * scale.view(-1, 1)) @ b2)
    return (y, None) if case["stats"] else y
