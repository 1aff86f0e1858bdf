"""Performance cases: what users of this package run, through its public entry points.

  linear    kernels.matmul_q40, the Q4_0 linear as one operator on checkpoint-layout weights
  convert   fp16_to_int4.quantize_linear_weight_gpu, one linear of a checkpoint -> Q4_0 (the converter and the direct loader)
  dequant   kernels.deq_int40, Q4_0 -> fp16
  expand    kernels.sample_topk_counts + kernels.tree_step, one expansion of the tree sampler
  paged     kernels.page_flash_attn, tree attention through a page table
  shared    kernels.shared_prefix_attn, one query per branch over a shared prompt and the branch's own rows
  decode    Transformer.forward(tokens, start_pos) with one token per branch
  steps     BucketedForward, consecutive decode steps of a tree search (begin, then step after step)
  prefill   Transformer.forward(prompt, 0)

Models have the 7B architecture of the headline workload at full depth, or three of the 80 layers of the 70B architecture
(GQA, 8 queries a kv head); weights are normal with deviation 0.02 quantised to Q4_0, as in bench.py.
"""
import math

import torch

from spec_mcts_amd import ModelArgs, Transformer, kernels as K
from spec_mcts_amd.decode import BucketedForward
from spec_mcts_amd.fp16_to_int4 import quantize_linear_weight_gpu
from spec_mcts_amd.mcts import EOS, TERMINAL_SEQ

DEV = "cuda:0"
VOCAB = 32016
MAX_BRANCHES, MAX_ROWS = 100, 128                # suffix cache of the models: branches x rows per branch
ARCHS = {
    "7b": dict(dim=4096, n_layers=32, n_heads=32, n_kv_heads=None, multiple_of=256, ffn_dim_multiplier=None),
    "70b": dict(dim=8192, n_layers=3, n_heads=64, n_kv_heads=8, multiple_of=4096, ffn_dim_multiplier=1.3),
}
FFN = {"7b": 11008, "70b": 28672}
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # one token through one attention projection: the smallest call of the operator, latency and host path
        dict(name="linear_1x4096x4096", kind="linear", M=1, N=4096, K=4096, residual=False),
        # the gate projection for a full tree of branches
        dict(name="linear_100x11008x4096", kind="linear", M=100, N=11008, K=4096, residual=False),
        # converting a bfloat16 checkpoint: one FFN weight
        dict(name="convert_bf16_11008x4096", kind="convert", N=11008, K=4096, dtype="bf16"),
        # one expansion of a search over 80 branches (the reference's batch)
        dict(name="expand_80", kind="expand", B=80, vocab=VOCAB, top_k=32, temp=0.8, grown=True),
        # the reference's tree-attention benchmark at its largest: 99 branches, 512 positions, half of them a shared prompt
        dict(name="paged_99x512", kind="paged", B=99, L=512, prompt=256, H=32, ids="int16"),
        # 64 branches over a 1024-token prompt with ragged fp16 suffixes
        dict(name="shared_64x1024", kind="shared", B=64, P=1024, S=256, H=32, Hkv=32, fmt="f16"),
        # a chat turn: one branch after a 512-token prompt, in the middle of its answer
        dict(name="decode_7b_b1", kind="decode", arch="7b", B=1, P=512, t=63, forked=False),
        # a growing tree: an odd number of branches that share ancestors, issued step by step
        dict(name="decode_7b_b37_forked", kind="decode", arch="7b", B=37, P=221, t=40, forked=True),
        # the headline workload: 100 branches from captured graphs
        dict(name="steps_7b_b100", kind="steps", arch="7b", B=100, P=512, n=8),
        # grouped queries and a long prompt
        dict(name="decode_70b_b10", kind="decode", arch="70b", B=10, P=2047, t=31, forked=False),
        # the headline prompt
        dict(name="prefill_7b_512", kind="prefill", arch="7b", S=512),
        # the longest prompt in use, of no round length
        dict(name="prefill_7b_2047", kind="prefill", arch="7b", S=2047),
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(lo, min(hi, int(v) // step * step))


def draw(rng):
    kind = rng.choice(("linear", "linear", "convert", "dequant", "expand", "paged", "shared", "decode", "decode", "decode", "steps", "prefill", "prefill"))
    if kind == "linear":
        return dict(kind=kind, M=_log(rng, 1, 512), N=_log(rng, 1024, 32128, 128), K=_log(rng, 1024, 28672, 8), residual=rng.random() < 0.5)
    if kind == "convert":
        return dict(kind=kind, N=_log(rng, 1024, 28672, 128), K=_log(rng, 1024, 8192), dtype=rng.choice(("bf16", "bf16", "f16", "f32")))
    if kind == "dequant":
        return dict(kind=kind, N=_log(rng, 1024, 28672, 128), K=_log(rng, 1024, 8192))
    if kind == "expand":
        return dict(kind=kind, B=_log(rng, 2, 128), vocab=VOCAB, top_k=_log(rng, 4, 128), temp=round(rng.uniform(0.3, 1.2), 2), grown=rng.random() < 0.7)
    if kind == "paged":
        L = _log(rng, 96, 768)
        return dict(kind=kind, B=_log(rng, 1, 99), L=L, prompt=max(1, int(L * rng.uniform(0.3, 0.9))), H=32, ids=rng.choice(("int32", "int64")))
    if kind == "shared":
        Hkv = rng.choice((32, 8))
        return dict(kind=kind, B=_log(rng, 1, 100), P=_log(rng, 16, 2048), S=_log(rng, 16, 256), H=32 if Hkv == 32 else 64, Hkv=Hkv, fmt=rng.choice(("f16", "q40")))
    if kind == "decode":
        return dict(kind=kind, arch=rng.choice(("7b", "7b", "70b")), B=_log(rng, 1, 100), P=_log(rng, 16, 2048), t=rng.randint(1, MAX_ROWS - 1), forked=rng.random() < 0.4)
    if kind == "steps":
        return dict(kind=kind, arch=rng.choice(("7b", "7b", "70b")), B=_log(rng, 1, 100), P=_log(rng, 16, 2048), n=rng.randint(2, 8))
    return dict(kind=kind, arch=rng.choice(("7b", "7b", "70b")), S=_log(rng, 16, 2047))


# ---- inputs ------------------------------------------------------------------------------------------------------------
def _normal(g, shape, std=1.0, dtype=torch.float16):
    return torch.randn(shape, device=DEV, generator=g, dtype=dtype) * std


def _model(arch, g, P):
    a = ARCHS[arch]
    model = Transformer(ModelArgs(**a, vocab_size=VOCAB, norm_eps=1e-5, rope_theta=1e6, max_batch_size=MAX_BRANCHES, max_seq_len=MAX_ROWS,
                                  max_prompt_seq_len=max(512, P)))
    ones = lambda: torch.ones(a["dim"], device=DEV, dtype=torch.float16)
    sd = {"tok_embeddings.weight": _normal(g, (VOCAB, a["dim"]), 0.02), "output.weight": _normal(g, (VOCAB, a["dim"]), 0.02), "norm.weight": ones()}
    for i in range(a["n_layers"]):
        sd["layers.%d.attention_norm.weight" % i] = ones()
        sd["layers.%d.ffn_norm.weight" % i] = ones()
    model.load_state_dict(sd, strict=False, assign=True)
    for layer in model.layers:
        att, ff = layer.attention, layer.feed_forward
        for lin in (att.wq, att.wk, att.wv, att.wo, ff.w1, ff.w2, ff.w3):
            n, k = lin.shape
            lin.w, lin.s = K.quantize_q40(_normal(g, (k, n), 0.02))
            lin.shape = torch.Size((n, k))
    model.to(device=DEV, dtype=torch.float16)
    model.eval()
    return model


def _prompt_rows(model, g, P):
    """The shared prompt's keys and values, as a prefill leaves them."""
    for layer in model.layers:
        att = layer.attention
        att.cache_prompt_k[0, :P] = _normal(g, (P, att.n_kv_heads, 128), 1.28)
        att.cache_prompt_v[0, :P] = _normal(g, (P, att.n_kv_heads, 128), 1.28)
        att.cache_prompt_len = P


def _suffix(att, cache, width):
    return cache.view(MAX_BRANCHES, MAX_ROWS, att.n_kv_heads, width)


def _suffix_rows(model, g, B, t):
    """The branches' own rows, as t decode steps leave them."""
    for layer in model.layers:
        att = layer.attention
        for c, s in ((att.cache_k, att.cache_k_s), (att.cache_v, att.cache_v_s)):
            qw, qs = K.quantize_q40(_normal(g, (B, t, att.n_kv_heads, 128), 1.28))
            _suffix(att, c, 64)[:B, :t] = qw.view(B, t, att.n_kv_heads, 64)
            _suffix(att, s, 2)[:B, :t] = qs.view(B, t, att.n_kv_heads, 2)


def _tokens(g, *shape):
    return torch.randint(0, VOCAB, shape, device=DEV, generator=g)


def _pager(B, L, prompt, ids):
    """Page ids of B branches of which one is forked off per step behind the prompt (a fork shares its ancestor's pages)."""
    pages = torch.zeros((B, L), dtype=torch.int64)
    pages[:, :prompt] = torch.arange(prompt)
    used, b = prompt, 1
    for i in range(prompt, L):
        if b < B:
            pages[b, :i] = pages[b - 1, :i]
            b += 1
        pages[:b, i] = used + torch.arange(b)
        used += b
    return pages.to(getattr(torch, ids)), used


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind = case["kind"]
    s = dict(case)
    if kind == "linear":
        M, N, Kd = case["M"], case["N"], case["K"]
        s["w"], s["s"] = K.quantize_q40(_normal(g, (Kd, N), 0.02))
        s["x"] = _normal(g, (M, Kd))
        s["r"] = _normal(g, (M, N)) if case["residual"] else None
    elif kind == "convert":
        s["v"] = _normal(g, (case["N"], case["K"]), 0.02, DTYPES[case["dtype"]])
    elif kind == "dequant":
        s["w"], s["s"] = K.quantize_q40(_normal(g, (case["K"], case["N"]), 0.02))
    elif kind == "expand":
        B = case["B"]
        i32 = dict(dtype=torch.int32, device=DEV)
        if case["grown"]:                          # the tree has its full batch: one draw per branch
            live, counts = B, torch.ones(B, **i32)
        else:                                      # it still grows: B draws over the live branches
            live = max(1, B // 3)
            counts = torch.bincount(torch.randint(0, live, (B - live,), device=DEV, generator=g), minlength=B).to(torch.int32)
            counts[:live] += 1
        s.update(logits=_normal(g, (B, case["vocab"]), 2.0), u=torch.rand(B, device=DEV, generator=g), draws=torch.zeros(B, dtype=torch.int64, device=DEV),
                 counts=torch.stack((_tokens(g, B).to(torch.int32), counts)).contiguous(), alive=torch.ones(B, dtype=torch.uint8, device=DEV),
                 curr=torch.full((1,), live, **i32), results=_tokens(g, B, 127), t=torch.full((1,), 40, **i32),
                 pages=torch.arange(B * MAX_ROWS, **i32).view(B, MAX_ROWS), origin=torch.empty(B, **i32), state=torch.zeros(B, **i32),
                 term=torch.tensor(TERMINAL_SEQ, dtype=torch.int64, device=DEV), length=torch.full((B,), 40, **i32),
                 next=torch.zeros(B, dtype=torch.int64, device=DEV), summary=torch.zeros(2, **i32))
    elif kind == "paged":
        pages, used = _pager(case["B"], case["L"], case["prompt"], case["ids"])
        pool = (case["H"], 1 << used.bit_length(), 128)
        s.update(pages=pages.to(DEV), pool=pool[1], q=_normal(g, (case["B"], case["H"], 128), 0.5), k=_normal(g, pool, 0.5), v=_normal(g, pool, 0.5))
    elif kind == "shared":
        B, P, S, H, Hkv = (case[k] for k in ("B", "P", "S", "H", "Hkv"))
        s.update(q=_normal(g, (B, H, 128)), pk=_normal(g, (P, Hkv, 128)), pv=_normal(g, (P, Hkv, 128)), sks=None, svs=None,
                 lens=torch.randint(0, S + 1, (B,), device=DEV, generator=g, dtype=torch.int32))
        s["sk"], s["sv"] = _normal(g, (B, S, Hkv, 128)), _normal(g, (B, S, Hkv, 128))
        if case["fmt"] == "q40":
            s["sk"], s["sks"] = K.quantize_q40(s["sk"])
            s["sv"], s["svs"] = K.quantize_q40(s["sv"])
    elif kind == "decode":
        B, P, t = case["B"], case["P"], case["t"]
        m = s["model"] = _model(case["arch"], g, P)
        _prompt_rows(m, g, P)
        _suffix_rows(m, g, B, t)
        s["tokens"] = _tokens(g, B, 1)
        m(s["tokens"], P + t - 1)                  # the step before
        if case["forked"] and B > 1:
            m.fork(0, 1, B // 2)
    elif kind == "steps":
        B, P = case["B"], case["P"]
        m = _model(case["arch"], g, P)
        _prompt_rows(m, g, P)
        s["tokens"] = _tokens(g, B, case["n"])
        fwd = s["fwd"] = BucketedForward(m, MAX_BRANCHES)
        fwd.begin()
        for i in range(2):                         # two steps of which half the branches inherit the first branch's rows
            fwd.step(s["tokens"][:, i:i + 1])
        if B > 1:
            m.fork(0, 1, B // 2)
    else:
        m = s["model"] = _model(case["arch"], g, case["S"])
        s["tokens"] = _tokens(g, 1, case["S"])
        m(s["tokens"][:, :16], 0)                  # an earlier, short prompt
    return s


def run(s):
    kind = s["kind"]
    if kind == "linear":
        return K.matmul_q40(s["x"], s["w"], s["s"], (s["K"], s["N"]), residual=s["r"])
    if kind == "convert":
        w, sc, _ = quantize_linear_weight_gpu(s["v"])
        return w, sc
    if kind == "dequant":
        return K.deq_int40(s["w"], s["s"], 64, (s["K"], s["N"]))
    if kind == "expand":
        K.sample_topk_counts(s["logits"], s["temp"], s["top_k"], s["counts"][1], s["u"], out=s["draws"])
        K.tree_step(s["draws"], s["counts"], s["alive"], s["curr"], s["results"], s["t"], s["pages"], s["origin"], s["state"], s["term"],
                    s["length"], s["next"], s["summary"], EOS)
        return [s[k] for k in ("draws", "counts", "alive", "curr", "results", "pages", "origin", "state", "length", "next", "summary")]
    if kind == "paged":
        return K.page_flash_attn(s["pages"], s["q"], s["k"], s["v"], s["pool"], s["B"], s["L"], s["H"], 128)
    if kind == "shared":
        return K.shared_prefix_attn(s["q"], s["pk"], s["pv"], s["P"], suffix_k=s["sk"], suffix_v=s["sv"], suffix_ks=s["sks"], suffix_vs=s["svs"],
                                    Smax=s["S"], lens=s["lens"], lens_stride=1)
    if kind == "decode":
        m, B, t = s["model"], s["B"], s["t"]
        logits = m(s["tokens"], s["P"] + t)
        att = m.layers[0].attention                # (the first layer's new rows: whole values that depend on no long sum)
        return [logits] + [_suffix(att, c, w)[:B, t] for c, w in ((att.cache_k, 64), (att.cache_k_s, 2), (att.cache_v, 64), (att.cache_v_s, 2))]
    if kind == "steps":
        fwd = s["fwd"]
        fwd.begin()
        for i in range(s["n"]):
            logits = fwd.step(s["tokens"][:, i:i + 1])
        return logits
    m, S = s["model"], s["S"]
    logits = m(s["tokens"], 0)
    att = [m.layers[i].attention for i in (0, len(m.layers) // 2, -1)]
    return [logits] + [a.cache_prompt_k[0, :S] for a in att] + [a.cache_prompt_v[0, :S] for a in att]


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------
def _weights(arch):
    """(values in the Q4_0 linears, query heads, kv heads, layers) of a model"""
    a = ARCHS[arch]
    d, f, H = a["dim"], FFN[arch], a["n_heads"]
    Hkv = a["n_kv_heads"] or H
    return a["n_layers"] * (d * (2 * H + 2 * Hkv) * 128 + 3 * d * f), H, Hkv, a["n_layers"]


def _decode_work(arch, B, P, t, forked):
    n, H, Hkv, L = _weights(arch)
    d = ARCHS[arch]["dim"]
    rows = B * t if not forked else (B - B // 2) * t          # forked branches read their ancestor's rows
    nbytes = n * 17 / 32 + VOCAB * d * 2 + L * (2 * P * Hkv * 256 + rows * 2 * Hkv * 68 + B * 2 * Hkv * 68) + B * (d + VOCAB) * 2
    return nbytes, 2.0 * B * (n + VOCAB * d) + 4.0 * B * L * H * 128 * (P + t + 1)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, Kd = case["M"], case["N"], case["K"]
        return {"bytes": N * Kd * 17 / 32 + 2 * M * (Kd + N * (2 if case["residual"] else 1)), "flops": 2.0 * M * N * Kd}
    if kind in ("convert", "dequant"):
        n = case["N"] * case["K"]
        return {"bytes": n * 17 / 32 + n * (4 if case.get("dtype") == "f32" else 2), "flops": 2.0 * n}
    if kind == "expand":
        return {"bytes": case["B"] * (case["vocab"] * 2 + 64), "flops": case["B"] * case["vocab"] * 1.0}
    if kind == "paged":
        B, L, p = case["B"], case["L"], case["prompt"]
        used = p + sum(min(B, i - p + 2) for i in range(p, L))                  # pages that exist
        return {"bytes": used * case["H"] * 512 + B * L * (2 if case["ids"] == "int16" else 4 if case["ids"] == "int32" else 8) + B * case["H"] * 512,
                "flops": 4.0 * B * L * case["H"] * 128}
    if kind == "shared":
        B, P, S, H, Hkv = (case[k] for k in ("B", "P", "S", "H", "Hkv"))
        rows = B * S / 2                                                        # lengths are uniform in 0 .. S
        return {"bytes": 2 * P * Hkv * 256 + rows * 2 * Hkv * (256 if case["fmt"] == "f16" else 68) + 2 * B * H * 256, "flops": 4.0 * H * 128 * (B * P + rows)}
    if kind == "decode":
        nbytes, flops = _decode_work(case["arch"], case["B"], case["P"], case["t"], case["forked"] and case["B"] > 1)
        return {"bytes": nbytes, "flops": flops}
    if kind == "steps":
        each = [_decode_work(case["arch"], case["B"], case["P"], t, False) for t in range(case["n"])]
        return {"bytes": sum(e[0] for e in each), "flops": sum(e[1] for e in each)}
    n, H, Hkv, L = _weights(case["arch"])
    S, d = case["S"], ARCHS[case["arch"]]["dim"]
    return {"bytes": n * 17 / 32 + VOCAB * d * 2 + S * (d + VOCAB) * 2 + L * 2 * S * Hkv * 256,
            "flops": 2.0 * S * (n + VOCAB * d) + 2.0 * L * H * 128 * S * (S + 1)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("convert", "dequant", "expand"):
        return "exact"                             # whole codes, scales and tokens
    if kind == "linear":
        return {"rel": 1e-3}                       # fp32 sums, one rounding to fp16
    if kind in ("paged", "shared"):
        return {"rel": 2e-3}                       # probabilities and outputs rounded to fp16
    # every linear, norm and residual rounds to fp16: two sound evaluations drift apart layer by layer (an evaluation with all
    # sums in double precision moves the 32-layer model's logits by 0.07 at most, at a deviation of about 1.3)
    return {"rel": 2e-2 if case["arch"] == "7b" else 1e-2, "differ": 5e-3}
