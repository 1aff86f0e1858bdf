"""The drop-in model where the decode step leaves the small-batch kernels: more than 16 branches (LDS/MFMA
GEMM, K-slice slabs, their consumers) and the layer shapes of the 70B architecture (BASELINE
dim 8192, 64 heads over 8 KV heads, FFN 28672), each against the oracle's dense restatement.

Branches are given DIFFERENT tokens, so a row mix-up between branches cannot cancel out, and several decode
steps are taken, so the later ones read suffix rows the earlier ones appended."""
import ctypes

import pytest
import torch

from oracle import q40_oracle as O
from tests.sync_state import sync_prefix, sync_suffix_row

pytestmark = pytest.mark.gpu


def _build(cfg, seed, std):
    from spec_mcts_amd import ModelArgs
    from spec_mcts_amd.load_q40 import load_q40
    oargs = O.OracleArgs(**cfg)
    sd = O.random_q40_state_dict(oargs, seed=seed, std=std)
    model = load_q40(dict(sd), ModelArgs(**cfg), device="cuda:0")
    return oargs, sd, model


def _steps(cfg, seed, B, P, std, rtol, atol, steps=3, forks={}):
    oargs, sd, model = _build(cfg, seed, std)
    oracle = O.OracleTransformer(oargs, sd, dense=True)
    gen = torch.Generator().manual_seed(seed + 100)
    prompt = torch.randint(0, cfg["vocab_size"], (1, P), generator=gen)
    want0 = oracle.forward(prompt, 0)
    got0 = model(prompt.cuda(), 0).cpu()
    assert torch.allclose(got0.float(), want0.float(), rtol=rtol, atol=atol)
    # Every step starts from the oracle's cache state (tests/sync_state.py), so every step and every branch is held to
    # the tolerance: steps after the first read the suffix rows the earlier ones appended.
    sync_prefix(model, oracle)
    for step in range(steps):
        if step in forks:                              # from here on the branches read an ancestor's rows through the page table
            model.fork(*forks[step])
            oracle.fork(*forks[step])
        tok = torch.randint(0, cfg["vocab_size"], (B, 1), generator=gen)
        want = oracle.forward(tok, P + step)
        got = model(tok.cuda(), P + step).cpu()
        assert got.shape == want.shape and got.dtype == torch.float16
        diff = (got.float() - want.float()).abs().reshape(B, -1)
        bound = atol + rtol * want.float().abs().reshape(B, -1)
        row_ok = (diff <= bound).all(dim=1)
        print(f"B={B} step {step}: largest logit difference {float(diff.max()):.4f}, branches within tolerance {int(row_ok.sum())}/{B}")
        assert bool(row_ok.all()), f"step {step}: largest difference {float(diff.max())}, branches outside the tolerance {torch.nonzero(~row_ok).flatten().tolist()}"
        sync_suffix_row(model, oracle, B, step)


MANY = dict(dim=256, n_layers=2, n_heads=2, vocab_size=320, multiple_of=128, max_batch_size=40, max_seq_len=8,
            max_prompt_seq_len=32)
MANY_GQA = dict(dim=512, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=384, multiple_of=128, max_batch_size=112,
                max_seq_len=8, max_prompt_seq_len=48)


@pytest.mark.parametrize("cfg,seed,B", [(MANY, 70, 17), (MANY, 71, 40), (MANY_GQA, 72, 33), (MANY_GQA, 73, 100)])
def test_decode_logits_above_16_branches(cfg, seed, B):
    _steps(cfg, seed, B, P=21, std=0.05, rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("forks", [{}, {2: (3, 9, 6), 4: (16, 0, 3)}])
@pytest.mark.parametrize("cfg,seed,B,P", [(MANY, 74, 17, 97), (MANY, 75, 37, 150), (MANY, 76, 40, 512), (MANY_GQA, 77, 65, 100), (MANY_GQA, 78, 100, 300), ("7b", 79, 70, 96),
                                          ("7b", 80, 100, 130), ("70b", 81, 40, 100)])
def test_decode_logits_behind_longer_prompts(cfg, seed, B, P, forks):
    """From 96 prompt rows on, where such steps take their attention in one launch (eight queries a workgroup; 16 with the heads of the 7B and the 70B
    architecture): per branch and step against the oracle, branches with rows of their own and branches that share an ancestor's."""
    cfg = {"7b": LAYER_7B, "70b": ARCH_70B_LAYER}.get(cfg, cfg) if isinstance(cfg, str) else cfg
    std = 0.05 if cfg["dim"] <= 512 else 0.02
    _steps(dict(cfg, n_layers=min(cfg["n_layers"], 2), max_batch_size=B, max_prompt_seq_len=P), seed, B, P, std=std, rtol=1e-2, atol=1e-2, steps=6, forks=forks)


ARCH_70B_LAYER = dict(dim=8192, n_layers=1, n_heads=64, n_kv_heads=8, vocab_size=512, multiple_of=4096,
                      ffn_dim_multiplier=1.3, max_batch_size=20, max_seq_len=8, max_prompt_seq_len=16)


@pytest.mark.parametrize("B,P", [(3, 9), (20, 9), (100, 2048)])
def test_70b_architecture_layer(B, P):
    """One layer with the 70B shapes (wq 8192x8192, wk/wv 1024x8192, w1/w3 28672x8192, w2 8192x28672, 8 query
    heads per KV head) through prefill and decode steps: GEMV at B=3, GEMM at B=20, and the workload of BASELINE
    configs[4] - 100 branches over a 2048-token shared prompt - at B=100."""
    cfg = dict(ARCH_70B_LAYER, max_batch_size=max(B, 20), max_prompt_seq_len=max(P, 16))
    assert O.ffn_hidden_dim(cfg["dim"], cfg["multiple_of"], cfg["ffn_dim_multiplier"]) == 28672
    _steps(cfg, 74, B, P=P, std=0.02, rtol=1e-2, atol=1e-2, steps=2 if P > 100 else 3)


def test_rmsnorm_inside_a_launch_whose_slices_do_not_fit():
    """The 70B shape's w1|w3 (K-slices of 4096 rows): up to three branches fit next to the rings, from four on each step is normalised on its way into the
    matrix core.  The same bits as with launches of RMSNorm's own."""
    _, _, model = _build(ARCH_70B_LAYER, 83, 0.02)
    gen = torch.Generator().manual_seed(84)
    prompt = torch.randint(0, 512, (1, 9), generator=gen).cuda()
    for B in (1, 3, 4, 10, 16):
        tok = torch.randint(0, 512, (B, 1), generator=gen).cuda()
        outs = []
        for inside in (True, False):
            model.norm_in_matmul = inside
            model.resetSeq()
            outs.append([model(prompt, 0).clone(), model(tok, 9).clone(), model(tok, 10).clone()])
        for x, y in zip(*outs):
            assert x.isfinite().all() and torch.equal(x, y), B


def test_rmsnorm_inside_wq_wk_wv_of_many_rows():
    """16 rows of 6144: more than fits next to the rings row by row.  The same bits as with launches of RMSNorm's own."""
    _, _, model = _build(dict(dim=6144, n_layers=2, n_heads=48, vocab_size=512, multiple_of=256, ffn_dim_multiplier=0.25, max_batch_size=16, max_seq_len=8,
                              max_prompt_seq_len=16), 87, 0.02)
    gen = torch.Generator().manual_seed(88)
    prompt, tok = torch.randint(0, 512, (1, 9), generator=gen).cuda(), torch.randint(0, 512, (16, 1), generator=gen).cuda()
    outs = []
    for inside in (True, False):
        model.norm_in_matmul = inside
        model.resetSeq()
        outs.append([model(prompt, 0).clone(), model(tok, 9).clone(), model(tok, 10).clone()])
    assert model._norm_in_ok and all(model._norm_in_ok.values())
    for x, y in zip(*outs):
        assert x.isfinite().all() and torch.equal(x, y)


@pytest.mark.parametrize("B", [2, 5, 16])
def test_norm_weights_that_are_not_aligned_to_16_bytes(B):
    """Launches of GEMVs that normalise themselves read 16 bytes of them at a time; such weights go to the launch of RMSNorm's own: the same bits."""
    _, _, model = _build(MANY, 85, 0.05)
    gen = torch.Generator().manual_seed(86)
    prompt, tok = torch.randint(0, 320, (1, 9), generator=gen).cuda(), torch.randint(0, 320, (B, 1), generator=gen).cuda()
    outs = []
    for offset in (0, 4):
        for layer in model.layers:
            for norm in (layer.attention_norm, layer.ffn_norm):
                buf = torch.empty(256 + offset, dtype=torch.float16, device="cuda:0")
                buf[offset:] = norm.weight
                norm.weight.data = buf[offset:]
        model.resetSeq()
        outs.append([model(prompt, 0).clone(), model(tok, 9).clone(), model(tok, 10).clone()])
    for x, y in zip(*outs):
        assert x.isfinite().all() and torch.equal(x, y)


LAYER_7B = dict(dim=4096, n_layers=2, n_heads=32, vocab_size=512, multiple_of=256, max_seq_len=8, max_prompt_seq_len=16)


@pytest.mark.parametrize("cfg,B,swiglu", [(LAYER_7B, 129, True), (LAYER_7B, 257, True), (LAYER_7B, 257, False), (LAYER_7B, 400, True), (ARCH_70B_LAYER, 641, True)])
def test_decode_above_128_branches(cfg, B, swiglu):
    """Decode steps of more branches than one row block of the GEMM holds: from 257 rows of the 7B shape (385 of the 70B one) the
    wq|wk|wv launch stores fp16 itself, from 641 rows of the 70B shape wo and w2 do too - no slabs are reserved for such launches."""
    cfg = dict(cfg, max_batch_size=B)
    P = 9
    oargs, sd, model = _build(cfg, 75, 0.02)
    model.swiglu_in_matmul = swiglu
    oracle = O.OracleTransformer(oargs, sd, dense=True)
    gen = torch.Generator().manual_seed(175)
    prompt = torch.randint(0, cfg["vocab_size"], (1, P), generator=gen)
    oracle.forward(prompt, 0)
    model(prompt.cuda(), 0)
    sync_prefix(model, oracle)
    for step in range(2):
        tok = torch.randint(0, cfg["vocab_size"], (B, 1), generator=gen)
        want = oracle.forward(tok, P + step).float()
        got = model(tok.cuda(), P + step).cpu().float()
        print(f"B={B} step {step}: largest logit difference {float((got - want).abs().max()):.4f}", flush=True)
        assert torch.allclose(got, want, rtol=1e-2, atol=1e-2)
        sync_suffix_row(model, oracle, B, step)


def _layer_pass(model, h, t, pages, from_qkv=1, **fields):
    """One decode step of a model of one layer by smh_decode_layer; fields: of its smh_pass, in place of the model's own."""
    from spec_mcts_amd import kernels as K
    p, B, dev = model.params, h.shape[0], h.device
    s = model._layer_struct(model.layers[0])
    run = K.LayerPass(s, B, h, *model._tables(dev), True)
    state = torch.tensor([s.prompt_len + t, t], dtype=torch.int32, device=dev)
    one = B * s.heads <= 16 * s.kv_heads
    run.decode_step((state[:1], state[1:]), K.attn_workspace(dev, B, s.heads, s.prompt_len), K.attn_qkv_workspace(dev, B, s.heads, s.prompt_len) if one else None,
                    p.max_seq_len, p.max_batch_size * p.max_seq_len, None, 0, 0, from_qkv)
    if pages is not None:
        run.p.pages, run.p.pages_stride = pages.data_ptr(), pages.stride(0)
    for name, value in fields.items():
        setattr(run.p, name, value)
    run.decode(s)
    return run.finish(s, model.norm.weight, model.norm.eps)


@pytest.mark.parametrize("heads,kv_heads,B,P,change", [(2, 2, 17, 100, "narrow table"), (4, 2, 40, 300, "narrow table"), (2, 2, 10, 800, "no row count"), (4, 2, 5, 300, "no row count"),
                                                       (2, 2, 10, 800, "small workspace"), (4, 2, 5, 900, "small workspace")])
def test_passes_that_only_some_forms_of_the_attention_take(heads, kv_heads, B, P, change):
    """A table of fewer columns than a branch has rows (t lies in it), no number of cache rows, a workspace for the one-launch form only: what the
    forms a layer is usually given to ask for, and others do not.  The result is that of the form that takes it, bit for bit."""
    cfg = dict(dim=128 * heads, n_layers=1, n_heads=heads, n_kv_heads=kv_heads, vocab_size=320, multiple_of=128, max_batch_size=B, max_seq_len=8, max_prompt_seq_len=1024)
    _, _, model = _build(cfg, 90 + B, 0.05)
    att, t = model.layers[0].attention, 3
    g = torch.Generator(device="cuda:0").manual_seed(B)
    normal = lambda *shape: torch.randn(shape, generator=g, device="cuda:0", dtype=torch.float16)
    att.cache_prompt_k[0, :P], att.cache_prompt_v[0, :P] = normal(P, kv_heads, 128), normal(P, kv_heads, 128)
    att.cache_prompt_len = P
    h = normal(B, cfg["dim"])
    rows = torch.arange(B, dtype=torch.int32, device="cuda:0")[:, None] * 8 + torch.arange(8, dtype=torch.int32, device="cuda:0")
    for i in range(t):
        _layer_pass(model, normal(B, cfg["dim"]), i, None)
    if change == "narrow table":
        want = _layer_pass(model, h, t, rows, from_qkv=0)
        got = _layer_pass(model, h, t, rows[:, :6].contiguous())
    else:                                              # (with neither, only the one-launch form takes it)
        want = _layer_pass(model, h, t, rows, attn_ws=None, cache_rows=0)
        got = _layer_pass(model, h, t, rows, **(dict(cache_rows=0) if change == "no row count" else dict(attn_ws_bytes=256)))
    torch.cuda.synchronize()
    assert want.isfinite().all() and torch.equal(got, want)


@pytest.mark.parametrize("B,P", [(5, 96), (6, 130), (11, 300), (16, 100), (17, 97), (32, 96), (5, 95), (16, 95), (24, 95)])
def test_few_branches_behind_a_prompt(B, P):
    """Layers of the 7B shape for 5 .. 32 branches: from 96 prompt rows on 128-column blocks and SwiGLU inside w1|w3 (one row tile up to 16 branches, two from
    17 on), before that GEMVs, or slabs of w1|w3.  Against the same tokens among 48 branches, which take the blocks anyway: no more than flips of a
    rounding apart.  (Against the oracle: the test below.)"""
    cfg = dict(LAYER_7B, max_batch_size=48, max_prompt_seq_len=320)
    _, _, model = _build(cfg, 77, 0.02)
    att = [layer.attention for layer in model.layers]
    g = torch.Generator(device="cuda:0").manual_seed(B + P)
    for a in att:
        for c in (a.cache_prompt_k, a.cache_prompt_v):
            c[0, :P] = torch.randn((P, 32, 128), generator=g, device="cuda:0", dtype=torch.float16)
        a.cache_prompt_len = P
    tok = torch.randint(0, cfg["vocab_size"], (B, 1), generator=g, device="cuda:0")
    outs = []
    for step in range(2):                              # (the second reads what the first appended)
        got = model(tok, P + step)[:, 0].float()
        rows = [(a.cache_k.clone(), a.cache_k_s.clone(), a.cache_v.clone(), a.cache_v_s.clone()) for a in att]
        wide = model(tok.repeat(48 // B + 1, 1)[:48], P + step)[:B, 0].float()
        for a, saved in zip(att, rows):                # (what the wider step appended, taken back)
            for c, r in zip((a.cache_k, a.cache_k_s, a.cache_v, a.cache_v_s), saved):
                c.copy_(r)
        outs.append((got, wide))
    for got, wide in outs:
        assert got.isfinite().all()
        # fp16 roundings at the same points, fp32 sums in another order: a flip now and then moves a logit by a few 2^-11 of the deviation, two layers deep
        assert float((got - wide).norm() / wide.norm()) < 4e-3


LAYER_8B = dict(LAYER_7B, n_kv_heads=8, multiple_of=1024, ffn_dim_multiplier=1.3)


def _form(cfg, B, P):
    """smh_decode_layer_form of a model's layers behind P prompt rows, and the slabs of wq|wk|wv, wo, w1|w3 and w2"""
    from spec_mcts_amd import _lib
    layer, slabs = _lib.SmhLayer(), (ctypes.c_int * 4)()
    layer.dim, layer.heads, layer.kv_heads, layer.prompt_len = cfg["dim"], cfg["n_heads"], cfg.get("n_kv_heads") or cfg["n_heads"], P
    layer.ffn = O.ffn_hidden_dim(cfg["dim"], cfg["multiple_of"], cfg.get("ffn_dim_multiplier"))
    return _lib.load().smh_decode_layer_form(layer, B, 1, slabs), list(slabs)


@pytest.mark.parametrize("forked", [False, True])
@pytest.mark.parametrize("cfg,B,P,form,slabs", [(LAYER_7B, 5, 96, 3, [2, 8, 0, 8]), (LAYER_7B, 10, 130, 3, [2, 8, 0, 8]), (LAYER_7B, 16, 97, 3, [2, 8, 0, 8]), (LAYER_7B, 24, 100, 2, [2, 8, 0, 8]),
                                                (LAYER_7B, 10, 95, 0, [10, 16, 5, 16]), (LAYER_8B, 5, 96, 3, [5, 8, 0, 8]), (LAYER_8B, 16, 129, 3, [5, 8, 0, 8]),
                                                (LAYER_8B, 9, 260, 3, [5, 8, 0, 8])])
def test_decode_logits_of_few_branches_behind_longer_prompts(cfg, B, P, form, slabs, forked):
    """5 .. 32 branches of the 7B shape, and of 32 heads over 8, on 128-column blocks with SwiGLU inside w1|w3 from 96 prompt rows on (asked of the library): per
    branch and step against the oracle, branches with rows of their own and branches that share an ancestor's."""
    assert _form(cfg, B, P) == (form, slabs)
    cfg = dict(cfg, n_layers=1, max_batch_size=B, max_prompt_seq_len=P)
    _steps(cfg, 91, B, P, std=0.02, rtol=1e-2, atol=1e-2, steps=5, forks={2: (1, 3, B - 3), 4: (B - 1, 0, 1)} if forked else {})


@pytest.mark.parametrize("cfg,P", [(LAYER_7B, 4), (LAYER_7B, 5), (LAYER_7B, 16), (LAYER_7B, 17), (LAYER_7B, 32), (LAYER_8B, 13)])
def test_prefill_of_few_rows(cfg, P):
    """Prompts of 5 .. 32 rows take the launches that as many branches behind a longer prompt do."""
    _steps(dict(cfg, n_layers=1, max_batch_size=2, max_prompt_seq_len=32), 92, 2, P, std=0.02, rtol=1e-2, atol=1e-2, steps=1)
