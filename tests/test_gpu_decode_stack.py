"""All layers of a decode step of a few branches in one launch (smh_decode_stack), against the oracle's dense restatement and
the layer-by-layer launches."""
import ctypes

import pytest
import torch

from oracle import q40_oracle as O
from tests.sync_state import sync_prefix, sync_suffix_row

# layers, dim, ffn columns / 256 -> where it can go wrong
CASES = [
    (dict(dim=256, n_layers=33, n_heads=2), 1, 1, 3),       # more layers than a launch holds; runs of two tiles, most workgroups without any
    (dict(dim=512, n_layers=2, n_heads=4), 2, 33, 4),       # two slices of the prompt, the second of one row
    (dict(dim=1024, n_layers=2, n_heads=8), 3, 131, 3),     # runs that touch two column units
    (dict(dim=1280, n_layers=1, n_heads=10), 4, 70, 3),     # the most rows; units that no number of equal runs divides
    (dict(dim=2048, n_layers=1, n_heads=16), 1, 300, 30),   # more own rows than the attention's waves take at once
]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,B,P,steps", CASES)
def test_stack_matches_the_oracle(shape, B, P, steps, monkeypatch):
    from spec_mcts_amd import ModelArgs, kernels as K
    from spec_mcts_amd.load_q40 import load_q40
    cfg = dict(shape, vocab_size=320, multiple_of=256, max_batch_size=5, max_seq_len=steps + 2, max_prompt_seq_len=320)
    std = 0.8 / shape["dim"] ** 0.5
    oargs = O.OracleArgs(**cfg)
    sd = O.random_q40_state_dict(oargs, seed=B + P, std=std)
    model = load_q40(dict(sd), ModelArgs(**cfg), device="cuda:0")
    model.decode_stack_min_prompt = 0                  # (behind short prompts too: the kernel, not the rule)
    oracle = O.OracleTransformer(oargs, sd, dense=True)
    calls = []
    monkeypatch.setattr(K.LayerPass, "decode_stack", lambda self, structs, ws, _f=K.LayerPass.decode_stack: (calls.append(len(structs)), _f(self, structs, ws)))
    gen = torch.Generator().manual_seed(P)
    prompt = torch.randint(0, cfg["vocab_size"], (1, P), generator=gen)
    oracle.forward(prompt, 0)
    model(prompt.cuda(), 0)
    sync_prefix(model, oracle)
    for step in range(steps):
        tok = torch.randint(0, cfg["vocab_size"], (B, 1), generator=gen)
        want = oracle.forward(tok, P + step).float()
        got = model(tok.cuda(), P + step)
        assert calls.pop() == cfg["n_layers"]
        model.decode_stack = False
        layers = model(tok.cuda(), P + step).float().cpu()
        model.decode_stack = True
        again = model(tok.cuda(), P + step)
        calls.clear()
        assert torch.equal(got, again), "the order of the sums depends on nothing but the sizes"
        got = got.float().cpu()
        # Both round to fp16 at the same points and differ from the oracle in the order of fp32 sums alone, so by flipped roundings that
        # add up over the layers: as far from the oracle as the layers' launches are, with room for the flips that fall the other way.
        far, near = float((got - want).norm() / want.norm()), float((layers - want).norm() / want.norm())
        print("step %d: from the oracle %.2e, layer by layer %.2e" % (step, far, near))
        assert far <= 2 * near + 2e-3
        sync_suffix_row(model, oracle, B, step)
    # a fork: the branches share their ancestor's rows through the page table
    model.fork(0, B, 1)
    tok = tok[:1].expand(B + 1, 1).cuda()
    if B < K.DECODE_STACK_MAX_ROWS:
        got = model(tok, P + steps)
        assert calls and torch.equal(got[0], got[B])


def test_refused_sizes_and_arguments():
    """No workspace, and an error instead of a launch, for what the kernel is not made for (no GPU needed)."""
    from spec_mcts_amd import _lib
    lib = _lib.load()

    def layer(dim, heads, kv_heads, ffn, P=7):
        s = _lib.SmhLayer()
        s.dim, s.heads, s.kv_heads, s.ffn, s.prompt_len = dim, heads, kv_heads, ffn, P
        return s

    for rows in (1, 2, 3, 4):
        for dim, heads, ffn in ((4096, 32, 11008), (5120, 40, 13824), (256, 2, 768)):
            assert lib.smh_decode_stack_workspace_bytes(layer(dim, heads, heads, ffn), rows) > 0
    for rows, s in ((0, layer(4096, 32, 32, 11008)), (5, layer(4096, 32, 32, 11008)), (1, layer(8192, 64, 8, 28672)), (1, layer(4096, 32, 32, 11008 + 32)),
                    (1, layer(4096 + 128, 33, 33, 11008)), (1, layer(128, 1, 1, 256)), (1, layer(256, 0, 0, 256))):
        assert lib.smh_decode_stack_workspace_bytes(s, rows) == 0
        p = _lib.SmhPass()
        p.rows, p.smax = rows, 8
        for field in ("h", "pos_dev", "t_dev", "cos_tab", "sin_tab", "scratch"):
            setattr(p, field, 256)                     # (never read: the sizes are refused first)
        arr = (ctypes.POINTER(_lib.SmhLayer) * 1)(ctypes.pointer(s))
        assert lib.smh_decode_stack(arr, 1, p, 256, 1 << 30, None) != 0


def _pointers(dim=256, heads=2, ffn=768, P=7):
    from spec_mcts_amd import _lib
    s = _lib.SmhLayer()
    s.dim, s.heads, s.kv_heads, s.ffn, s.prompt_len = dim, heads, heads, ffn, P
    for i, (name, _) in enumerate(_lib.SmhLayer._fields_[6:-1]):
        setattr(s, name, 1 << 20 | i << 12)            # (never read)
    return s


@pytest.mark.parametrize("name,align", [(n, 16) for n in ("wq", "wk", "wv", "wo", "w1", "w2", "w3")] + [("prompt_k", 8), ("prompt_v", 8)]
                         + [(n, 4) for n in ("cache_k", "cache_v", "cache_ks", "cache_vs", "att_norm", "ffn_norm")])
def test_alignments_that_the_stack_takes(name, align):
    """... are asked for before the pass is built (no GPU needed): what is refused goes to the layers' own launches."""
    from spec_mcts_amd import kernels as K
    for at in (0, 1, 2):                               # in any layer
        layers = [_pointers() for _ in range(3)]
        assert K.decode_stack_layers(layers, 2) is not None
        good = getattr(layers[at], name)
        setattr(layers[at], name, good + align)
        assert K.decode_stack_layers(layers, 2) is not None
        setattr(layers[at], name, good + align // 2)
        assert K.decode_stack_layers(layers, 2) is None
        setattr(layers[at], name, None)
        assert K.decode_stack_layers(layers, 2) is None
    layers = [_pointers(P=0) for _ in range(2)]
    if name.startswith("prompt"):                      # without a prompt there is no cache to read
        setattr(layers[1], name, None)
        assert K.decode_stack_layers(layers, 2) is not None
    assert K.decode_stack_layers([_pointers(), _pointers(ffn=1024)], 2) is None
    assert K.decode_stack_layers([_pointers(), _pointers(P=-1)], 2) is None


def _offset(t, elements):
    """the same values, so many elements behind an aligned address"""
    buf = torch.empty(t.numel() + elements, dtype=t.dtype, device=t.device)
    out = buf[elements:].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("name,elements,stack", [("cache_k", 4, True), ("cache_v_s", 2, True), ("cache_prompt_k", 4, True), ("cache_prompt_v", 2, False)])
def test_views_as_caches(name, elements, stack, monkeypatch):
    """A cache that is a view at an offset runs, in one launch where the kernel's loads allow it, else layer by layer."""
    from spec_mcts_amd import ModelArgs, kernels as K
    from spec_mcts_amd.load_q40 import load_q40
    cfg = dict(dim=512, n_layers=2, n_heads=4, vocab_size=320, multiple_of=256, max_batch_size=2, max_seq_len=4, max_prompt_seq_len=128)
    model = load_q40(dict(O.random_q40_state_dict(O.OracleArgs(**cfg), seed=5, std=0.04)), ModelArgs(**cfg), device="cuda:0")
    tokens = torch.randint(0, 320, (2, 101), generator=torch.Generator().manual_seed(7)).cuda()
    model(tokens[:1, :100], 0)
    calls = []
    monkeypatch.setattr(K.LayerPass, "decode_stack", lambda self, layers, ws, _f=K.LayerPass.decode_stack: (calls.append(len(layers)), _f(self, layers, ws)))
    one = model(tokens[:, 100:], 100)
    assert calls == [2]
    model.decode_stack = False
    want = one if stack else model(tokens[:, 100:], 100)
    model.decode_stack = True
    att = model.layers[1].attention
    setattr(att, name, _offset(getattr(att, name), elements))
    got = model(tokens[:, 100:], 100)
    assert calls == [2] + [2] * stack and torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("eps", [(1e-5, 1e-3, 1e-3), (float("nan"), 1e-5, 1e-5), (1e-5, 1e-5, float("nan"))])
def test_layers_of_different_eps(eps):
    """take a launch each time it changes; one that is NaN (which equals nothing, itself included) a launch of its own"""
    from spec_mcts_amd import ModelArgs
    from spec_mcts_amd.load_q40 import load_q40
    cfg = dict(dim=512, n_layers=3, n_heads=4, vocab_size=320, multiple_of=256, max_batch_size=2, max_seq_len=4, max_prompt_seq_len=128)
    model = load_q40(dict(O.random_q40_state_dict(O.OracleArgs(**cfg), seed=6, std=0.04)), ModelArgs(**cfg), device="cuda:0")
    tokens = torch.randint(0, 320, (2, 101), generator=torch.Generator().manual_seed(8)).cuda()
    model(tokens[:1, :100], 0)
    for layer, e in zip(model.layers, eps):
        layer.ffn_norm.eps = e
    got = model(tokens[:, 100:], 100).float()
    model.decode_stack = False
    want = model(tokens[:, 100:], 100).float()
    if any(e != e for e in eps):
        assert got.isnan().all() and want.isnan().all()
    else:
        assert float((got - want).norm() / want.norm()) < 4e-3


def _model(cfg, seed, std=0.04):
    from spec_mcts_amd import ModelArgs
    from spec_mcts_amd.load_q40 import load_q40
    oargs = O.OracleArgs(**cfg)
    sd = O.random_q40_state_dict(oargs, seed=seed, std=std)
    model = load_q40(dict(sd), ModelArgs(**cfg), device="cuda:0")
    model.decode_stack_min_prompt = 0
    return oargs, sd, model


# workgroups launched, us the first wait for the others (0: the list is closed before most have started, and ids go by arrival)
@pytest.mark.gpu
@pytest.mark.parametrize("workgroups,join_us", [(1, 50), (2, 50), (7, 50), (100, 50), (255, 50), (256, 0), (40, 0), (256, 50)])
def test_any_number_of_workgroups_finishes_the_work(workgroups, join_us, monkeypatch):
    """Fewer workgroups than tasks deal themselves the rest: the same bits from however many took part."""
    from spec_mcts_amd import kernels as K
    from spec_mcts_amd._lib import check
    _, _, model = _model(dict(dim=768, n_layers=2, n_heads=6, vocab_size=320, multiple_of=256, max_batch_size=4, max_seq_len=12, max_prompt_seq_len=128), seed=9)
    tokens = torch.randint(0, 320, (3, 110), generator=torch.Generator().manual_seed(9)).cuda()
    model(tokens[:1, :100], 0)
    calls = []

    def launch(self, layers, ws):
        calls.append(workgroups)
        check(self.lib.smh_decode_stack_of(layers, len(layers), self.p, ws.data_ptr(), ws.numel(), workgroups, join_us, self.stream), "smh_decode_stack_of")

    for i in range(5):                                 # several steps on one workspace, between launches of all workgroups
        want = model(tokens[:, 100 + i:101 + i], 100 + i)
        caches = [model.layers[1].attention.cache_k.clone(), model.layers[1].attention.cache_v.clone()]
        with monkeypatch.context() as m:
            m.setattr(K.LayerPass, "decode_stack", launch)
            got = model(tokens[:, 100 + i:101 + i], 100 + i)
        assert calls.pop() == workgroups and torch.equal(got, want) and bool(got.isfinite().all())
        assert torch.equal(caches[0], model.layers[1].attention.cache_k) and torch.equal(caches[1], model.layers[1].attention.cache_v)


def test_number_of_workgroups_is_checked():
    from spec_mcts_amd import _lib, kernels as K
    p = _lib.SmhPass()
    p.rows, p.smax, p.h = 2, 8, 256
    layers = [_pointers()]
    for workgroups, join_us in ((0, 50), (257, 50), (-1, 50), (256, -1), (256, 1000001)):
        assert _lib.load().smh_decode_stack_of(K.decode_stack_layers(layers, 2), 1, p, 256, 1 << 30, workgroups, join_us, None) != 0
        assert b"workgroups" in _lib.load().smh_last_error_string()


@pytest.mark.gpu
@pytest.mark.parametrize("B,forks", [(2, [(0, 1, 1)]), (3, [(0, 2, 1), (2, 1, 1)]), (4, [(1, 2, 2), (3, 0, 1)])])
def test_rows_through_the_page_table_match_the_oracle(B, forks, monkeypatch):
    """Branches that read their ancestors' rows through the page table, and their own behind them (as test_stack_matches_the_oracle)."""
    from spec_mcts_amd import kernels as K
    P, steps = 45, 2
    cfg = dict(dim=512, n_layers=2, n_heads=4, vocab_size=320, multiple_of=256, max_batch_size=5, max_seq_len=40, max_prompt_seq_len=64)
    oargs, sd, model = _model(cfg, seed=20 + B, std=0.8 / 512 ** 0.5)
    oracle = O.OracleTransformer(oargs, sd, dense=True)
    calls = []
    monkeypatch.setattr(K.LayerPass, "decode_stack", lambda self, layers, ws, _f=K.LayerPass.decode_stack: (calls.append(len(layers)), _f(self, layers, ws)))
    gen = torch.Generator().manual_seed(B)
    prompt = torch.randint(0, 320, (1, P), generator=gen)
    oracle.forward(prompt, 0)
    model(prompt.cuda(), 0)
    sync_prefix(model, oracle)
    at = 0
    for fork in [None] + forks:
        if fork is not None:
            model.fork(*fork)
            oracle.fork(*fork)
            assert model._pages(torch.device("cuda:0")) is not None
        for _ in range(steps):
            tok = torch.randint(0, 320, (B, 1), generator=gen)
            want = oracle.forward(tok, P + at).float()
            got = model(tok.cuda(), P + at)
            assert calls.pop() == cfg["n_layers"]
            model.decode_stack = False
            layers = model(tok.cuda(), P + at).float().cpu()
            model.decode_stack = True
            got = got.float().cpu()
            far, near = float((got - want).norm() / want.norm()), float((layers - want).norm() / want.norm())
            print("row %d: from the oracle %.2e, layer by layer %.2e" % (at, far, near))
            assert far <= 2 * near + 2e-3              # (as above)
            sync_suffix_row(model, oracle, B, at)
            at += 1


def _poison(model, kind):
    """Writes something that is not finite where one decode step reads it; returns the branches that must not notice."""
    att, inf, nan = model.layers[0].attention, float("inf"), float("nan")
    p, H = model.params, att.n_kv_heads
    own = lambda c, w: c.view(p.max_batch_size, p.max_seq_len, H, w)
    if kind == "query":                                # of branch 1: token 7's embedding
        model.tok_embeddings.weight.data[7, 3] = nan
    elif kind == "own_k_nan":
        own(att.cache_k_s, 2)[1, 2, 1] = nan
    elif kind == "own_v_inf":
        own(att.cache_v_s, 2)[1, 2, 1] = inf
    elif kind == "behind_the_rows":                    # rows that no branch has yet
        own(att.cache_k_s, 2)[:, 4:], own(att.cache_v_s, 2)[:, 4:] = nan, inf
        att.cache_prompt_k[0, 70:], att.cache_prompt_v[0, 70:] = nan, inf
        return [0, 1, 2]
    elif kind == "prompt_k_inf":                       # the last row of an odd number: a score of +inf or -inf, by the query's sign
        att.cache_prompt_k[0, 69, 2, 5] = inf
        return []
    elif kind == "prompt_k_lowest":
        att.cache_prompt_k[0, :, 2] = -65504.0
        return []
    elif kind == "prompt_v_inf":
        att.cache_prompt_v[0, 33, 2, 5] = -inf
        return []
    return [0, 2]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["query", "own_k_nan", "own_v_inf", "behind_the_rows", "prompt_k_inf", "prompt_k_lowest", "prompt_v_inf"])
def test_values_that_are_not_finite_stay_where_they_are(kind):
    """A branch with a NaN or an infinity among what it reads has the result that the layers' launches give it; the others' bits do not move."""
    cfg = dict(dim=512, n_layers=1, n_heads=4, vocab_size=320, multiple_of=256, max_batch_size=3, max_seq_len=8, max_prompt_seq_len=96)
    _, _, model = _model(cfg, seed=31, std=0.8 / 512 ** 0.5)
    gen = torch.Generator().manual_seed(31)
    model(torch.randint(0, 320, (1, 70), generator=gen).cuda(), 0)
    tokens = torch.tensor([[3], [7], [11]]).cuda()
    for i in range(4):
        clean = model(tokens, 70 + i)
    untouched = _poison(model, kind)
    got = model(tokens, 73)
    model.decode_stack = False
    want = model(tokens, 73)
    for b in untouched:
        assert torch.equal(got[b], clean[b]), b
    finite = [bool(want[b].isfinite().all()) for b in range(3)]
    print(kind, finite)
    assert [bool(got[b].isfinite().all()) for b in range(3)] == finite
    assert torch.equal(got.isnan(), want.isnan())
    for b in range(3):
        if finite[b]:
            assert float((got[b].float() - want[b].float()).norm() / want[b].float().norm()) < 4e-3
