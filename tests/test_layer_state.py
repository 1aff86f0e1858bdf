"""What a layer call reads of a transformer block is looked at again at every pass, natively (kernels.layer_state; no GPU needed)."""
import pytest
import torch
from torch import nn

CFG = dict(dim=256, n_layers=1, n_heads=2, vocab_size=320, multiple_of=256, max_batch_size=2, max_seq_len=4, max_prompt_seq_len=8)
LINEARS = ("attention.wq", "attention.wk", "attention.wv", "attention.wo", "feed_forward.w1", "feed_forward.w2", "feed_forward.w3")


def _block():
    from spec_mcts_amd import ModelArgs, Transformer, kernels as K
    model = Transformer(ModelArgs(**CFG))
    block = model.layers[0]
    for name in LINEARS:
        lin = block.get_submodule(name)
        lin._tiled = K.TiledQ40(lin.w.clone(), lin.shape[1], lin.shape[0])
    return model, block


def _replace(owner, name):
    setattr(owner, name, getattr(owner, name).clone())


def _new_parameter(norm):
    norm.weight = nn.Parameter(norm.weight.detach().clone())


def _new_data(norm):
    norm.weight.data = norm.weight.detach().clone()


CHANGES = ([("a cache", lambda b, n=n: _replace(b.attention, n)) for n in ("cache_prompt_k", "cache_prompt_v", "cache_k", "cache_k_s", "cache_v", "cache_v_s")]
           + [("%s of %s" % (a, n), lambda b, n=n, a=a: _replace(b.get_submodule(n), a)) for n in LINEARS for a in ("w", "s")]
           + [("tiled buffer of " + n, lambda b, n=n: _replace(b.get_submodule(n)._tiled, "buf")) for n in LINEARS]
           + [("no tiled copy of " + n, lambda b, n=n: b.get_submodule(n).invalidate()) for n in LINEARS]
           + [("parameter of " + n, lambda b, n=n: _new_parameter(getattr(b, n))) for n in ("attention_norm", "ffn_norm")]
           + [("data of " + n, lambda b, n=n: _new_data(getattr(b, n))) for n in ("attention_norm", "ffn_norm")]
           + [("eps of " + n, lambda b, n=n: setattr(getattr(b, n), "eps", torch.tensor(1e-3))) for n in ("attention_norm", "ffn_norm")]
           + [("another linear", lambda b: setattr(b.attention, "wo", _block()[1].attention.wo)),
              ("another attention", lambda b: setattr(b, "attention", _block()[1].attention)),
              ("another norm", lambda b: setattr(b, "ffn_norm", _block()[1].ffn_norm))])


@pytest.mark.parametrize("change", [c for _, c in CHANGES], ids=[n for n, _ in CHANGES])
def test_every_change_is_seen(change):
    from spec_mcts_amd import kernels as K
    _, block = _block()
    block.attention.cache_prompt_len = 3
    key = bytearray(K.layer_key_bytes())
    assert K.layer_state(block, key) == -1 - 3             # nothing known yet
    assert K.layer_state(block, key) == 3
    before = [getattr(block.attention, n) for n in ("wo", "cache_k")], block.attention      # (alive: no address comes back)
    keep = [(block.get_submodule(n).w, block.get_submodule(n).s, block.get_submodule(n)._tiled, block.get_submodule(n)._tiled.buf) for n in LINEARS]
    norms = [block.attention_norm, block.ffn_norm, block.attention_norm.weight.detach(), block.ffn_norm.weight.detach()]
    caches = [v for v in vars(block.attention).values() if isinstance(v, torch.Tensor)]
    change(block)
    assert K.layer_state(block, key) == -1 - block.attention.cache_prompt_len
    assert K.layer_state(block, key) == block.attention.cache_prompt_len
    del before, keep, norms, caches


def test_the_prompt_length_is_read_and_checked():
    from spec_mcts_amd import kernels as K
    _, block = _block()
    key = bytearray(K.layer_key_bytes())
    K.layer_state(block, key)
    for rows in (0, 5, CFG["max_prompt_seq_len"]):
        block.attention.cache_prompt_len = rows
        assert K.layer_state(block, key) == rows
    block.attention.cache_prompt_len = CFG["max_prompt_seq_len"] + 1
    with pytest.raises(AssertionError):
        K.layer_state(block, key)
    with pytest.raises(AssertionError):
        K.layer_state(block, bytearray(8))


def test_attributes_kept_elsewhere_are_found():
    """weights that are no parameters and caches that are buffers: what attribute access finds"""
    from spec_mcts_amd import kernels as K
    _, block = _block()
    norm = block.ffn_norm
    weight = norm.weight.detach().clone()
    del norm.weight
    norm.weight = weight
    cache = block.attention.cache_k.clone()
    del block.attention.cache_k
    block.attention.register_buffer("cache_k", cache)
    key = bytearray(K.layer_key_bytes())
    K.layer_state(block, key)
    assert K.layer_state(block, key) == 0
    block.attention.cache_k = cache.clone()
    assert K.layer_state(block, key) == -1
    del block.attention.wq
    with pytest.raises(AttributeError):
        K.layer_state(block, key)


def test_an_unchanged_layer_costs_no_lookup_through_the_modules(monkeypatch):
    """A step in one launch waits for the look at all layers: nothing of it goes through nn.Module.__getattr__."""
    from spec_mcts_amd import _lib, kernels as K
    model, block = _block()
    monkeypatch.setattr(K, "layer_struct", lambda *a: _lib.SmhLayer())
    for name in LINEARS:
        lin = block.get_submodule(name)
        monkeypatch.setattr(lin, "operand", lambda tiled=True, lin=lin: lin._tiled)
    block.attention.cache_prompt_len = 2
    first = model._layer_struct(block)
    looked = []
    found = nn.Module.__getattr__
    monkeypatch.setattr(nn.Module, "__getattr__", lambda self, name: (looked.append(name), found(self, name))[1])
    again = model._layer_struct(block)
    assert again is first and again.prompt_len == 2 and looked == []
