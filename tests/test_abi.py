"""The C-ABI library loads and exports every symbol include/smh.h declares (no GPU needed)."""
import ctypes
import os
import re
import shutil
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "smh.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(smh_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_are_exported_and_bound():
    from spec_mcts_amd import _lib
    names = _declared()
    assert len(names) >= 15
    lib = _lib.load()
    for n in names:
        assert hasattr(lib, n), f"{n} declared in smh.h but not exported by libsmh.so"
        assert n in _lib.SIGNATURES, f"{n} has no ctypes signature in spec_mcts_amd/_lib.py"
    assert sorted(_lib.SIGNATURES) == names
    assert lib.smh_version() == 1


def test_argument_errors_are_reported_without_a_gpu():
    from spec_mcts_amd import _lib
    lib = _lib.load()
    # N not a multiple of 128 is rejected before anything touches the device
    st = lib.smh_q40_gemv(None, 1, 64, 64, None, None, 100, None, 100, 0, None, 0, None, 0, None)
    assert st < 0 and b"multiple of 128" in lib.smh_last_error_string()
    st = lib.smh_q40_quantize(None, None, None, 3, None)
    assert st < 0 and b"even" in lib.smh_last_error_string()
    with pytest.raises(_lib.SmhError):
        _lib.check(st, "smh_q40_quantize")
    assert lib.smh_q40_matmul_workspace_bytes(16, 4096) >= 16 * 16 * 4096 * 4
    import ctypes
    n = (ctypes.c_int * 3)(4096, 4096, 4096)
    ks = lib.smh_q40_matmul_plan(1, 4096, 3, n)
    assert 1 <= ks <= 16
    assert lib.smh_q40_matmul_plan(1, 4096, 1, (ctypes.c_int * 1)(100)) < 0      # N not a multiple of 128
    assert lib.smh_attn_workspace_bytes(64, 32, 1024) >= 32 * 64 * 32 * 130 * 4
    # SwiGLU inside the gate|up launch: 17 .. 128 rows, K a multiple of 64, at most 16384 columns per weight
    assert lib.smh_q40_swiglu_fits(100, 4096, 11008) == 1 and lib.smh_q40_swiglu_fits(16, 4096, 11008) == 0
    assert lib.smh_q40_swiglu_fits(100, 4096, 28672) == 0 and lib.smh_q40_swiglu_fits(100, 4096, 1024) == 0
    st = lib.smh_q40_matmul_tiled_swiglu(None, 5, 4096, 4096, None, None, 11008, None, 11008, None)
    assert st < 0 and b"17 .. 128" in lib.smh_last_error_string()
    # the entry point without a workspace refuses shapes beyond its static array before anything touches the device
    assert lib.smh_attn_static_scratch_bytes() == 16 << 20
    st = lib.smh_shared_prefix_attn_static(None, None, 4096, 64, 64, 128, None, None, 4096, 0, None, None, None, None, 0, None, 0,
                                           None, None, None)
    assert st < 0 and b"static array holds" in lib.smh_last_error_string()


@pytest.mark.parametrize("name,align", [("slabs", 16), ("prefix_k", 16), ("prefix_v", 16), ("out", 8), ("cos", 8), ("sin", 8), ("cache_k", 8), ("cache_v", 8), ("cache_ks", 4),
                                        ("cache_vs", 4), ("P", 0), ("cache_rows", 0), ("B", 0)])
def test_tile_attention_refuses_what_its_loads_cannot_take(name, align):
    """... before anything touches the device: the alignment of every tensor, sizes past 32-bit offsets, more tiles than a grid has."""
    from spec_mcts_amd import _lib
    lib = _lib.load()
    a = dict(slabs=1 << 20, ksplit=2, out=1 << 21, B=17, H=4, Hkv=4, D=128, cos=1 << 22, sin=1 << 22, pos=1 << 12, prefix_k=1 << 23, prefix_v=1 << 23, P=100,
             cache_k=1 << 24, cache_ks=1 << 25, cache_v=1 << 24, cache_vs=1 << 25, Smax=8, t=1 << 12, pages=1 << 13, pages_stride=8, cache_rows=136, stream=None)
    if align:
        a[name] += align // 2
    else:
        a.update({"P": dict(P=1 << 22), "cache_rows": dict(cache_rows=1 << 24), "B": dict(B=65535, H=68, cache_rows=65535 * 8)}[name])
    assert lib.smh_shared_prefix_attn_qkv_tiles(*a.values()) < 0
    assert {"P": b"32-bit", "cache_rows": b"32-bit", "B": b"grid"}.get(name, b"%d-byte aligned" % align) in lib.smh_last_error_string()


def _tile_tensors():
    from spec_mcts_amd import kernels as K
    half, i8, i32 = torch.float16, torch.int8, torch.int32
    B, H, Hkv, P, Smax = 5, 4, 2, 9, 8
    cache = lambda n, dtype: torch.zeros((B, Smax, Hkv, n), dtype=dtype)
    return dict(p=K.PartialProduct(torch.zeros((2, B, (H + 2 * Hkv) * 128)), 2, B, (H + 2 * Hkv) * 128), H=H, Hkv=Hkv, D=128, cos=torch.zeros((64, 64), dtype=half),
                sin=torch.zeros((64, 64), dtype=half), pos_dev=torch.zeros(1, dtype=i32), prefix_k=torch.zeros((P, Hkv, 128), dtype=half),
                prefix_v=torch.zeros((P, Hkv, 128), dtype=half), P=P, cache_k=cache(64, i8), cache_ks=cache(2, half), cache_v=cache(64, i8), cache_vs=cache(2, half),
                Smax=Smax, t_dev=torch.zeros(1, dtype=i32))


@pytest.mark.parametrize("name,change", [(n, f) for n in ("cos", "sin") for f in ("float", "strided", "narrow")] + [("pos_dev", "long"), ("t_dev", "long")]
                         + [(n, f) for n in ("prefix_k", "prefix_v") for f in ("float", "strided", "short", "narrow")]
                         + [(n, f) for n in ("cache_k", "cache_v", "cache_ks", "cache_vs") for f in ("float", "strided", "short")] + [(None, None)])
def test_tile_attention_checks_its_tensors(name, change, monkeypatch):
    """kernels.shared_prefix_attn_qkv_tiles raises where a tensor is of another type, stride or size than the kernel reads (no GPU needed: the library is
    stood in for)."""
    from spec_mcts_amd import _lib, kernels as K
    calls = []
    monkeypatch.setattr(_lib, "load", lambda: type("Lib", (), {"smh_shared_prefix_attn_qkv_tiles": lambda self, *a: calls.append(a) or 0})())
    monkeypatch.setattr(K, "_need_gpu", lambda *a: None)
    monkeypatch.setattr(K, "_stream", lambda: None)
    t = _tile_tensors()
    if name is not None:
        x = t[name]
        t[name] = {"float": lambda: x.float(), "long": lambda: x.long(), "strided": lambda: torch.stack((x, x), -1)[..., 0], "short": lambda: x[:-1],
                   "narrow": lambda: x[..., :-8].contiguous()}[change]()
        with pytest.raises(AssertionError):
            K.shared_prefix_attn_qkv_tiles(**t)
        assert not calls
    else:
        assert K.shared_prefix_attn_qkv_tiles(**t).shape == (5, 4, 128) and len(calls) == 1


def test_kernels_know_their_memory(tmp_path):
    """No flat load or store in any kernel: through a pointer of which the compiler does not know whether it is to global memory or to LDS, every access
    is waited for with both (a direct product of 300 rows took 1.5 % longer with flat stores)."""
    from spec_mcts_amd import build
    objdump = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(objdump) or not os.path.exists(build.LIB):
        pytest.skip("no disassembler, or nothing built")
    shutil.copy(build.LIB, tmp_path / "lib.so")
    subprocess.run([objdump, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    parts = sorted(tmp_path.glob("lib.so.*gfx950"))
    assert parts
    for part in parts:
        text = subprocess.run([objdump, "-d", part], check=True, capture_output=True, text=True).stdout
        assert "global_load" in text
        assert [l for l in text.splitlines() if "\tflat_" in l] == []


def test_matmul_plans_fit_the_workspace_the_library_asks_for():
    """the slabs of any planned launch (even split, or runs of steps across column units above 16 rows) fit the bytes
    smh_q40_matmul_workspace_bytes returns for the largest batch and width, and never exceed 16 slices"""
    from spec_mcts_amd import _lib
    lib = _lib.load()
    widths = ([4096], [4096, 4096, 4096], [11008, 11008], [11008], [32128], [8192, 1024, 1024], [28672, 28672], [16640, 16640],
              [7680, 7680, 7680], [128], [256, 128, 128])
    for K in (32, 256, 1024, 2048, 4096, 8192, 11008, 28672):
        for ns in widths:
            n = (ctypes.c_int * len(ns))(*ns)
            for M in (1, 2, 10, 16, 17, 64, 100, 128):
                for plan in (lib.smh_q40_matmul_plan, lib.smh_q40_matmul_plan_tiled):
                    ks = plan(M, K, len(ns), n)
                    assert 1 <= ks <= 16, (M, K, ns, ks)
                    assert ks * M * sum(ns) * 4 <= lib.smh_q40_matmul_workspace_bytes(M, sum(ns)), (M, K, ns, ks)
                if M <= 16:
                    assert lib.smh_q40_matmul_plan(M, K, len(ns), n) == lib.smh_q40_matmul_plan_tiled(M, K, len(ns), n)
    # the plans the GPU tests and the design notes name: checkpoint layout ...
    three, two, one = (ctypes.c_int * 3)(4096, 4096, 4096), (ctypes.c_int * 2)(11008, 11008), (ctypes.c_int * 1)(4096)
    assert lib.smh_q40_matmul_plan(100, 4096, 2, two) == 4      # range cut: 256 runs of 43 steps
    assert lib.smh_q40_matmul_plan(100, 4096, 3, three) == 5
    # ... and tiled weights at 100 rows: 128-column blocks with two K-groups a workgroup
    assert lib.smh_q40_matmul_plan_tiled(100, 4096, 1, one) == 4         # wo: 32 blocks x 2 row blocks x 4 slices
    assert lib.smh_q40_matmul_plan_tiled(100, 11008, 1, one) == 8        # w2: 32 blocks x 8 slices
    assert lib.smh_q40_matmul_plan_tiled(100, 4096, 3, three) == 2       # wq|wk|wv: 96 blocks x 2 slices
    assert lib.smh_q40_matmul_plan_tiled(100, 4096, 2, two) == 1         # w1|w3: 172 blocks, K uncut
    assert lib.smh_q40_matmul_plan_tiled(32, 4096, 2, two) == 4          # wide and at most 64 rows: the 256-column units' plan


def test_host_quantiser_matches_oracle():
    """spec_mcts_amd.quant (the converter's quantiser) against the oracle on the host"""
    import torch
    from oracle import q40_oracle as O
    from spec_mcts_amd import quant
    g = torch.Generator().manual_seed(5)
    v = (torch.randn((256, 128), generator=g) * 0.02).to(torch.float16)
    w, s, shp = quant.quantize_linear_weight(v)
    w2, s2, shp2 = O.quantize_weight(v)
    assert torch.equal(w, w2) and torch.equal(s, s2) and shp == shp2
    assert torch.equal(quant.dequantize_q40_torch(w, s, 64, (128, 256)), O.dequantize_q40(w, s, 64, (128, 256)))
    vb = v.to(torch.bfloat16)
    wb, sb = quant.quantize_q40_torch(vb.t(), 64)
    wb2, sb2 = O.quantize_q40(vb.t(), 64)
    assert torch.equal(wb, wb2) and torch.equal(sb, sb2)


def test_converter_and_loader_host_logic():
    import torch
    from spec_mcts_amd import fp16_to_int4 as C
    from spec_mcts_amd.load_q40 import load_q40
    from spec_mcts_amd import ModelArgs
    g = torch.Generator().manual_seed(6)
    hf = {"model.embed_tokens.weight": torch.randn((320, 256), generator=g).half(),
          "model.norm.weight": torch.ones(256).half(), "lm_head.weight": torch.randn((320, 256), generator=g).half()}
    for name, shape in (("self_attn.q_proj", (256, 256)), ("self_attn.k_proj", (256, 256)), ("self_attn.v_proj", (256, 256)),
                        ("self_attn.o_proj", (256, 256)), ("mlp.gate_proj", (768, 256)), ("mlp.down_proj", (256, 768)),
                        ("mlp.up_proj", (768, 256))):
        hf[f"model.layers.0.{name}.weight"] = (torch.randn(shape, generator=g) * 0.02).half()
    hf["model.layers.0.input_layernorm.weight"] = torch.ones(256).half()
    hf["model.layers.0.post_attention_layernorm.weight"] = torch.ones(256).half()
    sd = C.quantize_state_dict(C.remap_state_dict(hf))
    assert "layers.0.attention.wq.w" in sd and "layers.0.feed_forward.w2.shape" in sd and "tok_embeddings.weight" in sd
    assert "layers.0.attention.wq.weight" not in sd and tuple(sd["layers.0.feed_forward.w1.shape"]) == (768, 256)
    args = ModelArgs(dim=256, n_layers=1, n_heads=2, vocab_size=320, multiple_of=128, max_batch_size=2, max_seq_len=4,
                     max_prompt_seq_len=8)
    model = load_q40(sd, args, device="cpu")
    lin = model.layers[0].feed_forward.w2
    assert tuple(lin.shape) == (256, 768) and lin.w.shape == (768 * 256 // 128, 64) and lin.s.numel() == 768 * 256 // 64
    assert model.tok_embeddings.weight.dtype == torch.float16 and model.output.weight.shape == (320, 256)
    # the hot path refuses to run without a GPU instead of falling back
    with pytest.raises(AssertionError):
        model(torch.zeros((1, 4), dtype=torch.int64), 0)


def test_layer_scratch_holds_every_slab_of_a_pass():
    """smh_decode_scratch_bytes against the plans of the launches a layer makes: the fp16 buffers, and the slabs of every linear
    whose launch does not store fp16 itself"""
    from spec_mcts_amd import _lib
    lib = _lib.load()

    def slabs(M, K, *ns):
        n = (ctypes.c_int * len(ns))(*ns)
        return 0 if lib.smh_q40_matmul_tiled_direct_fits(M, K, len(ns), n) == 1 else lib.smh_q40_matmul_plan_tiled(M, K, len(ns), n) * M * sum(ns) * 4

    for dim, heads, kv_heads, ffn in ((4096, 32, 32, 11008), (5120, 40, 40, 13824), (8192, 64, 8, 28672), (256, 2, 2, 768)):
        layer = _lib.SmhLayer()
        layer.dim, layer.heads, layer.kv_heads, layer.ffn = dim, heads, kv_heads, ffn
        nq, nkv = heads * 128, kv_heads * 128
        for swiglu in (0, 1):
            for M in range(1, 1025):
                gate_up = 0 if M > 128 and swiglu and lib.smh_q40_swiglu_fits(M, dim, ffn) else lib.smh_q40_matmul_plan_tiled(M, dim, 2, (ctypes.c_int * 2)(ffn, ffn)) * M * 2 * ffn * 4
                need = 2 * M * (3 * dim + 2 * nq + 2 * nkv + ffn) + max(slabs(M, dim, nq, nkv, nkv), gate_up) + max(slabs(M, nq, dim), slabs(M, ffn, dim))
                assert lib.smh_decode_scratch_bytes(layer, M, swiglu) >= need, (dim, swiglu, M)


def test_rmsnorm_inside_the_launches_of_a_layer():
    """up to 16 rows wherever a K-slice's norm weights fit, one row where they do or the row does; _norm_in of the model asks the same"""
    from spec_mcts_amd import ModelArgs, Transformer, _lib, kernels as K
    lib = _lib.load()
    fits = lambda M, Kd, *ns: lib.smh_decode_norm_in_fits(M, Kd, len(ns), (ctypes.c_int * len(ns))(*ns))
    for M in range(1, 17):
        for Kd, ns in ((4096, (4096,) * 3), (6656, (6656,) * 3), (8192, (8192,) * 3), (8192, (28672, 28672)), (7168, (7168, 1024, 1024)), (14336, (512,))):
            assert fits(M, Kd, *ns) == 1
            assert lib.smh_q40_norm_in_fits(M, Kd, len(ns), (ctypes.c_int * len(ns))(*ns)) in (0, 1)
        assert fits(M, 16384, 131072) == 0                 # (one K-slice of 16384 rows)
    assert fits(1, 12288, 131072) == 1 and fits(2, 12288, 131072) == 0
    assert fits(0, 4096, 4096) == fits(17, 4096, 4096) == fits(4, 4096 + 8, 4096) == 0 and fits(4, 4096, 100) < 0
    model = Transformer(ModelArgs(dim=256, n_layers=1, n_heads=2, vocab_size=320, multiple_of=128))
    for M, Kd in ((1, 4096), (12, 6144), (16, 6656), (9, 8192), (16, 8192)):
        assert model._norm_in(M, Kd, [K.TiledQ40(None, Kd, Kd)] * 3)
    assert not model._norm_in(17, 4096, [K.TiledQ40(None, 4096, 4096)] * 3)


def test_form_of_a_layer():
    """5 .. 16 branches on 128-column blocks, and up to 32 with SwiGLU inside w1|w3, behind 96 prompt rows and more where all linears have them; whatever the
    form leaves, the scratch holds"""
    from spec_mcts_amd import _lib
    lib = _lib.load()

    def form(dim, heads, kv_heads, ffn, P, M, swiglu=1):
        layer, slabs = _lib.SmhLayer(), (ctypes.c_int * 4)()
        layer.dim, layer.heads, layer.kv_heads, layer.ffn, layer.prompt_len = dim, heads, kv_heads, ffn, P
        f = lib.smh_decode_layer_form(layer, M, swiglu, slabs)
        n = (heads + 2 * kv_heads) * 128
        need = 2 * M * (3 * dim + n + heads * 128 + ffn) + 4 * M * (max(slabs[0] * n, slabs[2] * 2 * ffn) + max(slabs[1], slabs[3]) * dim)
        assert f < 0 or lib.smh_decode_scratch_bytes(layer, M, swiglu) >= need
        return f, list(slabs)

    L7, L8, L13, L70 = (4096, 32, 32, 11008), (4096, 32, 8, 14336), (5120, 40, 40, 13824), (8192, 64, 8, 28672)
    for L, wide in ((L7, [2, 8, 0, 8]), (L8, [5, 8, 0, 8])):
        for M in (1, 4, 5, 10, 16, 17, 32, 33, 100):
            for P in (0, 95, 96, 512):
                f, slabs = form(*L, P, M)
                assert f == (3 if 5 <= M <= 16 and P >= 96 else 2 if M > 32 or (M > 16 and P >= 96) else 0), (L, M, P)
                assert f == 0 or M == 100 or slabs == wide
                assert form(*L, P, M, 0)[0] == 0           # (SwiGLU switched off: as before, whatever the rows)
    assert [form(*L13, 96, M)[0] for M in (5, 16, 17, 32)] == [0, 0, 2, 2]             # (wo and w2 of 5120 columns have no such blocks)
    assert [form(*L70, 512, M)[0] for M in (1, 5, 16, 17, 100, 129)] == [0, 0, 0, 0, 0, 2]
    for L in (L7, L8, L13, L70, (256, 2, 2, 768)):
        for P in (0, 100):
            for M in range(1, 700, 3):
                assert form(*L, P, M)[0] >= 0
    assert form(*L7, 96, 0)[0] < 0 and form(4096, 32, 5, 11008, 96, 8)[0] < 0 and form(100, 32, 32, 11008, 96, 8)[0] < 0


@pytest.mark.parametrize("dim,heads,kv_heads,ffn,wide_from", [(4096, 32, 32, 8192, 33), (3072, 24, 8, 8192, 33), (4096, 32, 32, 9088, 33), (4096, 32, 32, 9216, 25), (3584, 28, 28, 9728, 25),
                                                              (4096, 32, 8, 10240, 25), (5120, 40, 8, 10240, 25), (4096, 32, 32, 10880, 25), (4096, 32, 32, 11008, 17), (3072, 24, 24, 12288, 17)])
def test_swiglu_of_17_to_32_rows_wants_wide_weights(dim, heads, kv_heads, ffn, wide_from):
    """SwiGLU inside w1|w3 up to 32 rows only where its workgroups fill the compute units far enough; slabs below, as behind short prompts"""
    from spec_mcts_amd import _lib
    lib, layer, slabs = _lib.load(), _lib.SmhLayer(), (ctypes.c_int * 4)()
    layer.dim, layer.heads, layer.kv_heads, layer.ffn = dim, heads, kv_heads, ffn
    for P in (95, 96, 1024):
        layer.prompt_len = P
        for M in (17, 20, 24, 25, 31, 32, 33, 100):
            inside = M > 32 or (P >= 96 and M >= wide_from)
            assert lib.smh_decode_layer_form(layer, M, 1, slabs) == (2 if inside else 0), (P, M)
            assert (slabs[2] == 0) == inside


def _asks(dim, heads, kv_heads, ffn, P, M, swiglu=1):
    from spec_mcts_amd import _lib
    layer = _lib.SmhLayer()
    layer.dim, layer.heads, layer.kv_heads, layer.ffn, layer.prompt_len = dim, heads, kv_heads, ffn, P
    return _lib.load().smh_decode_layer_asks(layer, M, swiglu)


@pytest.mark.parametrize("dim,heads,kv_heads,ffn,some", [(4096, 32, 32, 11008, True), (3840, 30, 30, 10240, True), (3584, 28, 28, 9728, False), (3072, 24, 8, 8192, False),
                                                         (2048, 16, 16, 5632, False), (4608, 36, 36, 12288, False), (5120, 40, 40, 13824, False), (5120, 40, 8, 10240, False),
                                                         (6144, 48, 48, 16384, False), (8192, 64, 8, 28672, False)])
def test_dims_whose_launches_ask_for_weights_ahead(dim, heads, kv_heads, ffn, some):
    """where asking was the slower way nothing is asked for, whatever the rows and the prompt; nor of up to 16 rows on GEMVs"""
    for P in (0, 96, 1024):
        for M in (1, 5, 16, 17, 33, 48, 65, 100, 128):
            asks = _asks(dim, heads, kv_heads, ffn, P, M)
            assert asks == 0 or (some and (M > 16 or P >= 96)), (P, M, asks)
        assert (_asks(dim, heads, kv_heads, ffn, P, 33) == 15) == some
        assert _asks(dim, heads, kv_heads, ffn, P, 33, 0) == (4 if some else 0)
    assert _asks(dim, heads, kv_heads, ffn, 96, 0) < 0


@pytest.mark.parametrize("ffn", [8192, 11008, 16384])
def test_attention_of_many_branches_asks_for_nothing(ffn):
    """wo's weights are asked for up to three row tiles, with 32 kv heads and with 8"""
    for kv_heads in (32, 8):
        for M in (17, 32, 47, 48, 49, 64, 65, 100, 128):
            for swiglu in (0, 1):
                assert (_asks(4096, 32, kv_heads, ffn, 512, M, swiglu) & 4 != 0) == (M <= 48), (kv_heads, M)


@pytest.mark.parametrize("ffn,asks", [(9216, 11), (11008, 11), (13824, 11), (13952, 3), (14336, 3), (14464, 0), (16384, 0)])
def test_swiglu_that_fills_the_chip_asks_for_nothing(ffn, asks):
    """w2 is asked for from 40 idle compute units on, by the norms where 32 are idle in SwiGLU's launch (bits: wq|wk|wv, w1|w3, wo, w2)"""
    for kv_heads in (32, 8):
        for M in (5, 16, 25, 33, 100):
            assert _asks(4096, 32, kv_heads, ffn, 512, M) & ~4 == asks, (kv_heads, M)


def test_columns_of_a_workgroup_above_128_rows():
    """which of the launches above 128 rows a shape takes (the GPU tests of each ask here), 0 where there is none"""
    from spec_mcts_amd import _lib
    lib = _lib.load()

    def direct(M, K, *ns):
        return lib.smh_q40_matmul_tiled_direct_columns(M, K, len(ns), (ctypes.c_int * len(ns))(*ns))

    assert direct(128, 4096, 4096) == 0 and direct(512, 4096 + 8, 11008) == 0 and direct(512, 4096, 100) == 0
    assert direct(2047, 4096, 11008 + 64) == 0
    for M in (129, 300, 512, 1024, 2047):
        for K, ns in ((4096, (4096, 4096, 4096)), (11008, (4096,)), (96, (10624,)), (8192, (8192, 1024, 1024))):
            fits = lib.smh_q40_matmul_tiled_direct_fits(M, K, len(ns), (ctypes.c_int * len(ns))(*ns))
            columns = direct(M, K, *ns)
            assert columns in ((192, 256, 384) if fits else (0,)) and not (columns == 192 and K % 64)
    # six pieces where they promise 3 %, against whichever of the others promises most (here 256 columns; 4 % at these sizes)
    assert direct(1600, 4096, 4096, 4096, 4096) == 384 and direct(1961, 5120, 5120, 5120, 5120) == 384 and direct(1929, 4096, 11008) == 384
    assert lib.smh_q40_swiglu_columns(16, 4096, 11008) == 0 and lib.smh_q40_swiglu_columns(300, 4096 + 8, 11008) == 0
    assert lib.smh_q40_swiglu_columns(100, 4096, 11008) == 128
    assert {lib.smh_q40_swiglu_columns(M, 4096, 11008) for M in range(129, 600)} == {256, 384}
    # two launches where the last round of one would be a poor one: 48 workgroups of three pieces, then the columns behind them
    assert lib.smh_q40_swiglu_first_columns(128, 4096, 11008) == 0 and lib.smh_q40_swiglu_first_columns(2047, 4096 + 8, 11008) == 0
    assert lib.smh_q40_swiglu_first_columns(512, 4096, 11008) == 0 and lib.smh_q40_swiglu_first_columns(2047, 4096, 11008) == 48 * 192


def test_columns_of_a_workgroup_on_the_checkpoint_layout():
    """which of its two launches above 16 rows smh_q40_matmul takes"""
    from spec_mcts_amd import _lib
    columns = _lib.load().smh_q40_matmul_columns
    assert columns(16, 4096, 4096) == 0 and columns(100, 4096, 100) < 0
    assert columns(17, 4096, 4096) == 128 and columns(100, 4096, 11008) == 256 and columns(512, 4096, 4096) == 128 and columns(512, 11008, 4096) == 256
    assert columns(100, 4096 + 32, 4096) == 256                # (half a stage past the end of K)


@pytest.mark.parametrize("M,K,ns,swiglu", [(37, 4096, [4096, 4096, 4096], 0), (100, 4096, [4096], 0), (100, 11008, [4096], 0), (17, 4096, [4096], 0),
                                           (128, 8192, [8192, 1024, 1024], 0), (64, 4096, [5248, 1152, 1152], 0), (48, 13824, [5120], 0),
                                           (100, 4096, [11008, 11008], 1), (33, 5120, [13824, 13824], 1), (64, 64, [8320, 8320], 1),
                                           (5, 4096, [4096, 4096, 4096], 2), (10, 4096, [4096, 1024, 1024], 2), (16, 11008, [4096], 2), (5, 14336, [4096], 2), (16, 4096, [4096], 2),
                                           (5, 4096, [11008, 11008], 3), (16, 4096, [14336, 14336], 3), (10, 5120, [13824, 13824], 3)])
def test_weights_asked_for_ahead_are_those_of_the_launch(M, K, ns, swiglu):
    """a few stages stay inside the weights; all stages are every line of every tile once (the padded half of a last unit included)"""
    from spec_mcts_amd import _lib
    lib = _lib.load()
    n = (ctypes.c_int * len(ns))(*ns)
    out = [(ctypes.c_long * len(ns))() for _ in range(3)]
    for stages in (1, 3, 16):
        assert lib.smh_q40_warm_span(M, K, len(ns), n, swiglu, stages, *out) == 1
        for i, N in enumerate(ns):
            assert out[0][i] > 0 and 0 <= out[1][i] < out[2][i] <= lib.smh_q40_tiled_bytes(K, N)
    assert lib.smh_q40_warm_span(M, K, len(ns), n, swiglu, 1 << 20, *out) == 1
    for i, N in enumerate(ns):
        # 34 lines a tile; its scales are asked for with each half of it (128-column blocks), with each piece (SwiGLU)
        pieces, lines = (2 * (N // 128), 10) if swiglu & 1 else (2 * ((N + 255) // 256), 18)
        assert out[0][i] == pieces * lines * (K // 32)
        assert out[1][i] == 0 and (out[2][i] == lib.smh_q40_tiled_bytes(K, N) or N % 256)


@pytest.mark.parametrize("M,K,ns,swiglu", [(16, 4096, [4096], 0), (129, 4096, [4096], 0), (100, 4096 + 32, [4096], 0), (32, 4096, [11008, 11008], 0),
                                           (100, 28672, [8192], 0), (100, 8192, [28672, 28672], 1), (200, 4096, [11008, 11008], 1)])
def test_nothing_is_asked_for_ahead_of_other_kernels(M, K, ns, swiglu):
    from spec_mcts_amd import _lib
    out = [(ctypes.c_long * len(ns))() for _ in range(3)]
    assert _lib.load().smh_q40_warm_span(M, K, len(ns), (ctypes.c_int * len(ns))(*ns), swiglu, 3, *out) == 0
