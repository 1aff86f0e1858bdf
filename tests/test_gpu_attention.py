"""GPU parity of the shared-prefix decode attention and the causal prefill attention against the
oracle (explicit fp32 softmax attention).  Tolerance: 1e-2 relative + 2e-3 absolute."""
import pytest
import torch

from oracle import q40_oracle as O

pytestmark = pytest.mark.gpu
RTOL, ATOL = 1e-2, 2e-3


def _g(seed):
    return torch.Generator().manual_seed(seed)


def _check(got, want):
    got, want = got.float().cpu(), want.float()
    err = (got - want).abs()
    tol = ATOL + RTOL * want.abs()
    assert bool((err <= tol).all()), f"max err {err.max():.4e}, worst excess {(err - tol).max():.4e}"


def _inputs(B, H, Hkv, D, P, S, seed, std=1.0):
    g = _g(seed)
    q = (torch.randn((B, H, D), generator=g) * std).to(torch.float16)
    pk = (torch.randn((max(P, 1), Hkv, D), generator=g) * std).to(torch.float16)
    pv = (torch.randn((max(P, 1), Hkv, D), generator=g) * std).to(torch.float16)
    sk = (torch.randn((B, max(S, 1), Hkv, D), generator=g) * std).to(torch.float16)
    sv = (torch.randn((B, max(S, 1), Hkv, D), generator=g) * std).to(torch.float16)
    lens = torch.randint(0, S + 1, (B,), generator=g, dtype=torch.int32)
    return q, pk, pv, sk, sv, lens


def test_config2_fp16_suffix():
    """B=64 branches, 32 heads, D=128, shared 1024-token prefix, ragged suffix 0..256, seed 2"""
    from spec_mcts_amd import kernels as K
    B, H, D, P, S = 64, 32, 128, 1024, 256
    q, pk, pv, sk, sv, lens = _inputs(B, H, H, D, P, S, 2)
    lens[0] = 0; lens[1] = S
    got = K.shared_prefix_attn(q.cuda(), pk.cuda(), pv.cuda(), P, suffix_k=sk.cuda(), suffix_v=sv.cuda(),
                               Smax=S, lens=lens.cuda(), lens_stride=1)
    want = O.shared_prefix_attention(q, pk, pv, sk, sv, lens.tolist())
    _check(got, want)


def test_config2_q40_suffix_as_the_model_stores_it():
    from spec_mcts_amd import kernels as K
    B, H, D, P, S = 64, 32, 128, 1024, 256
    q, pk, pv, sk, sv, lens = _inputs(B, H, H, D, P, S, 3)
    wk, sks = O.quantize_q40(sk, 64)
    wv, svs = O.quantize_q40(sv, 64)
    sk_deq = O.dequantize_q40(wk, sks, 64, sk.shape)
    sv_deq = O.dequantize_q40(wv, svs, 64, sv.shape)
    got = K.shared_prefix_attn(q.cuda(), pk.cuda(), pv.cuda(), P, suffix_k=wk.cuda(), suffix_v=wv.cuda(),
                               suffix_ks=sks.cuda(), suffix_vs=svs.cuda(), Smax=S, lens=lens.cuda(), lens_stride=1)
    want = O.shared_prefix_attention(q, pk, pv, sk_deq, sv_deq, lens.tolist())
    _check(got, want)


@pytest.mark.parametrize("B,H,Hkv,P,S", [(1, 2, 2, 1, 0), (3, 8, 2, 100, 5), (100, 8, 1, 512, 3), (17, 4, 4, 33, 9),
                                         (5, 2, 2, 0, 7), (2, 64, 8, 2048, 4)])
def test_shapes_gqa_empty_prefix_and_current_token(B, H, Hkv, P, S):
    from spec_mcts_amd import kernels as K
    D = 128
    q, pk, pv, sk, sv, lens = _inputs(B, H, Hkv, D, P, S, 10 + B)
    g = _g(99)
    ck = torch.randn((B, Hkv, D), generator=g).to(torch.float16)
    cv = torch.randn((B, Hkv, D), generator=g).to(torch.float16)
    # the new token is one more exact row after each branch's suffix
    sk2 = torch.cat((sk, torch.zeros_like(sk[:, :1])), 1); sv2 = torch.cat((sv, torch.zeros_like(sv[:, :1])), 1)
    for b in range(B):
        sk2[b, lens[b]] = ck[b]; sv2[b, lens[b]] = cv[b]
    want = O.shared_prefix_attention(q, pk[:P], pv[:P], sk2, sv2, (lens + 1).tolist())
    got = K.shared_prefix_attn(q.cuda(), pk.cuda() if P else None, pv.cuda() if P else None, P,
                               suffix_k=sk.cuda(), suffix_v=sv.cuda(), Smax=max(S, 1), lens=lens.cuda(), lens_stride=1,
                               cur_k=ck.cuda(), cur_v=cv.cuda(), n_kv_heads=Hkv)
    _check(got, want)


def test_uniform_length_from_device_counter():
    """lens_stride 0: every branch uses the same device-side step counter, as the model does"""
    from spec_mcts_amd import kernels as K
    B, H, D, P, S = 6, 4, 128, 64, 8
    q, pk, pv, sk, sv, _ = _inputs(B, H, H, D, P, S, 30)
    t = torch.tensor([5], dtype=torch.int32).cuda()
    got = K.shared_prefix_attn(q.cuda(), pk.cuda(), pv.cuda(), P, suffix_k=sk.cuda(), suffix_v=sv.cuda(), Smax=S,
                               lens=t, lens_stride=0)
    _check(got, O.shared_prefix_attention(q, pk, pv, sk, sv, [5] * B))


def test_special_cases():
    from spec_mcts_amd import kernels as K
    B, H, D, P, S = 4, 2, 128, 96, 8
    q, pk, pv, sk, sv, lens = _inputs(B, H, H, D, P, S, 31)
    lens[:] = S
    # q = 0 -> uniform weights -> mean of all V rows
    got = K.shared_prefix_attn(torch.zeros_like(q).cuda(), pk.cuda(), pv.cuda(), P, suffix_k=sk.cuda(),
                               suffix_v=sv.cuda(), Smax=S, lens=lens.cuda(), lens_stride=1).cpu()
    for b in range(B):
        assert torch.allclose(got[b].float(), torch.cat((pv, sv[b]), 0).float().mean(0), atol=2e-3)
    # one dominant prefix key -> its V row
    pk2 = pk.clone(); pk2[70] = 0; pk2[70, :, 0] = 200.0
    q2 = torch.zeros_like(q); q2[..., 0] = 50.0
    got = K.shared_prefix_attn(q2.cuda(), pk2.cuda(), pv.cuda(), P).cpu()
    assert torch.allclose(got[0].float(), pv[70].float(), atol=2e-3)
    # split invariance: moving the tail of the prefix into every branch's suffix changes nothing
    full = K.shared_prefix_attn(q.cuda(), pk.cuda(), pv.cuda(), P, suffix_k=sk.cuda(), suffix_v=sv.cuda(), Smax=S,
                                lens=lens.cuda(), lens_stride=1).cpu()
    cut = 40
    sk2 = torch.cat((pk[cut:][None].expand(B, -1, -1, -1), sk), 1).contiguous()
    sv2 = torch.cat((pv[cut:][None].expand(B, -1, -1, -1), sv), 1).contiguous()
    l2 = (lens + P - cut).to(torch.int32)
    moved = K.shared_prefix_attn(q.cuda(), pk[:cut].contiguous().cuda(), pv[:cut].contiguous().cuda(), cut,
                                 suffix_k=sk2.cuda(), suffix_v=sv2.cuda(), Smax=S + P - cut, lens=l2.cuda(),
                                 lens_stride=1).cpu()
    assert torch.allclose(full.float(), moved.float(), atol=2e-3, rtol=1e-2)


@pytest.mark.parametrize("S,H,Hkv", [(1, 2, 2), (19, 4, 2), (63, 2, 1), (64, 2, 2), (65, 4, 1), (200, 8, 2), (512, 32, 32), (1100, 8, 1)])
def test_prefill_causal(S, H, Hkv):
    from spec_mcts_amd import kernels as K
    g = _g(40 + S)
    q = torch.randn((S, H, 128), generator=g).to(torch.float16)
    k = torch.randn((S, Hkv, 128), generator=g).to(torch.float16)
    v = torch.randn((S, Hkv, 128), generator=g).to(torch.float16)
    got = K.prefill_attn(q.cuda(), k.cuda(), v.cuda())
    _check(got, O.causal_attention(q, k, v))


def test_prefill_causal_special_cases():
    """what the mathematics fixes: position 0 sees only itself (out = v[0]); equal keys give the running mean of v;
    one key that dominates every score makes every later position return that key's v"""
    from spec_mcts_amd import kernels as K
    S, H = 150, 2
    g = _g(77)
    q = torch.randn((S, H, 128), generator=g).half()
    k = torch.randn((S, H, 128), generator=g).half()
    v = torch.randn((S, H, 128), generator=g).half()
    out = K.prefill_attn(q.cuda(), k.cuda(), v.cuda()).cpu()
    assert torch.equal(out[0], v[0])
    k_same = k[:1].expand(S, H, 128).contiguous()
    out = K.prefill_attn(q.cuda(), k_same.cuda(), v.cuda()).cpu().float()
    mean = v.float().cumsum(0) / torch.arange(1, S + 1).view(S, 1, 1)
    assert torch.allclose(out, mean, atol=2e-3, rtol=1e-2)
    k_dom = (torch.randn((S, H, 128), generator=g) * 0.01).half()
    k_dom[70] = q[100] * 4                       # huge score for every query that resembles q[100]; use q = q[100] everywhere
    q_all = q[100:101].expand(S, H, 128).contiguous()
    out = K.prefill_attn(q_all.cuda(), k_dom.cuda(), v.cuda()).cpu().float()
    assert torch.allclose(out[70:], v[70:71].float().expand(S - 70, H, 128), atol=2e-3, rtol=1e-2)


def test_flash_attn_page_flash_attn_and_chunk_attn_drop_ins():
    """the reference's operator names (triton_kernels.py:621, :764) on top of the decode attention kernel, with
    the shapes of its own checks (triton_kernels_bench.py:294-330: B=100, L=512, H=32, D=128, atol 1e-2)"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(1)
    B, L, H, D = 100, 512, 32, 128
    q = torch.randn((B, H, D), generator=g).half()
    k = torch.randn((B, H, L, D), generator=g).half()
    v = torch.randn((B, H, L, D), generator=g).half()
    got = K.flash_attn(q.cuda(), k.cuda(), v.cuda(), B, L, H, D).cpu()
    want = torch.nn.functional.scaled_dot_product_attention(q.float()[:, :, None], k.float(), v.float())[:, :, 0]
    assert got.dtype == torch.float16 and torch.allclose(got.float(), want, rtol=1e-2, atol=2e-3)
    # paged: a pool of P pages per head, every branch an arbitrary list of L pages (pages may repeat)
    P, B2, L2 = 300, 27, 130
    kp = torch.randn((H, P, D), generator=g).half()
    vp = torch.randn((H, P, D), generator=g).half()
    pager = torch.randint(0, P, (B2, L2), generator=g).to(torch.int16)
    q2 = torch.randn((B2, H, D), generator=g).half()
    got2 = K.page_flash_attn(pager.cuda(), q2.cuda(), kp.cuda(), vp.cuda(), P, B2, L2, H, D).cpu()
    idx = pager.long()
    kk = kp.float()[:, idx].permute(1, 0, 2, 3)           # [B, H, L, D]
    vv = vp.float()[:, idx].permute(1, 0, 2, 3)
    want2 = torch.nn.functional.scaled_dot_product_attention(q2.float()[:, :, None], kk, vv)[:, :, 0]
    assert torch.allclose(got2.float(), want2, rtol=1e-2, atol=2e-3)
    # chunked: pool rows 0..offset-1 shared by every branch, then the branch's own pages; the shapes of the
    # reference's tree-attention check (triton_kernels_bench.py:479-493: 27 branches, 512 rows, 256 shared)
    for offset, L3 in ((256, 512), (0, 40), (40, 40)):
        pager3 = torch.randint(0, P, (B2, L3), generator=g).to(torch.int16)
        pager3[:, :offset] = torch.arange(offset, dtype=torch.int16)
        got3 = K.chunk_attn(pager3.cuda(), q2.cuda(), kp.cuda(), vp.cuda(), P, B2, L3, H, D, offset).cpu()
        idx3 = pager3.long()
        want3 = torch.nn.functional.scaled_dot_product_attention(
            q2.float()[:, :, None], kp.float()[:, idx3].permute(1, 0, 2, 3), vp.float()[:, idx3].permute(1, 0, 2, 3))[:, :, 0]
        assert got3.dtype == torch.float16 and torch.allclose(got3.float(), want3, rtol=1e-2, atol=2e-3)
        if offset:
            same = K.page_flash_attn(pager3.cuda(), q2.cuda(), kp.cuda(), vp.cuda(), P, B2, L3, H, D).cpu()
            assert torch.allclose(got3.float(), same.float(), rtol=1e-2, atol=2e-3)


@pytest.mark.parametrize("B,H,Hkv,P,t", [(1, 4, 4, 40, 0), (3, 4, 4, 40, 5), (16, 8, 2, 100, 9), (5, 8, 8, 0, 3)])
def test_attention_fed_by_the_qkv_product_matches_the_three_launch_sequence(B, H, Hkv, P, t):
    """smh_shared_prefix_attn_qkv (RoPE + KV append inside the attention kernels) against
    smh_partial_rope_append_kv + smh_shared_prefix_attn on the same slabs: same rounding points, so the
    outputs and the appended cache rows must be bit-identical."""
    from spec_mcts_amd import kernels as K
    dev = "cuda:0"
    D, Smax, dim = 128, 16, 512
    g = torch.Generator(device="cpu").manual_seed(900 + B + t)
    x = (torch.randn((B, dim), generator=g) * 0.5).half().to(dev)
    ws = []
    for n in (H * D, Hkv * D, Hkv * D):
        w = torch.randint(-128, 128, (dim * n // 2,), generator=g, dtype=torch.int16).to(torch.int8).to(dev)
        s = (torch.rand((dim * n // 64,), generator=g) * 0.02 + 0.005).half().to(dev)
        ws.append((w, s, n))
    qkv = K.matmul_q40_partial(x, ws)
    ang = torch.rand((64, 64), generator=g) * 6.28
    cos, sin = torch.cos(ang).half().to(dev), torch.sin(ang).half().to(dev)
    pos_dev = torch.tensor([P + t], dtype=torch.int32, device=dev) % 64
    t_dev = torch.tensor([t], dtype=torch.int32, device=dev)
    pk = (torch.randn((max(P, 1), Hkv, D), generator=g) * 0.5).half().to(dev)
    pv = (torch.randn((max(P, 1), Hkv, D), generator=g) * 0.5).half().to(dev)
    caches = []
    for _ in range(2):
        ck = torch.randint(-128, 128, (B, Smax, Hkv, 64), generator=torch.Generator().manual_seed(7), dtype=torch.int16).to(torch.int8).to(dev)
        cv = torch.randint(-128, 128, (B, Smax, Hkv, 64), generator=torch.Generator().manual_seed(8), dtype=torch.int16).to(torch.int8).to(dev)
        cks = (torch.rand((B, Smax, Hkv, 2), generator=torch.Generator().manual_seed(9)) * 0.1 + 0.01).half().to(dev)
        cvs = (torch.rand((B, Smax, Hkv, 2), generator=torch.Generator().manual_seed(10)) * 0.1 + 0.01).half().to(dev)
        caches.append((ck, cks, cv, cvs))
    ck, cks, cv, cvs = caches[0]
    q, k, v = K.partial_rope_append_kv(qkv, H, Hkv, D, cos, sin, pos_dev, ck, cks, cv, cvs, Smax, t_dev)
    want = K.shared_prefix_attn(q, pk if P else None, pv if P else None, P, suffix_k=ck, suffix_v=cv, suffix_ks=cks, suffix_vs=cvs,
                                Smax=Smax, lens=t_dev, lens_stride=0, cur_k=k, cur_v=v, n_kv_heads=Hkv)
    ck2, cks2, cv2, cvs2 = caches[1]
    got = K.shared_prefix_attn_qkv(qkv, H, Hkv, D, cos, sin, pos_dev, pk if P else None, pv if P else None, P,
                                   ck2, cks2, cv2, cvs2, Smax, t_dev, single_launch=False)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    for a, b_ in zip(caches[0], caches[1]):
        assert torch.equal(a, b_), "appended cache rows differ"
    # one launch: the partials are merged in another order, so equal up to fp32 summation order; three calls in a
    # row check that the arrival counters are left ready for the next call
    for rep in range(3):
        ck3, cks3, cv3, cvs3 = (x.clone() for x in caches[0])
        ck3[:, t], cks3[:, t], cv3[:, t], cvs3[:, t] = 0, 0, 0, 0
        one = K.shared_prefix_attn_qkv(qkv, H, Hkv, D, cos, sin, pos_dev, pk if P else None, pv if P else None, P,
                                       ck3, cks3, cv3, cvs3, Smax, t_dev, single_launch=True)
        torch.cuda.synchronize()
        assert torch.allclose(one.float(), want.float(), rtol=2e-3, atol=2e-3), f"call {rep}: {float((one.float() - want.float()).abs().max())}"
        for a, b_ in zip(caches[0], (ck3, cks3, cv3, cvs3)):
            assert torch.equal(a, b_), "appended cache rows differ"


def _tiles_against_launches(qkv, H, Hkv, P, t, Smax, paged, g, one=False):
    """smh_shared_prefix_attn_qkv_tiles (one: smh_shared_prefix_attn_qkv in one launch) and smh_partial_rope_append_kv + smh_shared_prefix_attn / smh_paged_prefix_attn on the same slabs and caches, of
    which nobody's rows are alike: the same rows appended, outputs within the bound of the tests below.  Returns the call and its output."""
    from spec_mcts_amd import kernels as K
    dev, D, B = "cuda:0", 128, qkv.M
    ang = torch.rand((64, 64), generator=g) * 6.28
    cos, sin = torch.cos(ang).half().to(dev), torch.sin(ang).half().to(dev)
    pos_dev = torch.tensor([P + t], dtype=torch.int32, device=dev) % 64
    t_dev = torch.tensor([t], dtype=torch.int32, device=dev)
    pk, pv = ((torch.randn((P + 5, Hkv, D), generator=g) * 0.5).half().to(dev) for _ in range(2))
    ck, cv = (torch.randint(-128, 128, (B, Smax, Hkv, 64), generator=g, dtype=torch.int16).to(torch.int8).to(dev) for _ in range(2))
    cks, cvs = ((torch.rand((B, Smax, Hkv, 2), generator=g) * 0.1 + 0.01).half().to(dev) for _ in range(2))
    for past in (pk[P:], pv[P:], cks[:, max(t, 1):], cvs[:, max(t, 1):]):
        past.fill_(float("nan"))
    pages = None
    if paged:                                      # rows of any branch, but for the new one
        pages = torch.randint(0, B, (B, Smax), generator=g, dtype=torch.int32) * Smax + torch.randint(0, max(t, 1), (B, Smax), generator=g, dtype=torch.int32)
        pages = pages.to(dev)
    mine = [c.clone() for c in (ck, cks, cv, cvs)]
    q, k, v = K.partial_rope_append_kv(qkv, H, Hkv, D, cos, sin, pos_dev, ck, cks, cv, cvs, Smax, t_dev)
    common = dict(lens=t_dev, lens_stride=0, cur_k=k, cur_v=v)
    prefix = (pk, pv) if P else (None, None)
    if paged:
        del common["lens"]
        want = K.paged_prefix_attn(q, pages, t_dev, ck.view(-1, Hkv, 64), cv.view(-1, Hkv, 64), cks.view(-1, Hkv, 2), cvs.view(-1, Hkv, 2), False, *prefix, P, **common)
    else:
        want = K.shared_prefix_attn(q, *prefix, P, suffix_k=ck, suffix_v=cv, suffix_ks=cks, suffix_vs=cvs, Smax=Smax, n_kv_heads=Hkv, **common)
    call = K.shared_prefix_attn_qkv if one else K.shared_prefix_attn_qkv_tiles
    tiles = lambda: call(qkv, H, Hkv, D, cos, sin, pos_dev, *prefix, P, *mine, Smax, t_dev, pages=pages)
    got = tiles()
    torch.cuda.synchronize()
    assert torch.isfinite(got).all()
    assert torch.allclose(got.float(), want.float(), rtol=2e-3, atol=2e-3), f"{qkv.ksplit} slabs: {float((got.float() - want.float()).abs().max())}"
    for a, b_ in zip((ck, cks, cv, cvs), mine):
        assert torch.equal(a.nan_to_num(-1.0), b_.nan_to_num(-1.0)) if a.dtype == torch.float16 else torch.equal(a, b_), "appended cache rows differ"
    return tiles, got


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("B,H,Hkv,P,t", [(1, 4, 4, 31, 0), (16, 9, 9, 32, 1), (17, 4, 4, 33, 5), (33, 8, 2, 511, 15), (7, 6, 2, 513, 9), (40, 2, 2, 1030, 14), (5, 8, 8, 0, 3),
                                         (100, 3, 3, 100, 8)])
def test_attention_of_sixteen_queries_a_workgroup_matches_the_three_launch_sequence(B, H, Hkv, P, t, paged):
    """smh_shared_prefix_attn_qkv_tiles against smh_partial_rope_append_kv + smh_shared_prefix_attn / smh_paged_prefix_attn on the same slabs (as many
    as the plans of 256 to 2048 rows come to): the same rows appended; outputs equal up to the order of fp32 sums and to which fp16 a probability of
    the prefix is rounded to (relative to another maximum), 2^-11 of a mean of values below 3: 2e-3 as in the test above.  Prefixes around the
    32 rows of a wave and the 512 of a workgroup's pass, tiles with one to eight queries (few heads: the form of eight), grouped heads that straddle a
    tile.  What lies past the prefix and past a branch's rows is NaN; then one branch's query is, and nobody else's output."""
    from spec_mcts_amd import kernels as K
    dev = "cuda:0"
    D, Smax = 128, 16
    for dim in (256, 2048):
        g = torch.Generator(device="cpu").manual_seed(900 + B + t)
        x = (torch.randn((B, dim), generator=g) * 0.5).half().to(dev)
        ws = []
        for n in (H * D, Hkv * D, Hkv * D):
            w = torch.randint(-128, 128, (dim * n // 2,), generator=g, dtype=torch.int16).to(torch.int8).to(dev)
            s = (torch.rand((dim * n // 64,), generator=g) * 0.02 + 0.005).half().to(dev)
            ws.append((w, s, n))
        qkv = K.matmul_q40_partial(x, ws)
        tiles, got = _tiles_against_launches(qkv, H, Hkv, P, t, Smax, paged, g)
        qkv.buf.view(qkv.ksplit, B, -1)[0, B // 2, 3] = float("nan")
        got_nan = tiles()
        assert got_nan[B // 2, 0].isnan().all()
        got_nan[B // 2, 0] = got[B // 2, 0]
        assert torch.equal(got_nan, got)


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("B,H,Hkv,queries,ksplit,P,t", [
    (100, 32, 32, 16, 2, 100, 65), (100, 32, 32, 16, 5, 512, 40), (65, 32, 32, 16, 1, 96, 127), (65, 32, 32, 16, 3, 222, 16), (33, 64, 8, 16, 6, 130, 33), (33, 64, 8, 16, 2, 600, 17),
    (40, 64, 8, 16, 12, 129, 31), (73, 29, 29, 16, 7, 97, 64), (65, 32, 32, 16, 16, 1100, 1), (31, 64, 8, 8, 5, 2047, 110), (37, 32, 32, 8, 5, 221, 40), (37, 32, 32, 8, 2, 100, 64),
    (17, 4, 4, 8, 16, 96, 127), (20, 8, 2, 8, 3, 222, 33), (64, 32, 32, 8, 1, 512, 32), (5, 64, 8, 8, 6, 500, 63)])
def test_tile_attention_over_long_branches(B, H, Hkv, queries, ksplit, P, t, paged):
    """Both numbers of queries a workgroup, each of their three kernels by the number of slabs, and branches of more rows than a turn of the walk (16 or 32)
    and than one request of page ids (32): lengths around both, with and without a table, no two branches' rows alike."""
    from spec_mcts_amd import kernels as K
    assert (16 if Hkv * -(-B * (H // Hkv) // 8) > 256 else 8) == queries          # (the rule of the entry point)
    g = torch.Generator().manual_seed(B + t)
    n = (H + 2 * Hkv) * 128
    qkv = K.PartialProduct((torch.randn((ksplit, B, n), generator=g) * 1.5 / ksplit ** 0.5).to("cuda:0"), ksplit, B, n)
    _tiles_against_launches(qkv, H, Hkv, P, t, 128, paged, g)


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("B,H,ksplit,P,t", [
    (1, 32, 2, 96, 5), (1, 32, 1, 97, 120), (2, 32, 2, 96, 1), (5, 32, 2, 95, 64), (5, 32, 1, 96, 0), (16, 32, 2, 97, 127), (10, 32, 3, 96, 31), (10, 32, 2, 129, 32), (11, 32, 2, 200, 33),
    (12, 32, 1, 193, 120), (14, 32, 2, 128, 16), (16, 32, 2, 256, 63), (5, 32, 5, 400, 100), (16, 32, 2, 400, 17), (13, 32, 2, 511, 90), (8, 32, 2, 512, 40), (16, 32, 2, 704, 65),
    (10, 40, 2, 96, 70), (12, 40, 16, 320, 40), (6, 64, 2, 128, 21), (12, 64, 9, 96, 50)])
def test_one_launch_of_many_heads(B, H, ksplit, P, t, paged):
    """smh_shared_prefix_attn_qkv in one launch from 32 kv heads on, against the three-launch sequence (bound: the test of sixteen queries a workgroup): its kernels by the
    number of slabs (up to two, 8, 12, 16), prompts around the rows from which slices are 64 rows wide, last slices of 1 to 64 rows, one, two and four waves a query's own
    rows with and without a table, of 0 rows, of one and of several turns of a walk.  What lies past the prompt and past a branch's rows is NaN, and the
    counters are left ready for the next call."""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(B + P + t)
    n = 3 * H * 128
    qkv = K.PartialProduct((torch.randn((ksplit, B, n), generator=g) * 1.5 / ksplit ** 0.5).to("cuda:0"), ksplit, B, n)
    again, got = _tiles_against_launches(qkv, H, H, P, t, 128, paged, g, one=True)
    for _ in range(2):
        assert torch.equal(again(), got)


@pytest.mark.parametrize("B,H,Hkv,P", [(17, 4, 4, 100), (20, 8, 2, 530), (100, 32, 32, 130), (40, 64, 8, 1030)])
@pytest.mark.parametrize("where", ["first", "last", "one of many", "both signs"])
def test_infinite_prompt_values_stay_infinite_in_one_launch(B, H, Hkv, P, where):
    """An infinity in a row of the prompt's V: that dimension is infinite in every branch's output (NaN where +inf and -inf meet, as a
    sum of the two is), all others are what they are with a finite value there - bit for bit but for what fp16 rounds off a probability (2^-11 of
    a mean of values below 3).  With eight queries a workgroup and with 16."""
    from spec_mcts_amd import kernels as K
    dev, D, Smax, t = "cuda:0", 128, 8, 3
    g = torch.Generator().manual_seed(40 + B)
    half = lambda *shape, std=0.5: (torch.randn(shape, generator=g) * std).half().to(dev)
    qkv = K.PartialProduct(torch.randn((2, B, (H + 2 * Hkv) * D), generator=g).to(dev), 2, B, (H + 2 * Hkv) * D)
    cos, sin = half(64, 64), half(64, 64)
    pos_dev, t_dev = (torch.tensor([x], dtype=torch.int32, device=dev) for x in (7, t))
    pk, pv = half(P, Hkv, D), half(P, Hkv, D)
    ck, cv = (torch.randint(-128, 128, (B, Smax, Hkv, 64), generator=g, dtype=torch.int16).to(torch.int8).to(dev) for _ in range(2))
    cks, cvs = ((torch.rand((B, Smax, Hkv, 2), generator=g) * 0.1 + 0.01).half().to(dev) for _ in range(2))
    run = lambda: K.shared_prefix_attn_qkv_tiles(qkv, H, Hkv, D, cos, sin, pos_dev, pk, pv, P, ck, cks, cv, cvs, Smax, t_dev)
    inf, row = float("inf"), {"first": 0, "last": P - 1}.get(where, P // 2)
    pv[row, 0, 77] = 1.0
    clean = run().view(B, Hkv, H // Hkv, D)
    pv[row, 0, 77] = -inf
    if where == "both signs":
        pv[row - 1, 0, 77] = inf
    got = run().view(B, Hkv, H // Hkv, D)
    torch.cuda.synchronize()
    assert clean.isfinite().all()
    hit = got[:, 0, :, 77]
    assert hit.isnan().all() if where == "both signs" else (hit == -inf).all()
    got[:, 0, :, 77] = clean[:, 0, :, 77]
    assert torch.equal(got[:, 1:], clean[:, 1:])
    assert torch.allclose(got.float(), clean.float(), rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("B,H,Hkv,P,L", [(100, 4, 4, 150, 9), (33, 8, 2, 70, 4), (5, 4, 4, 0, 6), (128, 2, 2, 40, 0)])
def test_one_launch_attention_matches_two_launches(B, H, Hkv, P, L):
    """smh_shared_prefix_attn_one against smh_shared_prefix_attn on the same inputs (Q4_0 suffix, new token):
    same partials, merged in another order; called three times to check the counters are left ready."""
    from spec_mcts_amd import kernels as K
    dev = "cuda:0"
    D, Smax = 128, 16
    g = torch.Generator().manual_seed(1200 + B)
    q = (torch.randn((B, H, D), generator=g) * 0.7).half().to(dev)
    pk = (torch.randn((max(P, 1), Hkv, D), generator=g) * 0.5).half().to(dev)
    pv = (torch.randn((max(P, 1), Hkv, D), generator=g) * 0.5).half().to(dev)
    ck = torch.randint(-128, 128, (B, Smax, Hkv, 64), generator=g, dtype=torch.int16).to(torch.int8).to(dev)
    cv = torch.randint(-128, 128, (B, Smax, Hkv, 64), generator=g, dtype=torch.int16).to(torch.int8).to(dev)
    cks = (torch.rand((B, Smax, Hkv, 2), generator=g) * 0.1 + 0.01).half().to(dev)
    cvs = (torch.rand((B, Smax, Hkv, 2), generator=g) * 0.1 + 0.01).half().to(dev)
    k = (torch.randn((B, Hkv, D), generator=g) * 0.5).half().to(dev)
    v = (torch.randn((B, Hkv, D), generator=g) * 0.5).half().to(dev)
    lens = torch.tensor([L], dtype=torch.int32, device=dev)
    kw = dict(suffix_k=ck, suffix_v=cv, suffix_ks=cks, suffix_vs=cvs, Smax=Smax, lens=lens, lens_stride=0, cur_k=k, cur_v=v,
              n_kv_heads=Hkv)
    want = K.shared_prefix_attn(q, pk if P else None, pv if P else None, P, **kw)
    for rep in range(3):
        got = K.shared_prefix_attn(q, pk if P else None, pv if P else None, P, single_launch=True, **kw)
        torch.cuda.synchronize()
        assert torch.allclose(got.float(), want.float(), rtol=2e-3, atol=2e-3), f"call {rep}: {float((got.float() - want.float()).abs().max())}"


@pytest.mark.parametrize("B,H,Hkv,P,S", [(1, 8, 8, 1, 5), (15, 8, 8, 31, 17), (16, 3, 3, 33, 64), (17, 16, 2, 127, 3), (65, 8, 8, 128, 33), (33, 16, 8, 129, 40),
                                         (5, 32, 32, 1000, 12), (130, 8, 1, 300, 16)])
@pytest.mark.parametrize("current", [False, True])
def test_fp16_suffix_beside_the_prefix_slices(B, H, Hkv, P, S, current):
    """slices and walks in one launch, then the merge: edges of slices (32 .. 128 rows) and of query tiles, grouped queries,
    branches without rows of their own; the workspace of the older size takes the prefix launch and then the walk"""
    from spec_mcts_amd import _lib, kernels as K
    g = torch.Generator().manual_seed(B + P)
    r = lambda *s: torch.randn(s, generator=g).half()
    q, pk, pv, sk, sv, ck, cv = r(B, H, 128), r(P, Hkv, 128), r(P, Hkv, 128), r(B, S, Hkv, 128), r(B, S, Hkv, 128), r(B, Hkv, 128), r(B, Hkv, 128)
    lens = torch.randint(0, S + 1, (B,), generator=g, dtype=torch.int32)
    lens[0] = 0
    want = torch.empty((B, H, 128), dtype=torch.float64)
    for b in range(B):
        parts = [(pk, pv), (sk[b, :lens[b]], sv[b, :lens[b]])] + ([(ck[b:b + 1], cv[b:b + 1])] if current else [])
        k, v = (torch.cat([x[i] for x in parts]).double().repeat_interleave(H // Hkv, 1) for i in range(2))
        p = torch.softmax(torch.einsum("hd,thd->ht", q[b].double(), k) / 128 ** 0.5, 1)
        want[b] = torch.einsum("ht,thd->hd", p, v)
    d = [t.cuda() for t in (q, pk, pv, sk, sv, lens, ck, cv)]
    kw = dict(suffix_k=d[3], suffix_v=d[4], Smax=S, lens=d[5], lens_stride=1, **(dict(cur_k=d[6], cur_v=d[7]) if current else {}))
    got = K.shared_prefix_attn(d[0], d[1], d[2], P, **kw).cpu().double()
    tol = 2e-3 + 1e-2 * want.abs()                       # the bound of the other attention tests: fp16 probabilities of the prefix, fp16 output
    assert bool(((got - want).abs() <= tol).all())
    lib, splits = _lib.load(), -(-P // 32)
    ws, out = torch.empty(splits * B * H * 130 * 4, dtype=torch.uint8, device="cuda"), torch.empty_like(d[0])
    K.check(lib.smh_shared_prefix_attn(d[0].data_ptr(), out.data_ptr(), B, H, Hkv, 128, d[1].data_ptr(), d[2].data_ptr(), P, K.SMH_KV_FP16, d[3].data_ptr(),
                                       d[4].data_ptr(), None, None, S, d[5].data_ptr(), 1, d[6].data_ptr() if current else None,
                                       d[7].data_ptr() if current else None, ws.data_ptr(), ws.numel(), K._stream()), "smh_shared_prefix_attn")
    assert bool(((out.cpu().double() - want).abs() <= tol).all())


@pytest.mark.parametrize("B,H,Hkv,P,S,L", [(2, 4, 4, 64, 20, 20), (2, 4, 4, 0, 20, 20), (2, 4, 4, 64, 20, 0), (20, 8, 2, 300, 70, 64), (3, 8, 2, 200, 9, 5)])
@pytest.mark.parametrize("q40", [False, True])
@pytest.mark.parametrize("single_launch", [False, True])
@pytest.mark.parametrize("current", [False, True])
def test_nan_in_a_query_stays_visible(B, H, Hkv, P, S, L, q40, single_launch, current):
    """a NaN in a query makes every score of it NaN: its output is NaN in every form of the attention (no partial has a maximum then),
    all others are what they are without it"""
    from spec_mcts_amd import kernels as K
    g = _g(300 + B + P)
    q = torch.randn((B, H, 128), generator=g).half()
    pk, pv = (torch.randn((max(P, 1), Hkv, 128), generator=g).half().cuda() if P else None for _ in range(2))
    kw = dict(Smax=S, lens=torch.full((B,), L, dtype=torch.int32).cuda(), n_kv_heads=Hkv, single_launch=single_launch)
    if q40:
        kw.update(zip(("suffix_k", "suffix_v"), (torch.randint(-128, 128, (B, S, Hkv, 64), generator=g, dtype=torch.int16).to(torch.int8).cuda() for _ in range(2))))
        kw.update(zip(("suffix_ks", "suffix_vs"), ((torch.rand((B, S, Hkv, 2), generator=g) * 0.1).half().cuda() for _ in range(2))))
    else:
        kw.update(zip(("suffix_k", "suffix_v"), (torch.randn((B, S, Hkv, 128), generator=g).half().cuda() for _ in range(2))))
    if current:
        kw.update(zip(("cur_k", "cur_v"), (torch.randn((B, Hkv, 128), generator=g).half().cuda() for _ in range(2))))
    clean = K.shared_prefix_attn(q.cuda(), pk, pv, P, **kw).cpu()
    q[B - 1, H - 1, 5] = float("nan")
    got = K.shared_prefix_attn(q.cuda(), pk, pv, P, **kw).cpu()
    assert bool(got[B - 1, H - 1].isnan().all())
    got[B - 1, H - 1] = clean[B - 1, H - 1] = 0
    assert torch.equal(got, clean)


@pytest.mark.parametrize("S,H", [(97, 4), (130, 256)])
@pytest.mark.parametrize("at", [5, 50, 96])
def test_prefill_values_that_are_not_finite_reach_no_earlier_block(S, H, at):
    """masked keys weigh 0, and 0 times an infinity is NaN: a value that is not finite must not reach the blocks of 32 queries before
    its own, whose products leave it out"""
    from spec_mcts_amd import kernels as K
    g = _g(77)
    q, k, v = (torch.randn((S, H, 128), generator=g).half() for _ in range(3))
    clean = K.prefill_attn(q.cuda(), k.cuda(), v.cuda()).cpu()
    v[at, 1, 3], v[at, 1, 4] = float("inf"), float("nan")
    got = K.prefill_attn(q.cuda(), k.cuda(), v.cuda()).cpu()
    assert torch.equal(got[: at // 32 * 32], clean[: at // 32 * 32])
    assert bool(got[at:, 1, 3].isinf().all()) and bool(got[at:, 1, 4].isnan().all())
    others = torch.ones((S, H, 128), dtype=torch.bool)
    others[:, 1, 3:5] = False
    assert torch.equal(got[others], clean[others])


@pytest.mark.parametrize("S", [1, 31, 32, 33, 63, 64, 65, 95, 127, 128, 129, 191, 193, 255, 257, 385])
@pytest.mark.parametrize("H,Hkv", [(256, 32), (2, 1)])
def test_prefill_lengths_around_the_tiles(S, H, Hkv):
    """every remainder class of the waves' 32 queries, the tiles of 64 keys and the workgroups' 64 and 128 queries: 256 heads fill the
    GPU with four query groups a workgroup, 2 heads take two groups"""
    from spec_mcts_amd import kernels as K
    g = _g(500 + S)
    q, k, v = (torch.randn((S, h, 128), generator=g).half() for h in (H, Hkv, Hkv))
    _check(K.prefill_attn(q.cuda(), k.cuda(), v.cuda()), O.causal_attention(q, k, v))


@pytest.mark.parametrize("P", [1, 128, 129, 256, 257, 512, 513, 1050])
@pytest.mark.parametrize("order", ["level", "rising", "falling", "below the suffix"])
def test_merge_at_every_number_of_partials_on_their_way(P, order):
    """fp16 suffixes: slices of 32 prompt rows and the suffix leave 2, 5, 6, 9, 10, 17, 18 and 34 partials a query; the merge has 5, 9 or 17 of them on
    their way at a time.  Scores that rise by 30 from slice to slice let the last one outweigh all before it (e^-30 and less), which the merge has
    scaled already; that fall by 30 leave it to the first; below the suffix the last partial, the suffix's, outweighs them.  A branch without rows"""
    from spec_mcts_amd import kernels as K
    B, S = 5, 9
    q, pk, pv, sk, sv, lens = _inputs(B, 1, 1, 128, P, S, 60 + P)
    lens[:] = torch.tensor([0, 9, 1, 4, 7])
    slices = (P + 31) // 32
    rank = torch.arange(P) // 32
    level = {"level": 0 * rank, "rising": rank, "falling": slices - 1 - rank, "below the suffix": -1 - rank}[order]
    if order != "level":                                   # a score's part of dimension 0 is its key's value there
        q[..., 0] = 128 ** 0.5
        pk[..., 0] = (30 * level).half()[:, None]
        sk[..., 0] = 0
    score = torch.einsum("bhd,lhd->bl", q.float(), pk.float()) / 128 ** 0.5
    top = torch.stack([score[:, rank == i].amax(1) for i in range(slices)], 1)
    own = torch.einsum("bhd,blhd->bl", q.float(), sk.float()) / 128 ** 0.5
    step = top[:, 1:] - top[:, :-1]
    assert {"level": bool((step.abs() < 10).all()), "rising": bool((step > 20).all()), "falling": bool((step < -20).all()),
            "below the suffix": bool((step < -20).all()) and bool((own.amin(1) > top.amax(1) + 20).all())}[order]
    want = O.shared_prefix_attention(q, pk, pv, sk, sv, lens.tolist())
    _check(K.shared_prefix_attn(q.cuda(), pk.cuda(), pv.cuda(), P, suffix_k=sk.cuda(), suffix_v=sv.cuda(), Smax=S, lens=lens.cuda(), lens_stride=1), want)
