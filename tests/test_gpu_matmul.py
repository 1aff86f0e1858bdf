"""GPU parity of the fused Q4_0 dequant+matmul (GEMV for M<=16, LDS/MFMA GEMM above) against the
oracle.  Tolerance is the one the task states for fp16 outputs: 1e-2 relative + 2e-3 absolute."""
import numpy as np
import pytest
import torch

from oracle import q40_oracle as O

pytestmark = pytest.mark.gpu
RTOL, ATOL = 1e-2, 2e-3


def _weights(N, K, seed, std=0.02):
    g = torch.Generator().manual_seed(seed)
    v = (torch.randn((N, K), generator=g) * std).to(torch.float16)
    w, s, _ = O.quantize_weight(v)
    return w, s


def _acts(M, K, seed):
    return torch.randn((M, K), generator=torch.Generator().manual_seed(seed)).to(torch.float16)


def _check(got, want):
    got, want = got.float().cpu(), want.float()
    err = (got - want).abs()
    tol = ATOL + RTOL * want.abs()
    assert bool((err <= tol).all()), f"max err {err.max():.4e}, worst excess {(err - tol).max():.4e}"


def test_config0_single_linear():
    """x[1,4096] . W[11008,4096]^T, seed 0: dequant bit-exact, output within tolerance"""
    from spec_mcts_amd import kernels as K
    N, Kd = 11008, 4096
    g = torch.Generator().manual_seed(0)
    x = torch.randn((1, Kd), generator=g).to(torch.float16)
    v = (torch.randn((N, Kd), generator=g) * 0.02).to(torch.float16)
    w, s, shp = O.quantize_weight(v)
    wd, sd_ = w.cuda(), s.cuda()
    deq = K.deq_int40(wd, sd_, 64, (Kd, N))
    assert torch.equal(deq.cpu().view(torch.int16), O.dequantize_q40(w, s, 64, (Kd, N)).view(torch.int16))
    y = K.matmul_q40(x.cuda(), wd, sd_, (Kd, N))
    assert y.shape == (1, N) and y.dtype == torch.float16
    _check(y, O.matmul_q40(x, w, s, (Kd, N)))
    _check(y, O.linear_q40_cpu_path(x, w, s, (N, Kd)))


def test_config0_as_worded_block32_flavour():
    """The first configuration as its text words it: W [11008, 4096] in 32-weight blocks, scale = absmax / 8, q in [0, 15],
    value = (q - 8) * scale (a format the reference's code does not have).  GPU quantiser = oracle quantiser byte for
    byte, dequant bit-exact, y = x . W^T within tolerance."""
    from spec_mcts_amd import kernels as K
    N, Kd = 11008, 4096
    g = torch.Generator().manual_seed(0)
    x = torch.randn((1, Kd), generator=g).to(torch.float16)
    v = (torch.randn((N, Kd), generator=g) * 0.02).to(torch.float16)
    packed, scale = O.quantize_gq40(v)
    pd, sd_ = K.quantize_gq40(v.cuda())
    assert torch.equal(pd.cpu(), packed) and torch.equal(sd_.cpu().view(torch.int16), scale.view(torch.int16))
    deq = K.dequantize_gq40(pd, sd_, (N, Kd))
    want = O.dequantize_gq40(packed, scale, (N, Kd))
    assert torch.equal(deq.cpu().view(torch.int16), want.view(torch.int16))
    assert float((want.float() - v.float()).abs().max()) <= float(scale.float().max())            # it is a quantisation of v
    y = K.linear_gq40(x.cuda(), pd, sd_, (N, Kd))
    _check(y, O.linear_gq40(x, packed, scale, (N, Kd)))
    # zeros, a lone spike and the largest fp16 value survive the round trip's edge cases
    e = torch.zeros((4, 64), dtype=torch.float16)
    e[1, 5], e[2, 40], e[3, :] = 3.0, -65504.0, 1e-7
    pe, se = K.quantize_gq40(e.cuda())
    po, so = O.quantize_gq40(e)
    assert torch.equal(pe.cpu(), po) and torch.equal(se.cpu().view(torch.int16), so.view(torch.int16))
    assert torch.equal(K.dequantize_gq40(pe, se, e.shape).cpu().view(torch.int16), O.dequantize_gq40(po, so, e.shape).view(torch.int16))


SHAPES = [(4096, 4096), (11008, 4096), (4096, 11008), (32128, 4096)]   # 32016 padded to 251*128


@pytest.mark.parametrize("idx", range(len(SHAPES)))
def test_config1_sweep(idx):
    from spec_mcts_amd import kernels as K
    N, Kd = SHAPES[idx]
    w, s = _weights(N, Kd, 1000 + idx)
    wd, sd_ = w.cuda(), s.cuda()
    deq = O.dequantize_q40(w, s, 64, (Kd, N)).float()
    for M in (1, 10, 100):
        a = _acts(M, Kd, 2000 + 10 * idx + M)
        got = K.matmul_q40(a.cuda(), wd, sd_, (Kd, N))
        want = (a.float() @ deq).to(torch.float16)
        _check(got, want)
        # a second launch reuses the self-cleaning workspace and must give the same bits
        again = K.matmul_q40(a.cuda(), wd, sd_, (Kd, N))
        assert torch.equal(got, again)


@pytest.mark.parametrize("M", [1, 3, 16, 17, 100, 130, 300])
def test_one_hot_rows_are_bit_exact(M):
    """x = e_k returns row k of the dequantised matrix exactly (covers every column-block boundary)"""
    from spec_mcts_amd import kernels as K
    N, Kd = 384, 512
    w, s = _weights(N, Kd, 7)
    deq = O.dequantize_q40(w, s, 64, (Kd, N))
    ks = torch.randint(0, Kd, (M,), generator=torch.Generator().manual_seed(M))
    ks[0] = 0
    ks[-1] = Kd - 1
    a = torch.zeros((M, Kd), dtype=torch.float16)
    a[torch.arange(M), ks] = 1.0
    got = K.matmul_q40(a.cuda(), w.cuda(), s.cuda(), (Kd, N)).cpu()
    assert torch.equal(got.view(torch.int16), deq[ks].view(torch.int16))
    zero = K.matmul_q40(torch.zeros((M, Kd), dtype=torch.float16).cuda(), w.cuda(), s.cuda(), (Kd, N))
    assert bool((zero == 0).all())


@pytest.mark.parametrize("M,N,Kd", [(2, 128, 8), (5, 256, 40), (16, 128, 72), (40, 256, 200), (129, 128, 1000),
                                    (33, 128, 32), (40, 256, 96), (100, 128, 160), (17, 256, 224), (100, 384, 416)])
def test_ragged_k_and_small_shapes(M, N, Kd):
    """K not a multiple of the 32-row step, single column block, M around the tile sizes"""
    from spec_mcts_amd import kernels as K
    w, s = _weights(N, Kd, 11, std=0.05)
    a = _acts(M, Kd, 12)
    got = K.matmul_q40(a.cuda(), w.cuda(), s.cuda(), (Kd, N))
    _check(got, O.matmul_q40(a, w, s, (Kd, N)))


@pytest.mark.parametrize("M,N,Kd", [(17, 128, 32), (33, 384, 160), (48, 128, 4096), (64, 11008, 256), (81, 640, 1056), (100, 20224, 512),
                                    (128, 384, 2048), (129, 128, 224), (250, 8192, 96), (300, 24704, 64),
                                    # K not a multiple of 32: 8, 16 and 24 rows of k in the last step, also as the only step of a slice
                                    (17, 128, 8), (33, 384, 168), (64, 11008, 264), (81, 640, 1048), (100, 4096, 4088), (100, 20224, 520),
                                    (128, 384, 2056), (129, 128, 232), (250, 8192, 88), (300, 24704, 72)])
def test_checkpoint_layout_by_workgroups(M, N, Kd):
    """eight waves and the DMA waves (one workgroup a compute unit, range cut among them) or four waves: column units of one block,
    few steps, edges of row tiles; fp32 sums of exact products, one rounding to fp16"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M + N)
    w, s = K.quantize_q40(torch.randn((Kd, N), device="cuda", generator=g).half())
    x = torch.randn((M, Kd), device="cuda", generator=g).half()
    d = K.deq_int40(w, s, 64, (Kd, N))
    want = x.double() @ d.double()
    got = K.matmul_q40(x, w, s, (Kd, N)).double()
    bound = want.abs() * 2.0 ** -11 + 2.0 ** -24 + (x.double().abs() @ d.double().abs()) * Kd * 2.0 ** -24      # the rounding; sums of Kd terms
    assert bool(((got - want).abs() <= bound).all())


@pytest.mark.parametrize("M", [4, 100])
def test_residual_epilogue(M):
    from spec_mcts_amd import kernels as K
    N, Kd = 512, 1024
    w, s = _weights(N, Kd, 13)
    a = _acts(M, Kd, 14)
    r = _acts(M, N, 15)
    got = K.matmul_q40(a.cuda(), w.cuda(), s.cuda(), (Kd, N), residual=r.cuda())
    want = r + O.matmul_q40(a, w, s, (Kd, N))            # fp16 add of the fp16 product, as h + wo(..)
    _check(got, want)


def test_linearity_at_full_size():
    """size-independent property at a BASELINE shape: f(x1) + f(x2) ~ f(x1 + x2), f(2x) = 2 f(x) exactly"""
    from spec_mcts_amd import kernels as K
    N, Kd = 11008, 4096
    w, s = _weights(N, Kd, 16)
    wd, sd_ = w.cuda(), s.cuda()
    x1, x2 = _acts(10, Kd, 17).cuda(), _acts(10, Kd, 18).cuda()
    y1 = K.matmul_q40(x1, wd, sd_, (Kd, N)).float()
    y2 = K.matmul_q40(x2, wd, sd_, (Kd, N)).float()
    y12 = K.matmul_q40((x1.float() * 0.5 + x2.float() * 0.5).half(), wd, sd_, (Kd, N)).float()
    assert torch.allclose(y12, 0.5 * (y1 + y2), rtol=RTOL, atol=2 * ATOL)
    # scaling the input scales the output (up to the fp16 rounding of the scaled activations)
    y = K.matmul_q40(x1, wd, sd_, (Kd, N)).float()
    yd = K.matmul_q40(x1 * 2, wd, sd_, (Kd, N)).float()
    assert torch.allclose(yd, 2 * y, rtol=RTOL, atol=2 * ATOL)


def test_argument_errors():
    from spec_mcts_amd import kernels as K
    w, s = _weights(128, 64, 19)
    a = _acts(2, 64, 20).cuda()
    with pytest.raises(AssertionError):
        K.matmul_q40(a, w.cuda(), s.cuda(), (32, 128))                    # K mismatch
    with pytest.raises(AssertionError):
        K.matmul_q40(a.t().contiguous().t(), w.cuda(), s.cuda(), (64, 128))  # non-contiguous A
    with pytest.raises(AssertionError):
        K.matmul_q40(a.cpu(), w, s, (64, 128))                            # no CPU fallback


@pytest.mark.parametrize("M", [1, 10, 100])
def test_fused_segments_and_consumers(M):
    """wq|wk|wv and w1|w3 as segments of one launch; slab consumers against the oracle's cast points"""
    from spec_mcts_amd import kernels as K
    Kd = 1024
    ws = [_weights(n, Kd, 50 + i) for i, n in enumerate((512, 256, 256))]
    a = _acts(M, Kd, 60 + M)
    lin = [(w.cuda(), s.cuda(), n) for (w, s), n in zip(ws, (512, 256, 256))]
    pp = K.matmul_q40_partial(a.cuda(), lin)
    assert pp.n_total == 1024 and pp.M == M
    want = torch.cat([O.matmul_q40(a, w, s, (Kd, n)) for (w, s), n in zip(ws, (512, 256, 256))], 1)
    got = K.partial_reduce(pp)
    _check(got, want)
    # column windows and the residual epilogue
    r = _acts(M, 256, 70)
    _check(K.partial_reduce(pp, 512, 256, residual=r.cuda()), r + want[:, 512:768])
    # SiLU(gate) * up with gate = columns [0,512), up = columns [512,1024)
    got_act = K.partial_silu_mul(pp).cpu()
    g16, u16 = got[:, :512].cpu(), got[:, 512:].cpu()
    want_act = O.silu_mul(g16, u16)
    assert torch.allclose(got_act.float(), want_act.float(), rtol=2e-3, atol=1e-4)
    # residual + RMSNorm consumer on a [M, 1024] product
    wt = (1 + 0.1 * torch.randn(1024, generator=torch.Generator().manual_seed(71))).to(torch.float16)
    hin = _acts(M, 1024, 72)
    h, xn = K.partial_rmsnorm(pp, hin.cuda(), wt.cuda(), 1e-5)
    h_want = hin + got.cpu()
    assert torch.equal(h.cpu(), h_want)
    xn_want = O.rmsnorm(h_want, wt, 1e-5)
    assert torch.allclose(xn.cpu().float(), xn_want.float(), rtol=2e-3, atol=1e-4)
    assert (xn.cpu() != xn_want).float().mean() < 0.01


def test_fused_rope_append_consumer_bit_exact():
    from spec_mcts_amd import kernels as K
    B, H, Hkv, D, Kd, Smax = 3, 4, 2, 128, 512, 4
    ws = [_weights(n, Kd, 80 + i, std=0.05) for i, n in enumerate((H * D, Hkv * D, Hkv * D))]
    a = _acts(B, Kd, 83)
    lin = [(w.cuda(), s.cuda(), n) for (w, s), n in zip(ws, (H * D, Hkv * D, Hkv * D))]
    pp = K.matmul_q40_partial(a.cuda(), lin)
    flat = K.partial_reduce(pp).cpu()
    q0 = flat[:, :H * D].view(B, 1, H, D); k0 = flat[:, H * D:(H + Hkv) * D].view(B, 1, Hkv, D)
    v0 = flat[:, (H + Hkv) * D:].view(B, Hkv, D)
    fc = O.precompute_freqs_cis(D, 32, 1e6)
    pos, t = 9, 2
    qe, ke = O.apply_rotary_emb(q0, k0, fc[pos:pos + 1])
    cos, sin = fc.real.to(torch.float16).contiguous().cuda(), fc.imag.to(torch.float16).contiguous().cuda()
    rows = B * Smax * Hkv
    ck = torch.zeros((rows, 64), dtype=torch.int8).cuda(); cks = torch.zeros((rows * 2, 1), dtype=torch.float16).cuda()
    cv = torch.zeros((rows, 64), dtype=torch.int8).cuda(); cvs = torch.zeros((rows * 2, 1), dtype=torch.float16).cuda()
    st = torch.tensor([pos, t], dtype=torch.int32).cuda()
    q, k, v = K.partial_rope_append_kv(pp, H, Hkv, D, cos, sin, st[0:1], ck, cks, cv, cvs, Smax, st[1:2])
    assert torch.equal(q.cpu().view(torch.int16), qe[:, 0].view(torch.int16))
    assert torch.equal(k.cpu().view(torch.int16), ke[:, 0].view(torch.int16))
    assert torch.equal(v.cpu().view(torch.int16), v0.view(torch.int16))
    wk, sk = O.quantize_q40(ke[:, 0], 64); wv, sv = O.quantize_q40(v0, 64)
    assert torch.equal(ck.cpu().view(B, Smax, Hkv, 64)[:, t], wk.view(B, Hkv, 64))
    assert torch.equal(cv.cpu().view(B, Smax, Hkv, 64)[:, t], wv.view(B, Hkv, 64))
    assert torch.equal(cks.cpu().view(B, Smax, Hkv, 2)[:, t].view(torch.int16), sk.view(B, Hkv, 2).view(torch.int16))
    assert torch.equal(cvs.cpu().view(B, Smax, Hkv, 2)[:, t].view(torch.int16), sv.view(B, Hkv, 2).view(torch.int16))


@pytest.mark.parametrize("M", [1, 16, 17, 100])
def test_matmul_workspace_serves_the_c_entry_point(M):
    """smh_q40_matmul on the workspace that matmul_workspace returns: what matmul_q40 returns, bit for bit"""
    from spec_mcts_amd import _lib, kernels as K
    N, Kd = 1024, 2048
    g = torch.Generator().manual_seed(60 + M)
    w, s = K.quantize_q40((torch.randn((Kd, N), generator=g) * 0.02).half().cuda())
    a = torch.randn((M, Kd), generator=g).half().cuda()
    ws = K.matmul_workspace(a.device, M, N)
    assert ws.numel() >= _lib.load().smh_q40_matmul_workspace_bytes(M, N) and K.matmul_workspace(a.device, 1, 128) is ws
    c = torch.empty((M, N), dtype=torch.float16, device=a.device)
    K.check(_lib.load().smh_q40_matmul(a.data_ptr(), M, Kd, Kd, w.data_ptr(), s.data_ptr(), N, c.data_ptr(), N, K.SMH_EPI_NONE, None, N,
                                       ws.data_ptr(), ws.numel(), K._stream()), "smh_q40_matmul")
    assert torch.equal(c, K.matmul_q40(a, w, s, (Kd, N)))


@pytest.mark.parametrize("M,N,K", [(33, 4352, 2880), (100, 4352, 2888), (17, 6400, 1920), (96, 2304, 1032), (257, 2688, 1040), (300, 5120, 1024)])
def test_matmul_with_few_column_units(M, N, K):
    """Column units that do not divide by the eight XCDs: launches of at most 256 workgroups of which one XCD would get more than 32
    (four waves a workgroup where its steps are few), K a multiple of 32 and not, and row blocks planned for the busiest XCD"""
    from spec_mcts_amd import kernels as K_
    w, s = _weights(N, K, seed=N + K)
    a = _acts(M, K, seed=M)
    r = _acts(M, N, seed=M + 1)
    want = O.matmul_q40(a, w, s, (K, N)).float()
    got = K_.matmul_q40(a.cuda(), w.cuda(), s.cuda(), (K, N)).cpu().float()
    assert torch.allclose(got, want, rtol=RTOL, atol=ATOL)
    got = K_.matmul_q40(a.cuda(), w.cuda(), s.cuda(), (K, N), residual=r.cuda()).cpu().float()
    assert torch.allclose(got, r.float() + want, rtol=RTOL, atol=2 * ATOL)


@pytest.mark.parametrize("ks", range(1, 17))
def test_consumers_at_every_number_of_slabs(ks):
    """Each consumer of a product's slabs against itself on one slab that holds their sum: the sums in slice order and nothing else, at
    numbers with a kernel of their own and at those between; what lies behind the last slab (NaN) is not added."""
    from spec_mcts_amd import _lib, kernels as K
    lib, dev = _lib.load(), "cuda:0"
    g = torch.Generator(device=dev).manual_seed(ks)
    for M, n in ((3, 768), (2, 5120), (2, 12288)):     # one, two and four passes of a row; two query heads and more, one kv head in three
        buf = torch.full((17, M, n), float("nan"), device=dev)
        buf[:ks] = torch.randn((ks, M, n), device=dev, generator=g)
        total = torch.zeros((M, n), device=dev)
        for s in range(ks):
            total = total + buf[s]
        both = K.PartialProduct(buf, ks, M, n), K.PartialProduct(total[None].contiguous(), 1, M, n)
        h, w = torch.randn((M, n), device=dev, generator=g).half(), torch.randn(n, device=dev, generator=g).half()
        odd = torch.empty(M * n + 1, dtype=torch.float16, device=dev)[1:].view(M, n).copy_(h)          # (a residual that is not aligned)
        heads = n // 128
        hkv = heads // 6
        H = heads - 2 * hkv
        angles = torch.randn((16, 64), device=dev, generator=g)
        cos, sin = angles.cos().half(), angles.sin().half()
        results = []
        for p in both:
            out = [K.partial_reduce(p), K.partial_reduce(p, 128, 256), K.partial_reduce(p, residual=h), K.partial_reduce(p, residual=odd)]
            out += [*K.partial_rmsnorm(p, h, w, 1e-5), *K.partial_rmsnorm(p, None, w, 1e-5), *K.partial_residual_sumsq(p, h), *K.partial_residual_sumsq(p, None)]
            out.append(K.partial_silu_mul(p))
            ck, cks = torch.zeros((M * 4 * hkv, 64), dtype=torch.int8, device=dev), torch.zeros((M * 8 * hkv, 1), dtype=torch.float16, device=dev)
            cv, cvs = ck.clone(), cks.clone()
            st = torch.tensor([9, 2], dtype=torch.int32, device=dev)
            out += [*K.partial_rope_append_kv(p, H, hkv, 128, cos, sin, st[0:1], ck, cks, cv, cvs, 4, st[1:2]), ck, cks, cv, cvs]
            q, k, v = (torch.empty((M, x, 128), dtype=torch.float16, device=dev) for x in (H, hkv, hkv))
            _lib.check(lib.smh_partial_rope_rows(p.buf.data_ptr(), p.ksplit, M, H, hkv, 128, q.data_ptr(), k.data_ptr(), v.data_ptr(), cos.data_ptr(),
                                                 sin.data_ptr(), 1, K._stream()), "smh_partial_rope_rows")
            results.append(out + [q, k, v])
        for i, (a, b) in enumerate(zip(*results)):
            assert bool(a.float().isfinite().all()) and torch.equal(a, b), (i, M, n)


@pytest.mark.parametrize("M", [17, 61, 80, 100, 128, 300])
@pytest.mark.parametrize("K,N", [(2056, 11008), (4112, 4096), (6168, 3712), (264, 8192), (8168, 16384), (4096, 4096), (224, 4096)])
def test_checkpoint_products_at_the_end_of_k(M, K, N):
    """17 rows and more on the checkpoint layout: the end of K (8, 16, 24 or 32 rows of its last step) lies in one slice of K, in whichever stage
    of the ring that slice's start makes it, and adds nothing past K.  Against 64 bits: half a unit of fp16 and the fp32 sums"""
    from spec_mcts_amd import kernels as Kn
    g = torch.Generator(device="cuda").manual_seed(M + K)
    w, s = Kn.quantize_q40(torch.randn((K, N), device="cuda", generator=g, dtype=torch.float16) * 0.02)
    x = torch.randn((M, K), device="cuda", generator=g, dtype=torch.float16)
    got = Kn.matmul_q40(x, w, s, (K, N)).double()
    want = x.double() @ Kn.deq_int40(w, s, 64, (K, N)).double()
    assert bool(((got - want).abs() <= want.abs() * 2.0 ** -11 + 2.0 ** -24 * K ** 0.5 * want.abs().max()).all())


@pytest.mark.parametrize("M,K,columns,stored", [(1040, 2048, 128, True), (900, 1536, 256, False), (300, 4096, 128, False)])
def test_checkpoint_product_over_its_own_activations(M, K, columns, stored):
    """A product whose K is cut reads all of its activations before the launch that writes the result, so the result may take their place: also where the
    plan's two slices become one slice of 128-column blocks, which apart is stored without slabs.  The same bits as apart"""
    from spec_mcts_amd import _lib, kernels as Kn
    ks = Kn.matmul_plan(M, K, [K])
    assert ks > 1 and _lib.load().smh_q40_matmul_columns(M, K, K) == columns
    g = torch.Generator(device="cuda").manual_seed(M + K)
    w, s = Kn.quantize_q40(torch.randn((K, K), device="cuda", generator=g, dtype=torch.float16) * 0.02)
    x = torch.randn((M, K), device="cuda", generator=g, dtype=torch.float16)
    apart = Kn.matmul_q40(x, w, s, (K, K))
    slabs, c = torch.full((ks * M * K,), float("nan"), device="cuda"), torch.empty((M, K), device="cuda", dtype=torch.float16)
    Kn.check(_lib.load().smh_q40_matmul(x.data_ptr(), M, K, K, w.data_ptr(), s.data_ptr(), K, c.data_ptr(), K, Kn.SMH_EPI_NONE, None, K, slabs.data_ptr(),
                                        slabs.numel() * 4, Kn._stream()), "smh_q40_matmul")
    assert torch.equal(c, apart) and bool(slabs.isnan().all()) == stored
    assert torch.equal(Kn.matmul_q40(x, w, s, (K, K), out=x), apart)


# row counts of the test below that keep 256 columns a workgroup
WIDE_ROWS = {(4104, 3840): (512,), (1928, 24064): (129, 200, 273, 512), (3000, 6400): (273, 512), (2072, 5760): (512,), (7168, 7168): (129, 200, 273, 512),
             (1496, 21760): (129, 200, 273, 512), (1024, 2944): (17, 48, 64)}


@pytest.mark.parametrize("M", [17, 48, 64, 65, 97, 128, 129, 200, 273, 512])
@pytest.mark.parametrize("K,N", [(4096, 4096), (4104, 3840), (1928, 24064), (3000, 6400), (2072, 5760), (7168, 7168), (1496, 21760), (1024, 2944)])
def test_checkpoint_products_in_blocks_of_128_columns(M, K, N):
    """Launches of 128-column blocks with two K-groups a workgroup: edges of the row tiles and of the two row blocks, odd numbers of blocks, K that ends in
    the first or the second half of a stage, one slice (stored without slabs) and several, with and without a residual, in rows of a larger output.  Against
    64 bits: half a unit of fp16 and the fp32 sums; with the residual another half.  Where the other launch is planned, the same"""
    from spec_mcts_amd import _lib, kernels as Kn
    assert _lib.load().smh_q40_matmul_columns(M, K, N) == (256 if M in WIDE_ROWS.get((K, N), ()) else 128)
    g = torch.Generator(device="cuda").manual_seed(7 * M + K)
    w, s = Kn.quantize_q40(torch.randn((K, N), device="cuda", generator=g, dtype=torch.float16) * 0.02)
    x = torch.randn((M, K), device="cuda", generator=g, dtype=torch.float16)
    r = torch.randn((M, N), device="cuda", generator=g, dtype=torch.float16)
    want = x.double() @ Kn.deq_int40(w, s, 64, (K, N)).double()
    err = want.abs() * 2.0 ** -11 + 2.0 ** -24 * K ** 0.5 * want.abs().max()
    got = Kn.matmul_q40(x, w, s, (K, N)).double()
    assert bool(((got - want).abs() <= err).all())
    sum_ = want + r.double()
    got = Kn.matmul_q40(x, w, s, (K, N), residual=r).double()
    assert bool(((got - sum_).abs() <= err + (sum_.abs() + err) * 2.0 ** -11).all())
    wide = torch.full((M, N + 12), float("nan"), device="cuda", dtype=torch.float16)
    ks = Kn.matmul_plan(M, K, [N])
    if ks > 1:                                             # (an output row of N + 12: a multiple of 4, which the slabs' sum takes)
        ws = torch.empty(ks * M * N * 4, dtype=torch.uint8, device="cuda")
        Kn.check(_lib.load().smh_q40_matmul(x.data_ptr(), M, K, K, w.data_ptr(), s.data_ptr(), N, wide.data_ptr(), N + 12, Kn.SMH_EPI_NONE, None, N, ws.data_ptr(),
                                            ws.numel(), Kn._stream()), "smh_q40_matmul")
        assert torch.equal(wide[:, :N], Kn.matmul_q40(x, w, s, (K, N))) and bool(wide[:, N:].isnan().all())
