"""GPU parity of the Q4_0 codec kernels against the oracle (bit-exact), through the C ABI."""
import numpy as np
import pytest
import torch

from oracle import q40_oracle as O

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _same_or_both_nan(a, b):
    fa, fb = a.view(np.float16), b.view(np.float16)
    return bool(np.all((a == b) | (np.isnan(fa) & np.isnan(fb))))


def test_dequant_exhaustive_bit_exact(cref):
    """every nibble pattern x every fp16 scale pattern, against the integer-only C table"""
    from spec_mcts_amd import kernels as K
    table = np.zeros(16 * 65536, dtype=np.uint16)
    cref.q40_ref_dequant_table(table.ctypes.data)
    table = table.reshape(16, 65536)
    # every row holds all 16 patterns in both nibble positions; row r uses scales (2r, 2r+1).
    # Two passes (the second with neighbouring scales swapped) cover all 16 x 65536 pairs for
    # both nibble positions.
    rows = 32768
    j = torch.arange(64)
    byte_row = ((j % 16) << 4) | ((j % 16 + j // 16) % 16)
    byte = byte_row[None, :].expand(rows, 64).contiguous()
    w = byte.to(torch.uint8).view(torch.int8)
    b = byte.numpy()
    r = np.arange(rows)[:, None]
    for swap in (0, 1):
        idx = torch.arange(65536, dtype=torch.int32) ^ swap
        scales = idx.to(torch.int16).view(torch.float16).view(-1, 1)
        got = _bits(K.deq_int40(w.cuda(), scales.cuda(), 64, (rows * 2, 64))).reshape(rows, 2, 64)
        assert _same_or_both_nan(got[:, 0, :], table[b >> 4, (2 * r) ^ swap])
        assert _same_or_both_nan(got[:, 1, :], table[b & 15, (2 * r + 1) ^ swap])


@pytest.mark.parametrize("shape", [(11008, 4096), (128, 64), (2, 64)])
def test_dequant_random_weights_bit_exact(shape):
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(0)
    v = (torch.randn(shape, generator=g) * 0.02).to(torch.float16)
    w, s = O.quantize_q40(v, 64)
    want = O.dequantize_q40(w, s, 64, shape)
    got = K.deq_int40(w.cuda(), s.cuda(), 64, shape)
    assert got.shape == tuple(shape) and got.dtype == torch.float16
    assert np.array_equal(_bits(got), _bits(want))


def test_quantize_matches_torch_rounding():
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(1)
    x = (torch.randn((4096, 64), generator=g) * 0.5).to(torch.float16)
    x[3] = 0                                            # 0/0 -> code 0, scale 0
    x[5, 7] = 6.0e4
    x[6] = x[6] * 1e-4                                   # subnormal scales
    x[8, :8] = torch.tensor([0.5, -0.5, 1.5, -1.5, 2.5, -2.5, 3.5, 7.0], dtype=torch.float16)
    x[8, 8:] = 0                                         # exact ties: round half to even
    w_want, s_want = O.quantize_q40(x, 64)
    w_got, s_got = K.q_int40(x.cuda(), 64)
    assert w_got.shape == w_want.shape and s_got.shape == s_want.shape
    assert np.array_equal(_bits(s_got), _bits(s_want))
    assert torch.equal(w_got.cpu(), w_want)
    # round trip on the device reproduces the oracle's dequantised values
    back = K.deq_int40(w_got, s_got, 64, x.shape)
    assert np.array_equal(_bits(back), _bits(O.dequantize_q40(w_want, s_want, 64, x.shape)))
    # idempotence at full size: quantising dequantised data is the identity on (codes, scales)
    w2, s2 = K.q_int40(back, 64)
    assert torch.equal(w2, w_got) and torch.equal(s2, s_got)


def test_quantize_dispatch_host_tensor():
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(2)
    x = torch.randn((8, 64), generator=g).to(torch.bfloat16)
    w, s = K.quantize_q40(x, 64)
    w2, s2 = O.quantize_q40(x, 64)
    assert torch.equal(w, w2) and torch.equal(s, s2)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,Kd", [(128, 1), (128, 63), (256, 64), (384, 65), (640, 200), (1024, 129)])
def test_quantize_of_the_transpose_matches_the_oracle(dtype, N, Kd):
    """edges of the 128 x 64 tile, rows of odd length, zero groups, subnormal and infinite scales, quotients at rounding ties"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(N + Kd)
    v = torch.randn((N, Kd), generator=g) * 0.02
    v[:64, 0] = 0
    v[64:128, -1] *= 1e-4
    v[:17, Kd // 2] = torch.tensor([7.0, 0.5, -0.5, 1.5, -1.5, 2.5, -2.5, 3.5, 6.5, -6.5, 4.5, 5.5, 2.4995, 2.5005, 1.4995, 1.5005, 0.50012])
    v[17:64, Kd // 2] = 0
    v = v.to(dtype)
    if dtype != torch.float16 and Kd > 2:
        v[70, 1] = 1e6                                    # the scale overflows fp16
    w_want, s_want = O.quantize_q40(v.t().contiguous(), 64)
    w_got, s_got = K.quantize_q40_t(v.cuda())
    assert np.array_equal(_bits(s_got).reshape(-1), _bits(s_want).reshape(-1))
    assert torch.equal(w_got.cpu(), w_want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,Kd", [(128, 31), (384, 33), (8192, 65), (8320, 70)])
def test_quantize_of_the_transpose_next_to_ties(dtype, N, Kd):
    """quotients on and next to points where a code changes, under scales from 2^-14 (the smallest that is multiplied by, not divided) to 2^7, in blocks
    of outputs taken all or two at a time (65: the last one alone): the oracle's bytes"""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(N + Kd)
    half_steps = torch.randint(-14, 15, (N, Kd), generator=g).float() / 2
    half_steps[::64] = 7.0
    step = 2.0 ** torch.randint(-14, 8, (1, Kd), generator=g).float()
    ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7, torch.float32: 2.0 ** -23}[dtype]
    near = 1 + torch.randint(-4, 5, (N, Kd), generator=g).float() * ulp
    for v in (half_steps * step, half_steps * step * near, half_steps * step * 1.3717 * near):
        v = v.to(dtype)
        w_want, s_want = O.quantize_q40(v.t().contiguous(), 64)
        w_got, s_got = K.quantize_q40_t(v.cuda())
        assert np.array_equal(_bits(s_got).reshape(-1), _bits(s_want).reshape(-1))
        assert torch.equal(w_got.cpu(), w_want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_quantize_nan_values(dtype):
    """A NaN has code 0, whatever its payload.  In a group of fp32 or bfloat16 values it does not count towards the scale (the bytes are
    those of the group with a zero in its place); a group of fp16 values with a NaN has a NaN scale and codes 0."""
    from spec_mcts_amd import kernels as K
    g = torch.Generator().manual_seed(9)
    v = (torch.randn((256, 70), generator=g) * 0.02).to(dtype)
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    exponent = {torch.float16: 0x7C00, torch.bfloat16: 0x7F80, torch.float32: 0x7F800000}[dtype]
    at = [(5, 0), (63, 0), (64, 7), (130, 33), (131, 33), (255, 69)]
    for i, (n, k) in enumerate(at):
        v.view(bits)[n, k] = exponent + 1 + 2 * i                 # payloads with low bits set
    v.view(bits)[200, 50] = -1                                    # all ones
    assert int(torch.isnan(v).sum()) == len(at) + 1
    clean = torch.where(torch.isnan(v), torch.zeros_like(v), v)
    w_want, s_want = O.quantize_q40(clean.t().contiguous(), 64)
    forms = [K.quantize_q40_t(v.cuda()), K.quantize_q40(v.t().contiguous().cuda())]
    if dtype == torch.float16:
        groups = torch.isnan(v.t().reshape(-1, 64)).any(1)
        nib = w_want.view(torch.uint8).clone().view(-1, 64)
        nib[groups[0::2]] &= 15                                   # even groups: high nibbles
        nib[groups[1::2]] &= 240
        w_want = nib.view(torch.int8).view_as(w_want)
        s_want = s_want.clone()
        s_want.view(-1)[groups] = float("nan")
    for w, s in forms:
        assert torch.equal(w.cpu(), w_want)
        assert _same_or_both_nan(_bits(s).reshape(-1), _bits(s_want).reshape(-1))
