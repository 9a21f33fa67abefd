"""GPU parity of the small-output GEMM kernels at the edges of their tiles and of the rules that choose them.

wf_gemm_bf16: the few-row kernel (1-16 rows; to 64 with SiLU on the input), the LDS tiles of gemm_small.hpp (32 x 64
and 64 x 64 with loading waves of their own, 64 x 128, 128 x 128) and the direct kernel behind them, which all give
a row the same bits; sizes one off a tile, K tails inside a 64-element step, rows and columns past the end,
strided A and y, a bias that is only 2-byte aligned, no bias.

Bound per element, against the product in 64 bits: fp32 accumulation in any order, K 2^-23 sum |a w| (with
margin 2 over (K - 1) 2^-24), then one bf16 rounding (half an ulp of 8 significand bits: 2^-8 of the value); an
activation has slope at most 1.13 and adds a rounding of its own and the hardware exponential's and reciprocal's few ulps (2^-20).
"""

import pytest
import torch

from waveforcing_amd import _lib
from waveforcing_amd.dit import gemm_bf16
from waveforcing_amd.fp8 import gemm_fp8_pertensor, gemm_i8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rand(shape, seed, std=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * std).to(torch.bfloat16).to(DEV)


def _check_bf16(got, a, w, b, silu_in, act):
    a64, w64 = a.double(), w.double()
    if silu_in:  # rounded to bf16 as the module's output; the kernel's own rounding may differ by an ulp
        slack = (a64 * torch.sigmoid(a64)).abs() * 2.0 ** -8
        a64 = a64 * torch.sigmoid(a64)
    else:
        slack = torch.zeros_like(a64)
    pre = a64 @ w64.t() + (0 if b is None else b.double())
    err = a.shape[1] * 2.0 ** -23 * (a64.abs() @ w64.abs().t()) + slack @ w64.abs().t() + 2.0 ** -8 * pre.abs()
    ref = pre
    if act == "silu":
        ref = pre * torch.sigmoid(pre)
    elif act == "gelu":
        ref = torch.nn.functional.gelu(pre, approximate="tanh")
    bound = (1.13 * err + (2.0 ** -8 + 2.0 ** -20) * ref.abs() if act else err) * 1.01 + 1e-30
    worst = ((got.double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, f"{worst:.3f} of the bound"


@pytest.mark.parametrize("M,K,N,silu_in,act", [
    (1, 8, 4, False, None), (1, 256, 1536, False, "silu"), (3, 1536, 9216, True, None), (8, 72, 20, True, "gelu"),
    (9, 1544, 60, False, "gelu"), (16, 520, 17 * 4, True, "silu"), (16, 1536, 16, False, None),
    (17, 64, 64, True, None), (33, 200, 36, True, "silu"), (64, 136, 132, True, None), (65, 264, 68, True, "gelu"),
    (17, 72, 60, False, None), (32, 512, 64, False, "gelu"), (33, 1032, 68, False, "silu"), (300, 4096, 1536, False, "gelu"),
    (512, 4096, 1536, False, "gelu"), (513, 1544, 1540, False, None), (780, 1536, 1536, False, None),
    (1100, 520, 2052, False, None), (4680, 64, 1536, False, None), (129, 192, 4100, False, "silu"),
    (2000, 328, 2500, False, None), (4680, 1536, 64, False, None),
])
def test_gemm_bf16_tiles(M, K, N, silu_in, act):
    a, w, b = _rand((M, K), M + K), _rand((N, K), N, 0.05), _rand((N,), 7)
    _check_bf16(gemm_bf16(a, w, b, silu_in=silu_in, act_out=act), a, w, b, silu_in, act)


@pytest.mark.parametrize("M,K,N", [(3, 264, 20), (40, 264, 36), (300, 264, 500), (700, 1032, 3000)])
def test_gemm_bf16_strides_bias_and_edges(M, K, N):
    """A with a row stride, y with an odd multiple of 4, a bias 2 bytes off, no bias; nothing past y's columns or
    rows is written."""
    big = _rand((M, K + 40), 11)
    a, w = big[:, :K], _rand((N, K), 12, 0.05)
    bias = _rand((N + 1,), 13)[1:]
    assert bias.data_ptr() % 4 == 2
    for b in (bias, None):
        y = torch.full((M + 2, N + 12), 3.0, dtype=torch.bfloat16, device=DEV)
        gemm_bf16(a, w, b, out=y[:M, :N])
        _check_bf16(y[:M, :N], a, w, b, False, None)
        assert bool((y[M:] == 3.0).all()) and bool((y[:, N:] == 3.0).all())


def _bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("K,N,act,bias", [(1536, 1536, None, True), (1544, 9220, "silu", True), (4096, 1540, "gelu", False),
                                          (72, 20, None, True), (8, 64, None, False), (520, 260, "gelu", True)])
def test_gemm_bf16_rows_have_the_same_bits_in_any_call(K, N, act, bias):
    """The first rows of calls of every size (few-row kernel at 8 and 16 rows and its 32-column workgroups, every
    tile) against the direct kernel, which rows 8 MB apart reach (32-bit offsets end at 2 GiB)."""
    a, w, b = _rand((2600, K), 21), _rand((N, K), 22, 0.05), _rand((N,), 23) if bias else None
    apart = torch.zeros((20, 1 << 22), dtype=torch.bfloat16, device=DEV)
    apart[:, :K] = a[:20]
    ref = gemm_bf16(apart[:, :K], w, b, act_out=act)
    _check_bf16(ref, a[:20], w, b, False, act)
    for M in (1, 3, 8, 9, 16, 17, 20, 64, 300, 512, 1100, 2600):
        got = gemm_bf16(a[:M], w, b, act_out=act)
        assert torch.equal(_bits(got[:20]), _bits(ref[:M])), M


@pytest.mark.parametrize("K,N", [(1536, 9216), (1544, 1540), (264, 8196), (72, 20), (5120, 256)])
def test_gemm_bf16_silu_rows_have_the_same_bits_in_any_call(K, N):
    """With SiLU on the input: the few-row kernel (8, 16 and 32 rows at a time) against the direct one at 65 rows."""
    a, w, b = _rand((65, K), 24), _rand((N, K), 25, 0.05), _rand((N,), 26)
    ref = gemm_bf16(a, w, b, silu_in=True)
    _check_bf16(ref, a, w, b, True, None)
    for M in (1, 7, 8, 9, 16, 17, 31, 32, 33, 64):
        assert torch.equal(_bits(gemm_bf16(a[:M], w, b, silu_in=True)), _bits(ref[:M])), M


def test_gemm_bf16_at_the_end_of_32_bit_offsets():
    """The largest row stride that each form takes and the next one, which goes to the direct kernel: same bits."""
    K, N = 264, 68
    a, w, b = _rand((17, K), 27), _rand((N, K), 28, 0.05), _rand((N,), 29)
    ref = gemm_bf16(a, w, b)
    span = (1 << 31) - 16
    for rows, most in ((17, 17 + 256), (3, 32)):
        last = (span - 1) // (2 * most) // 8 * 8   # rows of the form's own count stay below the span
        for lda in (last, last + 8):
            x = torch.empty((rows * lda,), dtype=torch.bfloat16, device=DEV).as_strided((rows, K), (lda, 1))
            x.copy_(a[:rows])
            assert torch.equal(_bits(gemm_bf16(x, w, b)), _bits(ref[:rows])), (rows, lda)


def test_flags_and_shapes_still_refused():
    a, w = _rand((4, 64), 1), _rand((8, 64), 2)
    y = torch.empty((4, 8), dtype=torch.bfloat16, device=DEV)
    st = _lib.stream_handle(torch.device(DEV))
    for args in ((4, 60, 64, 8, 8, 0), (4, 64, 64, 6, 8, 0), (4, 64, 64, 8, 8, 8), (4, 64, 64, 8, 8, 6), (4, 64, 60, 8, 8, 0)):
        m, k, lda, n, ldy, flags = args
        with pytest.raises(RuntimeError):
            _lib.call("wf_gemm_bf16", a.data_ptr(), m, k, lda, w.data_ptr(), n, None, y.data_ptr(), ldy, flags, st)


# 32 x 64 tiles, 64 x 64, 64 x 128, 128 x 128, and one shape past them, each off the tile's edges
W8A8_SHAPES = [(1, 4, 16), (31, 60, 112), (33, 68, 144), (77, 1536, 8960), (300, 1540, 1552), (512, 1536, 1536),
               (150, 5120, 5120), (513, 1500, 400), (780, 1536, 1536), (790, 1540, 272), (1560, 1536, 1536),
               (2047, 1924, 656), (4680, 1536, 1536)]


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("M,N,K", W8A8_SHAPES)
def test_gemm_i8_small_tiles_equal_the_large_ones(M, N, K, gelu):
    """The same bits as the 128 x 256 tiles, which a call that asks for the int32 accumulators runs (checked
    against the oracle on their own), with and without a bias and into strided rows."""
    g = torch.Generator().manual_seed(M + 3 * N + K)
    qx = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8).to(DEV)
    qw = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).to(DEV)
    sx = (torch.rand(M, generator=g) * 0.01 + 1e-3).to(DEV)
    sw = (torch.rand(N, generator=g) * 0.01 + 1e-3).to(DEV)
    for b in (_rand((N,), 5), None):
        acc = torch.empty((M, N), dtype=torch.int32, device=DEV)
        ref = gemm_i8(qx, qw, sx, sw, b, gelu=gelu, acc_out=acc)
        y = torch.full((M + 1, N + 4), 3.0, dtype=torch.bfloat16, device=DEV)
        gemm_i8(qx, qw, sx, sw, b, gelu=gelu, out=y[:M, :N])
        assert torch.equal(y[:M, :N].contiguous().view(torch.int16), ref.view(torch.int16))
        assert bool((y[M:] == 3.0).all()) and bool((y[:, N:] == 3.0).all())


# past one round of 128 x 128 tiles: the 128 x 256 and 256 x 256 ones, with M, N and K tails and one or two K steps
LARGE_SHAPES = [(3000, 3204, 272), (2050, 8196, 160), (4680, 8956, 1552), (4680, 8960, 16), (4680, 8960, 144)]


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("M,N,K", LARGE_SHAPES)
def test_gemm_i8_large_tiles_without_accumulators(M, N, K, gelu):
    """The large tiles as a linear calls them, without acc_out: the same bits as with it, with and without a bias,
    into rows that only allow 8-byte stores."""
    g = torch.Generator().manual_seed(M + 3 * N + K)
    qx = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8).to(DEV)
    qw = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).to(DEV)
    sx = (torch.rand(M, generator=g) * 0.01 + 1e-3).to(DEV)
    sw = (torch.rand(N, generator=g) * 0.01 + 1e-3).to(DEV)
    acc = torch.empty((M, N), dtype=torch.int32, device=DEV)
    for b in (_rand((N,), 5), None):
        ref = gemm_i8(qx, qw, sx, sw, b, gelu=gelu, acc_out=acc)
        assert torch.equal(_bits(gemm_i8(qx, qw, sx, sw, b, gelu=gelu)), _bits(ref))
        y = torch.full((M + 1, N + 4), 3.0, dtype=torch.bfloat16, device=DEV)
        y = y.view(-1)[4:4 + M * (N + 4)].view(M, N + 4)
        assert y.data_ptr() % 16 == 8
        gemm_i8(qx, qw, sx, sw, b, gelu=gelu, out=y[:, :N])
        assert torch.equal(_bits(y[:, :N]), _bits(ref))
        assert bool((y[:, N:] == 3.0).all())


@pytest.mark.parametrize("M", [20, 50, 150, 300, 4680])
def test_gemm_i8_zero_without_bias_keeps_its_sign(M):
    """A sum of 0 under a negative scale is -0, and stays -0 without a bias (a bias of -0 in the small tiles)."""
    qx = torch.zeros((M, 64), dtype=torch.int8, device=DEV)
    qw = torch.ones((8960, 64), dtype=torch.int8, device=DEV)
    sx, sw = torch.ones((M,), device=DEV), -torch.ones((8960,), device=DEV)
    got = gemm_i8(qx, qw, sx, sw, None)
    assert bool((_bits(got) == -32768).all())
    assert bool((_bits(gemm_i8(qx, qw, sx, sw, torch.zeros(8960, dtype=torch.bfloat16, device=DEV))) == 0).all())


@pytest.mark.parametrize("M,N,K", LARGE_SHAPES + [(4680, 8960, 4112)])
def test_gemm_e4m3_small_tiles_equal_the_large_ones(M, N, K):
    """The first and last rows of a call on the large tiles, against calls of these rows alone, which take the small
    ones (32 x 64, 64 x 64, 64 x 128, 128 x 128): one order of the fp32 sums."""
    x, w, b = _rand((M, K), K), _rand((N, K), N), _rand((N,), 9)
    a8, w8 = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
    sa, sw = torch.tensor([0.0123], device=DEV), torch.tensor([-0.0456], device=DEV)
    for bias in (b, None):
        ref = gemm_fp8_pertensor(a8, w8, sa, sw, bias)
        for rows in (1, 31, 50, 64, 150, 300):
            assert torch.equal(_bits(gemm_fp8_pertensor(a8[:rows], w8, sa, sw, bias)), _bits(ref[:rows])), rows
            tail = a8[M - rows:].clone()
            assert torch.equal(_bits(gemm_fp8_pertensor(tail, w8, sa, sw, bias)), _bits(ref[M - rows:])), rows


@pytest.mark.parametrize("M,N,K", W8A8_SHAPES + LARGE_SHAPES)
def test_gemm_e4m3_small_tiles(M, N, K):
    """Small and large tiles against the product of the codes in 64 bits.  Beside the bound above, the fp8 matrix
    instruction does not add its products in full fp32: with 16 products in it, outputs err by up to 2^-13.7 of
    sum |a w| (the largest of 42 million at K = 16, the same in every tile; less with more products); 2^-13 of it
    is allowed."""
    x, w, b = _rand((M, K), M + K), _rand((N, K), N + K), _rand((N,), 9)
    a8, w8 = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
    sa, sw = torch.tensor([0.0123], device=DEV), torch.tensor([0.0456], device=DEV)
    s = float(sa) * float(sw)
    a64, w64 = a8.float().double(), w8.float().double()
    sums = (2.0 ** -13 + (K + 8) * 2.0 ** -23) * s * (a64.abs() @ w64.abs().t())
    for bias in (b, None):
        got = gemm_fp8_pertensor(a8, w8, sa, sw, bias).double()
        pre = (a64 @ w64.t()) * s + (0 if bias is None else bias.double())
        assert bool(((got - pre).abs() <= (sums + (2.0 ** -8 + 2.0 ** -22) * pre.abs()) * 1.01 + 1e-30).all())
