"""The quantized-QK attention's running maxima, which move only for a raise of more than 8 log2 units.

Keys grow from the third 64-key tile on, so that later scores exceed the first tile's maximum by a few, by tens and
by more than 128 (weights that would overflow fp32) in log2 units, in a whole tile, a ragged last tile and for half
of the queries only.  4680 queries run 256-query workgroups (no staging waves), the slices the finer split with
them; both give the same bits.
"""

import math

import pytest
import torch

from oracle import attention as oat
from oracle import kv as okv
from waveforcing_amd import inputs
from waveforcing_amd.backend import attn_paged_fp8
from waveforcing_amd.kv import Fp8PagePool, PagedKV

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LQ, H, D, PAGE = 4680, 12, 128, 100


@pytest.mark.parametrize("grow", [4.0, 32.0, 128.0])
@pytest.mark.parametrize("n_kv", [130, 200, 256])
def test_maxima_move_with_growing_keys(grow, n_kv):
    g = torch.Generator().manual_seed(int(grow) + n_kv)
    q = torch.randn((LQ, H, D), generator=g)
    q[::2] /= 64.0  # these queries' maxima hardly move
    q = q.to(torch.bfloat16)
    k = torch.randn((n_kv, H, D), generator=g)
    k[128:] *= grow
    k, v = k.to(torch.bfloat16), torch.randn((n_kv, H, D), generator=g).to(torch.bfloat16)
    n_pages = -(-n_kv // PAGE)
    ids = inputs.page_table(n_pages, n_pages + 2, seed=3)
    pool = Fp8PagePool(n_pages + 2, H, D, PAGE, DEV)
    table = pool.page_table(ids)
    pool.pack(k.to(DEV), v.to(DEV), table)
    ctx = PagedKV(pool, table, n_kv)
    out = attn_paged_fp8(q.to(DEV), ctx, quantized_qk=True)
    for a, b in ((0, 33), (1000, 1300)):
        assert torch.equal(attn_paged_fp8(q[a:b].to(DEV), ctx, quantized_qk=True), out[a:b])
    kp, vp = okv.new_pool(n_pages + 2, PAGE, H, D), okv.new_pool(n_pages + 2, PAGE, H, D)
    okv.pack(k, ids, PAGE, *kp)
    okv.pack(v, ids, PAGE, *vp)
    rows = torch.cat([torch.arange(40), torch.arange(LQ - 40, LQ)])
    ref = oat.paged_fp8_qk8(q[rows], kp, vp, ids, n_kv, PAGE)
    err = ((out[rows.to(DEV)].cpu().float() - ref).abs() / ref.abs().clamp(min=1.0)).max().item()
    print(f"grow {grow} n_kv {n_kv}: max rel err {err:.3e}")
    # bf16 weights and results (5e-3), and the fp32 scores' own error: summing 128 products of N(0, 1) queries and
    # grow x N(0, 1) keys errs by up to 128 * 2^-24 * sum |q k| * scale * log2 e = 1e-2 at grow = 128 in the exponent,
    # so 0.7 % of a weight, against values that differ by about 2
    assert err <= 2e-2


def test_maxima_stay_for_small_raises():
    """A key that raises a query's maximum by less than 8 log2 units leaves the reference of the exponents where it
    was: its weight is bf16(2^x), not 1.

    K is one value per key at d = 0 beside a constant 448 at d = 1 (so every row's scale is 1 and its codes are the
    values); a query one e4m3 value at d = 0.  Keys 0..63 score 0, key 64 raises the
    exponent by x = q c u, u = fp32(scale log2 e), the other keys of the second tile score 0 with V = 0.  V is -r for
    keys 0..63 and v for key 64 with 64 r within a few percent of 2^x v, so that the weight's own rounding (2^-9 of
    it) is many bf16 steps of the difference.  The bound: one bf16 rounding of the result, and 2^-20 of the two
    terms for the fp32 sums and the hardware exponential.
    """
    n_kv = 128
    u = float(torch.tensor(1 / math.sqrt(D)) * torch.tensor(math.log2(math.e)))
    cs = torch.tensor([3.5, 5.0, 7.0, 11.0, 13.0, 15.0, 22.0, 26.0, 28.0, 36.0, 44.0, 52.0, 60.0, 9.0, 18.0, 30.0])
    q = torch.zeros((len(cs), H, D))
    q[:, :, 0] = (cs / 32)[:, None]               # a query's score against key 64 (32 there) is cs
    k = torch.zeros((n_kv, H, D))
    k[:, :, 1] = 448.0
    k[64, :, 0] = 32.0
    x = cs.double() * u
    w = torch.exp2(x)
    wb = w.to(torch.float32).to(torch.bfloat16).double()
    ulp = torch.exp2(torch.floor(torch.log2(w)) - 7)
    tie = ((w / ulp) % 1.0 - 0.5).abs() < 1e-3     # a weight that either rounding may take
    sharp = ~tie & ((wb - w).abs() / w > 2.0 ** -11)
    assert int(sharp.sum()) >= 8
    # r: every e4m3 mantissa from 2^-6 on, among them some next to 2^x v / 64
    r = torch.tensor([(1 + (d % 8) / 8) * 2.0 ** ((d // 8) - 6) for d in range(D)]).clamp(max=448.0)
    v = torch.zeros((n_kv, H, D))
    v[:64] = -r
    v[:64, :, D - 1] = -448.0                     # row scale 1
    v[64] = 448.0
    pool = Fp8PagePool(4, H, D, PAGE, DEV)
    table = pool.page_table([2, 0])
    pool.pack(k.to(torch.bfloat16).to(DEV), v.to(torch.bfloat16).to(DEV), table)
    out = attn_paged_fp8(q.to(torch.bfloat16).to(DEV), PagedKV(pool, table, n_kv), quantized_qk=True).cpu().double()
    vv = (v[0, 0].double(), v[64, 0].double())
    seen = 0
    for i in torch.nonzero(sharp).flatten().tolist():
        ref = (64 * vv[0] + wb[i] * vv[1]) / (127 + wb[i])
        other = (64 * vv[0] + w[i] * vv[1]) / (127 + w[i])       # the reference moved to key 64
        bound = 2.0 ** -8 * ref.abs() + 2.0 ** -20 * (64 * vv[0].abs() + w[i] * vv[1].abs()) / 127
        assert bool(((out[i] - ref).abs() <= bound).all()), float(((out[i] - ref).abs() / bound).max())
        seen += int(((other - ref).abs() > 2 * bound).sum())
    assert seen > 0                               # dims in which a moved reference would show
