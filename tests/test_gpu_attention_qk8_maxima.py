"""The quantized-QK attention's running maxima, which are taken from the exponents against the maximum so far.

Keys grow from the third 64-key tile on, so that later scores exceed the first tile's maximum by a few, by tens and
by more than 128 (weights that would overflow fp32) in log2 units, in a whole tile, a ragged last tile and for half
of the queries only.  4680 queries run 256-query workgroups (no staging waves), the slices the finer split with
them; both give the same bits.
"""

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
