"""The splits of the attention over workgroups (256, 128, 96, 64 or 32 queries each, chosen by the grid they make)
give every query the same bits.

A call of 4680 queries and 12 heads runs 256-query workgroups; calls of its first rows run the finer splits (2400
rows 128, 1560 rows 96, 1000 rows 64, 300 rows and fewer 32 on a 256-CU device), whose staging waves and
barriers are the code under test: odd and even tile counts, one tile, a ragged last tile and pages that
start inside a tile.
"""

import pytest
import torch

from waveforcing_amd import inputs
from waveforcing_amd.backend import attn_dense_bf16, attn_paged_fp8
from waveforcing_amd.kv import Fp8PagePool, PagedKV

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
H, D, LQ, PAGE = 12, 128, 4680, 200
FORMS = {"exact": {}, "quantized_qk": {"quantized_qk": True}, "fp8_pv": {"fp8_pv": True}, "dense": None}


def _normal(shape, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV).to(torch.bfloat16)


@pytest.mark.parametrize("n_kv", [1, 64, 65, 130, 1000])
@pytest.mark.parametrize("form", list(FORMS))
def test_every_split_gives_the_same_rows(form, n_kv):
    q, k, v = _normal((LQ, H, D), 70), _normal((n_kv, H, D), 71 + n_kv), _normal((n_kv, H, D), 72 + n_kv)
    k[n_kv // 2:] *= 4  # raises the running maxima on the way
    if form == "dense":
        attend = lambda x: attn_dense_bf16(x, k, v)
    else:
        n_pages = -(-n_kv // PAGE)
        pool = Fp8PagePool(n_pages + 3, H, D, PAGE, DEV)
        table = pool.page_table(inputs.page_table(n_pages, n_pages + 3, seed=73))
        pool.pack(k, v, table)
        ctx = PagedKV(pool, table, n_kv)
        attend = lambda x: attn_paged_fp8(x, ctx, **FORMS[form])
    full = attend(q)
    assert torch.isfinite(full).all()
    for rows in (1, 31, 33, 300, 1000, 1560, 2400):
        assert torch.equal(attend(q[:rows]), full[:rows]), rows
