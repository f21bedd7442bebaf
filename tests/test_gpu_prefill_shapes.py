"""Every workgroup shape of the prefill kernel (heads per workgroup, slices of its waves) against the
oracle.  The shape follows from the number of waves a launch has, so the batch sets it: fewer than two
waves per CU (four slices), three (two slices), six (one slice); blocks of 16 (sub-block masks) and 64,
head dims 64 and 128, ragged lengths and chunked queries, and scores that outgrow the first tile's."""
import sys

import pytest
import torch

from oracle import attention as oa
from sparseattentioninfer_amd import ops
from sparseattentioninfer_amd.patterns import bernoulli_block_mask, block_mask_to_csr
from tests.helpers import assert_close_bf16, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("per_cu", [1, 3, 6])
@pytest.mark.parametrize("heads,kv,rows", [(3, 3, 3), (4, 2, 2), (4, 1, 4), (4, 1, 1)])
@pytest.mark.parametrize("D,bs,T_q,T_k,dtype", [(128, 64, 200, 200, torch.bfloat16), (64, 16, 150, 1100, torch.float16),
                                                (128, 16, 90, 1000, torch.bfloat16), (64, 64, 129, 129, torch.bfloat16)])
def test_shapes_match_the_oracle(per_cu, heads, kv, rows, D, bs, T_q, T_k, dtype):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    tiles = -(-T_q // 64)
    B = max(1, per_cu * cus // (2 * tiles * heads))
    print(f"[prefill shapes] {per_cu} waves per CU: B={B} heads={heads}/{kv} rows={rows} D={D} bs={bs} T={T_q}/{T_k}", flush=True)
    sys.stdout.flush()
    nqb, nkb = -(-T_q // bs), -(-T_k // bs)
    bm = bernoulli_block_mask(rows, nqb, nkb, density=0.4, seed=per_cu, q_block_offset=(T_k - T_q) // bs)
    pairs, offsets = block_mask_to_csr(bm)
    g = torch.Generator(device=DEV).manual_seed(7)
    q = torch.randn(B, heads, T_q, D, generator=g, device=DEV).to(dtype)
    k, v = (torch.randn(B, kv, T_k, D, generator=g, device=DEV).to(dtype) for _ in range(2))
    # later keys outgrow the first tile's scores: the row references are raised on the way
    k[:, :, T_k // 2:] *= torch.linspace(1, 6, B, device=DEV).to(dtype)[:, None, None, None]
    out = ops.universal_sparse_attn(q, k, v, pairs.to(DEV), offsets.to(DEV), bs)
    want = oa.block_sparse_attention(q, k, v, pairs, offsets, bs)
    assert torch.isfinite(out.float()).all()
    # Rounding every probability to the element type moves a row by at most u max|v| (u: half an ulp at 1),
    # rounding the output by at most 2 u |out|; 2e-3 for the fp32 sums and exponentials.  (Rows that one key
    # dominates have outputs of 4, beyond what the fixed 2e-2 of order-1 outputs is meant for.)
    u = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    err = (out.float() - want.to(out.device)).abs()
    bound = u * v.float().abs().amax() + 2 * u * want.to(out.device).abs() + 2e-3
    assert (err <= bound).all(), f"max-abs {err.max():.3e}, {(err / bound).max():.2f} of the bound"
    assert err.mean() <= 2e-3


@pytest.mark.parametrize("heads,kv,rows", [(4, 2, 2), (4, 4, 4), (4, 1, 1)])
@pytest.mark.parametrize("D,bs,T_q,T_k", [(128, 64, 40, 40), (64, 16, 2, 33), (128, 64, 300, 300), (64, 64, 70, 2118),
                                          (128, 128, 200, 200)])
def test_lists_of_one_tile_match_the_oracle(heads, kv, rows, D, bs, T_q, T_k):
    """Few items, diagonal blocks only (one tile per item, or two with blocks of 128)."""
    print(f"[prefill shapes] one tile: heads={heads}/{kv} rows={rows} D={D} bs={bs} T={T_q}/{T_k}", flush=True)
    sys.stdout.flush()
    nqb, nkb = -(-T_q // bs), -(-T_k // bs)
    bm = (torch.arange(nkb)[None] == torch.arange(nqb)[:, None] + (T_k - T_q) // bs).expand(rows, -1, -1)
    pairs, offsets = block_mask_to_csr(bm)
    q = seeded((2, heads, T_q, D), 1, torch.bfloat16)
    k, v = (seeded((2, kv, T_k, D), s, torch.bfloat16) for s in (2, 3))
    out = ops.universal_sparse_attn(q.to(DEV), k.to(DEV), v.to(DEV), pairs.to(DEV), offsets.to(DEV), bs)
    assert_close_bf16(out, oa.block_sparse_attention(q, k, v, pairs, offsets, bs), "one tile")
