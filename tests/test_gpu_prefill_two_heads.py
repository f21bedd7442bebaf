"""Two query heads per schedule row: the two-head workgroups' pairs of K/V buffers, over lists of no, one,
two, three and up to nine tiles per item (which pair an item ends in, and where its output is staged),
several items per workgroup, against the oracle."""
import sys

import pytest
import torch

from oracle import attention as oa
from sparseattentioninfer_amd import ops
from sparseattentioninfer_amd.patterns import block_mask_to_csr
from tests.helpers import assert_close_bf16, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bs", [16, 64])
@pytest.mark.parametrize("windows", [[1] * 8, [2] * 8, [0, 1, 2, 3, 5, 9, 0, 9]])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_two_head_items_match_the_oracle(D, bs, windows, dtype):
    B, Hq, Hkv, T = 8, 16, 8, 571
    n = -(-T // bs)
    print(f"[two heads] D={D} bs={bs} windows={windows} {dtype}", flush=True)
    sys.stdout.flush()
    qb, kb = torch.arange(n)[:, None] * bs // 64, torch.arange(n)[None] * bs // 64
    bm = torch.stack([(kb <= qb) & (kb > qb - w) for w in windows])     # windows of 64-key tiles
    bm[:, ::3] &= (kb > 0)                                              # and some lists one tile shorter
    pairs, offsets = block_mask_to_csr(bm)
    q = seeded((B, Hq, T, D), 1, dtype)
    k, v = (seeded((B, Hkv, T, D), s, dtype) for s in (2, 3))
    out = ops.universal_sparse_attn(q.to(DEV), k.to(DEV), v.to(DEV), pairs.to(DEV), offsets.to(DEV), bs)
    assert_close_bf16(out, oa.block_sparse_attention(q, k, v, pairs, offsets, bs), "two heads")
    if 0 in windows:
        assert (out[:, :2] == 0).all()                                  # no visible key: 0
