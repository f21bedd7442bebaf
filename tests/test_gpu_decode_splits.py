"""Contiguous decode (``universal_sparse_attn`` with one query) around the list lengths from which a
block list is split over workgroups: just below and at 512 KB of K and V, lists of a few blocks more than the
splits, the 32-split cap, ragged last blocks; and the paged entry point's own choice (``num_splits=0``)."""
import sys

import pytest
import torch

from oracle import attention as oa
from sparseattentioninfer_amd import ops
from sparseattentioninfer_amd.patterns import block_mask_to_csr
from tests.helpers import assert_close_bf16, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,Hq,Hkv,rows,D,bs,T", [
    (1, 8, 2, 2, 128, 64, 959), (1, 8, 2, 2, 128, 64, 961), (1, 8, 2, 8, 128, 64, 1025), (2, 6, 3, 3, 64, 16, 1024),
    (1, 4, 1, 1, 128, 64, 4480), (1, 4, 1, 1, 64, 128, 9000), (3, 16, 2, 2, 128, 32, 2051), (40, 8, 8, 8, 64, 64, 1500), (1, 4, 1, 1, 64, 64, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_split_decode_matches_the_oracle(B, Hq, Hkv, rows, D, bs, T, dtype):
    print(f"[decode splits] B={B} heads={Hq}/{Hkv} rows={rows} D={D} bs={bs} T={T} {dtype}", flush=True)
    sys.stdout.flush()
    nkb = -(-T // bs)
    bm = torch.ones(rows, 1, nkb, dtype=torch.bool)
    bm[0, 0, 1::3] = False                                 # rows of different lengths
    pairs, offsets = block_mask_to_csr(bm)
    q = seeded((B, Hq, 1, D), 1, dtype).to(DEV)
    k, v = (seeded((B, Hkv, T + 70, D), s, dtype).to(DEV)[:, :, :T] for s in (2, 3))   # a cache's views
    out = ops.universal_sparse_attn(q, k, v, pairs.to(DEV), offsets.to(DEV), bs)
    want = oa.block_sparse_attention(q, k, v, pairs, offsets, bs)
    assert_close_bf16(out, want, "contiguous")
    if T % bs == 0 or bs > 64 or B > 3:
        return
    # the same lists over pages, split count chosen from the shapes
    pad = torch.zeros(B, Hkv, nkb * bs - T, D, dtype=dtype, device=DEV)
    kp, vp = (torch.cat([x, pad], 2).reshape(B, Hkv, nkb, bs, D).transpose(1, 2).reshape(B * nkb, Hkv, bs, D).contiguous()
              for x in (k, v))
    table = torch.arange(B * nkb, dtype=torch.int32, device=DEV).reshape(B, nkb)
    got = ops.paged_sparse_decode(q, kp, vp, table, torch.full((B,), T, dtype=torch.int32, device=DEV),
                                  pairs.to(DEV)[None].expand(B, -1, -1), offsets.to(DEV)[None].expand(B, -1, -1),
                                  num_splits=0)
    assert_close_bf16(got, want, "paged")


@pytest.mark.parametrize("B,Hq,Hkv,n", [(1, 32, 8, 100), (1, 8, 2, 64), (8, 32, 8, 27)])
def test_chosen_split_count_fits_a_workspace_of_either_rule(B, Hq, Hkv, n):
    """``num_splits=0`` with a caller's workspace, sized by either public count."""
    D, page = 128, 16
    print(f"[decode splits] workspace: B={B} heads={Hq}/{Hkv} {n} blocks", flush=True)
    sys.stdout.flush()
    q = seeded((B, Hq, D), 1, torch.bfloat16).to(DEV)
    kp, vp = (seeded((B * n, Hkv, page, D), s, torch.bfloat16).to(DEV) for s in (2, 3))
    table = torch.arange(B * n, dtype=torch.int32, device=DEV).reshape(B, n)
    lens = torch.full((B,), n * page, dtype=torch.int32, device=DEV)
    sel = torch.arange(n, dtype=torch.int32, device=DEV).expand(B, Hkv, n).contiguous()
    off = torch.tensor([0, n], dtype=torch.int32, device=DEV).expand(B, Hkv, 2).contiguous()
    args = (q, kp, vp, table, lens, sel, off)
    for splits in (ops.auto_decode_splits(B, Hkv, n), ops.decode_splits(B, Hq, Hkv, n)):
        ws = torch.empty(ops.decode_workspace_bytes(B, Hq, D, splits), dtype=torch.uint8, device=DEV)
        got = ops.paged_sparse_decode(*args, num_splits=0, workspace=ws)
        assert_close_bf16(got, ops.paged_sparse_decode(*args), "workspace")
    with pytest.raises(AssertionError, match="workspace too small"):
        ops.paged_sparse_decode(*args, num_splits=0, workspace=ws[:1024])
