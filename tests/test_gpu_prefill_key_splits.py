"""Four-head prefill launches whose few query tiles divide their keys over workgroups, against the
oracle: two to many splits, chunk lengths around a query tile, key counts that cut the last tile,
schedules with empty query blocks and with splits that hold no block, blocks of 16, 64 and 128, both
head dims, scores that outgrow an earlier split's."""
import sys

import pytest
import torch

from oracle import attention as oa
from sparseattentioninfer_amd import _lib, ops
from sparseattentioninfer_amd.patterns import block_mask_to_csr

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,Hq,Hkv,D,bs,T_q,T_k,dtype,hole", [
    (1, 8, 2, 128, 64, 2, 4096, torch.bfloat16, 0), (1, 8, 2, 128, 64, 64, 2048, torch.bfloat16, 0),
    (2, 16, 2, 128, 64, 65, 3001, torch.float16, 0), (1, 32, 8, 128, 64, 1000, 5000, torch.bfloat16, 0),
    (1, 4, 1, 64, 128, 500, 4500, torch.bfloat16, 0), (2, 8, 2, 64, 16, 130, 3200, torch.float16, 0),
    (1, 8, 2, 128, 64, 300, 6000, torch.bfloat16, 40), (1, 4, 1, 128, 64, 4096, 4096, torch.bfloat16, 0)])
def test_key_splits_match_the_oracle(B, Hq, Hkv, D, bs, T_q, T_k, dtype, hole):
    nqb, nkb = -(-T_q // bs), -(-T_k // bs)
    off = T_k - T_q
    last = torch.tensor([(off + min(T_q, (i + 1) * bs) - 1) // bs for i in range(nqb)])
    bm = (torch.arange(nkb)[None, :] <= last[:, None])[None].expand(Hkv, -1, -1).clone()
    if hole:
        bm[0, :, 3:3 + hole] = False          # whole splits of row 0 hold nothing
        bm[1, 1] = False                      # an empty query block
    pairs, offsets = block_mask_to_csr(bm)
    n = int(_lib.load().sa_prefill_partial_bytes(Hkv, B, Hq, T_q, T_k, D, bs, max(1, pairs.size(1))))
    print(f"[key splits] B={B} heads={Hq}/{Hkv} D={D} bs={bs} T={T_q}/{T_k}: {n} bytes of partials", flush=True)
    sys.stdout.flush()
    assert n > 0
    g = torch.Generator(device=DEV).manual_seed(T_q)
    q = torch.randn(B, Hq, T_q, D, generator=g, device=DEV).to(dtype)
    k, v = (torch.randn(B, Hkv, T_k, D, generator=g, device=DEV).to(dtype) for _ in range(2))
    k[:, :, T_k // 3:T_k // 2] *= 3           # splits whose row references differ
    out = ops.universal_sparse_attn(q, k, v, pairs.to(DEV), offsets.to(DEV), bs)
    want = oa.block_sparse_attention(q, k, v, pairs, offsets, bs).to(DEV)
    assert torch.isfinite(out.float()).all()
    # rounding of the probabilities (u max|v|) and of the output (2 u |out|), 2e-3 for the fp32 part
    u = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    err = (out.float() - want).abs()
    assert (err <= u * v.float().abs().amax() + 2 * u * want.abs() + 2e-3).all(), f"max-abs {err.max():.3e}"
    assert err.mean() <= 2e-3
    if hole:
        assert (out[:, Hq // Hkv:2 * Hq // Hkv, bs:2 * bs] == 0).all()     # no visible key: 0


def test_key_splits_in_a_graph_give_the_eager_bits():
    B, Hq, Hkv, T_q, T_k, D, bs = 1, 8, 2, 200, 4000, 128, 64
    nqb, nkb = -(-T_q // bs), -(-T_k // bs)
    pairs, offsets = (x.to(DEV) for x in block_mask_to_csr(torch.ones(Hkv, nqb, nkb, dtype=torch.bool)))
    g = torch.Generator(device=DEV).manual_seed(5)
    q = torch.randn(B, Hq, T_q, D, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(B, Hkv, T_k, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        want = ops.universal_sparse_attn(q, k, v, pairs, offsets, bs)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = ops.universal_sparse_attn(q, k, v, pairs, offsets, bs)
    for rep in range(3):
        out.zero_()
        other = ops.universal_sparse_attn(q * 2, k, v, pairs, offsets, bs)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep
        assert not torch.equal(other, want)
