"""Skinny products on either side of the size from which W is read non-temporally (64 MiB)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# N K = 2^25 elements is the line: the first of each pair of row counts lies on or just past it.  The
# products of both run on the matrix-core kernel (N >= 24 per CU, K a multiple of 128); 13,108 and 13,107
# columns leave a ragged last tile, K = 128 is a single stage.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,below,K", [(8, 13108, 13107, 2560), (1, 8192, 8191, 4096), (5, 262144, 262143, 128)])
def test_streamed_weights_give_the_same_bits(M, N, below, K, dtype):
    print(f"[skinny-stream] M={M} N={N} K={K} {dtype}", flush=True)
    from sparseattentioninfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(N + M)
    x = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    w = (0.05 * torch.randn(N, K, generator=g, device="cuda")).to(dtype)
    out = ops.gemm_skinny(x, w)
    assert torch.equal(out[:, :below], ops.gemm_skinny(x, w[:below]))
    # one rounding of the output (half an ulp) and fp32 sums in another order
    want = x.float() @ w.float().t()
    ulp = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(1e-30))) - (7 if dtype is torch.bfloat16 else 10))
    bound = 0.5 * ulp + 1e-5 * (x.float().abs() @ w.float().abs().t())
    assert not ((out.float() - want).abs() > bound).any()


@pytest.mark.parametrize("M,half,K", [(8, 6554, 2560), (3, 4096, 4096)])
def test_streamed_swiglu_gives_the_bits_of_the_smaller_product(M, half, K):
    print(f"[skinny-stream] swiglu M={M} I={half} K={K}", flush=True)
    from sparseattentioninfer_amd import ops
    g = torch.Generator(device="cuda").manual_seed(half + M)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (0.05 * torch.randn(2 * half, K, generator=g, device="cuda")).bfloat16()
    out = ops.gemm_skinny_swiglu(x, w)
    assert torch.equal(out[:, :half - 1], ops.gemm_skinny_swiglu(x, w[:2 * half - 2]))
