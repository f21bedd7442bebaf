"""Time of persistent prefill launches whose work items differ much in length: CSR rows of different
densities, dense causal prompts.  The same schedule launched as one workgroup per item, which the hardware
hands out as workgroups end, is the yardstick: dealing the first items by index or keeping a KV head's items
on one XCD must not leave most of the chip idle (three neighbouring items per workgroup took 2.1 times the
yardstick, a queue per XCD with one dense KV head among eight 2.2 times)."""
import math
import sys

import pytest
import torch

from sparseattentioninfer_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
PROFILES = {"dense": [0] * 8, "one dense": [0] + [5] * 7, "last dense": [5] * 7 + [0], "half dense": [0] * 4 + [5] * 4}
SLACK = 1.3


def _time(launch):
    for _ in range(3):
        launch()
    best = math.inf
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(4):
            launch()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / 4 * 1e3)
    return best


def _ratio(Hq, rows, B, T, profile, ws_bytes):
    """Time with a workspace of ``ws_bytes`` over the time without one; both outputs have the same bits."""
    Hkv, D, bs = 8, 128, 64
    n = -(-T // bs)
    qb, kb = torch.arange(n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    groups = [(kb <= qb) & ((kb > qb - w) | (w == 0)) for w in PROFILES[profile]]
    pairs, offsets = ops.block_mask_to_csr_gpu(torch.stack(groups).repeat_interleave(rows // Hkv, 0))
    g = torch.Generator(device=DEV).manual_seed(T)
    q = torch.randn(B, Hq, T, D, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(B, Hkv, T, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    ws = torch.zeros(ws_bytes // 4, dtype=torch.int32, device=DEV)
    lib = _lib.load()

    def launch(o, words):
        st = lib.sa_prefill_split(0, q.data_ptr(), *q.stride()[:3], k.data_ptr(), *k.stride()[:3], v.data_ptr(),
                                  *v.stride()[:3], o.data_ptr(), *o.stride()[:3], pairs.data_ptr(), pairs.stride(0),
                                  offsets.data_ptr(), offsets.stride(0), None, 0, rows, n, B, Hq, Hkv, T, T, D, bs, 0,
                                  1.0 / math.sqrt(D), words.data_ptr() if words is not None else None,
                                  4 * words.numel() if words is not None else 0, None, 0,
                                  torch.cuda.current_stream().cuda_stream)
        assert st == 0, lib.sa_last_error()

    plain, dealt = torch.empty_like(q), torch.empty_like(q)
    us = _time(lambda: launch(dealt, ws)), _time(lambda: launch(plain, None))
    print(f"[prefill balance] heads {Hq}/{Hkv} rows {rows} B={B} T={T} {profile} {ws_bytes} B: {us[0]:.1f} us, "
          f"one workgroup per item {us[1]:.1f} us", flush=True)
    sys.stdout.flush()
    assert not ws.any()
    assert torch.equal(plain, dealt)
    return us[0] / us[1]


@pytest.mark.parametrize("B,T", [(1, 8192), (2, 4096), (1, 6016)])
@pytest.mark.parametrize("profile", list(PROFILES))
def test_one_queue_four_heads(B, T, profile):
    """Four items per workgroup, the first three dealt by index, and three."""
    assert _ratio(32, 8, B, T, profile, int(_lib.load().sa_prefill_workspace_bytes())) <= SLACK


@pytest.mark.parametrize("Hq,rows,B,T", [(32, 8, 1, 8192), (32, 8, 2, 4096), (32, 32, 1, 8192), (32, 32, 4, 4096),
                                         (16, 8, 2, 8192), (16, 8, 1, 12000)])
@pytest.mark.parametrize("profile", list(PROFILES))
def test_queue_workspace(Hq, rows, B, T, profile):
    """With room for a queue per XCD: four, one and two heads to an item, even and uneven rows."""
    assert _ratio(Hq, rows, B, T, profile, int(_lib.load().sa_prefill_queue_workspace_bytes())) <= SLACK
