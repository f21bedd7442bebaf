"""How a persistent prefill launch deals its work items: counts around one, two and three items per
resident workgroup, where the items fixed by the workgroup's index end and the counter's claims begin.
Every item must be processed once (the status word stays clear, the counters end at zero) and the
output must have the bits of the one-workgroup-per-item launch."""
import math
import sys

import pytest
import torch

from sparseattentioninfer_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(n, rows):
    """``n`` query tiles of four heads sharing one KV head (block 0 and the diagonal block of each)."""
    Hq, D, T = 4, 64, 64 * n - 5
    R = 1 if rows == "group" else Hq
    g = torch.Generator(device=DEV).manual_seed(n)
    q = torch.randn(1, Hq, T, D, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(1, 1, T, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    qb = torch.arange(n)
    counts = torch.where(qb > 0, 2, 1)
    flat = torch.stack([torch.zeros_like(qb), qb], 1).reshape(-1)[1:].to(torch.int32)
    offsets = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)]).to(torch.int32)
    return q, k, v, flat.expand(R, -1).contiguous().to(DEV), offsets.expand(R, -1).contiguous().to(DEV), R, 64


def _launch(q, k, v, pairs, offsets, R, bs, ws):
    lib = _lib.load()
    o = torch.full_like(q, float("nan"))
    B, Hq, T, D = q.shape
    st = lib.sa_prefill(0, q.data_ptr(), *q.stride()[:3], k.data_ptr(), *k.stride()[:3], v.data_ptr(), *v.stride()[:3],
                        o.data_ptr(), *o.stride()[:3], pairs.data_ptr(), pairs.stride(0), offsets.data_ptr(),
                        offsets.stride(0), None, 0, R, offsets.size(1) - 1, B, Hq, k.shape[1], T, T, D, bs, 0,
                        1.0 / math.sqrt(D), ws.data_ptr() if ws is not None else None, 32 if ws is not None else 0,
                        torch.cuda.current_stream().cuda_stream)
    assert st == 0, lib.sa_last_error()
    return o


@pytest.mark.parametrize("rows", ["group", "head"])
@pytest.mark.parametrize("rounds,extra", [(0, 1), (1, -1), (1, 0), (1, 1), (2, -1), (2, 3), (3, -1), (3, 0), (3, 1), (5, 7)])
def test_item_counts_around_the_workgroup_count(rows, rounds, extra):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = max(1, rounds * cus + extra)              # query tiles = items of the four-head kernel
    print(f"[prefill items] {rows} rows, {n} tiles on {cus} CUs", flush=True)
    sys.stdout.flush()
    case = _case(n, rows)
    ws = torch.zeros(8, dtype=torch.int32, device=DEV)
    want = _launch(*case, None)
    for _ in range(2):
        got = _launch(*case, ws)
        torch.cuda.synchronize()
        assert ws.tolist() == [0] * 8
        assert torch.equal(got, want)
    assert torch.isfinite(want.float()).all()


@pytest.mark.parametrize("rows", ["group", "head"])
@pytest.mark.parametrize("rounds", [1, 5])
@pytest.mark.parametrize("word,value", [(0, 3), (0, 1 << 20), (1, 2)])
def test_claims_word_that_was_not_zero_is_reported(rows, rounds, word, value):
    """Dealt launches (one round) and claimed ones (five): the status bit is set, and a workspace
    zeroed afterwards serves the next launch."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    case = _case(rounds * cus, rows)
    print(f"[prefill items] {rows} rows, {rounds} rounds, word {word} = {value}", flush=True)
    want = _launch(*case, None)
    ws = torch.zeros(8, dtype=torch.int32, device=DEV)
    ws[word] = value
    _launch(*case, ws)
    torch.cuda.synchronize()
    assert int(ws[3]) == 1
    ws.zero_()
    got = _launch(*case, ws)
    torch.cuda.synchronize()
    assert ws.tolist() == [0] * 8
    assert torch.equal(got, want)


def test_workspace_aligned_to_four_bytes_only():
    case = _case(5 * torch.cuda.get_device_properties(0).multi_processor_count + 3, "group")
    buf = torch.zeros(16, dtype=torch.int32, device=DEV)
    want = _launch(*case, None)
    for _ in range(2):
        got = _launch(*case, buf[1:9])
        torch.cuda.synchronize()
        assert buf.tolist() == [0] * 16
        assert torch.equal(got, want)
