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
                        1.0 / math.sqrt(D), ws.data_ptr() if ws is not None else None,
                        4 * ws.numel() if ws is not None else 0,
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


@pytest.mark.parametrize("Hq,Hkv,rows,B", [(16, 8, 16, 1), (8, 8, 8, 2), (32, 8, 8, 1), (12, 4, 12, 2), (6, 6, 6, 4), (24, 8, 24, 3)])
@pytest.mark.parametrize("skew", [False, True])
def test_queues_per_xcd_process_every_item_once(Hq, Hkv, rows, B, skew):
    """Launches with claims and a KV-head count that the XCDs divide evenly (or not: one queue then), even
    and skewed row lengths (queues that run out early claim from the others): the bits of the launch
    without a workspace, and a workspace that is zero afterwards."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    per_item = 4 if Hq // rows == 4 else 1
    n = -(-(8 if per_item == 1 else 4) * 4 * cus * per_item // (Hq * B))     # query tiles: several items per workgroup
    D, bs, T = 64, 64, 64 * n - 9
    print(f"[prefill items] queues: heads {Hq}/{Hkv} rows {rows} B={B} T={T} skew={skew}", flush=True)
    sys.stdout.flush()
    g = torch.Generator(device=DEV).manual_seed(n)
    q = torch.randn(B, Hq, T, D, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(B, Hkv, T, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    qb = torch.arange(n)
    lists = []
    for r in range(rows):
        w = (1 + 12 * r // rows) if skew else 2                               # blocks of the window
        lists.append([list(range(max(0, int(i) - w + 1), int(i) + 1)) for i in qb])
    width = max(sum(map(len, row)) for row in lists)
    pairs = torch.zeros(rows, width, dtype=torch.int32)
    offsets = torch.zeros(rows, n + 1, dtype=torch.int32)
    for r, row in enumerate(lists):
        flat = [x for e in row for x in e]
        pairs[r, :len(flat)] = torch.tensor(flat, dtype=torch.int32)
        offsets[r, 1:] = torch.tensor([len(e) for e in row]).cumsum(0)
    case = (q, k, v, pairs.to(DEV), offsets.to(DEV), rows, bs)
    nbytes = int(_lib.load().sa_prefill_queue_workspace_bytes())
    ws = torch.zeros(nbytes // 4, dtype=torch.int32, device=DEV)
    want = _launch(*case, None)
    for _ in range(3):
        got = _launch(*case, ws)
        torch.cuda.synchronize()
        assert not ws.any()
        assert torch.equal(got, want)
    assert torch.isfinite(want.float()).all()
