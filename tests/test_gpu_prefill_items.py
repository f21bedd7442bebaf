"""How a persistent prefill launch deals its work items: counts around one, two and three items per
resident workgroup, where the items fixed by the workgroup's index end and the counter's claims begin.
Every item must be processed once (the status word stays clear, the counters end at zero) and the
output must have the bits of the one-workgroup-per-item launch."""
import math
import sys

import pytest
import torch

from sparseattentioninfer_amd import _lib, ops

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


def _windows(B, Hq, Hkv, T, D, windows):
    """Row r keeps the last ``windows[r]`` blocks of 64 keys."""
    n = -(-T // 64)
    g = torch.Generator(device=DEV).manual_seed(n)
    q = torch.randn(B, Hq, T, D, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(B, Hkv, T, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    qb, kb = torch.arange(n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    pairs, offsets = ops.block_mask_to_csr_gpu(torch.stack([(kb <= qb) & (kb > qb - w) for w in windows]))
    return q, k, v, pairs, offsets


def _launch(q, k, v, pairs, offsets, R, bs, ws, split=False):
    """``sa_prefill``, or with ``split`` ``sa_prefill_split`` (queues, in a workspace with room for them)."""
    lib = _lib.load()
    o = torch.full_like(q, float("nan"))
    B, Hq, T, D = q.shape
    fn, partials = (lib.sa_prefill_split, (None, 0)) if split else (lib.sa_prefill, ())
    st = fn(0, q.data_ptr(), *q.stride()[:3], k.data_ptr(), *k.stride()[:3], v.data_ptr(), *v.stride()[:3],
            o.data_ptr(), *o.stride()[:3], pairs.data_ptr(), pairs.stride(0), offsets.data_ptr(),
            offsets.stride(0), None, 0, R, offsets.size(1) - 1, B, Hq, k.shape[1], T, T, D, bs, 0,
            1.0 / math.sqrt(D), ws.data_ptr() if ws is not None else None,
            4 * ws.numel() if ws is not None else 0, *partials, torch.cuda.current_stream().cuda_stream)
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


def test_only_the_workspace_bytes_of_a_larger_buffer_are_used():
    """``sa_prefill`` asks for its 32 bytes to be zero, whatever the size of the buffer they are in."""
    T, Hkv, B = 4091, 8, 12
    print("[prefill items] larger buffer", flush=True)
    q, k, v, pairs, offsets = _windows(B, 8, Hkv, T, 64, [2] * 8)
    buf = torch.full((1024,), 0x5a5a5a5a, dtype=torch.int32, device=DEV)
    buf[:8] = 0
    want = _launch(q, k, v, pairs, offsets, Hkv, 64, None)
    for _ in range(2):
        got = _launch(q, k, v, pairs, offsets, Hkv, 64, buf)
        torch.cuda.synchronize()
        assert not buf[:8].any() and (buf[8:] == 0x5a5a5a5a).all()
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


FINISH, ALL, QUEUE = 2, 4, 16      # 64-bit words of a queue workspace: a queue's finish word, the queues', per queue


@pytest.mark.parametrize("Hq,Hkv,rows,B,D,T", [
    (16, 8, 16, 1, 64, 32759), (8, 8, 8, 2, 64, 32759), (24, 8, 24, 3, 64, 7295),       # one head to an item
    (16, 8, 8, 8, 64, 4091), (16, 8, 8, 6, 128, 4091),                                  # two, units of four and two heads
    (32, 8, 8, 4, 64, 4091), (32, 8, 8, 4, 128, 4091), (64, 8, 8, 2, 128, 4091),        # four; two items per head
    (32, 8, 8, 1, 128, 16379), (20, 5, 5, 4, 128, 4091), (5, 5, 5, 20, 64, 4091),       # one queue: K/V past the L2; 20 heads
    (12, 4, 12, 2, 64, 21832), (6, 6, 6, 4, 64, 21832)])
@pytest.mark.parametrize("windows", ["even", "nearly", "uneven"])
def test_queues_per_xcd_process_every_item_once(Hq, Hkv, rows, B, D, T, windows):
    """Launches with claims, with and without a queue per XCD, rows of one length, of nearly one (queues that
    run out early claim from others) and of very different ones (small workgroups claim every item): the
    bits of the launch without a workspace, and a workspace that is zero afterwards.  Whether a launch used queues shows in a finish
    word that was not zero, which only they look at."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    per_row = Hq // rows
    heads = 4 if per_row % 4 == 0 else 2 if per_row % 2 == 0 else 1
    items = -(-T // 64) * rows * B * per_row // heads
    assert items > 3 * cus * {1: 6, 2: 3, 4: 1}[heads]         # more than the dealt ones at any occupancy
    w = {"even": [2] * rows, "nearly": [21 if r == rows // 2 else 20 for r in range(rows)],
         "uneven": [1 + 12 * r // rows for r in range(rows)]}[windows]
    case = (*_windows(B, Hq, Hkv, T, D, w), rows, 64)
    queues = B * Hkv % 8 == 0 and (heads < 4 or T * D * 4 <= 4 << 20)
    if queues and windows == "uneven":      # uneven rows: only where the queues hold about the same, and not with four heads
        load = case[4][:, -1].float().view(Hkv, -1).sum(1).repeat(B).view(8, -1).sum(1)
        queues = heads < 4 and bool(load.max() <= {1: 1.75, 2: 1.25}[heads] * load.mean())
    print(f"[prefill items] queues: heads {Hq}/{Hkv} rows {rows} B={B} D={D} T={T} {windows}: {queues}", flush=True)
    sys.stdout.flush()
    ws = torch.zeros(int(_lib.load().sa_prefill_queue_workspace_bytes()) // 4, dtype=torch.int32, device=DEV)
    want = _launch(*case, None)
    for _ in range(3):
        got = _launch(*case, ws, split=True)
        torch.cuda.synchronize()
        assert not ws.any()
        assert torch.equal(got, want)
    assert torch.isfinite(want.float()).all()
    ws.view(torch.int64)[5 * QUEUE + FINISH] = 1 << 20
    got = _launch(*case, ws, split=True)
    torch.cuda.synchronize()
    assert int(ws[3]) == int(queues)
    assert torch.equal(got, want)


@pytest.mark.parametrize("word,value", [(5 * QUEUE, 2), (0, 1 << 20), (3 * QUEUE, 1 << 33), (FINISH, 1 << 20),
                                        (7 * QUEUE + FINISH, 3), (2 * QUEUE + FINISH, 1 << 33), (ALL, 8), (ALL, 3),
                                        (ALL, 1 << 33)])
def test_queue_words_that_were_not_zero_are_reported(word, value):
    """A claims or finish word of a queue, or the queues' finish word: the status bit is set, and a
    workspace zeroed afterwards serves the next launch."""
    print(f"[prefill items] queue word {word} = {value}", flush=True)
    sys.stdout.flush()
    case = (*_windows(4, 32, 8, 4091, 64, [3] * 8), 8, 64)
    ws = torch.zeros(int(_lib.load().sa_prefill_queue_workspace_bytes()) // 4, dtype=torch.int32, device=DEV)
    want = _launch(*case, None)
    ws.view(torch.int64)[word] = value
    _launch(*case, ws, split=True)
    torch.cuda.synchronize()
    assert int(ws[3]) == 1
    ws.zero_()
    got = _launch(*case, ws, split=True)
    torch.cuda.synchronize()
    assert not ws.any()
    assert torch.equal(got, want)
