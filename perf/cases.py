"""Timed workloads of the block-sparse attention framework, through its public entry points.

``listed()`` names twelve calls that stand for what a program built on the framework has it do;
``draw(rng)`` gives further ones of the same ranges.  A case is a plain dict; its ``kind`` says
which path it takes:

* ``prefill``   attention of a prompt over a CSR block schedule (``ops.universal_sparse_attn``);
* ``backend``   the same through ``get_backend(...).forward`` with a pattern's metadata, as the
                decoder layers call it: BigBird budgets, local windows, dense causal layers, whole
                prompts, chunks of a prompt over a cached prefix, and single decode tokens over a
                contiguous cache;
* ``paged``     one decode token per sequence over a paged cache (``ops.paged_sparse_decode``);
* ``attn_step`` the attention half of a decode step, and
* ``mlp_step``  its feed-forward half with the output head, each captured in a HIP graph as the
                graph decoder does with a whole step;
* ``schedule``  building a pattern's block schedule on the GPU.

``prepare`` makes the inputs on the GPU from a seed, ``run`` is one pass, ``work`` the bytes and
operations a pass cannot do without, and ``exact`` the same results in float64 from plain torch.
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

from sparseattentioninfer_amd import get_backend, ops
from sparseattentioninfer_amd.models.kv_cache import KVCache, PagedKVStore
from sparseattentioninfer_amd.patterns import (BernoulliBlockPattern, BigBirdPattern, DenseCausalPattern,
                                                LocalWindowPattern, SeededBigBirdPattern, block_mask_to_csr)

DEV = "cuda"
_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
EPS = 1e-6
ROPE_THETA = 1e6


def listed():
    return [
        # The long prompt of the benchmark: 32K tokens, 32 query and 8 KV heads of 128, one BigBird
        # schedule per KV group with its own number of random blocks.
        dict(name="prefill_long", kind="prefill", B=1, Hq=32, Hkv=8, D=128, T=32768, block=64, dtype="bf16",
             mask="bigbird", window=3, globals=2, randoms="0,1,2,3,3,4,6,8"),
        # An arbitrary schedule, as block-selection methods produce them: a batch of 8K prompts, each
        # KV group keeping a random tenth of the blocks.
        dict(name="prefill_arbitrary", kind="prefill", B=4, Hq=32, Hkv=8, D=128, T=8192, block=64, dtype="bf16",
             mask="bernoulli", density=0.10),
        # The project's own BigBird pattern on a prompt: a budget of 1024 keys, so blocks of 32, with a
        # schedule per query head.
        dict(name="prefill_topk_heads", kind="backend", pattern="bigbird", topk=1024, B=1, Hq=32, Hkv=8, D=128,
             T_q=8192, T_k=8192, dtype="bf16"),
        # The small layer benchmark: 8 heads of 64, about a thousand tokens, blocks of 16, fp16.
        dict(name="prefill_topk_small", kind="backend", pattern="bigbird", topk=256, B=1, Hq=8, Hkv=8, D=64,
             T_q=1000, T_k=1000, dtype="fp16"),
        # The default pattern of the model integration: a window of 512 tokens, blocks of 64, a
        # schedule per query head.
        dict(name="prefill_local", kind="backend", pattern="local", window=512, block=64, B=1, Hq=32, Hkv=8, D=128,
             T_q=4096, T_k=4096, dtype="bf16"),
        # A dense causal layer on one chunk of a prompt, over the prefix that the cache already holds.
        dict(name="chunk_dense", kind="backend", pattern="dense", B=1, Hq=32, Hkv=8, D=128, T_q=1000, T_k=5000,
             dtype="bf16"),
        # Serving: 64 sequences of 16K cached tokens, 14 blocks kept of each.
        dict(name="decode_paged", kind="paged", B=64, Hq=32, Hkv=8, D=128, page=64, L=16384, ragged=False,
             local=4, globals=2, randoms=8, dtype="bf16"),
        # A dense layer decoding a few sequences over a contiguous cache.
        dict(name="decode_dense", kind="backend", pattern="dense", B=4, Hq=32, Hkv=8, D=128, T_q=1, T_k=8191,
             dtype="bf16"),
        # The smallest call: one token of one sequence, 8 heads of 64, the layer benchmark's decode mode.
        dict(name="decode_small", kind="backend", pattern="bigbird", topk=256, B=1, Hq=8, Hkv=8, D=64, T_q=1,
             T_k=1000, dtype="bf16"),
        # Attention half of a decode step: norm, q|k|v projection, rotary embedding and page write,
        # attention over a dense layer's pages, output projection.
        dict(name="decode_attn_step", kind="attn_step", B=8, hidden=2560, Hq=32, Hkv=8, D=128, page=64, L=4100,
             dense=True, dtype="bf16"),
        # Feed-forward half of a decode step and the output head.
        dict(name="decode_mlp_step", kind="mlp_step", B=8, hidden=2560, inter=9728, vocab=151936, dtype="bf16"),
        # A new prompt length: a BigBird block schedule built from nothing on the GPU.
        dict(name="schedule_new", kind="schedule", pattern="seeded", rows=8, T=32768, block=64, window=3, globals=2,
             randoms=3),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "topk", "local", "dense", "paged", "decode", "decode", "attn_step",
                       "mlp_step", "schedule"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind in ("prefill", "topk", "local", "dense"):
        Hq, Hkv = rng.choice([(32, 8), (32, 8), (16, 8), (8, 2), (8, 8), (12, 4)])
        D = rng.choice([64, 128, 128])
        B = rng.choice([1, 1, 2, 3, 4])
        cap = 8192 if kind in ("prefill", "topk", "local") else 4096
        T = max(2, min(_log_int(rng, 130, cap), cap * 32 // (B * Hq) if kind != "local" else cap))
        if kind == "prefill":
            c = dict(kind="prefill", B=B, Hq=Hq, Hkv=Hkv, D=D, T=T, block=rng.choice([64, 64, 128]), dtype=dtype)
            if rng.random() < 0.6:
                return dict(c, mask="bigbird", window=rng.choice([2, 3, 5]), globals=rng.choice([1, 2]),
                            randoms=rng.randint(0, 8))
            return dict(c, mask="bernoulli", density=round(rng.uniform(0.03, 0.3), 3))
        T_q = T if rng.random() < 0.6 else max(2, _log_int(rng, 2, T))
        if kind == "topk":
            return dict(kind="backend", pattern="bigbird", topk=rng.choice([64, 256, 512, 1024, 4096]), B=B, Hq=Hq,
                        Hkv=Hkv, D=D, T_q=T, T_k=T, dtype=dtype)
        if kind == "local":
            return dict(kind="backend", pattern="local", window=_log_int(rng, 64, 1024), block=rng.choice([32, 64, 64, 128]),
                        B=min(B, 2), Hq=Hq, Hkv=Hkv, D=D, T_q=T_q, T_k=T, dtype=dtype)
        return dict(kind="backend", pattern="dense", B=B, Hq=Hq, Hkv=Hkv, D=D, T_q=T_q, T_k=T, dtype=dtype)
    if kind == "paged":
        B = _log_int(rng, 1, 64)
        return dict(kind="paged", B=B, Hq=32, Hkv=rng.choice([8, 8, 4]), D=rng.choice([64, 128, 128]),
                    page=rng.choice([16, 32, 64, 64, 128]), L=_log_int(rng, 500, 16000), ragged=rng.random() < 0.7,
                    local=rng.randint(1, 8), globals=rng.randint(1, 2), randoms=rng.randint(0, 16), dtype=dtype)
    if kind == "decode":
        Hq, Hkv = rng.choice([(32, 8), (16, 8), (8, 8), (8, 2)])
        B = rng.choice([1, 1, 2, 4, 8])
        c = dict(kind="backend", B=B, Hq=Hq, Hkv=Hkv, D=rng.choice([64, 128, 128]), T_q=1,
                 T_k=min(_log_int(rng, 100, 32000), 64000 // B), dtype=dtype)
        p = rng.choice(["dense", "bigbird", "local"])
        if p == "bigbird":
            return dict(c, pattern=p, topk=rng.choice([64, 256, 1024, 4096]))
        if p == "local":
            return dict(c, pattern=p, window=_log_int(rng, 128, 4096), block=64)
        return dict(c, pattern=p)
    if kind == "attn_step":
        Hq, Hkv = rng.choice([(32, 8), (16, 8), (8, 2)])
        return dict(kind="attn_step", B=rng.randint(1, 8), hidden=rng.choice([1024, 2048, 2560, 4096]), Hq=Hq, Hkv=Hkv,
                    D=128, page=64, L=_log_int(rng, 70, 8000), dense=rng.random() < 0.5, dtype=dtype)
    if kind == "mlp_step":
        hidden = rng.choice([512, 1024, 2048, 2560, 4096])
        return dict(kind="mlp_step", B=rng.randint(1, 8), hidden=hidden, inter=8 * rng.randint(hidden // 4, min(1216, hidden // 2)),
                    vocab=rng.choice([5000, 32000, 151936 // 2]), dtype=dtype)
    c = dict(kind="schedule", rows=rng.choice([2, 8, 8, 32]), T=_log_int(rng, 3000, 32768), block=rng.choice([64, 64, 128]))
    if rng.random() < 0.3:
        return dict(c, pattern="bernoulli", density=round(rng.uniform(0.03, 0.3), 3))
    return dict(c, pattern="seeded", window=rng.choice([2, 3, 5]), globals=rng.choice([1, 2]), randoms=rng.randint(1, 8))


# ------------------------------------------------------------------------------------ schedules

def _mask_generator(case, seed):
    return torch.Generator().manual_seed(7919 * seed + 17)


def _block_mask(case, seed):
    """Retained blocks ``[rows, NQB, NKB]`` (CPU, bool) of a ``prefill`` case, one row per KV group:
    BigBird rows with uniformly drawn random blocks, or independent draws with the diagonal kept."""
    g = _mask_generator(case, seed)
    n, R = -(-case["T"] // case["block"]), case["Hkv"]
    qb, kb = torch.arange(n)[:, None], torch.arange(n)[None, :]
    if case["mask"] == "bernoulli":
        m = torch.rand(R, n, n, generator=g) < case["density"]
        return (m & (kb < qb)) | (kb == qb)
    base = (((kb > qb - case["window"]) | (kb < case["globals"])) & (kb <= qb)).expand(R, n, n)
    free = (kb <= qb) & ~base
    counts = [int(x) for x in str(case["randoms"]).split(",")]     # one count, or one per KV group
    counts = counts * R if len(counts) == 1 else counts
    keys = torch.where(free, torch.rand(R, n, n, generator=g), torch.full((), -1.0))
    top = torch.topk(keys, k=min(max(counts), n), dim=2)
    take = (torch.arange(top.indices.shape[2]) < torch.tensor(counts)[:, None, None]) & (top.values >= 0)
    return base | torch.zeros_like(base).scatter_(2, top.indices, take)


def _topk_layout(T, topk):
    """Block size of the schedule and the (global, window, random) block counts of a key budget."""
    bs = max(1, min(T, math.isqrt(max(1, topk))))
    budget = max(1, -(-topk // bs))
    window = min(2, budget)
    return max(16, 1 << (bs - 1).bit_length()), 1, window, max(0, budget - 1 - window)


def _topk_mask(H, T_q, T_k, topk, device):
    """The BigBird pattern's retained blocks ``[H, NQB, NKB]``: the first block, the window, and a run
    of the blocks between them that starts at a hash of head, query block and block count."""
    bs, g, s, r = _topk_layout(T_k, topk)
    nqb, nkb = -(-T_q // bs), -(-T_k // bs)
    head = torch.arange(H, device=device)[:, None, None]
    qb = ((T_k - T_q) // bs + torch.arange(nqb, device=device))[None, :, None]
    kb = torch.arange(nkb, device=device)[None, None, :]
    end = torch.minimum(qb, (qb - s + 1).clamp(min=g))
    n = (end - g).clamp(min=0)
    rank = (kb - g - (131 * head + 17 * qb + 7 * nkb) % n.clamp(min=1)) % n.clamp(min=1)
    rand = (kb >= g) & (kb < end) & (rank < r)
    return ((kb < g) | ((kb > qb - s) & (kb <= qb)) | rand), bs


def _local_mask(T_q, T_k, window, bs, device):
    """Blocks that the window of any row of a query block overlaps, ``[NQB, NKB]``."""
    nqb, nkb = -(-T_q // bs), -(-T_k // bs)
    first = T_k - T_q + bs * torch.arange(nqb, device=device)[:, None]
    last = T_k - T_q + (bs * torch.arange(1, nqb + 1, device=device)).clamp(max=T_q)[:, None] - 1
    kb = torch.arange(nkb, device=device)[None, :]
    return (kb * bs <= last) & (torch.clamp(kb * bs + bs, max=T_k) - 1 >= first - window + 1)


def _pattern(case):
    if case["pattern"] == "bigbird":
        return BigBirdPattern(top_k=case["topk"], n_heads=case["Hq"])
    if case["pattern"] == "local":
        return LocalWindowPattern(window_size=case["window"], block_size=case["block"])
    return DenseCausalPattern()


def _seeded_pattern(case, seed):
    if case["pattern"] == "bernoulli":
        return BernoulliBlockPattern(rows=case["rows"], density=case["density"], block_size=case["block"], seed=seed,
                                     rng="philox")
    return SeededBigBirdPattern(rows=case["rows"], block_size=case["block"], window=case["window"],
                                global_blocks=case["globals"], random_blocks=case["randoms"], seed=seed, rng="philox")


def _backend_mask(case, device):
    """Retained blocks ``[rows, NQB, NKB]`` and the block size of a ``backend`` case."""
    if case["pattern"] == "bigbird":
        return _topk_mask(case["Hq"], case["T_q"], case["T_k"], case["topk"], device)
    if case["pattern"] == "local":
        return _local_mask(case["T_q"], case["T_k"], case["window"], case["block"], device)[None], case["block"]
    return torch.ones(1, 1, 1, dtype=torch.bool, device=device), max(case["T_q"], case["T_k"])


def _selection(case, seed):
    """Kept logical blocks of each sequence and KV head (ascending), and the sequence lengths."""
    g = _mask_generator(case, seed)
    B, R, page, L = case["B"], case["Hkv"], case["page"], case["L"]
    lens = torch.full((B,), L, dtype=torch.int32)
    if case["ragged"]:
        lens = torch.randint(-(-L // 2), L + 1, (B,), generator=g).to(torch.int32)
    n = (-(-lens // page))[:, None, None]
    kb = torch.arange(int(n.max()))[None, None, :]
    base = (((kb >= n - case["local"]) | (kb < case["globals"])) & (kb < n)).expand(B, R, kb.shape[2])
    keys = torch.where((kb < n) & ~base, torch.rand(base.shape, generator=g), torch.full((), -1.0))
    top = torch.topk(keys, k=min(case["randoms"], base.shape[2]), dim=2)
    keep = base | torch.zeros_like(base).scatter_(2, top.indices, top.values >= 0)
    count = keep.sum(2)
    width = int(count.max())
    ids = torch.where(keep, kb, kb.shape[2]).sort(dim=2).values[:, :, :width]
    sel = torch.where(torch.arange(width) < count[:, :, None], ids, 0).to(torch.int32).contiguous()
    off = torch.stack([torch.zeros_like(count), count], dim=2).to(torch.int32).contiguous()
    return sel, off, lens


# ---------------------------------------------------------------------------------- preparation

def _normal(g, dtype, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=dtype)


def _qkv(case, seed, T_q, T_k):
    """q, k with a spread of scales over the head dims (as projections give them), v ~ N(0, 1)."""
    g = torch.Generator(device=DEV).manual_seed(1000003 * seed + 11)
    dt = _DTYPES[case["dtype"]]
    B, Hq, Hkv, D = case["B"], case["Hq"], case["Hkv"], case["D"]
    scale = torch.empty(D, device=DEV).uniform_(0.5, 1.5, generator=g).to(dt)
    return (_normal(g, dt, B, Hq, T_q, D) * scale, _normal(g, dt, B, Hkv, T_k, D) * scale,
            _normal(g, dt, B, Hkv, T_k, D))


def _prepare_prefill(case, seed):
    q, k, v = _qkv(case, seed, case["T"], case["T"])
    pairs, offsets = block_mask_to_csr(_block_mask(case, seed))
    return dict(q=q, k=k, v=v, pairs=pairs.to(DEV), offsets=offsets.to(DEV))


def _prepare_backend(case, seed):
    q, k, v = _qkv(case, seed, case["T_q"], case["T_k"])
    if case["T_q"] < case["T_k"]:     # a cached prefix: the views a cache with room to grow hands out
        cache = KVCache(1, max_len=case["T_k"] + 128)
        cache.init([k], [v])
        k, v = cache.get(0)
    pattern = _pattern(case).build(q, k, causal=True)
    return dict(q=q, k=k, v=v, pattern=pattern, backend=get_backend("hip_block_sparse"))


def _prepare_paged(case, seed):
    g = torch.Generator(device=DEV).manual_seed(1000003 * seed + 13)
    dt = _DTYPES[case["dtype"]]
    sel, off, lens = _selection(case, seed)
    B, page = case["B"], case["page"]
    nblk = -(-case["L"] // page)
    table = torch.randperm(B * nblk, generator=_mask_generator(case, seed + 1)).to(torch.int32).reshape(B, nblk)
    return dict(q=_normal(g, dt, B, case["Hq"], case["D"]),
                k_pages=_normal(g, dt, B * nblk, case["Hkv"], page, case["D"]),
                v_pages=_normal(g, dt, B * nblk, case["Hkv"], page, case["D"]),
                table=table.to(DEV), lens=lens.to(DEV), sel=sel.to(DEV), off=off.to(DEV))


def _capture(step):
    """A HIP graph of ``step``, after two eager passes, as the graph decoder captures a decode step."""
    for _ in range(2):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return graph


def _prepare_attn_step(case, seed):
    g = torch.Generator(device=DEV).manual_seed(1000003 * seed + 17)
    dt = _DTYPES[case["dtype"]]
    B, hidden, Hq, Hkv, D, page, L = (case[x] for x in ("B", "hidden", "Hq", "Hkv", "D", "page", "L"))
    s = dict(case=case, x=_normal(g, dt, B, hidden), w_in=1 + 0.1 * _normal(g, dt, hidden),
             w_q=1 + 0.1 * _normal(g, dt, D), w_k=1 + 0.1 * _normal(g, dt, D),
             w_qkv=_normal(g, dt, (Hq + 2 * Hkv) * D, hidden) * 0.02, w_o=_normal(g, dt, hidden, Hq * D) * 0.02)
    store = PagedKVStore(B, Hkv, D, L + page, page=page, dtype=dt, device=DEV, shuffle_seed=seed)
    store.k_pages.zero_()
    store.v_pages.zero_()
    # L tokens in the cache and room for the new one at position L
    store.write(_normal(g, dt, B, Hkv, L + 1, D), _normal(g, dt, B, Hkv, L + 1, D))
    nblk = -(-(L + 1) // page)
    if case["dense"]:
        sel = torch.arange(nblk, dtype=torch.int32).expand(Hkv, nblk).contiguous()
    else:     # the first two blocks, the last three, three of the others
        mid = sorted(random.Random(seed).sample(range(2, nblk - 3), min(3, nblk - 5))) if nblk > 5 else []
        ids = sorted({*range(min(2, nblk)), *mid, *range(max(0, nblk - 3), nblk)})
        sel = torch.tensor(ids, dtype=torch.int32).expand(Hkv, len(ids)).contiguous()
    off = torch.tensor([0, sel.shape[1]], dtype=torch.int32).expand(Hkv, 2).contiguous()
    s.update(store=store, sel_row=sel, sel=sel.to(DEV)[None].expand(B, -1, -1), off=off.to(DEV)[None].expand(B, -1, -1),
             pos=torch.full((1,), L, dtype=torch.long, device=DEV),
             inv_freq=1.0 / ROPE_THETA ** (torch.arange(0, D, 2, device=DEV, dtype=torch.float32) / D),
             normed=torch.empty(B, hidden, dtype=dt, device=DEV),
             qkv=torch.empty(B, (Hq + 2 * Hkv) * D, dtype=dt, device=DEV),
             q=torch.empty(B, Hq, D, dtype=dt, device=DEV), att=torch.empty(B, Hq, D, dtype=dt, device=DEV),
             out=torch.empty(B, hidden, dtype=dt, device=DEV))
    splits = ops.auto_decode_splits(B, Hkv, sel.shape[1])
    work = torch.empty(max(1, ops.decode_workspace_bytes(B, Hq, D, splits)), dtype=torch.uint8, device=DEV)

    def step():
        ops.rmsnorm(s["x"], s["w_in"], EPS, out=s["normed"])
        ops.gemm_skinny(s["normed"], s["w_qkv"], out=s["qkv"])
        ops.qk_rope_kv(s["qkv"], s["w_q"], s["w_k"], s["inv_freq"], s["pos"], store, s["q"], num_heads=Hq, eps=EPS)
        ops.paged_sparse_decode(s["q"], store.k_pages, store.v_pages, store.block_table, store.kv_lens, s["sel"],
                                s["off"], num_splits=splits, workspace=work, out=s["att"])
        ops.gemm_skinny(s["att"].view(B, -1), s["w_o"], out=s["out"])

    s["graph"] = _capture(step)
    s["keep"] = work
    return s


def _prepare_mlp_step(case, seed):
    g = torch.Generator(device=DEV).manual_seed(1000003 * seed + 19)
    dt = _DTYPES[case["dtype"]]
    B, hidden, inter, vocab = (case[x] for x in ("B", "hidden", "inter", "vocab"))
    gate, up = (_normal(g, dt, inter, hidden) * 0.02 for _ in range(2))
    s = dict(x=_normal(g, dt, B, hidden), h0=_normal(g, dt, B, hidden), w_post=1 + 0.1 * _normal(g, dt, hidden),
             w_norm=1 + 0.1 * _normal(g, dt, hidden), w_gu=ops.interleave_gate_up(gate, up),
             w_down=_normal(g, dt, hidden, inter) * 0.02, w_head=_normal(g, dt, vocab, hidden) * 0.02)
    new = lambda n: torch.empty(B, n, dtype=dt, device=DEV)  # noqa: E731
    s.update(h=new(hidden), normed=new(hidden), mid=new(inter), down=new(hidden), logits=new(vocab))

    def step():
        s["h"].copy_(s["h0"])
        ops.rmsnorm(s["x"], s["w_post"], EPS, residual=s["h"], out=s["normed"])
        ops.gemm_skinny_swiglu(s["normed"], s["w_gu"], out=s["mid"])
        ops.gemm_skinny(s["mid"], s["w_down"], out=s["down"])
        ops.rmsnorm(s["down"], s["w_norm"], EPS, residual=s["h"], out=s["normed"])
        ops.gemm_skinny(s["normed"], s["w_head"], out=s["logits"])

    s["graph"] = _capture(step)
    return s


def _prepare_schedule(case, seed):
    q = torch.empty(1, case["rows"], case["T"], 0, device=DEV)      # a pattern reads shapes only
    return dict(q=q, k=q, seed=seed)


_PREPARE = dict(prefill=_prepare_prefill, backend=_prepare_backend, paged=_prepare_paged,
                attn_step=_prepare_attn_step, mlp_step=_prepare_mlp_step, schedule=_prepare_schedule)


def prepare(case, seed):
    return dict(_PREPARE[case["kind"]](case, seed), case=case)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "prefill":
        return ops.universal_sparse_attn(s["q"], s["k"], s["v"], s["pairs"], s["offsets"], case["block"])
    if kind == "backend":
        return s["backend"].forward(s["q"], s["k"], s["v"], s["pattern"])
    if kind == "paged":
        return ops.paged_sparse_decode(s["q"], s["k_pages"], s["v_pages"], s["table"], s["lens"], s["sel"], s["off"],
                                       num_splits=0)
    if kind == "attn_step":
        s["graph"].replay()
        return dict(out=s["out"], k_pages=s["store"].k_pages, v_pages=s["store"].v_pages)
    if kind == "mlp_step":
        s["graph"].replay()
        return dict(logits=s["logits"], residual=s["h"])
    p = _seeded_pattern(case, s["seed"]).build(s["q"], s["k"], causal=True)      # a new object: nothing cached
    return dict(pairs=p.block_pairs, offsets=p.block_pair_offsets)


# -------------------------------------------------------------------------------- work and limits

def _visible(mask, bs, T_q, T_k):
    """Visible (query, key) pairs of retained blocks under the causal limit, over all mask rows, and
    the keys below T_k that any query block of a row retains (for the bytes of K and V)."""
    R, nqb, nkb = mask.shape
    t = T_k - T_q + torch.arange(T_q)                          # absolute positions
    qb = torch.arange(T_q) // bs
    kb = torch.arange(nkb)
    # keys of block kb at or before position t
    seen = (t[:, None] + 1 - kb[None, :] * bs).clamp(min=0, max=bs)
    seen = torch.minimum(seen, (T_k - kb * bs).clamp(max=bs)[None, :])
    per_block = torch.zeros(nqb, nkb, dtype=torch.long).index_add_(0, qb, seen)
    used = mask.any(dim=1).long() * (T_k - kb * bs).clamp(min=0, max=bs)
    return int((mask.long() * per_block).sum()), int(used.sum())


def work(case):
    kind = case["kind"]
    if kind in ("prefill", "backend"):
        B, Hq, Hkv, D = case["B"], case["Hq"], case["Hkv"], case["D"]
        T_q, T_k = case.get("T_q", case.get("T")), case.get("T_k", case.get("T"))
        if kind == "prefill":
            m, bs = _block_mask(case, 0), case["block"]
        elif case["pattern"] == "dense":
            m, bs = None, 0
        else:
            m, bs = _backend_mask(case, "cpu")
        if m is None:
            pairs, keys, index = B * Hq * (T_q * (T_k - T_q) + T_q * (T_q + 1) // 2), B * Hkv * T_k, 0
        else:
            pairs, _ = _visible(m, bs, T_q, T_k)
            pairs *= B * (Hq // m.shape[0])
            # keys that any head of a KV group keeps
            group = m.reshape(min(m.shape[0], Hkv), -1, *m.shape[1:]).any(dim=1)
            keys = _visible(group, bs, T_q, T_k)[1] * B * (Hkv // group.shape[0])
            index = 4 * int(m.sum()) * (Hq // m.shape[0] if kind == "backend" else 1)
        return dict(bytes=4 * B * Hq * T_q * D + 4 * keys * D + index, flops=4 * D * pairs)
    if kind == "paged":
        sel, off, lens = _selection(case, 0)
        live = torch.arange(sel.shape[2]) < off[:, :, 1:]
        keys = int(((lens[:, None, None] - sel * case["page"]).clamp(max=case["page"]) * live).sum())
        group = case["Hq"] // case["Hkv"]
        return dict(bytes=4 * keys * case["D"] + 4 * case["B"] * case["Hq"] * case["D"] + 8 * int(live.sum()),
                    flops=4 * keys * group * case["D"])
    if kind == "attn_step":
        B, hidden, Hq, Hkv, D, page, L = (case[x] for x in ("B", "hidden", "Hq", "Hkv", "D", "page", "L"))
        nblk = -(-(L + 1) // page)
        keys = B * (L + 1 if case["dense"] or nblk <= 8 else L + 1 - (nblk - 8) * page)
        weights = hidden * D * (2 * Hq + 2 * Hkv)
        return dict(bytes=2 * weights + 4 * B * hidden + 4 * keys * Hkv * D, flops=2 * B * weights + 4 * keys * Hq * D)
    if kind == "mlp_step":
        weights = case["hidden"] * (3 * case["inter"] + case["vocab"])
        return dict(bytes=2 * weights + 2 * case["B"] * (4 * case["hidden"] + case["vocab"]), flops=2 * case["B"] * weights)
    n = -(-case["T"] // case["block"])
    kept = min(n, case["window"] + case["globals"] + case["randoms"]) if case["pattern"] == "seeded" \
        else 1 + case["density"] * n / 2
    return dict(bytes=4 * case["rows"] * (int(kept * n) + n), flops=case["rows"] * n * n)      # one test per block


def tolerance(case):
    if case["kind"] == "schedule":
        return "exact"
    # 16-bit results: one rounding of the output and, in attention, one of each probability.
    fine = case["dtype"] == "fp16"
    if case["kind"] in ("attn_step", "mlp_step"):      # several roundings to 16 bits one after the other
        return {"rel": 2.5e-3 if fine else 2e-2, "max": 0.05 if fine else 0.4}
    return {"rel": 1.2e-3 if fine else 1e-2, "max": 0.02 if fine else 0.12}


# ------------------------------------------------------------------------------------- float64

def _attention64(q, k, v, mask, bs, rows_per_step=64 * 1024 * 1024):
    """Causal attention over retained blocks in float64, ``mask [R, NQB, NKB]`` (R divides or equals
    the heads); a row that sees no key gives 0."""
    B, Hq, T_q, D = q.shape
    Hkv, T_k = k.shape[1], k.shape[2]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    key = torch.arange(T_k, device=q.device)
    kcol = key // bs
    step = max(1, rows_per_step // T_k)
    for b in range(B):
        for hk in range(Hkv):
            kt = k[b, hk].double().t().contiguous()
            vd = v[b, hk].double().contiguous()
            for h in range(hk * (Hq // Hkv), (hk + 1) * (Hq // Hkv)):
                m = mask[h * mask.shape[0] // Hq]
                for t0 in range(0, T_q, step):
                    t1 = min(T_q, t0 + step)
                    t = torch.arange(t0, t1, device=q.device)
                    s = torch.mm(q[b, h, t0:t1].double().contiguous(), kt).div_(math.sqrt(D))
                    keep = m[t // bs][:, kcol] & (key[None, :] <= (T_k - T_q + t)[:, None])
                    s.masked_fill_(~keep, -math.inf)
                    s.sub_(s.amax(dim=1, keepdim=True).nan_to_num_(neginf=0.0)).exp_()
                    total = s.sum(dim=1, keepdim=True)
                    out[b, h, t0:t1] = torch.mm(s, vd) / total.clamp(min=1e-300)
    return out


def _gathered64(q, k, v, sel, off, lens, table, page):
    """Decode attention in float64 of ``q [B, Hq, D]`` over the kept blocks of a paged cache."""
    B, Hq, D = q.shape
    Hkv = k.shape[1]
    out = torch.zeros(q.shape, dtype=torch.float64, device=q.device)
    live = torch.arange(sel.shape[2], device=q.device) < off[:, :, 1:]
    for b in range(B):
        blk = sel[b].long()                                                     # [Hkv, n]
        pg = table[b].long()[blk]
        pos = blk[:, :, None] * page + torch.arange(page, device=q.device)
        ok = (live[b][:, :, None] & (pos < lens[b])).reshape(Hkv, -1)
        head = torch.arange(Hkv, device=q.device)[:, None].expand_as(pg)
        kk, vv = (x[pg, head].double().reshape(Hkv, -1, D) for x in (k, v))
        s = (q[b].double().reshape(Hkv, -1, 1, D) * kk[:, None]).sum(-1) / math.sqrt(D)
        p = torch.softmax(s.masked_fill(~ok[:, None], -math.inf), dim=-1)
        out[b] = (p[..., None] * vv[:, None]).sum(2).reshape(Hq, D)
    return out


def _rms64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _exact_attn_step(case, s):
    B, Hq, Hkv, D, page, L = (case[x] for x in ("B", "Hq", "Hkv", "D", "page", "L"))
    store = s["store"]
    qkv = _rms64(s["x"].double(), s["w_in"]) @ s["w_qkv"].double().t().contiguous()
    q, k, v = qkv.reshape(B, Hq + 2 * Hkv, D).split([Hq, Hkv, Hkv], dim=1)
    ang = s["inv_freq"].double() * L
    cos, sin = torch.cat([ang.cos()] * 2), torch.cat([ang.sin()] * 2)
    turn = lambda x: x * cos + torch.cat([-x[..., D // 2:], x[..., :D // 2]], dim=-1) * sin  # noqa: E731
    q, k = turn(_rms64(q, s["w_q"])), turn(_rms64(k, s["w_k"]))
    kp, vp = store.k_pages.double(), store.v_pages.double()
    page_of = store.block_table[:, L // page].long()
    kp[page_of, :, L % page] = k
    vp[page_of, :, L % page] = v
    lens = torch.full((B,), L + 1, device=DEV)
    att = _gathered64(q, kp, vp, s["sel"], s["off"], lens, store.block_table, page)
    return dict(out=att.reshape(B, -1) @ s["w_o"].double().t().contiguous(), k_pages=kp, v_pages=vp)


def _exact_mlp_step(s):
    h = s["h0"].double() + s["x"].double()
    x = _rms64(h, s["w_post"])
    gu = x @ s["w_gu"].double().t().contiguous()
    h = h + (F.silu(gu[:, 0::2]) * gu[:, 1::2]) @ s["w_down"].double().t().contiguous()
    return dict(logits=_rms64(h, s["w_norm"]) @ s["w_head"].double().t().contiguous(), residual=h)


def exact(case, seed):
    kind = case["kind"]
    if kind == "schedule":
        return None
    s = prepare(case, seed)
    if kind == "prefill":
        return _attention64(s["q"], s["k"], s["v"], _block_mask(case, seed).to(DEV), case["block"])
    if kind == "backend":
        mask, bs = _backend_mask(case, DEV)
        return _attention64(s["q"], s["k"], s["v"], mask, bs)
    if kind == "paged":
        return _gathered64(s["q"], s["k_pages"], s["v_pages"], s["sel"], s["off"], s["lens"], s["table"], case["page"])
    return _exact_attn_step(case, s) if kind == "attn_step" else _exact_mlp_step(s)
