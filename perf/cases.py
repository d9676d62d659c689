"""Work that users have this framework do, as cases for timing: what is prepared once, what one pass
calls, and what a pass cannot do without.

Every tensor is bf16 with N(0, 1) entries, [batch, tokens, heads, 128]; token counts are multiples of
the 128-row kernel tile.  Families of cases:

* ``dense``  one rectangle through the flash-attention signatures: what the executors call for every
  chunk pair, and what any model calls for full or causal attention.
* ``ring``   one rank's loop over the K/V chunks it is sent: dense calls whose partial outputs are
  folded with ``update_out_and_lse`` and whose gradients are added up in fp32.
* ``sparse`` block-sparse attention over a block mask, the plan kept (one ``TileList`` per mask) or the
  mask handed over with every call (masks that depend on the data).
* ``stream`` the query shard of a long streaming context, as key-range kernel tiles that are merged.
* ``fused``  a fused rectangle of row and column chunks on packed buffers, with the layout changes
  around it and the reductions of the partial results that other devices send.
* ``plan``   block mask to tile lists on the device.
"""
import math

import numpy as np
import torch

from ultraattn_amd import masks, packed
from ultraattn_amd.executor import BlockSparseExecutor
from ultraattn_amd.flash_attn_interface import _flash_attn_backward, _flash_attn_forward
from ultraattn_amd.ops import bsa_bwd, bsa_fwd, grad_accumulate, update_out_and_lse
from ultraattn_amd.tilelist import TILE, build_tile_list, build_tile_list_device

DEVICE = "cuda:0"
DIM = 128
SCALE = 1.0 / math.sqrt(DIM)
TOKENS_MAX = 131072          # the longest sequence of the benchmark masks
FLOPS_MAX = 7.0e13           # just under the largest listed case


def _dense(batch, heads, seq_q, seq_k, causal, backward, packed_kv=False, in_place=False):
    return dict(kind="dense", batch=batch, heads=heads, seq_q=seq_q, seq_k=seq_k, causal=causal, backward=backward,
                packed_kv=packed_kv, in_place=in_place)


def _sparse(pattern, blocks, block, heads, backward, keep_plan):
    return dict(kind="sparse", pattern=pattern, blocks=blocks, block=block, heads=heads, backward=backward, keep_plan=keep_plan)


def listed():
    cases = [
        # the smallest entry of the planner's cost table: all latency
        ("tiny_causal_fwd", _dense(1, 1, 256, 256, True, False)),
        # one 512 x 512 chunk pair of the executors' loop, results written into the plan's buffers
        ("chunk_512_fwd_bwd", _dense(1, 32, 512, 512, False, True, in_place=True)),
        # one head, few query rows, a long key range: little parallelism in the rows
        ("one_head_1k_4k_fwd_bwd", _dense(1, 1, 1024, 4096, False, True)),
        # an ordinary training step's attention
        ("causal_8k_fwd_bwd", _dense(1, 32, 8192, 8192, True, True)),
        # odd tile and head counts, a batch, K and V as views of one projection's output, a cached prefix
        ("ragged_prefix_fwd_bwd", _dense(2, 5, 1408, 2688, True, True, packed_kv=True)),
        # the last rank of a four-way ring
        ("ring_rank_fwd_bwd", dict(kind="ring", rank=3, chunk=1024, heads=8)),
        # a mask that comes with the call
        ("mask_per_call_8k_fwd", _sparse("strided", 16, 512, 8, False, False)),
        # the benchmark's two training masks at full size
        ("strided_128k_fwd_bwd", _sparse("strided", 256, 512, 32, True, True)),
        ("global_local_128k_fwd_bwd", _sparse("global_local", 256, 512, 32, True, True)),
        # the benchmark's streaming shard: the last 64k queries of a 512k context in four kernel tiles
        ("streaming_shard_fwd", dict(kind="stream", q_blocks=128, k_blocks=1024, window=16, heads=32, kernel_tiles=4)),
        # 2 row chunks x 3 column chunks, three partial results per row chunk to reduce
        ("fused_rectangle_fwd_bwd", dict(kind="fused", rows=2, cols=3, chunk=1152, heads=32, peers=2)),
        # planning on the device at the benchmark's size
        ("device_plan_128k", dict(kind="plan", pattern="strided", blocks=256, block=512)),
    ]
    return [dict(c, name=n) for n, c in cases]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choices(("dense", "ring", "sparse", "stream", "fused", "plan"), (5, 1, 3, 1, 1, 1))[0]
    heads = rng.choice((1, 2, 3, 5, 8, 16, 24, 32))
    if kind == "dense":
        tiles_q = _log_int(rng, 1, 128)
        square = rng.random() < 0.6
        tiles_k = tiles_q if square else max(1, int(tiles_q * rng.choice((0.25, 0.5, 1.5, 2, 3, 4))))
        batch = rng.choice((1, 1, 1, 2, 3))
        return _dense(batch, heads, tiles_q * TILE, tiles_k * TILE, rng.random() < 0.5, rng.random() < 0.7,
                      packed_kv=rng.random() < 0.3, in_place=rng.random() < 0.3)
    if kind == "ring":
        return dict(kind=kind, rank=rng.randint(1, 7), chunk=TILE * _log_int(rng, 2, 32), heads=heads)
    if kind == "sparse":
        block = rng.choice((128, 256, 512, 512))
        keep_plan = rng.random() < 0.75
        # a mask per call is for contexts where the call is not far longer than the planning
        blocks = _log_int(rng, 8, min(256 if keep_plan else 96, TOKENS_MAX // block))
        return _sparse(rng.choice(("strided", "global_local", "causal")), blocks, block, heads, rng.random() < 0.6, keep_plan)
    if kind == "stream":
        q_blocks = _log_int(rng, 4, 128)
        return dict(kind=kind, q_blocks=q_blocks, k_blocks=q_blocks * rng.randint(2, 8), window=rng.randint(2, 16), heads=heads,
                    kernel_tiles=rng.choice((1, 2, 3, 4, 8)))
    if kind == "fused":
        return dict(kind=kind, rows=rng.randint(1, 4), cols=rng.randint(2, 4), chunk=TILE * _log_int(rng, 2, 32), heads=heads,
                    peers=rng.randint(1, 3))
    return dict(kind=kind, pattern=rng.choice(("strided", "global_local", "causal")), blocks=_log_int(rng, 8, 256),
                block=rng.choice((128, 256, 512)))


def draw(rng):
    while True:
        case = _draw_once(rng)
        if work(case)["flops"] <= FLOPS_MAX:
            return case


def _mask(pattern, blocks):
    """uint8 block table: 0 empty, 1 full, 2 causal."""
    if pattern == "strided":
        return masks.config_strided(blocks)
    if pattern == "global_local":
        return masks.config_global_local(blocks)
    return masks.config_causal(blocks)


class _Maker:
    """Seeded tensors on the device."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE).manual_seed(int(seed))

    def normal(self, *shape):
        return torch.empty(*shape, dtype=torch.bfloat16, device=DEVICE).normal_(generator=self.g)

    def rows(self, batch, tokens, heads):
        return self.normal(batch, tokens, heads, DIM)

    def lse(self, batch, heads, tokens):
        # a partial over a thousand N(0, 1) keys: log(1000) + 1/2, spread over neighbouring rows
        return torch.empty(batch, heads, tokens, dtype=torch.float32, device=DEVICE).normal_(7.4, 0.3, generator=self.g)


def prepare(case, seed):
    m, kind = _Maker(seed), case["kind"]
    heads = case.get("heads", 1)
    s = dict(case=case)
    if kind == "dense":
        B, sq, sk = case["batch"], case["seq_q"], case["seq_k"]
        s["q"] = m.rows(B, sq, heads)
        if case["packed_kv"]:
            kv = m.normal(B, sk, 2, heads, DIM)
            s["k"], s["v"] = kv[:, :, 0], kv[:, :, 1]
        else:
            s["k"], s["v"] = m.rows(B, sk, heads), m.rows(B, sk, heads)
        s["out"] = torch.empty_like(s["q"]) if case["in_place"] else None
        if case["backward"]:
            s["do"] = m.rows(B, sq, heads)
            s["dq"] = torch.empty_like(s["q"]) if case["in_place"] else None
            if case["packed_kv"]:                      # gradients of the projection's output
                dkv = torch.empty_like(kv)
                s["dk"], s["dv"] = dkv[:, :, 0], dkv[:, :, 1]
            else:
                s["dk"], s["dv"] = (torch.empty_like(s["k"]) if case["in_place"] else None for _ in range(2))
    elif kind == "ring":
        n, c = case["rank"] + 1, case["chunk"]
        s["q"], s["do"] = m.rows(1, c, heads), m.rows(1, c, heads)
        s["k"], s["v"] = [m.rows(1, c, heads) for _ in range(n)], [m.rows(1, c, heads) for _ in range(n)]
    elif kind == "sparse":
        n = case["blocks"] * case["block"]
        s["q"], s["k"], s["v"] = (m.rows(1, n, heads) for _ in range(3))
        if case["backward"]:
            s["do"] = m.rows(1, n, heads)
        s["mask"] = _mask(case["pattern"], case["blocks"])
        if case["keep_plan"]:
            s["mask"] = build_tile_list(s["mask"], block=case["block"])
            s["mask"].on(DEVICE)
    elif kind == "stream":
        s["q"] = m.rows(1, case["q_blocks"] * 512, heads)
        s["k"], s["v"] = m.rows(1, case["k_blocks"] * 512, heads), m.rows(1, case["k_blocks"] * 512, heads)
        table = masks.config_streaming_shard(case["q_blocks"], case["k_blocks"], case["window"])
        s["executor"] = BlockSparseExecutor(table, 512, SCALE, kernel_tiles=case["kernel_tiles"])
        for t in s["executor"].kernel_tiles or [s["executor"].tiles]:
            t.on(DEVICE)
    elif kind == "fused":
        X, Y, c, peers = case["rows"], case["cols"], case["chunk"], case["peers"]
        q_shape, kv_shape = (1, X * c, heads, DIM), (1, Y * c, heads, DIM)
        # receive buffers: [Q | dO | D | lse] of the rows, [K | V] chunk by chunk, the peers' partial results
        s["row"] = packed.InputRowBwd(m.normal(packed.InputRowBwd.numel(q_shape)), q_shape)
        s["cols"] = m.normal(2 * Y * c * heads * DIM)
        s["peer_out"] = [packed.OutputRowFwd(m.normal(math.prod(q_shape)), q_shape, lse=m.lse(1, heads, X * c)) for _ in range(peers)]
        s["peer_dq"] = [packed.OutputRowBwd(m.normal(math.prod(q_shape)), q_shape) for _ in range(peers)]
        s["out_row"] = torch.empty(math.prod(q_shape), dtype=torch.bfloat16, device=DEVICE)
        s["dq_row"] = packed.OutputRowBwd(torch.empty_like(s["out_row"]), q_shape)
        s["dkv_col"] = packed.OutputColBwd(torch.empty(2 * math.prod(kv_shape), dtype=torch.bfloat16, device=DEVICE), kv_shape)
        s["q_shape"] = q_shape
    else:
        table = _mask(case["pattern"], case["blocks"])
        # another seed: another selection, one full block in ten dropped as data-dependent masks do
        table = table.copy()
        drop = np.random.default_rng(int(seed)).permutation(np.flatnonzero(table == masks.FULL))
        table.flat[drop[:len(drop) // 10]] = masks.EMPTY
        rate = case["block"] // TILE
        full, diag = masks.block_counts(table)
        s["nnz"] = full * rate * rate + diag * (rate * (rate + 1) // 2)
        s["mask"] = torch.from_numpy(table).to(DEVICE)
    return s


def _run_dense(s):
    c = s["case"]
    res = _flash_attn_forward(s["q"], s["k"], s["v"], 0.0, SCALE, c["causal"], out=s["out"])
    out, lse = res[0], res[5]
    if not c["backward"]:
        return out, lse
    dq, dk, dv, delta = _flash_attn_backward(s["do"], s["q"], s["k"], s["v"], out, lse, s["dq"], s["dk"], s["dv"], 0.0, SCALE,
                                             c["causal"])
    return out, lse, dq, dk, dv, delta


def _run_ring(s):
    q, do, rank = s["q"], s["do"], s["case"]["rank"]
    out = lse = None
    for step in range(rank + 1):                        # K/V of rank `rank - step` have arrived
        j = rank - step
        res = _flash_attn_forward(q, s["k"][j], s["v"][j], 0.0, SCALE, step == 0)
        out, lse = update_out_and_lse(out, lse, res[0], res[5])
    out = out.to(torch.bfloat16)
    lse = lse.squeeze(dim=-1).transpose(1, 2).contiguous()
    dq = torch.zeros(q.shape, dtype=torch.float32, device=q.device)
    grads = [None] * (rank + 1)
    block_dq = torch.empty_like(q)
    for step in range(rank + 1):
        j = rank - step
        _, dk, dv, _ = _flash_attn_backward(do, q, s["k"][j], s["v"][j], out, lse, block_dq, None, None, 0.0, SCALE, step == 0)
        grad_accumulate(block_dq, None, acc=dq)
        grads[j] = (dk, dv)                             # sent on with their chunk
    return out, lse, dq.to(torch.bfloat16), grads


def _run_sparse(s):
    c = s["case"]
    out, lse = bsa_fwd(s["q"], s["k"], s["v"], s["mask"], SCALE, block=c["block"])
    if not c["backward"]:
        return out, lse
    return (out, lse) + tuple(bsa_bwd(s["do"], s["q"], s["k"], s["v"], out, lse, s["mask"], SCALE, block=c["block"]))


def _run_fused(s):
    c, row = s["case"], s["row"]
    Y, k_shape = c["cols"], (1, c["chunk"], c["heads"], DIM)
    col = packed.gather_cols(s["cols"], Y, k_shape)
    own = packed.OutputRowFwd(s["out_row"], s["q_shape"])
    res = _flash_attn_forward(row.Q, col.K, col.V, 0.0, SCALE, False, out=own.O)
    own.lse = res[5]
    for other in s["peer_out"]:                         # the rows' result over all devices' keys
        own.reduce(other)
    row.fill_delta(own.O)
    dq, dkv = s["dq_row"], s["dkv_col"]
    _flash_attn_backward(row.dO, row.Q, col.K, col.V, None, own.lse, dq.dQ, dkv.dK, dkv.dV, 0.0, SCALE, False, softmax_d=row.D)
    dq.begin_reduce()
    for other in s["peer_dq"]:
        dq.reduce(other)
    dq.end_reduce()
    return own.O, own.lse, row.D, dq.dQ, packed.scatter_cols(dkv, Y, k_shape)


def run(state):
    kind = state["case"]["kind"]
    if kind == "dense":
        return _run_dense(state)
    if kind == "ring":
        return _run_ring(state)
    if kind == "sparse":
        return _run_sparse(state)
    if kind == "stream":
        return state["executor"].forward(state["q"], state["k"], state["v"])
    if kind == "fused":
        return _run_fused(state)
    lists = build_tile_list_device(state["mask"], block=state["case"]["block"], nnz=state["nnz"])
    return {name: lists[name] for name in ("row_ptr", "col_idx", "flag", "col_ptr", "row_idx", "cflag", "q_order", "k_order")}


def _causal_pairs(seq_q, seq_k):
    """Visible (query, key) pairs with the diagonal in the bottom-right corner."""
    first = max(0, seq_q - seq_k)                       # rows before it see no key
    n = seq_q - first
    return n * (seq_k - seq_q + first + 1) + n * (n - 1) // 2


def _attention(pairs, rows_q, rows_k, backward):
    """flops and bytes of one attention over `pairs` visible pairs; rows_* count (token, head) rows.
    The forward is two products over the pairs, the backward five."""
    row, stat = DIM * 2, 4
    flops = 2 * 2 * pairs * DIM * (3.5 if backward else 1.0)
    moved = rows_q * (2 * row + stat) + rows_k * 2 * row                       # Q, O, LSE; K, V
    if backward:                                                               # dO, dQ; dK, dV
        moved += rows_q * 2 * row + rows_k * 2 * row
    return flops, moved


def work(case):
    kind = case["kind"]
    heads = case.get("heads", 1)
    row = DIM * 2
    if kind == "dense":
        bh = case["batch"] * heads
        pairs = _causal_pairs(case["seq_q"], case["seq_k"]) if case["causal"] else case["seq_q"] * case["seq_k"]
        flops, moved = _attention(bh * pairs, bh * case["seq_q"], bh * case["seq_k"], case["backward"])
    elif kind == "ring":
        c, n = case["chunk"], case["rank"] + 1
        flops, moved = _attention(heads * (_causal_pairs(c, c) + (n - 1) * c * c), heads * c, heads * c * n, True)
    elif kind in ("sparse", "stream"):
        if kind == "sparse":
            table, block, backward = _mask(case["pattern"], case["blocks"]), case["block"], case["backward"]
        else:
            table, block, backward = masks.config_streaming_shard(case["q_blocks"], case["k_blocks"], case["window"]), 512, False
        full, diag = masks.block_counts(table)
        pairs = full * block * block + diag * (block * (block + 1) // 2)
        used = int(table.any(0).sum())                  # key blocks that anybody attends
        flops, moved = _attention(heads * pairs, heads * table.shape[0] * block, heads * used * block, backward)
    elif kind == "fused":
        nq, nk = heads * case["rows"] * case["chunk"], heads * case["cols"] * case["chunk"]
        flops, moved = _attention(nq * case["cols"] * case["chunk"], nq, nk, True)
        moved += case["peers"] * nq * (2 * row + 4)     # the peers' O, LSE and dQ
    else:
        table, rate = _mask(case["pattern"], case["blocks"]), case["block"] // TILE
        full, diag = masks.block_counts(table)
        lines = 2 * case["blocks"] * rate
        flops, moved = 0.0, table.size + 10 * 0.9 * (full * rate * rate + diag * (rate * (rate + 1) // 2)) + 8 * lines
    return {"bytes": float(moved), "flops": float(flops)}


def tolerance(case):
    if case["kind"] == "plan":
        return "exact"
    # bf16 products and results with fp32 accumulation: two bf16 roundings (P or dS, and the result)
    return {"rel": 1e-2, "max": 0.25}
