"""Choice of attention kernel for a step.

The true 32-bit path, and shapes that the matrix-core kernels do not take, run the vector-unit
kernel over all entries. The bfloat16 path sends entries that bring one token to the split-key
decode kernel and portions to the tiled prefill kernel.
"""

from __future__ import annotations

import functools
from typing import Any, Callable, Optional

import numpy as np
import torch

from ..kernels import ops

# From decode steps at batch 1 to 64: two workgroups per compute unit, and at 4K keys at most 16
# runs, were ahead of more of either (the partial results cost a merge that grows with them); a
# request with 32K keys did better with 64 runs than with 16, so the limit grows with the keys.
# Runs of at least 256 keys: with 128, steps at contexts of 512 to 2,048 keys were 0.5 to 2% slower
# at the 1B and 3B sizes and 6% at four kv heads (8 requests of 2,048 keys: 16 runs of 128 keys
# against 8 of 256); with 512 they were 1 to 3% slower again.
WORKGROUPS_PER_UNIT = 2
MIN_KEYS_PER_SPLIT = 256
FEW_SPLITS = 16          # the limit up to 8K keys
KEYS_PER_EXTRA_SPLIT = 512
MAX_SPLITS = 64
ONE_RUN_KEYS, ONE_RUN_KEYS_WIDE, ONE_RUN_KEYS_ALONE = 576, 544, 528   # heads up to 64; wider; wider, one request


def choose_splits(requests: int, kv_head_tiles: int, max_keys: int, units: int = 256) -> int:
    """How many runs to cut each request's keys into for the decode kernel: enough workgroups
    to give every compute unit two workgroups, never runs under 256 keys (reference's rule of the
    same kind: src/dli/model/paged_attention.py:63-74). ``units``: the device's compute units."""
    programs = max(1, requests * kv_head_tiles)
    want = -(-WORKGROUPS_PER_UNIT * units // programs)
    most = max(1, max_keys // MIN_KEYS_PER_SPLIT)
    limit = min(MAX_SPLITS, max(FEW_SPLITS, max_keys // KEYS_PER_EXTRA_SPLIT))
    return max(1, min(want, most, limit))


@functools.lru_cache(maxsize=256)
def one_run_keys(requests: int, q_heads: int, kv_heads: int, head_dim: int, units: int = 256) -> int:
    """Up to how many keys one run serves a recorded step better than two, where every workgroup has a compute unit to itself. It
    then has eight waves, which walk up to 512 keys in one round of what they have on their way; what follows costs more the
    wider the heads are. Passes of 8 steps, two runs and one, ms: 1B sizes, 8 requests, 520 keys 6.52 and 6.48, 568 6.52 and 6.51, 632
    6.54 and 6.58; 135M sizes, 16 requests, 520 6.51 and 6.46, 568 6.55 and 6.55, 600 6.59 and 6.63. Heads of 128: 24 on 8, 4
    requests, 552 14.1 and 14.1; 16 on 2, 8 requests, 536 4.39 and 4.36, 552 4.42 and 4.42. Heads of 96: 16 on 8, 8 requests, 536 3.48
    and 3.49, 552 3.49 and 3.52. Groups whose states do not fit (heads of 128, 16 on one) have four waves: 2 requests, 568 4.21 and
    4.02; 16 requests, 552 5.17 and 4.95.

    One request asks here only where its o projection does not merge the runs (:func:`runs_for_the_product` answers else), with a
    merge in the attention's launch: 135M sizes, 520 5.24 and 5.18, 568 5.23 and 5.24; 24 on 8 of 128, 520 13.1 and 13.7; 16 on
    2, 536 3.81 and 3.84; 16 on one, 552 4.02 and 3.80."""
    workgroups = requests * head_tiles(q_heads, kv_heads)
    if workgroups > units:
        return 0
    alone = requests == 1
    if ops.attention_decode_waves(workgroups, q_heads // kv_heads, head_dim, units) == 4:
        return 0 if alone else ONE_RUN_KEYS
    return ONE_RUN_KEYS if head_dim <= 64 else ONE_RUN_KEYS_ALONE if alone else ONE_RUN_KEYS_WIDE


def planned_splits(requests: int, q_heads: int, kv_heads: int, head_dim: int, max_keys: int, units: int = 256) -> int:
    """:func:`choose_splits` rounded up to a power of two: the coarse form of the rule, for steps
    that are recorded once and replayed for a range of lengths (each distinct answer is a
    recording of its own). Up to :func:`one_run_keys` keys one run."""
    if max_keys <= ONE_RUN_KEYS and max_keys <= one_run_keys(requests, q_heads, kv_heads, head_dim, units):
        return 1
    kv_head_tiles = head_tiles(q_heads, kv_heads)
    splits, coarse = choose_splits(requests, kv_head_tiles, max_keys, units), 1
    while coarse < splits:
        coarse *= 2
    return coarse


def runs_for_the_product(q_heads: int, kv_heads: int, max_keys: int, units: int = 256) -> Optional[int]:
    """Runs of keys in a recorded step of one request whose o projection merges them: about 256 keys each, which eight waves have on
    their way at once, in powers of two; no more workgroups than compute units, since a run is ``q_heads * (4 * head_dim + 8)`` bytes
    (2.4 KB at the 135M sizes, 12.5 at the 3B sizes) that each workgroup of the product reads. None where that makes more runs than the
    product merges: :func:`planned_splits` decides then. Passes of eight steps, ms, with 1, 2, 4, ... runs: 135M sizes, 312
    keys 4.88 and 4.87, 408 5.09 and 4.85, 520 5.17, 4.91 and 4.95, 648 5.53, 5.11 and 4.98, 1,008 (from 2 on) 5.27, 5.05 and 5.11, 2,008
    (from 4 on) 5.39, 5.19 and 5.46; 1B sizes, 520 5.61 and 5.54, 2,008 (from 4 on) 5.78 and 5.64, with 16 5.78; 1.7B sizes, 4,008 (from 4
    on) 9.01, 8.86 and 9.06, 32,008 (from 8 on) 15.9 and 16.4; 3B sizes, 520 13.4, 13.1 and 13.2, 2,008 (from 4 on) 13.8, 13.6 and 14.1.

    So a request alone may have its keys in other runs than the same request among others, and the last bit of a rounding
    differ (as it may between steps of 8 and of 64 requests, whose runs differ too): what a row's sums do not depend on is the
    other rows of a product."""
    want, runs = max(1, (max_keys + 128) // 256), 1
    most = units // head_tiles(q_heads, kv_heads)
    while runs < want and 2 * runs <= most:
        runs *= 2
    return runs if runs <= ops.MERGED_SPLITS else None


# A launch of fewer workgroups than this per compute unit is as long as its longest workgroup, and
# cutting the keys of its longest tiles into runs, each a workgroup, shortens that (one prompt of
# 2,048 tokens at the 1B sizes: 43 -> 33 us a layer); with more, the workgroups queue anyway and
# the cut only costs its merge (3,072 tokens: 62 -> 69 us with room for four a unit). A run is not
# shorter than MIN_RUN_TILES tiles of 32 keys, and a tile has at most MAX_RUNS runs (the kernel's
# limit is asked at the first use).
CUT_BELOW_WORKGROUPS_PER_UNIT = 3
MIN_RUN_TILES = 8
MAX_RUNS = 8
LONE_TILE_COST = 1.5   # a tile of a workgroup alone on its SIMDs, in tiles of a busy compute unit


def runs_of_tiles(key_tiles: np.ndarray, workgroups_per_tile: int, units: int, most: int = MAX_RUNS) -> np.ndarray:
    """Into how many runs each tile of a launch has its keys cut (1: whole; ``key_tiles``: the
    number of 32-key tiles that each query tile walks). While the launch stays under three
    workgroups a compute unit, and the longest workgroup is still what the launch waits for (it
    takes longer than the units' work in all), the tile with the longest run gets one more, as long
    as its runs stay long enough; nothing is cut where that does not make the longest workgroup at
    least 15% shorter (tiles of much the same length and no room for all of them: a large portion on top of
    a long context)."""
    import heapq

    runs = np.ones(key_tiles.size, np.int64)
    spare = CUT_BELOW_WORKGROUPS_PER_UNIT * units // max(1, workgroups_per_tile) - key_tiles.size
    if spare <= 0 or key_tiles.size == 0:
        return runs
    # (Python's own numbers: one of an array's takes five times as long)
    tiles, count = key_tiles.tolist(), [1] * key_tiles.size
    heap = [(-t, i) for i, t in enumerate(tiles)]        # (the tile's longest run, negative)
    heapq.heapify(heap)
    # What a compute unit has to do in all, in tiles of 32 keys of one workgroup. Under a causal
    # mask from the prompt's start, the short tiles' workgroups leave early and the longest runs end
    # alone on their SIMDs, where a tile takes about one and a half times what a full unit needs
    # per tile: cutting stops when the longest run is no longer what the launch waits for. Tiles of
    # much the same length (a portion on top of a long context) all live to the end, and more runs
    # pay until the units are full (512 tokens on 8,192 keys: 155 us whole, 66 with four runs
    # a tile, 57 with six; one prompt of 2,048 tokens: 31.6 us with 21 tiles cut, 33.0 with 32).
    per_unit = float(key_tiles.sum()) * workgroups_per_tile / units
    lone_cost = LONE_TILE_COST if float(key_tiles.mean()) < 0.75 * float(key_tiles.max()) else 2 * LONE_TILE_COST
    while spare > 0:
        longest_run, i = heap[0]
        if -longest_run * lone_cost <= per_unit:
            break   # the launch is as long as its work by now, not as its longest workgroup
        if count[i] >= most or tiles[i] // (count[i] + 1) < MIN_RUN_TILES:
            break   # the longest workgroup cannot get shorter
        count[i] += 1
        spare -= 1
        heapq.heapreplace(heap, (-(-(-tiles[i] // count[i])), i))
    if -heap[0][0] * 20 > max(tiles) * 17:
        return runs
    return np.asarray(count, np.int64)


def round_about(order: np.ndarray, per_round: int) -> np.ndarray:
    """``order`` with every second run of ``per_round`` entries turned round."""
    order = order.copy()
    for r0 in range(per_round, order.size, 2 * per_round):
        order[r0:r0 + per_round] = order[r0:r0 + per_round][::-1].copy()
    return order


class PrefillTiles:
    """The tile list of a step's portions for :func:`ops.attention_prefill`, with what the kernel
    needs for the tiles whose keys are cut (``cut`` None: none are)."""

    def __init__(self, entry: torch.Tensor, q0: torch.Tensor, cut: Optional[torch.Tensor] = None, cut_tiles: int = 0,
                 cut_room: int = 0, cut_buf: Optional[torch.Tensor] = None,
                 cut_count: Optional[torch.Tensor] = None) -> None:
        self.entry, self.q0, self.cut, self.cut_tiles, self.cut_room = entry, q0, cut, cut_tiles, cut_room
        self.cut_buf, self.cut_count = cut_buf, cut_count

    @property
    def tiles(self) -> int:
        return int(self.entry.shape[0])


def list_tiles(q_len: np.ndarray, kv_len: np.ndarray, first_entry: int, rows: int, workgroups_per_tile: int,
               units: int, may_cut: bool) -> tuple[np.ndarray, np.ndarray, Optional[np.ndarray], int, int]:
    """The tiles of entries ``first_entry..`` (``q_len`` new tokens over ``kv_len`` keys each) in the
    order in which the prefill kernel wants them: ``(entry, first query, cut code or None, number of
    cut tiles, most runs of a tile)``. Those that see the most keys come first: workgroups start in the order of the list,
    and under a causal mask a tile's work grows with its place in the request; listed by place, the
    longest workgroups start last and the launch ends with a few of them alone on the device (a
    prompt of 8,192 tokens at the 1B sizes: 521 us a layer by place, 393 us longest first). Within
    the sorted list every second run of as many tiles as give every compute unit one workgroup (a
    tile becomes ``workgroups_per_tile`` workgroups, one per group of query heads) is turned round,
    so that a unit that got a long tile in one round gets a short one in the next. A cut tile is
    listed once per run, each time with its share of the keys."""
    def counted(counts: np.ndarray) -> np.ndarray:   # 0, 1, .. count - 1 of each
        return np.arange(int(counts.sum())) - np.repeat(np.cumsum(counts) - counts, counts)

    of_entry = np.maximum(-(-q_len[first_entry:].astype(np.int64) // rows), 0)
    ent_a = np.repeat(np.arange(first_entry, q_len.size, dtype=np.int32), of_entry)
    q0_a = (counted(of_entry) * rows).astype(np.int32)
    if ent_a.size == 0:
        return ent_a, q0_a, None, 0, 0
    length = q_len[ent_a].astype(np.int64)
    keys = kv_len[ent_a].astype(np.int64) - length + np.minimum(q0_a + rows, length)
    key_tiles = -(-keys // 32)
    runs = runs_of_tiles(key_tiles, workgroups_per_tile, units) if may_cut else np.ones(ent_a.size, np.int64)
    per_round = max(1, units // max(1, workgroups_per_tile))
    cut = runs > 1
    n_cut = int(cut.sum())
    if n_cut == 0:
        order = round_about(np.argsort(-keys, kind="stable"), per_round)
        return ent_a[order], q0_a[order], None, 0, 0
    # the list's entries: a tile once per run, each with its share of the keys
    which = np.repeat(np.arange(ent_a.size), runs)
    run = counted(runs)
    place = np.cumsum(cut) - 1                       # the cut tiles numbered in list order
    code = np.where(cut[which], run | runs[which] << 4 | place[which] << 8, -1)
    share = -(-key_tiles[which] // runs[which])
    order = round_about(np.argsort(-share, kind="stable"), per_round)
    return ent_a[which][order], q0_a[which][order], code[order].astype(np.int32), n_cut, int(runs.max())


def prefill_tiles(ctx: Any, head_dim: int, q_heads: int, kv_heads: int, first_entry: int, device: torch.device,
                  window: int = 0, pieces: Optional["ChunkPieces"] = None) -> PrefillTiles:
    """The tile list of the step's portions for :func:`ops.attention_prefill` (made once per step
    and shape; the buffers of the cut tiles serve every layer of that shape in turn). ``pieces``: of these in place
    of the entries."""
    rows = ops.attention_prefill_tile_rows(head_dim, q_heads, kv_heads)
    units = ops.compute_units(device)
    cut_floats = ops.attention_prefill_cut_floats(head_dim, q_heads, kv_heads)
    # a workgroup takes a tile for 4 * 32 / rows query heads where the kernel's waves share key
    # tiles (heads of 32 and more: the kernel that can also cut a tile's keys), else for one
    per_tile = q_heads * rows // 128 if cut_floats > 0 else q_heads
    may_cut = window == 0 and cut_floats > 0

    def make_lists() -> tuple:
        q_start, kv_len, first = ((ctx.q_start_host, np.asarray(ctx.kv_len_host), first_entry) if pieces is None
                                  else (pieces.q_start_host, pieces.kv_len_host, 0))
        q_len = (q_start[1:] - q_start[:-1]).astype(np.int64)
        ent, q0, code, n_cut, room = list_tiles(q_len, kv_len, first, rows, per_tile, units, may_cut)
        return (*ctx.upload([ent, q0] if code is None else [ent, q0, code]), *([None] if code is None else []), n_cut, room)

    # (the lists do not depend on the head size, which layers of one step may differ in; a cut tile's buffers do)
    shape = ("prefill tiles", rows, per_tile, first_entry, may_cut, 0 if pieces is None else pieces.chunk)

    def make() -> PrefillTiles:
        entry_t, q0_t, code_t, n_cut, room = ctx.step_lists(shape, make_lists)
        if code_t is None:
            return PrefillTiles(entry_t, q0_t)
        return PrefillTiles(entry_t, q0_t, code_t, n_cut, room,
                            torch.empty(n_cut * room * cut_floats, device=device, dtype=torch.float32),
                            torch.zeros(n_cut * q_heads, device=device, dtype=torch.int32))

    return ctx.step_lists((*shape, q_heads, cut_floats), make)


def chunk_pieces(q_start: np.ndarray, kv_len: np.ndarray, first_entry: int, chunk: int) -> tuple[np.ndarray, ...]:
    """The portions ``first_entry..`` of a step under a chunked mask as pieces that are causal by themselves: the rows of an
    entry that lie in one chunk see that chunk's keys and no others. Returns each piece's entry, its first key's position, where its rows
    begin (and the last one's end) and how many keys it has."""
    entry, first_key, begin, keys = [], [], [], []
    for e in range(first_entry, kv_len.size):
        row, end, pos = int(q_start[e]), int(q_start[e + 1]), int(kv_len[e]) - int(q_start[e + 1] - q_start[e])
        while row < end:
            low = pos // chunk * chunk
            n = min(end - row, low + chunk - pos)
            entry.append(e)
            first_key.append(low)
            begin.append(row)
            keys.append(pos + n - low)
            row, pos = row + n, pos + n
    begin.append(int(q_start[-1]))
    return tuple(np.asarray(a, np.int32) for a in (entry, first_key, begin, keys))


class ChunkPieces:
    """:func:`chunk_pieces` of a step on the device, with each piece's pages."""

    def __init__(self, ctx: Any, grp: Any, first_entry: int, chunk: int) -> None:
        entry, first_key, self.q_start_host, self.kv_len_host = chunk_pieces(ctx.q_start_host, np.asarray(ctx.kv_len_host), first_entry, chunk)
        self.chunk = chunk
        width = max(1, -(-int(self.kv_len_host.max()) // ctx.page_size))
        at = np.minimum(first_key[:, None] // ctx.page_size + np.arange(width, dtype=np.int32), grp.block_tables.shape[1] - 1)
        self.q_start, self.kv_len, where = ctx.upload([self.q_start_host, self.kv_len_host, entry[:, None] * grp.block_tables.shape[1] + at])
        self.block_tables = grp.block_tables.view(-1)[where]


# Pairs of a query head's row and a key from which a step's portions take that kernel. Below, the lists of its tiles, which the host makes
# while the step's first kernels wait to be launched, cost as much as it gives. In steps whose attention is narrower than 2,048 the device
# is done sooner and waits for them longer: two thirds more there. Prompts alone, from the call to their logits, us, the kernel for changed
# scores and this one (millions of pairs): 2,048 wide Miberax 1 x 1,600 (39) 4,147 4,072, 2 x 1,300 (52) 5,611 5,502; Rurorax 1 x 1,600 (39)
# 3,301 3,224, 1 x 2,200 (74) 4,180 4,054; Betepel 1 x 1,700 (44) 4,679 4,635, 2 x 1,500 (69) 6,534 6,491; 1,024 wide Miberax 1 x 2,300 (36)
# 3,042 3,096, 4 x 1,150 (40) 4,491 4,554, 4 x 1,400 (60) 4,953 4,958, 3 x 2,000 (92) 5,457 5,351; Rurorax 1 x 2,600 (41) 2,270 2,414, 2 x
# 1,700 (44) 2,632 2,728, 4 x 1,500 (69) 3,759 3,702; Betepel 3 x 1,300 (39) 4,024 4,006, 2 x 2,500 (78) 5,087 5,039.
PLAIN_FROM_PAIRS = 36 << 20
# How many times as many where chunks fill no more than half a tile's rows, which are 32, 64 or 128 for groups of a multiple of four, two
# or one query heads: the rest of a tile is work for nothing, in every chunk, so never. Steps of 41 million pairs, us a layer, by the
# kernel for changed scores and by this one: 32 heads of 64 on 32, chunks of 32 191 270, 48 157 157, 64 100 100, 80 99 80, 96 78 58; of 48,
# 64 84 93, 80 92 73; 24 of 64 on 8, 48 151 152, 64 97 88, 80 98 76; 16 of 64 on 8, 32 101 99, 48 130 94; 32 of 128 on 16, 16 412 523, 32 346
# 288, 48 277 176; 32 of 64 on 8, 16 195 193, 32 168 119. (The host's lists of the pieces, 240 us for 64 tokens each and 480 for 32, aside.)
SHORT_CHUNKS = 1 << 20


def plain_pays(head_dim: int, q_heads: int, kv_heads: int, pairs: int, chunk: int) -> bool:
    """Whether the kernel that shares key tiles is the one for a step's portions of so many pairs, cut into chunks of ``chunk`` (0: not
    cut). Heads of 16 have no such kernel: 32 on 8, 2,048 tokens 91 us by the kernel for changed scores, 101 by theirs."""
    if not ops.attention_prefill_cut_floats(head_dim, q_heads, kv_heads):
        return False
    short = 0 < 2 * chunk <= ops.attention_prefill_tile_rows(head_dim, q_heads, kv_heads)
    narrow = q_heads * head_dim < 2048
    return pairs >= (PLAIN_FROM_PAIRS * 5 // 3 if narrow else PLAIN_FROM_PAIRS) * (SHORT_CHUNKS if short else 1)


def plain_portions(q: torch.Tensor, k_pages: torch.Tensor, v_pages: torch.Tensor, out: torch.Tensor, ctx: Any, cache: Any,
                   q_heads: int, scale: float, *, chunk: int = 0, window: int = 0, keep_first: int = 0) -> bool:
    """The attention of the step's portions by the kernel that shares key tiles through LDS, where a chunked mask or a
    window is all that changes it: under a mask that no row of the step meets, a window that keeps no first positions, or
    chunks of whole pages, whose rows are entries by themselves. False (nothing has run) elsewhere. (The kernel for
    changed scores takes blocks of 64 keys by way of registers, one barrier a block: a prompt of 4,096 tokens in chunks of 2,048, 32
    heads of 64 on 8, 149 us a layer and 74.)"""
    def make() -> tuple:
        grp, nd = ctx.groups[cache.group], ctx.num_decode
        pages, kv_heads, page_size, head_dim = k_pages.shape
        if (tuple(v_pages.shape) != (pages, kv_heads, head_dim, page_size) or scale <= 0.0
                or not ops.attention_mfma_supports(head_dim, page_size, k_pages.dtype)):
            return ()
        new, keys = np.diff(ctx.q_start_host)[nd:].astype(np.int64), np.asarray(ctx.kv_len_host)[nd:].astype(np.int64)
        seen = np.minimum(keys, max(chunk, window)) if chunk or window else keys   # (by the last row, or one in the middle)
        longest = int(keys.max())
        met_chunk, met_window = (n if 0 < n < longest else 0 for n in (chunk, window))
        if not plain_pays(head_dim, q_heads, kv_heads, q_heads * int((new * np.minimum(seen, keys - new // 2)).sum()), met_chunk):
            return ()
        if met_window and (keep_first or met_chunk) or met_chunk % page_size:
            return ()
        if not met_chunk:
            return ctx.q_start, ctx.kv_len, grp.block_tables, prefill_tiles(ctx, head_dim, q_heads, kv_heads, nd, q.device, met_window), met_window
        pieces = ctx.step_lists(("chunk pieces", met_chunk, nd, cache.group), lambda: ChunkPieces(ctx, grp, nd, met_chunk))
        return (pieces.q_start, pieces.kv_len, pieces.block_tables,
                prefill_tiles(ctx, head_dim, q_heads, kv_heads, nd, q.device, 0, pieces), 0)

    if out.dtype != k_pages.dtype:
        return False
    # (asked once a step, also where the answer is no: a step of few tokens waits for its launches, and layers are alike)
    plan = ctx.step_lists(("plain portions", q_heads, tuple(k_pages.shape), tuple(v_pages.shape), cache.group, scale, chunk, window, keep_first), make)
    if not plan:
        return False
    q_start, kv_len, tables, t, met_window = plan
    ops.attention_prefill(q, k_pages, v_pages, out, q_start, kv_len, tables, t.entry, t.q0, q_heads, scale, met_window, t.cut, t.cut_tiles,
                          t.cut_room, t.cut_buf, t.cut_count, top_exact=True)
    return True


def paged_attention(q: torch.Tensor, k_pages: torch.Tensor, v_pages: torch.Tensor, out: torch.Tensor,
                    ctx: Any, grp: Any, q_heads: int, scale: float, window: int = 0,
                    arrival_counters: Optional[Callable[[int], Optional[torch.Tensor]]] = None,
                    planned: Optional[int] = None) -> None:
    """Attention of every row of the step over its request's pages, into ``out``.
    ``arrival_counters(n)``: the caller's ``n`` counters with which the decode kernel merges its
    runs of keys by itself (see ``ops.attention_decode``), or None. ``planned``: the number of
    runs that the mixer promised for this step when it was recorded (``Mixer.decode_plan``)."""
    if ctx.num_tokens == 0:
        return
    _, kv_heads, page_size, head_dim = k_pages.shape
    if not ops.attention_mfma_supports(head_dim, page_size, k_pages.dtype):
        rows = ops.attention_generic_tile_rows(head_dim)
        tile_entry, tile_q0 = ctx.q_tiles(rows)
        ops.attention_generic(q, k_pages, v_pages, out, ctx.q_start, ctx.kv_len, grp.block_tables,
                              tile_entry, tile_q0, q_heads, scale, window)
        return
    nd = ctx.num_decode
    if nd > 0:
        splits, part_o, part_ml = _decode_splits(ctx, nd, q_heads, kv_heads, head_dim, q.device, planned)
        arrivals = None
        if arrival_counters is not None and 1 < splits <= ops.SELF_MERGING_SPLITS:
            arrivals = arrival_counters(nd * kv_heads * (-(-(q_heads // kv_heads) // 16)))
        ops.attention_decode(q[:nd], k_pages, v_pages, out[:nd], ctx.kv_len, grp.block_tables, q_heads,
                             scale, window, splits, part_o, part_ml, arrivals=arrivals)
    if ctx.num_entries > nd:
        t = prefill_tiles(ctx, head_dim, q_heads, kv_heads, nd, q.device, window)
        ops.attention_prefill(q, k_pages, v_pages, out, ctx.q_start, ctx.kv_len, grp.block_tables, t.entry, t.q0,
                              q_heads, scale, window, t.cut, t.cut_tiles, t.cut_room, t.cut_buf, t.cut_count)


def decode_attention_unmerged(q: torch.Tensor, k_pages: torch.Tensor, v_pages: torch.Tensor, ctx: Any, grp: Any,
                              q_heads: int, scale: float, window: int, wanted,
                              planned: Optional[int] = None) -> Any:
    """Attention of a step in which every row is one request's single token, without the kernel
    that merges the runs of keys: ``(splits, part_o, part_ml)`` for the product that merges while
    it loads (``ops.skinny_gemm_merged``), or None (nothing has run) where the step's keys are
    not split or ``wanted(splits)`` says that this product does not take them."""
    _, kv_heads, page_size, head_dim = k_pages.shape
    nd = ctx.num_decode
    if nd != ctx.num_tokens or not ops.attention_mfma_supports(head_dim, page_size, k_pages.dtype):
        return None
    splits, part_o, part_ml = _decode_splits(ctx, nd, q_heads, kv_heads, head_dim, q.device, planned)
    if splits < 2 or not wanted(splits):
        return None
    ops.attention_decode(q[:nd], k_pages, v_pages, None, ctx.kv_len, grp.block_tables, q_heads, scale, window,
                         splits, part_o, part_ml, merge=False)
    return splits, part_o, part_ml


def head_tiles(q_heads: int, kv_heads: int) -> int:
    """Workgroups that one request's token gives the decode kernel per run of keys: a workgroup
    takes up to 16 query heads of one kv head."""
    return kv_heads * -(-(q_heads // kv_heads) // 16)


def step_splits(ctx: Any, nd: int, q_heads: int, kv_heads: int, device: torch.device,
                planned: Optional[int] = None) -> int:
    """Runs of keys for the ``nd`` single-token rows of this step: what was planned when the step
    was recorded, else the rule applied to the step's own lengths."""
    return planned or choose_splits(nd, head_tiles(q_heads, kv_heads), ctx.max_decode_kv_len,
                                    ops.compute_units(device))


def _decode_splits(ctx: Any, nd: int, q_heads: int, kv_heads: int, head_dim: int, device: torch.device,
                   planned: Optional[int] = None):
    splits = step_splits(ctx, nd, q_heads, kv_heads, device, planned)
    part_o = part_ml = None
    if splits > 1:
        part_o = torch.empty(nd * q_heads * splits * head_dim, device=device, dtype=torch.float32)
        part_ml = torch.empty(nd * q_heads * splits * 2, device=device, dtype=torch.float32)
    return splits, part_o, part_ml
