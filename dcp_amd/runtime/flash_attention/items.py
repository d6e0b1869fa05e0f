"""The work items of a forward launch whose rows are shorter than their blocks (``dcp_attn_fwd_items``).

An item is 128 queries of a row and one head.  The kernel can count them from the block size alone, but a row
shorter than its block then has items without queries, and each costs a workgroup a ticket and a chain of table
reads.  Forward (us) without and with a table of the items there are, by the share of them: 0.37 (4476 tokens in
sequences of 290, blocks of 1024, 8 heads of size 64) 31.6 / 13.9; 0.52 (3477 tokens, 16 heads) 32.1 / 16.8; 5323
tokens in sequences of 67 in two partials, 40 heads, 76.9 / 44.9; 0.87 (5269 tokens, 40 heads) 149.9 / 149.6; 0.98
(12678 tokens, 8 heads) between 100.2 / 103.5 and 95.9 / 94.7.
"""

from __future__ import annotations

from math import gcd
from typing import Optional, Sequence

import numpy as np

N_XCD = 8
MAX_SHARE = 0.8  # of the blocks' tiles: with more of them than that in use the table does not pay
MAX_TILES_WITHOUT_QUEUE = 64  # per slot


def deal_to_xcds(row: np.ndarray, n_kv_heads: int) -> np.ndarray:
    """The order of items of rows ``row`` (rows' items together, rows in the order they should start in), as a
    permutation.  Items go to the eight XCDs in turn, ``n_kv_heads`` streams each; the items of a row read the same
    K and V, so that they take positions that one XCD (one L2) serves, while the rows are dealt to the
    XCDs forth and back."""
    lanes = N_XCD // gcd(N_XCD, n_kv_heads)
    n = len(row)
    if lanes == 1 or n == 0:
        return np.arange(n)
    starts = np.flatnonzero(np.concatenate(([True], row[1:] != row[:-1])))
    turn = np.arange(len(starts)) % (2 * lanes)
    lane = np.repeat(np.where(turn < lanes, turn, 2 * lanes - 1 - turn), np.diff(np.append(starts, n)))
    by_lane = np.argsort(lane, kind="stable")
    counts = np.bincount(lane, minlength=lanes)
    place = np.empty(n, dtype=np.int64)  # of an item among its lane's
    place[by_lane] = np.arange(n) - np.repeat(np.cumsum(counts) - counts, counts)
    return np.argsort(place * lanes + lane, kind="stable")


def pays(seqlens_q: Sequence[int], block_size: int, n_heads: int, n_slots: int, tile: int = 128) -> bool:
    """Whether few enough of the tiles that the blocks have room for hold queries, and not all of them find a
    workgroup slot at once (where they do, the table is only one more thing to read: 773 tokens of 8 heads
    in blocks of 1024, 9.4 us without and 9.5 with it)."""
    used, room = sum(-(-n // tile) for n in seqlens_q), len(seqlens_q) * -(-block_size // tile)
    return 0 < used <= MAX_SHARE * room and room * n_heads > n_slots


def one_workgroup_each(seqlens_q: Sequence[int], seqlens_kv: Sequence[int], n_heads: int, n_slots: int, tile: int = 128) -> bool:
    """Whether a launch of more items than workgroup slots starts a workgroup for every item, instead of one per slot
    that takes item after item from a queue.  The queue wins by what it takes out of the gaps between workgroups,
    some 5 % of the launch, and costs a kernel that clears its counters, 4-5 us.  Forward (us) with and
    without it, by key tiles (64) per slot: 36 and 27 (two launches; 15480 tokens, 8 heads) 183 / 170; 43 (12678
    tokens, 8 heads) 103 / 96; 44 (18701 tokens) 76 / 65; 53 and 41 (two; 12926 tokens, size 64) 145 / 129; 53
    (5323 tokens, 40 heads of 64) 56.9 / 44.0; 56 (7604 tokens, 40 heads) 114 / 109; 98 (5269 tokens, 40 heads) 149 /
    152; 103 (16384 tokens, 16 heads) 197 / 199; 122 (28012 tokens, 32 heads) 348 / 363; 183 (32768 tokens, 8
    heads) 340 / 356; 2297 (65536 tokens, 32 heads) 3762 / 3933.  The line is on the low side: of ten launches of 65
    to 102 tiles per slot one is better off with the queue (78: 153.9 / 156.5), one indifferent (93) and eight are
    better off without it (65: 65.9 / 48.6; 74: 158.6 / 153.2; 82: 101.6 / 85.7; 85: 178.5 / 175.1; 98: 197.5 / 191.3;
    102: 134.8 / 123.6).  Tiles are counted from the rows' keys: under a window or a shared prefix a row sees a part
    of them, and such launches keep the queue at less work than the line says."""
    items = [-(-n // tile) for n in seqlens_q]
    return (sum(items) * n_heads > n_slots
            and sum(n * -(-k // 64) for n, k in zip(items, seqlens_kv)) * n_heads <= MAX_TILES_WITHOUT_QUEUE * n_slots)


def forward_items(seqlens_q: Sequence[int], seqlens_kv: Sequence[int], n_kv_heads: int, tile: int = 128,
                  parts: Optional[np.ndarray] = None) -> np.ndarray:
    """The table: int32 ``[items, 4]``.  ``parts``: the entries of ``fwd_parts.split_rows``; else the rows, the
    ones with the most keys first."""
    if parts is None:
        order = np.argsort(-np.asarray(seqlens_kv, dtype=np.int64), kind="stable")
        parts = np.stack([order, 0 * order, 0 * order + 1, 0 * order], axis=1)
    tiles = -(-np.asarray(seqlens_q, dtype=np.int64)[parts[:, 0]] // tile)
    entry = np.repeat(np.arange(len(parts)), tiles)
    # a row's last queries first: with a causal mask they see the most keys
    q_tile = np.repeat(np.cumsum(tiles), tiles) - 1 - np.arange(len(entry))
    order = deal_to_xcds(entry, n_kv_heads)
    part = parts[entry[order]]
    return np.stack([part[:, 0], q_tile[order], part[:, 1] + (part[:, 2] << 16), part[:, 3]], axis=1).astype(np.int32)
