"""Which rows of a forward launch are split along their keys (``dcp_attn_fwd_parts``).

A work item of the forward kernel -- 128 queries of one (row, head) -- walks its key tiles one after
the other.  A launch whose items all find a workgroup slot at once lasts as long as its longest item,
however idle the device is: 5120 tokens of 8 heads (352 items of 4 to 32 tiles on 512 slots, head size
64) take 31 us, and 26 in parts of up to 16 tiles, 5 of them for the kernel that adds those.
"""

from __future__ import annotations

from typing import List, Optional, Sequence, Tuple

import numpy as np

TILE = 64  # keys per step of the kernel
MIN_SHARE = 8  # tiles: a shorter part is mostly prologue


def share_of_a_part(tiles: Sequence[int], items_per_row: int, n_slots: int) -> Optional[int]:
    """How many key tiles a part takes, or None where nothing is split.  The shortest parts that are all
    on the device at once; if the rows alone are more than it holds, parts of the launch's mean work per
    slot (an item longer than that would end after all the others).  Partials and the kernel that adds
    them cost about as much as eight tiles, so the longest row has to get shorter by more than that.  (``tiles`` are
    counted from the rows' keys, whatever the mask leaves of them to see.)"""
    longest = max(tiles, default=0)
    share = max(MIN_SHARE, -(-sum(tiles) * items_per_row // n_slots))
    if len(tiles) * items_per_row <= n_slots:
        while share < longest and sum(-(-t // share) for t in tiles) * items_per_row > n_slots:
            share += 1
    return share if longest > share + MIN_SHARE and 2 * longest >= 3 * share else None


def split_rows(seqlens_kv: Sequence[int], items_per_row: int, n_slots: int) -> Optional[Tuple[np.ndarray, np.ndarray, int]]:
    """``(parts, splits, number of partials)`` of ``dcp_attn_fwd_parts``, longest parts first, or None."""
    tiles = [-(-n // TILE) for n in seqlens_kv]
    share = share_of_a_part(tiles, items_per_row, n_slots)
    if share is None:
        return None
    entries: List[Tuple[int, int, int, int]] = []
    splits: List[Tuple[int, int, int, int]] = []
    n_partials = 0
    for row, n in enumerate(tiles):
        parts = max(1, -(-n // share))
        entries += [(row, i, parts, n_partials if parts > 1 else 0) for i in range(parts)]
        if parts > 1:
            splits.append((row, parts, n_partials, 0))
            n_partials += parts
    entries.sort(key=lambda e: -(tiles[e[0]] / e[2]))
    return np.asarray(entries, dtype=np.int32), np.asarray(splits, dtype=np.int32), n_partials
