"""How many programs share the kv blocks of a pair of q blocks (SYN_ATTN_SPLIT_KV).

A workgroup of the paired kernel fills a compute unit and takes two q blocks, so a table with few of them leaves most
of the chip idle however long its kv range is.  Cut into parts, every pair's kv blocks are spread over several programs
whose sums are added up in 32 bits at the end.  Host logic on plain integers, like `work_plan`.

Two kinds of tables can be cut:

* consumer tables whose waves all list the same (z, h, q) ranges (the all-gather table): the parts are cut out of the kv
  blocks of all waves in a row, in wave order; or the blocks are dealt to the parts one by one, and a second kernel adds the
  parts up (SYN_ATTN_SPLIT_DEAL), for tables that would otherwise be single tiles;
* producer tables that visit every pair of q blocks once (attention that feeds an exchange), causal or not.
"""

from __future__ import annotations

from typing import Dict, NamedTuple, Optional, Sequence

BLOCK = 128
MAX_WAVES = 256           # wave-table rows that the kernel holds in LDS
MAX_PARTS = 16
MAX_SLOTS = 1024          # partial results in memory at a time: 136 KB each
# Microseconds, from kernel traces (256 programs of 8 blocks and three steps 66, 192 of 12 blocks and two steps 68, 256 of
# 16 blocks and one step 80): a kv block of a pair, what a segment costs beyond its blocks (launch, Q, first fills,
# epilogue), and a step of the tree that adds the parts (136 KB stored, handed over and loaded).
BLOCK_US, SEGMENT_US, STEP_US = 3.6, 14.0, 8.0
# The same where the blocks are dealt: a kv block on a nearly idle chip and what it takes longer where all units are busy, a
# segment, and the second kernel (its launch, and 136 KB of every part stored and loaded; 256 parts 6.8 us, 16 4.1).
# Measured: 32 pairs of 64 blocks as 1, 2, 4, 7, 8 parts 201, 112, 69, 54 and 51 us, 48 pairs of 48 as 2, 4, 5 90, 59 and 55.
DEAL_BLOCK_US, DEAL_FULL_US, DEAL_SEGMENT_US, DEAL_ADD_US, DEAL_ADD_FULL_US = 2.8, 0.9, 13.0, 4.0, 5.0
DEAL_BURST_US, DEAL_BURST_BLOCK_US = 20.0, 2.4         # 200 programs of 4 blocks 44 us, 154 of 2 36, 84 of 2 30
# Tiles that take less than the two launches of a cut table, with what lies around them, stay single.
DEAL_HOST_US = 24.0
MERGE_US = 5.0
MIN_GAIN_US = 10.0        # (the words and slots of the parts cost the host 3 us a launch, which small ones wait for)
RESERVED_UNITS = 32       # compute units that launches which wait leave to the copies that raise their flags
# Units that a producer does not count on: kernels that wait for its flags, one workgroup per side stream of an exchange, each
# keep a unit from a workgroup that wants all registers, and a program too many for its XCD costs a round.  128 pairs
# of 32 blocks as 256 programs: 85 us alone, 133 beside one such kernel; as single tiles, which share units with it, 96 and 95.
EXCHANGE_UNITS = 16


class KvSplit(NamedTuple):
    chain: bool           # parts of all waves in a row, else of the one visit
    pairs: int
    parts: int            # programs per pair
    blocks: int           # kv blocks per part

    @property
    def programs(self) -> int:
        return self.pairs * self.parts


def _steps(parts: int) -> int:
    return (parts - 1).bit_length()


def _deal_us(pairs: int, parts: int, blocks: int, units: int, burst: bool = True) -> float:
    """What `pairs` of `blocks` kv blocks take, dealt to `parts` programs each (`burst`: these are all the blocks there are)."""
    programs = pairs * parts
    share = min(programs / units, 1.0)
    each = -(-blocks // parts)
    us = -(-programs // units) * (each * (DEAL_BLOCK_US + DEAL_FULL_US * share) + DEAL_SEGMENT_US)
    if parts > 1 and burst:              # the sums of short parts go to memory all at once
        us += share * max(DEAL_BURST_US - DEAL_BURST_BLOCK_US * each, 0.0)
    return us + (DEAL_ADD_US + DEAL_ADD_FULL_US * programs / units if parts > 1 else 0.0)


def plan_kv_split(wave_offsets: Sequence[Sequence[int]], wave_sizes: Sequence[Sequence[int]], cum_wave_sizes: Sequence[int],
                  signal_offsets: Sequence[int], *, causal: bool, producer: bool, units: int,
                  always: bool) -> Optional[KvSplit]:
    """The split for these tables on `units` compute units, or None where they cannot be cut or gain nothing.

    `always`: the launch would otherwise take the kernel with one tile per program (uncut pairs may beat that too); else
    it would chain the uncut pairs, and None means that they stay whole."""
    if len(cum_wave_sizes) > MAX_WAVES or (causal and not producer):
        return None
    waves = _real_waves(wave_offsets, wave_sizes, cum_wave_sizes, causal=causal, producer=producer)
    if not waves:
        return None
    return _split_visits(waves, causal, units) if producer else _split_runs(waves, signal_offsets, units, always)


def plan_kv_deal(wave_offsets: Sequence[Sequence[int]], wave_sizes: Sequence[Sequence[int]], cum_wave_sizes: Sequence[int],
                 signal_offsets: Sequence[int], *, units: int) -> Optional[KvSplit]:
    """The split of a consumer's tables that `plan_kv_split` leaves to the kernel with one tile per program, as blocks that are dealt
    to the parts: there a late chunk is looked at as if its blocks were one part's, here as the parts share it.  (Tables that
    both would cut stay with the parts in wave order: a part that meets other blocks first rounds its probabilities against
    another running maximum, and the results of tables that were always cut do not change.  48 pairs of 48 blocks take 73
    us dealt and 79 in wave order.)"""
    if len(cum_wave_sizes) > MAX_WAVES:
        return None
    waves = _real_waves(wave_offsets, wave_sizes, cum_wave_sizes, causal=False, producer=False)
    return _split_dealt(waves, signal_offsets, units) if waves else None


def _real_waves(wave_offsets, wave_sizes, cum_wave_sizes, *, causal: bool, producer: bool):
    """The waves in front of the padding, None where they cannot be cut."""
    waves, align = [], 2 * BLOCK if causal else BLOCK
    for cum, off, size in zip(cum_wave_sizes, wave_offsets, wave_sizes):
        if cum == 0:
            break
        if not producer and waves and (off[:3] != waves[0][0][:3] or size[:3] != waves[0][1][:3]):
            return None
        if min(size) <= 0 or min(off) < 0 or size[2] % (2 * BLOCK) or size[3] % BLOCK or off[2] % align or off[3] % align:
            return None
        waves.append((off, size))
    return waves


def _split_runs(waves, signal_offsets: Sequence[int], units: int, always: bool) -> Optional[KvSplit]:
    size = waves[0][1]
    pairs = size[0] * size[1] * size[2] // (2 * BLOCK)
    lengths = [s[3] // BLOCK for _, s in waves]
    total = sum(lengths)
    # Programs that wait hold their compute unit with all its registers (eight wavefronts of 256), so that nothing else runs
    # there, a copy kernel that raises the flags among them.  Uncut pairs in fewer programs than units leave some free, and
    # the kernel with one tile per program room beside it however many tiles wait (two wavefronts of 232 registers per SIMD
    # of 512): what takes the place of either leaves units free, too, and from the start - with 256 programs of which 32 have
    # nothing to wait for the copies start when those end (8 heads x 1024 rows, eight chunks of 1024 that copies of 16
    # workgroups bring: 178 us, with 224 programs 148, single tiles 158; with 20 us between the copies 320, 290, 272).
    flagged = [n for n, signal in zip(lengths, signal_offsets) if signal >= 0]
    room = (always or pairs < units) and bool(flagged)
    best, best_us, whole_us = None, None, None
    for parts in range(1, min(MAX_PARTS, total) + 1):
        programs = pairs * parts
        if pairs * (parts - 1) > MAX_SLOTS or (room and (always or parts > 1) and programs > units - RESERVED_UNITS):
            continue
        # What is left to do when the last chunk arrives late: its blocks, on the one part of a pair that has them, and the
        # steps whose other sides are long there, against one round of its tiles.  (8 heads x 1024 rows, a chunk of 8 blocks
        # every 10 us: as 7 parts 41 us behind the last flag, as tiles 25; 2 heads, 16 blocks, as 16 parts 49 and 40.)
        if always and flagged and (min(-(-total // parts), flagged[-1]) * BLOCK_US + SEGMENT_US + 2.0 * _steps(parts) >
                                   _tiles_us(2 * pairs, flagged[-1], units)):
            continue
        us = -(-programs // units) * (-(-total // parts) * BLOCK_US + SEGMENT_US + STEP_US * _steps(parts))
        whole_us = whole_us or us
        if best is None or us < best_us:
            best, best_us = parts, us
    if always:
        tiles = 2 * pairs * len(waves)
        # visits to a q block that end at the same time are merged one after the other
        merges = min(len(waves), units // pairs) - 1 if tiles <= 2 * units else 0
        tiles_us = _tiles_us(tiles, -(-total // len(waves)), units) + MERGE_US * merges
        if best is None or best_us >= tiles_us:
            return None
        # Whole pairs that leave units idle (135 of 28 blocks 102 us, as tiles 89), or whose gain is within what the two
        # models are off (560 of 22 blocks 259 us, as tiles 225).  Over 1000 tables drawn anew (500 of them producers') four
        # lose more than 3 %, the most 7 % (324 pairs of 28 blocks), and the medians gain 20 to 39 %.
        if best == 1 and (8 * pairs < 7 * units or 1.05 * best_us >= tiles_us):
            return None
    elif best_us > min(0.85 * whole_us, whole_us - MIN_GAIN_US):
        return None
    return KvSplit(True, pairs, best, -(-total // best))


def _split_dealt(waves, signal_offsets: Sequence[int], units: int) -> Optional[KvSplit]:
    size = waves[0][1]
    pairs = size[0] * size[1] * size[2] // (2 * BLOCK)
    lengths = [s[3] // BLOCK for _, s in waves]
    total = sum(lengths)
    tiles = 2 * pairs * len(waves)
    merges = min(len(waves), units // pairs) - 1 if tiles <= 2 * units else 0          # as in _split_runs
    tiles_us = _tiles_us(tiles, -(-total // len(waves)), units) + MERGE_US * merges
    if tiles_us < DEAL_HOST_US:
        return None
    flagged = [n for n, signal in zip(lengths, signal_offsets) if signal >= 0]
    last_us = _tiles_us(2 * pairs, flagged[-1], units) if flagged else 0.0
    best, best_us = None, None
    for parts in range(1, min(MAX_PARTS, total) + 1):
        programs = pairs * parts
        if (parts > 1 and programs > MAX_SLOTS) or (flagged and programs > units - RESERVED_UNITS):
            break
        us = _deal_us(pairs, parts, total, units)
        # What is left to do when the last chunk arrives late - the share of a part and the second kernel - against one round
        # of its tiles: where that takes longer, the launch has to gain as much with every chunk there.
        if flagged:
            us += max(_deal_us(pairs, parts, flagged[-1], units, burst=False) - last_us, 0.0)
        if best is None or us < best_us:
            best, best_us = parts, us
    # Whole pairs that leave units idle (135 of 28 blocks 102 us, as tiles 89), and a gain within what the two models are off (75
    # of 172 as two parts 295 and 277).
    if best is None or (best == 1 and 8 * pairs < 7 * units) or 1.05 * best_us >= tiles_us:
        return None
    return KvSplit(True, pairs, best, -(-total // best))


def _split_visits(waves, causal: bool, units: int) -> Optional[KvSplit]:
    if len(waves) > 64:
        return None
    by_rows = sorted((off[2], off[2] + size[2], i) for i, (off, size) in enumerate(waves))
    for at, (_, end, i) in enumerate(by_rows):  # every pair of q blocks in one wave only
        (za, ha, *_), (nza, nha, *_) = waves[i]
        for start, _, j in by_rows[at + 1:]:
            if start >= end:
                break
            (zb, hb, *_), (nzb, nhb, *_) = waves[j]
            if za < zb + nzb and zb < za + nza and ha < hb + nhb and hb < ha + nha:
                return None
    walks: Dict[int, int] = {}                  # pairs that walk so many kv blocks
    for off, size in waves:
        for q in range(0, size[2] // BLOCK, 2):
            walked = size[3] // BLOCK
            if causal:
                walked = max(min(walked, off[2] // BLOCK + q + 2 - off[3] // BLOCK), 0)
            walks[walked] = walks.get(walked, 0) + size[0] * size[1]
    longest, pairs = max(walks), sum(walks.values())
    best, best_us = None, None
    tile_units, units = units, units - EXCHANGE_UNITS
    for parts in range(1, min(MAX_PARTS, max(longest, 1)) + 1):
        if pairs * (parts - 1) > MAX_SLOTS or (len(walks) > 1 and parts > 1 and pairs * parts > units):
            break
        blocks = max(-(-longest // parts), 1)
        one = blocks * BLOCK_US + SEGMENT_US + STEP_US * _steps(parts)
        # equal parts run in rounds; unequal ones (a causal mask) fill each other's gaps but for the last one's length
        if len(walks) == 1:
            us = -(-pairs * parts // units) * one
        else:
            whole = sum(count * (n * BLOCK_US + -(-n // blocks) * (SEGMENT_US + STEP_US * _steps(-(-n // blocks))))
                        for n, count in walks.items() if n)
            us = max(one, whole / units + one / 2)
        if best is None or us < best_us:
            best, best_us = (parts, blocks), us
    # Whole pairs lose to the kernel with one tile per program, whose tiles are half as long and share units (288 pairs of 10
    # blocks 96 us against 85, 672 causal ones of up to 32 328 against 258).  So do causal pairs cut into more programs than
    # units (152 pairs of up to 16 blocks, two parts: 87 against 55) and short ones (up to 8 blocks: 42 against 37); 48
    # pairs of up to 24 blocks as four parts take 48 against 67.
    if best[0] == 1 or (longest < 16 if len(walks) > 1 else best_us >= _tiles_us(2 * pairs, longest, tile_units)):
        return None
    return KvSplit(False, pairs, best[0], best[1])


def _tiles_us(tiles: int, blocks: int, units: int) -> float:
    """What the kernel with one tile per program takes, two programs to a unit: a block takes one that has the unit to itself
    2.4 us, two that share it 4.5 (256 tiles of 32 blocks: 85 us, 288 of 13: 54, 1408 of 21: 300).  Full rounds, and the rest as a
    launch of its own: over 815 tables of 16 to 30000 tiles 0.8 to 1.2 of what was measured, where a last round counted
    like a full one came to up to 1.55 just above a round (608 tiles of 22 blocks 163 us, not 214)."""
    full, rest = divmod(tiles, 2 * units)
    us = full * (blocks * 4.5 + 8.0)
    if rest > units:
        us += blocks * 3.5 + 8.0
    elif rest:
        us += blocks * 2.4 + 8.0
    return us
