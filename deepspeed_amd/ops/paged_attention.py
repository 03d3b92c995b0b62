"""Attention over the paged KV pool (reference:
inference/v2/kernels/ragged_ops/blocked_flash). The kernels read the
PagedKVCache pool through its block lists: the padded [n, Hkv, L, D] views are
never materialized, be the step single-token decoding, a portion of a prompt or
both (csrc/paged_attention.hip)."""

import itertools
import math
from dataclasses import dataclass
from typing import List, Optional

import numpy as np
import torch

from . import _loader
from ._loader import get_ext

# Workgroups wanted in flight: four waves each, two to three to a CU of 256. More splits
# than that only add partial results to write and merge.
WORKGROUPS = 1024
# Where they are known, splits fill whole rounds of the workgroups that the 256 CUs
# hold, three each of one tile of columns: a few more would begin when the others end,
# and read alone (us, 8 key heads, some 1024 of them / at most a round: 32 x 2000 59.6
# / 55.8, 8 x 16000 108.1 / 98.2, 16 x 8000 107.8 / 98.9, 40 x 3000 100.9 / 94.2). Of two
# tiles two each, two rounds (24 of 1000 and 200 rows 47.8 / 42.7, 29 of 2000 and 100
# rows 68.0 / 64.5). With less than KEYS keys each, two a CU: the rest merges longer
# than it reads (1 x 16000 27.0 / 21.1, 64 x 500 34.9 / 30.9, 15 of 200 and 250 rows
# 23.9 / 19.5).
ROUND, FEWER, KEYS = {1: 768, 2: 1024}, 512, 384
# But WORKGROUPS tiles and more stay whole, however their last round is filled (over 257
# steps of two tiles of columns, splits that fill it 1.05 of the time, 1.36 at worst; 93
# rows behind 382 beside 9 of as many, 32 key heads 50 / 39 us). And where rounds of two
# tiles' workgroups, as long as the longest of them, hold less than 0.7 of what they
# could, such as evenly long histories that do not fit in twice, parts of more than LONG
# keys are cut for WORKGROUPS if that is less by this measure (65 of 4600 steps, 0.91 of
# the time, 1.01 at worst; from 1024 keys on 91, 1.08 at worst; 319 rows behind 16000
# beside 2 of as many 605 / 482).
LONG = 2048
# Keys of the shortest split: one tile of 32 for each of a workgroup's waves.
MIN_SPLIT = 128
# Up to FEWER workgroups of whole histories are cut by what the parts would take
# (``_cost``, ns): for workgroups of ROOMS in all, up to the rounds above, or not at
# all, since a merge costs as much as reading 500 keys (us, 8 key heads, before / now:
# 32 of 2000 in 512 / whole 53.3 / 48.4; 24 of 150 17.0 / 11.3; 3 of 125 10.7 / 6.9; 8
# of 16000 in 768 / 512 92.4 / 91.2). STEP: a workgroup's 128 keys by tiles of columns,
# and for each workgroup a CU holds beside it, of HELD; BYTES a ns. Fitted to 8000 steps
# of 1 to 64 requests, half of them beside a run of up to 256 rows, 1 to 32 key heads:
# 0.90 of the time of the rounds alone, 1.01 of the fastest cut. A run of several rows
# alone keeps the rounds (its attention is 1 to 2% of such a step). So do blocks that
# hold no whole tile, for which a wave asks key by key: fewer parts are as much longer (16
# keys a block, by the rounds / by these: 31 of 1880, 8 key heads 54 / 69 us, 2 of 4541, 32
# key heads 36 / 45).
ROOMS = 64, 128, 192, 256, 384, 512, 768
STEP, HELD, BYTES, MERGE, MERGED = {1: (300, 1100), 2: (100, 1500)}, {1: 3, 2: 2}, \
    7500, 4400, 5
# Items of 128 columns (rows times heads a key head), eight waves of them a CU,
# take steps of runs of BLOCK columns and more each that have BLOCK_WORK columns
# times keys times key heads. us, 32 on 8 heads, tiles of 32 columns and of 128:
# 16 rows behind 4000 23 / 23, 32 behind 1500 19 / 20 and 4000 29 / 26, 64 behind
# 600 19 / 21 and 1500 26 / 25, 256 behind 64 19 / 23 and 600 37 / 30, 1024 behind
# 1500 112 / 82, 2048 behind 4000 445 / 290. Beside decoding requests a launch of
# their own is no gain (24 of 1000 and 200 rows 60 / 75).
BLOCK, BLOCK_WORK, CUS = 64, 1 << 21, 256


def _lines() -> List[int]:
    """As csrc/step_plan.cpp reads them."""
    return [ROUND[1], ROUND[2], FEWER, KEYS, MIN_SPLIT, BLOCK, BLOCK_WORK, CUS,
            WORKGROUPS, LONG, *STEP[1], *STEP[2], HELD[1], HELD[2], BYTES, MERGE,
            MERGED, *ROOMS]


def paged_decode_available(q: torch.Tensor, kpool: torch.Tensor) -> bool:
    return (get_ext() is not None and q.is_cuda
            and q.dtype == torch.bfloat16 and q.size(-1) == 128
            and q.size(1) % kpool.size(1) == 0
            and 1 <= q.size(1) // kpool.size(1) <= 16)


def aligned(x: torch.Tensor) -> torch.Tensor:
    """x as the kernels read it: contiguous, on 16 bytes."""
    x = x.contiguous()
    return x if x.data_ptr() % 16 == 0 else x.clone()


def paged_decode_attention(q: torch.Tensor, kpool: torch.Tensor,
                           vpool: torch.Tensor, block_table: torch.Tensor,
                           lens: torch.Tensor, splits: Optional[int] = None,
                           scale: Optional[float] = None) -> torch.Tensor:
    """q [n, H, 128] bf16; kpool/vpool [nb, Hkv, BS, 128] bf16;
    block_table [n, max_blocks] int32; lens [n] int32 -> o [n, H, 128].
    The lengths stay on the device, so every request is cut into the same
    number of splits; ``StepPlan`` cuts by length."""
    ext = get_ext()
    scale = scale if scale is not None else 1.0 / math.sqrt(q.size(-1))
    if splits is None:
        nw = max(1, q.size(0) * kpool.size(1))
        splits = max(1, min(32, WORKGROUPS // nw))
    return ext.paged_decode(aligned(q), aligned(kpool), aligned(vpool),
                            block_table.contiguous().int(),
                            lens.contiguous().int(), splits, scale)


@dataclass
class StepPlan:
    """One serving step for the kernels: where each new row goes (``dst``) and
    the work items of its attention (``meta``), both on the device."""

    dst: torch.Tensor
    meta: torch.Tensor
    items: int
    runs: int
    merges: int
    any_merge: bool
    nq: int

    @staticmethod
    def rows(slots: List[int], pos: np.ndarray, tables, block_size: int):
        """Pool row (block * block_size + offset) of every new token, and the
        block lists of the step's slots, one after another. A position is to lie
        in its own slot's blocks: the next ones are another request's."""
        used = list(dict.fromkeys(slots))
        lists = [tables[s] for s in used]
        flat = np.fromiter(itertools.chain.from_iterable(lists), np.int32,
                           sum(map(len, lists)))
        first, at = {}, 0
        for s, blocks in zip(used, lists):
            first[s] = at
            at += len(blocks)
        offs = np.array([first[s] for s in slots], np.int64)
        own = np.array([len(tables[s]) for s in slots], np.int64)
        if ((pos < 0) | (pos // block_size >= own)).any():
            raise IndexError("StepPlan: a position outside its slot's blocks")
        dst = flat[offs + pos // block_size].astype(np.int64) * block_size \
            + pos % block_size
        return dst, flat, offs

    @classmethod
    def build(cls, slots: List[int], pos: np.ndarray, tables, block_size: int,
              heads: int, kv_heads: int, device) -> "StepPlan":
        """``slots[i]`` and ``pos[i]``: request slot and position of row i.
        Neighbouring rows of one slot at following positions form a run and
        share the reads of its keys and values."""
        ext = _loader.get_ext()
        args = slots, pos, tables, block_size, heads, kv_heads
        values, items, runs, merges, any_merge, nq, head = _planned(*args) \
            if ext is None else ext.step_plan(
                *args, _lines(), torch.device(device).type == "cuda")
        # in the order of the current stream; from pageable memory the host would
        # wait there for all that the stream still has to do, the whole step before
        # (torch gives the pinned block to nobody else before it is read)
        meta = values.to(device, non_blocking=True)
        return cls(dst=meta[head:], meta=meta, items=items, runs=runs,
                   merges=merges, any_merge=any_merge, nq=nq)


def _rounds(end, n, kv_heads: int):
    """Keys of the longest part, and rounds of two tiles' workgroups."""
    return int((-(-end // n)).max()), -(-int(n.sum()) * kv_heads // FEWER)


def _parts(end, n, grain: int):
    """Parts of each tile in whole steps, and keys of a part."""
    step = -(-(-(-end // n)) // grain) * grain
    return -(-end // step), step


def _cost(end, n, kv_heads: int, nq: int) -> int:
    """ns that the tiles take in n parts each."""
    n, step = _parts(end, n, 32)
    count, total = int(n.sum()) * kv_heads, int(end.sum()) * kv_heads
    longest = -(-int(np.minimum(step, end).max()) // 128)
    room = HELD[nq] * CUS
    each = STEP[nq][0] + STEP[nq][1] * min(HELD[nq], -(-count // CUS))
    ns = max(longest * each, total * 512 // BYTES)
    if count > room:    # behind one another
        ns = max(ns, (total + 64 * count) // 128 * each // room
                 + 5 * longest * each // 8)
    return ns + (MERGE + MERGED * count if (n > 1).any() else 0)


def _planned(slots, pos, tables, block_size: int, heads: int, kv_heads: int):
    """``step_plan`` of csrc/step_plan.cpp, for a host without the extension."""
    T = len(slots)
    if T < 1 or pos.shape != (T,) or block_size < 1 or not 1 <= kv_heads <= heads:
        raise ValueError("StepPlan: a step of rows, each with its position")
    dst, flat, offs = StepPlan.rows(slots, pos, tables, block_size)
    sl = np.asarray(slots)
    cut = np.flatnonzero((sl[1:] != sl[:-1]) | (pos[1:] != pos[:-1] + 1))
    row0 = np.concatenate(([0], cut + 1))
    m = np.diff(np.append(row0, T))
    kv_len = pos[row0] + m
    runs = np.stack([row0, m, kv_len, offs[row0]], 1)
    G = heads // kv_heads
    # two tiles of 16 columns share the loads of a key tile where runs are
    # long enough, eight where they are longer
    nq = 2 if int(m.max()) * G > 16 else 1
    if int(m.min()) * G >= BLOCK and kv_heads * G * int(
            (m * (kv_len - m // 2)).sum()) >= BLOCK_WORK:
        nq = 8
    width = 16 * nq
    tiles = -(-m * G // width)
    run_of = np.repeat(np.arange(len(m)), tiles)
    tile = np.arange(len(run_of)) - np.repeat(np.cumsum(tiles) - tiles,
                                              tiles)
    tok = np.minimum((tile + 1) * width, m[run_of] * G) - 1
    end = kv_len[run_of] - m[run_of] + tok // G + 1
    # split long histories until the chip is full
    grain = 32
    if nq == 8:
        # the longest first; at most one round of workgroups, steps of 128
        order = np.argsort(-end, kind="stable")
        run_of, tile, end = run_of[order], tile[order], end[order]
        room, per, grain = CUS // kv_heads, int(end[0]), MIN_SPLIT
        if len(end) < room:
            per = max(MIN_SPLIT, int(end.sum()) // room)
            while per < end[0] and (-(-end // per)).sum() > room:
                per += MIN_SPLIT
        n = -(-end // per)
    elif len(end) * kv_heads >= WORKGROUPS:
        n = np.ones_like(end)
    else:
        total, full = int(end.sum()), ROUND[nq]
        if total * kv_heads < KEYS * full:
            full = FEWER
        room = -(-len(end) * kv_heads // full) * full // kv_heads
        # half a split more for each tile, where it ends unevenly
        per = max(MIN_SPLIT, total // max(1, room - len(end) // 2))
        n = -(-end // per)
        while n.sum() > max(room, len(end)):
            per += per // 16
            n = -(-end // per)
        if block_size % 32 == 0 and len(end) * kv_heads <= FEWER and (
                nq == 1 or len(m) > 1):
            n = np.ones_like(end)
            least = _cost(end, n, kv_heads, nq)
            for r in ROOMS:
                per = max(MIN_SPLIT, -(-total * kv_heads // r))
                other = -(-end // per)
                if r > full or int(other.sum()) > room:
                    continue
                ns = _cost(end, other, kv_heads, nq)
                if ns < least:
                    least, n = ns, other
        elif nq == 2:
            longest, rounds = _rounds(end, n, kv_heads)
            if rounds > 1 and longest > LONG and \
                    10 * total * kv_heads < 7 * rounds * FEWER * longest:
                other = -(-end // max(MIN_SPLIT, total * kv_heads // WORKGROUPS))
                if math.prod(_rounds(end, other, kv_heads)) < rounds * longest:
                    n = other
    n, step = _parts(end, n, grain)
    of = np.repeat(np.arange(len(end)), n)
    first = np.cumsum(n) - n
    part = np.arange(len(of)) - first[of]
    lo = part * step[of]
    hi = np.minimum(lo + step[of], end[of])
    hi = np.where(n[of] == 1, -hi, hi)
    items = np.stack([run_of[of], tile[of], lo, hi], 1)
    merges = np.stack([first, n], 1)
    meta = np.concatenate([items.ravel(), runs.ravel(), merges.ravel(), flat,
                           dst])
    return torch.from_numpy(meta.astype(np.int32)), len(items), len(runs), \
        len(merges), bool((n > 1).any()), nq, len(meta) - T


def paged_append(plan: StepPlan, q, k, v, kpool, vpool, cos=None, sin=None,
                 positions=None, seq: int = 1):
    """Write the step's new rows k, v [T, Hkv, 128] into the pool; with cos and
    sin tables, after the rotary embedding of k, and return that of q [T, H,
    128] (positions [T] int32, or row t at t % seq)."""
    return get_ext().paged_append(q, k, v, kpool, vpool, plan.dst, cos, sin,
                                  positions, seq)


def paged_attention(plan: StepPlan, q, kpool, vpool,
                    scale: Optional[float] = None):
    """q [T, H, 128] over the pool, each row up to its own position."""
    scale = scale if scale is not None else 1.0 / math.sqrt(q.size(-1))
    return get_ext().paged_rows(q, kpool, vpool, plan.meta, plan.items,
                                plan.runs, plan.merges, plan.any_merge,
                                plan.nq, scale)
