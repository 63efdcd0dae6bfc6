"""GEMM planning: tile shape / split-K choice for the MFMA kernel, plus optional autotune.

The projection GEMMs of a decode step are skinny (M = batch) and of a prefill step fat
(M = batch * prompt). The planner picks, per (M, N, K, epilogue):

* a tile from {64x64, 64x128, 128x128, 128x256, 256x128} sized to M,
* a split-K factor so the grid covers the 256 CUs (cdna_hip_programming.md §5 'Projection
  GEMM at M = 256': choose SPLITK so that tiles * SPLITK ~ 0.5-1x the CU count),
* every GEMM runs on our kernels (no vendor-library backend): decode GEMMs (the hipGraph
  steps) on tiles autotuned at graph capture (on by default; ``DLI_GEMM_AUTOTUNE=0``
  disables it); prefill GEMMs on the one-wave-per-SIMD kernel (gemm4w.h), whose tile and width the
  warmup measures per token bucket (``prefill_candidates``).

Split-K partial slabs live in a grow-only per-device workspace; engines warm every shape
up before hipGraph capture so no allocation happens inside a capture.
"""
from __future__ import annotations

import functools
import math
import os
import threading
import time
from dataclasses import dataclass

import numpy as np
import torch

# tile id -> (BM, BN); 0-4 stage K through 2 LDS buffers, 5-9 are the same tiles with 3
# buffers and one tile kept in flight across the K-step barrier (gemm.hip)
TILES = {0: (64, 64), 1: (64, 128), 2: (128, 128), 3: (128, 256), 4: (256, 128),
         5: (64, 64), 6: (64, 128), 7: (128, 128), 8: (128, 256), 9: (256, 128),
         10: (192, 128), 11: (192, 128), 12: (160, 128),
         # 8 waves / 512 threads (fewer L2 re-reads of A and W at M >= 256)
         13: (256, 256), 14: (256, 128), 15: (128, 256), 16: (256, 128), 17: (128, 256),
         # grid-filling tiles for N = 6144 / 4096 at M = 512
         18: (128, 96), 19: (128, 96), 20: (128, 64), 21: (128, 64),
         # 4 waves, one per SIMD (gemm4w.h): 256 columns, or fewer, or rows of 192 or 320, where they leave
         # less of a round of CUs empty (dense, not biased; gemm4w.hip's shape_of); the rarer epilogues on the
         # 8-phase ping-pong kernel (gemm8p.hip)
         22: (256, 256),
         # 192-wide, 8 waves: N = 6144 is 32 column tiles (fused QKV at M = 512 fills the chip
         # with split-K 2 / 4)
         23: (128, 192), 24: (128, 192), 25: (256, 192),
         # 256x224 ping-pong: N = 28672 (Llama-3 gate/up) at M = 512 = 256 tiles on 256 CUs
         26: (256, 224),
         # 256x128 of the same kernels: N = 4096 at M = 512 with split-K 4
         28: (256, 128),
         # 256x256, 4 waves (one per SIMD), 128x128 wave tiles, accumulators pinned in the AGPR
         # file, at most a workgroup a CU that walks its tiles (gemm4w.h)
         34: (256, 256), 41: (256, 256), 45: (256, 256),
         # 55: the same on tiles of 256, 192 or 160 columns by rounds of the chip, or of other
         # rows as 22; no split-K / grouped
         55: (256, 256)}
# weight-streaming tiles for up to 128 rows (gemm_stream.h): weights nontemporal, K loops turned from
# tile to tile, 3 to 6 stages; (BM, BN, K-tile: a split of K holds whole ones), so kept apart
STREAM_TILES = {60: (32, 32, 256), 61: (32, 128, 64), 62: (32, 64, 256), 63: (64, 128, 64),
                64: (64, 64, 64), 65: (64, 256, 64), 66: (96, 128, 64), 67: (128, 128, 64),
                68: (128, 256, 64), 69: (64, 32, 256), 70: (96, 64, 64), 71: (128, 64, 64),
                72: (128, 32, 128)}
STREAM_MAX_M = 128
# the plan of 256 columns throughout, raced against tile 22's width by rounds in the prefill autotune
PREFILL_4W_TILE = 45
# the persistent 4-wave tile (55) raced too
PREFILL_PERSIST = True
# prefill-sized grouped expert GEMMs (ops.moe_mlp's eager path): the 4-wave kernel on 256 columns, which
# tile 22 takes too where a product is grouped
MOE_PREFILL_TILE = 45
# weight-streaming skinny GEMM (gemm.hip gemv_kernel) for M <= GEMV_MAX_M rows: 16 / 32 output
# rows per workgroup (31 for the SiLU*up gate/up pairing); not an MFMA tile, so kept apart
GEMV_TILES = {30: 16, 31: 32, 32: 16, 33: 32,   # 32 / 33: 4 K-steps in flight per lane, M = 1
              29: 16,   # 29: SiLU*up on the 16-row grid (8 gate + 8 up rows), M <= 4
              56: 4, 57: 8,   # 4 / 8 rows a workgroup, 8 K-steps in flight (not SiLU)
              58: 4, 59: 8}   # SiLU*up pairing (2 + 2 / 4 + 4 rows), 8 K-steps in flight
GEMV_M1_ONLY = (32, 33)
GEMV_MAX_M = 4
# batch-1 decode without split-K reduces (ops.linear_residual, ops.NormedRows): the GEMVs that
# add into the residual (epi "res", full K per workgroup) and the tiles whose prologue applies
# a deferred RMSNorm to their input rows (gemv.hip dli_gemv_fused)
GEMV_RES_TILES = {30: 16, 32: 16, 56: 4, 57: 8}
GEMV_PRO_TILES = {"silu_mul": (29, 31, 33, 58, 59), "splitk": (30, 32, 56, 57),
                  "none": (30, 32, 56, 57)}
GEMV_PRO_M1_ONLY = (32, 33)
DEFER_NORM = os.environ.get("DLI_DEFER_NORM", "1") == "1"
# waves down and across a tile where they are not 2 x 2
TILE_WAVES = {13: (2, 4), 14: (4, 2), 15: (2, 4), 16: (4, 2), 17: (2, 4),
              23: (2, 4), 24: (2, 4), 25: (4, 2),
              26: (4, 2), 60: (2, 1), 66: (1, 4), 68: (2, 4), 69: (4, 1), 72: (4, 1)}


def tile_shape(tile: int):
    """(BM, BN) of an MFMA tile."""
    return STREAM_TILES[tile][:2] if tile in STREAM_TILES else TILES[tile]


def tile_step(tile: int) -> int:
    """The K-tile of an MFMA tile."""
    return STREAM_TILES[tile][2] if tile in STREAM_TILES else 64


def tile_ok(tile: int, epi: str) -> bool:
    """The SiLU*up epilogue pairs 16-column gate/up blocks inside a wave's column range,
    which must therefore be a multiple of 32."""
    if epi == "res":
        return tile in GEMV_RES_TILES
    if epi in ("gelu_erf", "clamp_mul", "relu_mul", "gelu_mul") and tile in (34, 41, 45, 55):
        return epi == "gelu_mul" and tile == 55     # the 4-wave families lack the others
    if tile in (29, 58, 59):
        return epi == "silu_mul"
    if tile in GEMV_TILES:
        return epi not in ("clamp_mul", "relu_mul", "gelu_mul") and (epi != "silu_mul" or tile in (31, 33))
    if epi not in PAIR_EPIS:
        return True
    if tile == 26:              # the straddling gate/up pair meets through LDS
        return True
    bn = tile_shape(tile)[1]
    return (bn // TILE_WAVES.get(tile, (2, 2))[1]) % 32 == 0


# "splitk": a plain GEMM whose fp32 partial slabs feed a fused reduce (ops.linear_add_rmsnorm,
# ops.linear_rope_cache); planned/tuned separately (a non-split winner runs unfused).
EPI = {"none": 0, "f32": 1, "silu_mul": 2, "bias_gelu": 3, "bias": 4, "splitk": 0,
       "slab16": 5, "gelu_erf": 6, "clamp_mul": 7, "relu_mul": 8, "gelu_mul": 9, "res_add": 16}
# the 4-wave kernel's tiles, whose unsplit product can add into its output (EPI "res_add")
RES_ADD_TILES = frozenset((22, 28, 34, 41, 45, 55))


# row strides that the 4-wave kernel reaches over a tile's 256 rows by 32-bit offsets
MAX_4W_STRIDE = 1 << 22


def spaced(x: torch.Tensor, w: torch.Tensor, tile: int):
    """(x, its row stride, w, its row stride) as the tile's kernel takes them: the 4-wave kernel reads a tile's rows by
    offsets within their range and so needs them at least their length apart, and not too far. Rows that overlap
    (expanded ones, windows) are copied; one row has no stride."""
    lda, ldw = x.stride(0), w.stride(-2)
    if tile in RES_ADD_TILES:
        n = x.shape[1]
        if not n <= lda < MAX_4W_STRIDE:
            x, lda = (x, n) if x.shape[0] == 1 else (x.contiguous(), n)
        if not n <= ldw < MAX_4W_STRIDE:
            w, ldw = (w, w.shape[-1]) if w.shape[-2] == 1 else (w.contiguous(), w.shape[-1])
    return x, lda, w, ldw


# epilogues over the interleaved gate/up weight: the output is half as wide
PAIR_EPIS = ("silu_mul", "clamp_mul", "relu_mul", "gelu_mul")
# tiles whose slab-only split-K call can store fp16 partials (EPI "slab16"); the fused consumers then
# read half the bytes. The weight-streaming GEMVs and tiles 34, 41, 45 and 55 keep fp32 slabs.
SLAB16_TILES = frozenset(list(range(0, 22)) + [22, 23, 24, 25, 26, 28] + list(STREAM_TILES))
SLAB16 = os.environ.get("DLI_SLAB_FP32", "0") != "1"      # A/B: fp32 partials everywhere
# tiles whose grouped SiLU*up GEMM can read its rows through a permutation (the generic
# family: dli_gemm_grouped_gather), so the MoE gate/up skips the gathered copy of its input
GATHER_TILES = frozenset(list(range(0, 22)) + [23, 24, 25] + list(STREAM_TILES))
NUM_CUS = 256


@dataclass(frozen=True)
class GemmPlan:
    backend: str      # "dli": our kernels (the only backend)
    tile: int
    splits: int


_plan_cache: dict = {}
_ws_lock = threading.Lock()
_workspaces: dict = {}
# buffers a larger workspace replaced: a captured hipGraph keeps the pointer it was captured
# with, so a replaced buffer must outlive every graph (the prefill autotune runs after the
# decode graphs are captured and grows the workspace; freeing the old buffer let eager
# tensors take its memory while graph replays still wrote split-K slabs into it)
_retired: list = []


def workspace(device: torch.device, nbytes: int) -> torch.Tensor:
    """Grow-only scratch (bytes) per device. Never freed: see ``_retired``. It at least doubles, so
    that all outgrown buffers together are smaller than the one in use: the sizes asked for follow
    the steps' lengths, and by exact sizes rising steps of recurrences (2.1 MB a segment and
    sequence, up to 256 MB) would leave 15 GB behind."""
    key = (device.type, device.index)
    with _ws_lock:
        ws = _workspaces.get(key)
        if ws is None or ws.numel() < nbytes:
            if ws is not None:
                _retired.append(ws)
            grown = max(nbytes, 1 << 20, 2 * ws.numel() if ws is not None else 0)
            ws = torch.empty(grown, dtype=torch.uint8, device=device)
            _workspaces[key] = ws
        return ws


LARGE_M = 1024


# (rows up to, tiles of 32, 64 and 128 columns, the head's)
STREAM_BANDS = ((32, 60, 62, 61, 62), (64, 69, 64, 63, 65), (96, 72, 70, 66, 68), (128, 72, 71, 67, 68))


def _stream_plan(M: int, N: int, K: int, epi: str):
    """Few rows: the weights' read is the product's time. One row of the weight-streaming tiles, as wide
    as still gives three quarters of the CUs a workgroup (a narrower one reads the rows more often, a
    second round costs as much as the first); where 32 columns are too wide too, 64 and K split until
    about one workgroup a CU. fp32 outputs, us on these against the best other tile: 24 rows: 4096 x 4096
    11.6 / 13.2, 8192 x 4096 13.9 / 17.6, 16384 x 4096 23.7 / 30.7, 4096 x 14336 24.2 / 27.4, 32000 x 4096 41.5 /
    56.3, 128256 x 4096 167 / 197; 64 rows: 14.1 / 13.8, 16.5 /
    20.0, 26.5 / 35.2, 28.5 / 29.0, 45 / 60, 177 / 209; 96 rows: 16.3 / 16.2, 23.8 / 24.4, 30.1 / 38.3, 31.9 / 33.0,
    47.5 / 63.5, 190 / 215. Above 96 rows the narrowest weights stay on two rows of tile 6 or one of tile 7
    (128 rows, 4096 x 4096 17.6 / 19.8, 4096 x 14336 35 / 39), from 65 rows the small ones on tile 5 (96 rows,
    2048 x 2048 11.2 / 14.0), above 96 rows all of short K (bias and GELU, 128 rows, 3072 x 768 7.7 / 10.9 on
    tile 6, 9.8 on tile 0), from 33 rows the up to 256 columns of a low-rank factor, K = 1024 split too (64 rows, 256 x
    1024 7.1 / 8.7 on tile 64 unsplit, 96 x 4096 8.6 / 9.2 on tile 64, 64 x 768 5.5 / 6.1)."""
    if K % 64:
        return None
    _, narrow, mid, wide, head = next(b for b in STREAM_BANDS if M <= b[0])
    fill = 3 * NUM_CUS // 4
    few = M > 32 and N <= 256
    split = False
    if N >= 256 * NUM_CUS:
        tile = head
    elif -(-N // 128) >= fill:
        tile = wide
    elif -(-N // 64) >= fill:
        tile = mid
    elif -(-N // 32) >= fill and K % tile_step(narrow) == 0:
        tile = narrow
    else:
        split = True
        tile = mid
        if M > 64 and N < 3072 or M > 96 and K <= 1024 or few:
            tile = 5
        elif M > 96 and N < 6144:
            tile = 7 if K > 8192 else 6
    if K % tile_step(tile):
        tile = wide
    step = tile_step(tile)
    bm, bn = tile_shape(tile)
    tiles, splits = -(-M // bm) * -(-N // bn), 1
    most = 2 * NUM_CUS if tile == 5 else NUM_CUS
    # (K <= 1024: the second launch costs more than the shorter loop saves, 4096 x 1024 at 24 rows 6.1 / 7.8)
    while (split and (K > 1024 or few and K == 1024) and tiles * splits * 2 <= most
           and K % (step * splits * 2) == 0 and K // (splits * 2) >= (256 if K == 1024 else 512)
           and splits < 8):
        splits *= 2
    if epi == "splitk" and splits == 1 and K % (2 * step) == 0 and K >= 1024:
        splits = 2            # the fused reduce consumes partial slabs: need >= 2 slices
    return GemmPlan("dli", tile, splits)


@functools.lru_cache(maxsize=8192)
def _heuristic(M: int, N: int, K: int, epi: str) -> GemmPlan:
    """Fitted to profiles/r1_gemm/gemm_bench.json and profiles/r1_gemm8p/ (MI355X, random
    bf16 operands): skinny decode GEMMs (M <= 512) on the 2/3-stage tiles below (autotuned
    at capture); fat prefill GEMMs (M >= LARGE_M) on 256-row tiles of the 4-wave kernel (22, 28, 55), with
    their fused epilogues (SiLU*up, bias+GELU, fp32); the prefill autotune (``prefill_candidates``) measures
    them per bucket."""
    # M > 512: mixed prefill+decode steps of a full batch and prefill — 256-row
    # tiles (the 128-row tiles below ran a 512 + 300-token mixed step's GEMMs ~2.5x slower
    # than the tuned decode step: 26.7 ms per mixed step end to end, profiles/r3/e2e/)
    if M >= LARGE_M or M > 512:
        # mid-sized steps (serving refills / mixed steps of ~1-2k rows): 256x256 tiles leave
        # most CUs idle on the N = 4096 / 6144 projections (M = 1200: 80 / 120 tiles), so
        # split K while the grid stays within one wave of the chip
        tiles = -(-M // 256) * -(-N // 256)
        if (epi == "f32" and tiles * 2 <= NUM_CUS and K <= 6144
                and -(-M // 256) * -(-N // 128) > NUM_CUS // 2):
            # half-width tiles fill the chip without a split and its reduce over fp32 slabs: M = 1100 /
            # 1536, N = K = 4096: 60 / 62 us against 78 / 80 unsplit
            return GemmPlan("dli", 28, 1)
        splits = 1
        if epi in ("none", "splitk", "f32"):
            # (f32, M = 1100, N = 4096, K = 14336: 240 us unsplit, 153 in two)
            while (tiles * splits * 2 <= NUM_CUS and K % (64 * splits * 2) == 0
                   and K // (splits * 2) >= 1024 and splits < 4):
                splits *= 2
        # 55 and 22 run one kernel (gemm4w.h), 55 on 256, 192 or 160 columns, 22 on 224 and 128 too, with any K, with
        # splits and, where biased, on 256. So they are equal where both choose one width (8192 x 6144, K = 4096 268
        # us, 4352 x 4096, K = 14336 371), and 22 is ahead where 128 or 224 columns fill a round better (1536 x 4096,
        # K = 4096 48 against 53, 1024 x 8192 pairs, K = 1024 18 against 22). The lines below are from kernels that
        # differed more: they cost up to that where they name 55
        if epi in PAIR_EPIS:
            pays = K > 2048 or (K >= 1024 and tiles > NUM_CUS) or N % 64 != 0   # (tile 22 takes no such N)
        else:
            pays = epi not in ("bias", "bias_gelu")
        # (long K from 4096 rows on where its narrower tiles save part of a round: as above)
        if (pays and splits == 1 and M >= LARGE_M and K % 128 == 0
                and (K <= 8192 or M < 4096 or persistent_width(M, N, epi in PAIR_EPIS, device_cus()) < 256)
                and (M < 16384 or N >= 16384) and tile_ok(55, epi)):
            return GemmPlan("dli", 55, 1)
        return GemmPlan("dli", 22, splits)
    if epi == "res":
        # residual-adding GEMV (full K): 4 rows a workgroup, 8 K-steps in flight per lane
        # (1024 workgroups on a 4096-wide projection)
        return GemmPlan("dli", 56, 1)
    # (up to 4 rows the fitted plans stay on the plain weight stream, whose sums do not depend on the
    # number of rows; a capture's timing may choose otherwise)
    if GEMV_MAX_M < M <= STREAM_MAX_M:
        p = _stream_plan(M, N, K, epi)
        if p is not None:
            return p
    if M <= GEMV_MAX_M and epi not in ("clamp_mul", "relu_mul", "gelu_mul"):   # (no GEMV has them)
        # batch-1 / tiny batches: stream the weights (gemv_kernel) with enough workgroups
        # (>= 512, two per CU) to keep ~64 KB of loads in flight per CU
        # gate/up at M <= 2: the 16-row SiLU grid (tile 29) 39.5 / 43.3 vs 49.0 / 51.0 us for
        # the 32-row tile 31 at M = 1 / 2 (profiles/r4/b1/s37_*, s38_gemv_sweep_m2.jsonl)
        tile = (29 if M <= 2 else 31) if epi == "silu_mul" else 30
        wgs = -(-N // GEMV_TILES[tile])
        splits = 1
        while (wgs * splits < 512 and K % (64 * splits * 2) == 0
               and K // (splits * 2) >= 1024 and splits < 8):
            splits *= 2
        if epi == "splitk" and splits == 1 and K % 128 == 0:
            splits = 2
        return GemmPlan("dli", tile, splits)
    if M <= 128:
        tile = 0 if N <= 8192 else 1
    elif M <= 256:
        tile = 1 if N <= 8192 else 2
    else:
        # (the last rows of a prefill wave through the head, K = 4096, N = 128256: 512 rows 447 us on
        # 256x256 tiles, 619 on 128x128. Up to 384 rows, which are three tiles of 128, where the last
        # round of tiles is nearly full and K is not short: 257 rows 419 and 438, but 1.05 times as long
        # at N = 102400, K = 2048 and 1.14 at 65536, K = 1024)
        tiles = -(-M // 256) * -(-N // 256)
        full = 10 * tiles >= 9 * NUM_CUS * -(-tiles // NUM_CUS) and K >= 2048
        tile = 22 if tiles >= 2 * NUM_CUS and (M > 384 or full) else 2
    bm, bn = TILES[tile]
    tiles = -(-M // bm) * -(-N // bn)
    splits = 1
    # split K until the grid is ~2-3 waves over the 256 CUs, keeping >= 512 K per slice
    while (tiles * splits * 2 <= 3 * NUM_CUS and K % (64 * splits * 2) == 0
           and K // (splits * 2) >= 512 and splits < 8):
        splits *= 2
    if epi == "splitk" and splits == 1 and K % 128 == 0 and K >= 1024:
        splits = 2            # the fused reduce consumes partial slabs: need >= 2 slices
    return GemmPlan("dli", tile, splits)


def grouped_tile(rows: int, groups: int) -> int:
    """Default tile for the grouped (MoE) GEMM over `rows` permuted rows in `groups` experts
    (autotune_grouped() replaces it at graph capture). Each expert's weights should be
    streamed ONCE, so the tile should cover one expert's rows (mean rows = rows / groups,
    plus headroom for routing imbalance) without doubling the MFMA work. Measured on
    Mixtral 8x7B at batch 512 (~128 rows per expert): 128-row tiles 8.5k tok/s (a second
    pass over most experts' weights), 160x128 14.4k, 192x128 10.2k, 256x128 4.8k, 3-stage
    variants slower (1 workgroup per CU)."""
    forced = os.environ.get("DLI_MOE_TILE")
    if forced:
        return int(forced)
    need = 1.25 * rows / max(1, groups)          # mean rows per expert + imbalance headroom
    for bm, tile in ((64, 1), (128, 2), (160, 12), (192, 10)):
        if need <= bm:
            return tile
    return 4              # 256 x 128


_grouped_cache: dict = {}


def grouped_plan(rows: int, N: int, K: int, epi: str, groups: int) -> GemmPlan:
    p = _grouped_cache.get((_bucket(rows), N, K, epi, groups))
    if p is not None:
        return p
    tile = grouped_tile(rows, groups)
    # experts of few rows: the streaming tile that covers them
    need = 1.25 * rows / max(1, groups)
    for t in (61, 63, 66) if "DLI_MOE_TILE" not in os.environ else ():
        if need <= tile_shape(t)[0]:
            if K % tile_step(t) == 0 and tile_ok(t, epi):
                tile = t
            break
    return GemmPlan("dli", tile, 1)


def autotune_grouped(rows: int, w: torch.Tensor, epi: str, iters: int = 5, log=None):
    """Pick the grouped-GEMM tile for `rows` permuted rows over the experts of `w`
    ([E, N, K]) with a random routing (what a decode step of rows/top_k tokens sees). The
    expert weights together exceed the Infinity Cache, so every call is cold."""
    from .. import ops
    E, N, K = w.shape
    key = (_bucket(rows), N, K, epi, E)
    if key in _grouped_cache or os.environ.get("DLI_MOE_TILE"):
        return _grouped_cache.get(key)
    dev = w.device
    # per-expert rows of a RANDOM routing (seeded multinomial), not an exactly even split: with
    # 1024 rows over 8 experts an even split fits 128-row tiles exactly, while in situ about
    # half the experts get more than 128 rows and take a second tile pass over their weights
    # (Mixtral b512: the even-split pick ran 13.6k tok/s, the 160-row tile 15.3k)
    counts = np.random.default_rng(1234).multinomial(rows, [1.0 / E] * E).tolist()
    off = torch.tensor([0] + list(__import__("itertools").accumulate(counts)),
                       dtype=torch.int32, device=dev)
    x = (torch.randn(max(rows, 1), K, device=dev) * 0.5).to(w.dtype)
    # the down projection is timed with what follows it (one pick per row, weight 1): the split plans on
    # the fp16-slab tiles fused with the combine, the residual add and, at the widths that take it, the
    # next norm (ops.MoEPending); the others with their kernels for the same. Timed alone, an unsplit
    # plan won at 64 tokens x 2 of 8 experts and cost the step 10 us a layer
    ones = torch.ones(max(rows, 1), 1, dtype=torch.float32, device=dev)
    ident = torch.arange(max(rows, 1), dtype=torch.int32, device=dev).view(-1, 1)
    comb = torch.empty(max(rows, 1), N, dtype=w.dtype, device=dev)
    res, nw = torch.zeros_like(comb), torch.ones(N, dtype=w.dtype, device=dev)
    best = None
    cands = []
    for tile in sorted(TILES) + sorted(STREAM_TILES):
        bm = tile_shape(tile)[0]
        if bm > 2 * max(64, rows // E + 32) or not tile_ok(tile, epi):
            continue                                  # far taller than an expert's rows
        if tile in STREAM_TILES and bm < rows // E:
            continue                                  # streams the weights once or not at all
        step = tile_step(tile)
        for splits in (1, 2, 4):                      # split-K for long-K expert GEMMs
            if K % (step * splits) == 0 and (splits == 1 or K // splits >= 2048):
                cands.append(GemmPlan("dli", tile, splits))
    for p in cands:
        fused = epi == "none" and ops.moe_slab_plan(p)

        def run(p=p, fused=fused):
            if fused:
                ops.moe_down_pending(x, w, off, rows, p, ones, ident, comb.shape).add_rmsnorm(res, nw, 1e-5)
                return
            y = ops._gemm_native(x, w, epi, plan=p, groups=E, group_off=off, rows_per_group=rows)
            if epi == "none":
                ops._native_call("dli_moe_combine", comb.data_ptr(), y.data_ptr(), ones.data_ptr(),
                                 ident.data_ptr(), rows, 1, N, ops._st())
                ops.add_rmsnorm(comb, res, nw, 1e-5)
        try:
            ms = ops.benchmark(run, iters=iters, warmup=1, graph=_GRAPH_TUNE)
        except Exception:  # noqa: BLE001
            continue
        if best is None or ms < best[1]:
            best = (p, ms)
    if best is not None:
        _grouped_cache[key] = best[0]
        if log:
            log(f"[gemm autotune] grouped rows={rows} E={E} N={N} K={K} {epi}: {best[0]} "
                f"{best[1]*1e3:.1f} us")
    return best


def _bucket(M: int) -> int:
    """Plan-cache key for M: exact up to 512 rows (decode graph buckets are a fixed small
    set and their best plans differ: one plan per power of two let M=320's plan run M=512),
    a multiple of 128 up to 1024 (the sizes of mixed prefill+decode steps of a full batch,
    tuned as a few buckets when serving: StageRunner.autotune_mixed), power-of-two above
    (prefill)."""
    if M <= 512:
        return M
    if M <= 1024:
        return -(-M // 128) * 128
    b = 1
    while b < M:
        b <<= 1
    return b


def plan(M: int, N: int, K: int, epi: str) -> GemmPlan:
    key = (_bucket(M), N, K, epi)
    # tuned and pinned plans by bucket; a fitted one by its own M (a bucket of prefill sizes spans a
    # factor of two, in which the best split differs)
    return _plan_cache.get(key) or _heuristic(M, N, K, epi)


@functools.lru_cache(maxsize=None)
def device_cus() -> int:
    """CUs of the current GPU as the kernels see them (a partition has fewer); 256 without one."""
    if torch.cuda.is_available():
        return torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count
    return NUM_CUS


@functools.lru_cache(maxsize=8192)
def persistent_width(M: int, N: int, pairs: bool, cus: int = NUM_CUS) -> int:
    """Columns of the tiles that the persistent kernel (tile 55) takes on ``cus`` CUs: gemm4w.hip's
    width_of."""
    best, least = 256, 0.0
    for nj, price in ((8, 1.0), (6, 0.794), (5, 0.684)):
        if pairs and nj & 1:
            continue
        whole, rest = divmod(-(-M // 256) * -(-N // (32 * nj)), cus)
        x = rest / cus
        last = 0.0 if not rest else 0.60 + 0.25 * x + 0.15 * x ** 3 if whole else 0.72 + 0.28 * x ** 3
        c = (whole + last) * price
        if nj == 8:
            least = 0.97 * c
        elif c < least:
            best, least = 32 * nj, c
    return best


@functools.lru_cache(maxsize=8192)
def row_cut(M: int, N: int, K: int) -> int:
    """Rows of a large product that run by themselves, in whole 256-row tiles, where the up to 128 rows
    past them would begin a round of the chip that they cannot fill; those then run on a streaming tile,
    bound by the weights' read. 0: all rows together. Reckoned in 256 x 256 tiles, of which the last round's price is
    0.73 of a full one even if nearly empty (fewer busy CUs clock higher): 0.017 us a K on one, the other
    side the weights at 5.5 TB/s and a launch. Not where as many rounds remain: 8199 x 6144 is 3.09 rounds, 4104 x
    6144 1.59. Nor where 512 rows would remain, which run on a decode step's tiles: 513 x 28672 168 and 186, 640 x 32000
    187 and 217. K = 4096, us together and cut: 4104 x 4096 109 and 107, 8199 x 4096 207 and 196, 8256 x 12288 608 and
    583, 8199 x 16384 803 and 775, 8199 x 28672 (SiLU pairs) 1302 and 1272; K = 14336: 4104 x 4096 356 and 332, 8199 x 4096
    736 and 659. The kernel's tiles of 192 and 320 rows, which this does not know, fill some such rounds as
    well or better: 1100 x 16384 129 and 140, 1537 x 28672 248 and 295, 3080 x 16384 313 and 329, 9220 x 28672 1440 and
    1497; of 53 sizes it cuts 21 lose by it, 5 % in the mean, and 32 gain 3. The rows past the cut are
    summed in another order than those before it (each order a valid fp32 one): a token's last bits depend on which
    side of it the step puts the token. Pinned and tuned plans apply to each part by its own rows."""
    rest = M % 256
    if M - rest <= 512 or not 0 < rest <= STREAM_MAX_M or K % 64:
        return 0
    rows, cols = M // 256, -(-N // 256)
    rounds = -(-(rows + 1) * cols // NUM_CUS) - -(-rows * cols // NUM_CUS)
    apart = (N * K * 2 / 5.5e6 + 8.0) * (1.0 if rest <= 64 else 1.25)
    return M - rest if rows * cols >= NUM_CUS // 2 and rounds * 0.017 * K > apart else 0


def set_plan(M: int, N: int, K: int, epi: str, p: GemmPlan) -> None:
    _plan_cache[(_bucket(M), N, K, epi)] = p


def clear_plans() -> None:
    _plan_cache.clear()
    _tuned.clear()


def autotune(shapes, weights: dict, device, iters: int = 6, log=None,
             cold_bytes: int = 1 << 30, qkv_heads=None, candidates=None,
             normed_in=()) -> dict:
    """Measure every candidate plan for each (M, N, K, epi) and pin the fastest
    ("measure, don't guess"). ``weights[(N, K)]`` is a real [N, K] weight of that shape.

    Measured the way a decode step sees it: the weight is COLD (each call reads a different
    copy; the copies together exceed the 256 MB Infinity Cache — timing one warm weight
    picked plans that ran 12 % slower in the model), and split-K plans pay their slab
    reduction (a "splitk" GEMM feeds a fused reduce that reads every slab). A non-split
    winner for a "splitk" shape also becomes that shape's plain plan (unfused path).
    ``qkv_heads`` = (hq, hkv, hd): the "splitk" shape with N = (hq + 2 hkv) hd is the fused
    QKV projection, whose consumer is the decode attention prologue (slab sum or bf16 read,
    RoPE, KV write), so its candidates are timed with the RoPE + cache-write kernel of the
    same input (``ops.linear_rope_cache``) instead of the add + RMSNorm one.
    ``candidates(M, N, K, epi)`` replaces the plan list (``prefill_candidates``).
    ``normed_in``: (N, K, epi) of the GEMMs whose input at M <= GEMV_MAX_M is a deferred
    RMSNorm (``ops.NormedRows``: the batch-1 QKV and gate/up), timed with that prologue.
    Returns {shape: (plan, ms)}."""
    from .. import ops  # local import: ops imports this module
    out = {}
    for (M, N, K, epi) in shapes:
        key = (_bucket(M), N, K, epi)
        if key in _tuned:
            continue
        w0 = weights[(N, K)]
        n_copies = max(2, min(16, -(-cold_bytes // (w0.numel() * w0.element_size()))))
        ws_ = [w0] + [w0.clone() for _ in range(n_copies - 1)]
        x = (torch.randn(M, K, device=device) * 0.5).to(w0.dtype)
        x_in = x
        if M <= GEMV_MAX_M and (N, K, epi) in normed_in:
            x_in = ops.NormedRows(x, torch.ones(K, dtype=w0.dtype, device=device), 1e-5)
        is_qkv = (epi == "splitk" and qkv_heads is not None
                  and N == (qkv_heads[0] + 2 * qkv_heads[1]) * qkv_heads[2])
        if epi == "splitk":
            # a "splitk" GEMM is timed WITH its consumer: split plans reduce their slabs in a
            # fused add+RMSNorm, unsplit plans write bf16 and run the separate add+RMSNorm
            # pass; timing the unsplit GEMM alone hid that pass and biased the choice
            res = torch.zeros(M, N, dtype=w0.dtype, device=device)
            nw = torch.ones(N, dtype=w0.dtype, device=device)
        if epi == "res":
            res_r = torch.zeros(M, N, dtype=w0.dtype, device=device)
        if is_qkv:
            from . import reference as R
            hq, hkv, hd = qkv_heads
            pos = torch.zeros(M, dtype=torch.int32, device=device)
            slots = torch.arange(M, dtype=torch.int32, device=device)
            kc = torch.empty(-(-M // 16), hkv, 16, hd, dtype=w0.dtype, device=device)
            vc = torch.empty_like(kc)
            cs = R.rope_cos_sin(16, hd, 10000.0, device=device)
            # decode-sized QKV: its consumer is the fused reduce + RoPE + KV write + attention
            # kernel where the plan's split count allows it (ops.linear_rope_attention), else
            # the RoPE/cache kernel + attention; time each plan with the path it will run
            # (one-token contexts: the launch and dependency structure, not the KV stream)
            decode_qkv = M <= 512 and candidates is None
            if decode_qkv:
                bt = (slots // 16).to(torch.int32).unsqueeze(1).contiguous()
                ctx = torch.ones(M, dtype=torch.int32, device=device)
                sc = 1.0 / math.sqrt(hd)
        # what the epilogue reads by address: clamp_mul's limit, a bias of the output's columns
        bias = (torch.ones(1, dtype=torch.float32, device=device) if epi == "clamp_mul" else
                torch.zeros(N, dtype=w0.dtype, device=device) if epi in ("bias", "bias_gelu") else None)
        best = None
        timed = []                                  # (ms, plan, run) of every valid candidate
        t_shape = time.perf_counter()
        for p in (candidates or candidate_plans)(M, N, K, epi):
            def run(p=p):
                for w in ws_:
                    if is_qkv and decode_qkv:
                        _qkv_decode(ops, x_in, w, p, pos, slots, cs, kc, vc, bt, ctx, hq, hkv,
                                    hd, sc)
                    elif x_in is not x:
                        ops.linear_normed(x_in, w, epi, plan=p)
                    elif is_qkv:
                        ops.linear_rope_cache(x, w, pos, slots, cs, kc, vc, hq, hkv, hd,
                                              plan=p)
                    elif epi == "splitk":
                        ops.linear_add_rmsnorm(x, w, res, nw, 1e-5, plan=p)
                    elif epi == "res":
                        ops.linear_residual(x, w, res_r, plan=p)
                    else:
                        ops._gemm_native(x, w, epi, bias=bias, plan=p)
            try:
                ms = ops.benchmark(run, iters=iters, warmup=1, graph=_GRAPH_TUNE) / len(ws_)
            except Exception:  # noqa: BLE001 — an invalid candidate is skipped
                continue
            timed.append((ms, p, run))
        best = _final_round(ops, timed, iters, len(ws_))
        del ws_, timed
        if best is not None:
            _plan_cache[key] = best[0]
            _tuned.add(key)
            if epi == "splitk" and best[0].splits == 1:
                _plan_cache[(_bucket(M), N, K, "none")] = best[0]
                _tuned.add((_bucket(M), N, K, "none"))
            out[(M, N, K, epi)] = best
            if log:
                log(f"[gemm autotune] M={M} N={N} K={K} {epi}: {best[0]} {best[1]*1e3:.1f} us "
                    f"({time.perf_counter() - t_shape:.1f} s)")
    return out


# finalists re-timed round-robin after the first pass: candidates within FINAL_BAND of the
# fastest, at most FINAL_N of them, FINAL_ROUNDS rounds; the lowest median wins. One pass in
# candidate order let drift and noise pick among plans a few % apart: two runs of the same
# tree on one box pinned different QKV plans (128x192 split 2 vs 128x96 unsplit,
# profiles/r4/prof vs profiles/r5/s06 wave summaries)
FINAL_BAND = 0.06
FINAL_N = 4
FINAL_ROUNDS = 3


def _final_round(ops, timed, iters: int, n_copies: int):
    """(plan, ms) of the winner among ``timed`` = [(ms, plan, run)] (None if empty)."""
    if not timed:
        return None
    timed.sort(key=lambda t: t[0])
    fin = [t for t in timed if t[0] <= timed[0][0] * (1 + FINAL_BAND)][:max(1, FINAL_N)]
    if len(fin) == 1 or FINAL_ROUNDS <= 0:
        return (fin[0][1], fin[0][0])
    samples = [[ms] for ms, _, _ in fin]
    for _ in range(FINAL_ROUNDS):
        for i, (_, _, run) in enumerate(fin):
            samples[i].append(ops.benchmark(run, iters=iters, warmup=1, graph=_GRAPH_TUNE)
                              / n_copies)
    med = [sorted(s)[len(s) // 2] for s in samples]
    i = min(range(len(fin)), key=lambda j: med[j])
    return (fin[i][1], med[i])


def _qkv_decode(ops, x, w, p, pos, slots, cs, kc, vc, bt, ctx, hq, hkv, hd, scale):
    """One decode step's QKV projection + attention under plan ``p``, as the model runs it
    (models/model.py ``_llama_layers``): the fused kernel when ``p`` allows it, else the
    RoPE/cache kernel and the decode attention."""
    with _forced_plan(x.shape[0], w.shape[0], x.shape[1], p):
        out = ops.linear_rope_attention(x, w, pos, slots, cs, kc, vc, bt, ctx, 1, hq, hkv, hd,
                                        scale)
        if out is None:
            qkv = ops.linear_rope_cache(x, w, pos, slots, cs, kc, vc, hq, hkv, hd, plan=p)
            ops.decode_attention(qkv, kc, vc, bt, ctx, 1, hq, hkv, hd, scale)


class _forced_plan:
    """Pin the plan of one shape for the duration of a timing call (the fused attention path
    reads its plan from the cache, not from an argument): the "splitk" entry, and for an
    unsplit plan also the "none" entry its plain GEMM takes."""

    def __init__(self, M, N, K, p):
        b = _bucket(M)
        self.keys = [(b, N, K, "splitk")] + ([(b, N, K, "none")] if p.splits == 1 else [])
        self.p = p

    def __enter__(self):
        self.old = [_plan_cache.get(k) for k in self.keys]
        for k in self.keys:
            _plan_cache[k] = self.p

    def __exit__(self, *exc):
        for k, o in zip(self.keys, self.old):
            if o is None:
                _plan_cache.pop(k, None)
            else:
                _plan_cache[k] = o


_tuned: set = set()
# candidates timed as graph replays (ops.benchmark graph=True)
_GRAPH_TUNE = True


def prefill_candidates(M: int, N: int, K: int, epi: str):
    """Prefill-sized GEMMs (M > 1024 rows): the one-wave-per-SIMD kernel on tile 22's width with the
    heuristic's split count, on 256 columns (PREFILL_4W_TILE) at the same split and, unsplit, on tile 55's
    width, measured per shape and bucket (a bucket's rows leave a part of a round empty that a step's own
    need not). At these sizes
    the GEMM is MFMA-bound, so the autotuner times them warm (``cold_bytes`` 1)."""
    base = _heuristic(M, N, K, epi)
    if base.tile == 55:                  # (its counterparts of other widths)
        base = GemmPlan("dli", 22, 1)
    out = [base]
    if base.tile == 22 and PREFILL_4W_TILE > 0:
        out.append(GemmPlan("dli", PREFILL_4W_TILE, base.splits))
    if base.tile == 22 and base.splits == 1 and K % 128 == 0 and PREFILL_PERSIST:
        out.append(GemmPlan("dli", 55, 1))
    return out


def candidate_plans(M: int, N: int, K: int, epi: str):
    if epi == "res":
        return [GemmPlan("dli", t, 1) for t in GEMV_RES_TILES
                if M <= GEMV_MAX_M and not (t == 32 and M > 1)]
    out = []
    # tiles kept out of the autotune candidates (DLI_GEMM_EXCLUDE="..." overrides, "" = none).
    # Default: 26 (256x224). It fills all 256 CUs on the gate/up GEMM and wins the isolated
    # autotune (98.8 vs ~106 us), but in the decode step it ran 97.9 vs 99.0 us per call and
    # the bench 0.3-0.7 % lower in three same-box A/B runs (profiles/r2_s2/README.md)
    excl_env = os.environ.get("DLI_GEMM_EXCLUDE")
    # 34, 41 and 45 are tile 22's kernel without its narrower widths and fp16 partial sums
    excl = {int(t) for t in (excl_env if excl_env is not None else "26,34,41,45,55").split(",")
            if t.strip()}
    # the persistent tile 55, whose stores drain under the next tile's loads, for the unsplit products of
    # many rows: the LM head of 512 456 -> 427 us in the step, which took 1571 and takes 1539
    if excl_env is None and M >= 192 and K % 128 == 0 and epi in ("f32", "silu_mul", "gelu_mul"):
        excl.discard(55)
    # ... except where 256x256 tiles take more than one wave of the chip and 256x224 tiles
    # land on a whole number of waves (Llama-3-70B gate/up at M = 512: N = 57344 is 448
    # 256x256 tiles = 1.75 waves, 512 256x224 tiles = 2 waves); an explicit
    # DLI_GEMM_EXCLUDE keeps the list as given
    if excl_env is None and 26 in excl:
        t256 = -(-M // 256) * -(-N // 256)
        t224 = -(-M // 256) * -(-N // 224)
        if t256 > NUM_CUS and t224 % NUM_CUS == 0:
            excl.discard(26)
    for tile in [*TILES, *STREAM_TILES]:
        bm, bn = tile_shape(tile)
        if not tile_ok(tile, epi) or tile in excl:
            continue
        if M <= 64 and bm > 64:
            continue
        if M > 512 and bm < 128:
            continue
        if tile in STREAM_TILES:
            # one row of tiles; for 2 to 4 rows beside the weight stream's own kernels, but for the
            # products whose partial sums those keep in fp32
            band = next((b for b in STREAM_BANDS if M <= b[0]), ())
            if (tile not in band[1:] or M < 2
                    or (M <= GEMV_MAX_M and epi in ("splitk", "none"))):
                continue
        elif M <= 64 and tile in (0, 1) and K % 128 == 0:
            continue                     # slower than their 3-stage and streaming forms
        for splits in (1, 2, 4, 8) if tile != 55 else (1,):
            if K % (tile_step(tile) * splits) or K // splits < 256:
                continue
            tiles = -(-M // bm) * -(-N // bn)
            if splits > 1 and tiles * splits > 4 * NUM_CUS:
                continue
            out.append(GemmPlan("dli", tile, splits))
    if M <= GEMV_MAX_M:
        for tile in GEMV_TILES:
            if tile in excl or not tile_ok(tile, epi) or (tile in GEMV_M1_ONLY and M > 1):
                continue
            for splits in (1, 2, 4, 8):
                if K % (64 * splits) == 0 and K // splits >= 512:
                    out.append(GemmPlan("dli", tile, splits))
    return out
