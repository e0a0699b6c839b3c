"""gfx950 launch-configuration search space, selection rules and the persisted tuning table.

This replaces the reference's candidate enumeration and ranking (tuner.py:181-235, 414-449,
503-517; mma.py:63-81). The reference compiles Triton candidates and ranks feasible ones by the
largest resource footprint without timing. Here the candidates are the tiles built into
libfa_gfx950.so; feasibility comes from the compiler's resource table (kernel_resources.json);
ranking comes from a timed sweep on an MI355X (``tune_table.json``, written by gfx950_tune.py),
with a fixed preference order when no measurement exists for a shape.

Tune arguments given by a caller (FlashAttenTuneArguments, or the BLOCK_* kwargs of a kernel
launch) are hints: a built tile that matches every given tile field is used; otherwise fields are
relaxed in the order NUM_STAGES, NUM_WARPS, BLOCK_N, BLOCK_M and the relaxation is recorded.
Tile choice never changes results, only speed.
"""
from __future__ import annotations

import functools
import json
import math
from dataclasses import dataclass
from pathlib import Path

import hip_lib

HERE = Path(__file__).resolve().parent
TUNE_TABLE_PATH = HERE / "tune_table.json"

VARIANT_BY_KERNEL = {
    "_flash_attn_fwd_kernel_basic": hip_lib.FA_VARIANT_BASIC,
    "_flash_attn_fwd_kernel_optimize_shared_mem": hip_lib.FA_VARIANT_OPT,
    "_flash_attn_fwd_kernel_block_d_nomask_contiguous": hip_lib.FA_VARIANT_SLICED,
}

# Attention tiles in preference order (used when the tuning table has no entry for a shape's variant,
# dtype, head dim and causality; the first ones are the fastest measured at large sizes):
# (block_m, block_n, waves, stages). stages selects the kernel pipeline:
#   1  the basic variant: the bodies of stages 9, 7 and 6 (64 keys, 32 rows per wave), else one K/V
#      buffer with two barriers per KV tile,
#   2  double-buffered K/V, one barrier per tile,
#   3  software-pipelined (QK of tile u+1 overlapped with the softmax of tile u inside each wave,
#      K/V brought into an LDS ring by LDS-DMA loads),
#   4  two-tile-ahead pipeline (QK of tile u+2 one for one with PV of tile u, the softmax of tile
#      u+1 spread over both; same LDS-DMA rings),
#   5  one tile per step in a 2-slot LDS-DMA ring, lean enough in registers for two waves per
#      SIMD at D = 256,
#   6  stages 5 with 16x16x32 MFMA tiles,
#   7  stages 3 with 16x16x32 MFMA tiles,
#   8  ping-pong: 8 waves in two groups of four that alternate MFMA phases and softmax phases
#      on the same SIMDs (16x16x32 MFMA tiles, 256 query rows per workgroup),
#   9  the ping-pong kernel in a persistent grid: one workgroup per CU walks a fixed sequence of
#      query blocks and fetches the next block's Q, K and V during the current block's last steps,
#  10  the ping-pong schedule with both groups on the same 128 rows and alternate KV tiles.
# The basic variant uses stages 1 (or 8, fa_launch_candidates); optimized and sliced use 2 to 10.
FA_TILE_SPACE = [
    (256, 64, 8, 8),
    (128, 32, 4, 6),
    (128, 64, 4, 7),
    (256, 64, 8, 9),
    (128, 64, 8, 10),
    (128, 64, 4, 3),
    (256, 64, 8, 3),
    (128, 32, 4, 3),
    (128, 64, 4, 4),
    (128, 32, 4, 4),
    (128, 32, 4, 5),
    (128, 64, 4, 5),
    (128, 64, 4, 6),
    (128, 32, 4, 7),
    (256, 64, 8, 2),
    (256, 64, 4, 2),
    (128, 64, 4, 2),
    (256, 128, 8, 2),
    (128, 128, 4, 2),
    (256, 32, 8, 2),
    (128, 32, 4, 2),
    (256, 64, 8, 1),
    (256, 64, 4, 1),
    (128, 64, 4, 1),
    (256, 128, 8, 1),
    (128, 128, 4, 1),
    (256, 32, 8, 1),
    (128, 32, 4, 1),
]
STAGES_BY_VARIANT = {
    hip_lib.FA_VARIANT_BASIC: (1,),
    hip_lib.FA_VARIANT_OPT: (3, 4, 5, 6, 7, 8, 9, 10, 2),
    hip_lib.FA_VARIANT_SLICED: (3, 4, 5, 6, 7, 8, 9, 10, 2),
}

# GEMM tiles in preference order: (block_m, block_n, block_k, waves).
GEMM_TILE_SPACE = [
    (256, 256, 64, 8),
    (256, 256, 64, 4),
    (256, 256, 32, 8),
    (256, 256, 32, 4),
    (256, 128, 64, 8),
    (128, 256, 64, 8),
    (128, 128, 64, 4),
    (128, 128, 32, 4),
    (128, 64, 32, 4),
    (64, 256, 32, 4),
    # K groups: 2 or 4 groups of 4 waves split one tile's K loop (shapes with few tiles)
    (128, 128, 32, 8),
    (128, 64, 32, 8),
    (128, 64, 32, 16),
    (64, 64, 32, 8),
]
GEMM_DEFAULT_GROUP_M = 8

# Time model of a GEMM tile, (c, lat, thr, e) in us and steps: c + (steps + e) * hypot(lat * ceil(tiles / 256),
# thr * tiles / 256), with steps the K slabs one K group multiplies, lat the time of a step of a round of one
# tile per CU, thr a step's share of a full chip and e what a tile's start and its C cost, in steps. All four
# are fitted, to timings of every tile at 500 sizes spread over M, N, K = 64 .. 8192; on 200 others the
# mean error is 3-8%. (With the C write left to c, and rounds of a fitted number of tiles per CU, it was
# 6-13%, and short-K products with a large C went to the 256x256 tiles: 7808x7104x64 22.0 -> 30.8 us.)
GEMM_COST = {
    (256, 256, 64, 8): (0.00, 1.014, 1.171, 5.3),
    (256, 256, 64, 4): (1.65, 1.140, 1.335, 4.7),
    (256, 256, 32, 8): (0.00, 0.541, 0.583, 10.8),
    (256, 256, 32, 4): (1.39, 0.526, 0.650, 10.6),
    (256, 128, 64, 8): (1.85, 0.619, 0.958, 3.2),
    (128, 256, 64, 8): (1.77, 0.615, 0.914, 3.2),
    (128, 128, 64, 4): (3.05, 0.439, 0.462, 2.2),
    (128, 128, 32, 4): (2.93, 0.211, 0.230, 3.7),
    (128, 64, 32, 4): (2.71, 0.218, 0.062, 1.1),
    (64, 256, 32, 4): (2.84, 0.233, 0.199, 3.9),
    (128, 128, 32, 8): (2.40, 0.354, 0.535, 5.2),
    (128, 64, 32, 8): (1.91, 0.279, 0.347, 5.2),
    (128, 64, 32, 16): (2.78, 0.474, 0.752, 3.8),
    (64, 64, 32, 8): (2.29, 0.216, 0.141, 3.8),
}
GEMM_GROUPS = {(128, 128, 32, 8): 2, (128, 64, 32, 8): 2, (128, 64, 32, 16): 4, (64, 64, 32, 8): 2}  # K groups
# Another tile than the nearest bucket's is taken when the model puts it the first margin ahead, the second
# where that bucket is within two octaves and its timing counts for more; a split of K when it is the third.
# Two of 685 timed sizes are then more than 2% slower than with the nearest bucket's tile alone (nine are
# without margins), and the choice is 3.4% slower than the fastest tile on average (the bucket's alone 38%).
GEMM_MODEL_MARGIN = 1.1
GEMM_NEAR_MARGIN = 1.27
GEMM_SPLIT_MARGIN = 1.15
# K split over the grid (hip_lib.gemm_f16 ksplits): the tiles it is built for, and its second launch's time
# (us) and partial-sum traffic (bytes per us). 74x608x6216 29.9 -> 9.2 us in 8 splits, 64x4096x4096 20.5 ->
# 12.1 in 4; 1000x1004x1000 (256 tiles) 8.6 -> 14 in 2, which the model refuses.
GEMM_SPLIT_TILES = ((64, 64, 32, 8), (128, 64, 32, 8))
GEMM_SPLITS = (2, 3, 4, 6, 8, 12, 16)
GEMM_SPLIT_US, GEMM_SPLIT_BYTES_PER_US = 2.7, 5e6

# The sliced variant splits KV until every CU holds as many workgroups as the kernel can keep
# resident (RESIDENT_DEFAULT when its resources are unknown); splitting further only adds merge
# traffic.
NUM_CUS = 256
RESIDENT_DEFAULT = 2
# Prefill-shaped sliced launches (full query tiles) split until each CU holds one workgroup, where
# prefill_splits finds that it pays. Times in us, from one-head to 32-head grids: a 64-key step of a
# 128-row tile by D (with 256 rows 1.5 times that); a split 2.5 for the merge launch, and its partials
# written and read back at 2.5 GB per ms. D = 128, 32 blocks of 128 rows, N=8192: 126 -> 37 us (81 with two
# splits); 128 blocks N=16384 279 -> 155, N=4096 70 -> 55; 64 blocks N=4096 75 -> 42; 64 blocks N=1024
# (22 against 26) and 128 blocks N=2048 (36 against 41) stay whole. D = 256, 6 heads 288x572 25 -> 21 in
# 4; with D = 128's step time it stayed whole.
PREFILL_SPLIT_CUS = NUM_CUS
PREFILL_STEP_US = {64: 0.55, 128: 0.95, 256: 2.6}
PREFILL_SPLIT_US = 2.5
PREFILL_SPLIT_BYTES_PER_US = 2.5e6
PREFILL_SPLIT_MARGIN = 1.1
# A single sequence with two kv heads needs 128 splits to fill the resident capacity (Qwen2.5
# B1 N32k: 18.7 us with 128 splits against 21.0 with 64, HIP-graph replay).
MAX_SPLITS = 128
LDS_PER_CU = 160 * 1024


@dataclass(frozen=True)
class FaTileChoice:
    block_m: int
    block_n: int
    waves: int
    stages: int
    splits: int = 1

    def to_c(self) -> hip_lib.FaTile:
        return hip_lib.make_tile(self.block_m, self.block_n, self.waves, self.stages, self.splits)


def stages_for(variant: int) -> int:
    """Default pipeline of a variant when no tile is chosen (the double-buffered one for
    optimized and sliced: it is built for every head dim)."""
    return 1 if variant == hip_lib.FA_VARIANT_BASIC else 2


def fa_candidates(variant: int, dtype, D: int) -> list[FaTileChoice]:
    """Built attention tiles for (variant, dtype, D), in preference order."""
    return list(_built_fa_tiles(variant, dtype, D))


def fa_launch_candidates(variant: int, dtype, D: int) -> list[FaTileChoice]:
    """The tiles a launch chooses among: the built ones and, in the basic variant, the dispatched ping-pong
    body behind its 256-row tile, as one more tile (stages 8), so that hints tell the two apart."""
    cands = fa_candidates(variant, dtype, D)
    if variant == hip_lib.FA_VARIANT_BASIC and FaTileChoice(256, 64, 8, 1) in cands:
        cands.append(FaTileChoice(256, 64, 8, 8))
    return cands


@functools.lru_cache(maxsize=256)
def _built_fa_tiles(variant: int, dtype, D: int) -> tuple[FaTileChoice, ...]:
    out = []
    allowed = STAGES_BY_VARIANT.get(variant, ())
    for bm, bn, waves, stages in FA_TILE_SPACE:
        if stages not in allowed:
            continue
        choice = FaTileChoice(bm, bn, waves, stages, 1)
        if not hip_lib.fa_fwd_supported(variant, dtype, D, choice.to_c()):
            continue
        # the sliced variant may split KV at run time: its split instantiation must exist as well
        if variant == hip_lib.FA_VARIANT_SLICED and not hip_lib.fa_fwd_supported(
                variant, dtype, D, FaTileChoice(bm, bn, waves, stages, 2).to_c()):
            continue
        out.append(choice)
    return tuple(out)


@functools.lru_cache(maxsize=1)
def _built_gemm_tiles() -> tuple[tuple[int, int, int, int], ...]:
    return tuple(t for t in GEMM_TILE_SPACE if hip_lib.gemm_supported(hip_lib.GemmTile(t[0], t[1], t[2], t[3], 1)))


def gemm_candidates() -> list[tuple[int, int, int, int]]:
    return list(_built_gemm_tiles())


# ---- hint resolution ----------------------------------------------------------------------------

_RELAX_ORDER = ("NUM_STAGES", "NUM_WARPS", "BLOCK_N", "BLOCK_M")


def _matches(choice: FaTileChoice, hints: dict[str, int]) -> bool:
    if "BLOCK_M" in hints and choice.block_m != hints["BLOCK_M"]:
        return False
    if "BLOCK_N" in hints and choice.block_n != hints["BLOCK_N"]:
        return False
    if "NUM_WARPS" in hints and choice.waves != hints["NUM_WARPS"]:
        return False
    if "NUM_STAGES" in hints and choice.stages != hints["NUM_STAGES"]:
        return False
    return True


def filter_by_hints(candidates: list[FaTileChoice], hints: dict[str, int | None]) -> tuple[list[FaTileChoice], list[str]]:
    """Candidates matching the given hints, relaxing hints in _RELAX_ORDER until some match.
    Returns (matching candidates, names of relaxed hints)."""
    active = {k: int(v) for k, v in hints.items() if v is not None and k in _RELAX_ORDER}
    relaxed: list[str] = []
    for key in _RELAX_ORDER:
        if any(_matches(c, active) for c in candidates):
            break
        if key in active:
            del active[key]
            relaxed.append(key)
    # Put back every dropped hint that some candidate still satisfies together with the rest.
    for key in list(relaxed):
        trial = dict(active)
        trial[key] = int(hints[key])
        if any(_matches(c, trial) for c in candidates):
            active = trial
            relaxed.remove(key)
    found = [c for c in candidates if _matches(c, active)]
    return (found or list(candidates)), relaxed


# ---- tuning table -------------------------------------------------------------------------------

_table_cache: dict | None = None


def load_tune_table(path: Path | None = None) -> dict:
    global _table_cache
    if path is None and _table_cache is not None:
        return _table_cache
    p = path or TUNE_TABLE_PATH
    table = json.loads(p.read_text()) if p.exists() else {"fa": {}, "gemm": {}}
    table.setdefault("fa", {})
    table.setdefault("gemm", {})
    if path is None:
        _table_cache = table
    return table


def reset_tune_table_cache() -> None:
    global _table_cache
    _table_cache = None
    _ranked.clear()


def _bucket(x: int) -> int:
    """Power-of-two bucket (>= 1) used to key shapes in the tuning table."""
    return 1 << max(0, math.ceil(math.log2(max(1, x))))


def fa_table_key(variant: int, dtype, D: int, causal: bool, B: int, H: int, M: int, N: int) -> str:
    dt = "bf16" if "bfloat16" in str(dtype) else "f16"
    return f"v{variant}|{dt}|D{D}|c{int(bool(causal))}|BH{_bucket(B * H)}|M{_bucket(M)}|N{_bucket(N)}"


def gemm_table_key(M: int, N: int, K: int) -> str:
    return f"M{_bucket(M)}|N{_bucket(N)}|K{_bucket(K)}"


def _split_key(key: str) -> tuple[str, list[int]]:
    """A table key's (variant, dtype, head dim, causality) part and its sizes."""
    prefix, *sizes = key.rsplit("|", 3)
    return prefix, [int(part.lstrip("BHMN")) for part in sizes]


_indexed: tuple[dict, int, dict] | None = None  # a table, its length and its index


def _bucket_index(table: dict) -> dict[str, list]:
    """The attention table's buckets by kind, as (sizes, their log2, entry) in key order: parsing every key
    at every new shape took 0.1-0.6 ms."""
    global _indexed
    if _indexed is None or _indexed[0] is not table or _indexed[1] != len(table):
        index: dict[str, list] = {}
        for key, entry in sorted(table.items()):
            prefix, sizes = _split_key(key)
            index.setdefault(prefix, []).append((sizes, [math.log2(x) for x in sizes], entry))
        _indexed = (table, len(table), index)
    return _indexed[2]


def _nearest_fa_entry(table: dict, key: str) -> dict | None:
    """The entry for `key`, else the swept bucket of the same (variant, dtype, D, causal) nearest to
    it: smallest sum of |log2| distances in B*H, M and N (ties: more work, then key order). Shapes
    between the swept sizes (the reference's B=1 H=28 pipeline cases, say) then run the tile timed on
    their neighbours instead of the fixed preference order. Decode buckets (fewer rows than a query
    tile: K/V streaming) and prefill buckets stand in for each other only when there is no other, and a
    decode bucket for a prefill shape not where the other 16-bit type, whose kernels are the same, has a
    prefill bucket (bf16 B1 H32/8 D128 N=4096 took a decode bucket's tile, 280 us against 228)."""
    entry = table.get(key)
    if entry is not None:
        return entry
    prefix, sizes = _split_key(key)
    want = [math.log2(x) for x in sizes]
    few = sizes[1] < FULL_TILE_ROWS
    index = _bucket_index(table)

    def swept(of: str) -> list[tuple[tuple, dict]]:
        """(rank, entry) of the buckets of one variant, dtype, head dim and causality; rank[0]: other kind."""
        return [(((have[1] < FULL_TILE_ROWS) != few, sum(abs(a - b) for a, b in zip(want, logs)),
                  -have[0] * have[1] * have[2]), ent) for have, logs, ent in index.get(of, ())]

    own = swept(prefix)
    if not few and own and all(rank[0] for rank, _ in own):
        swap = ("|f16|", "|bf16|") if "|f16|" in prefix else ("|bf16|", "|f16|")
        own += [item for item in swept(prefix.replace(*swap)) if not item[0][0]]
    return min(own, key=lambda item: item[0], default=(None, None))[1]


def _nearest_gemm_entry(table: dict, key: str) -> dict | None:
    """The entry for `key` ("M..|N..|K.."), else the swept GEMM bucket nearest to it: smallest sum
    of |log2| distances in M, N and K (ties: more work, then key order). A shape between the swept
    sizes (1024x4096x1024, say) then runs a tile timed on a shape of its scale, not the first built
    tile -- a 256x256 tile there leaves three quarters of the CUs idle."""
    entry = table.get(key)
    if entry is not None:
        return entry
    want = [int(part.lstrip("MNK")) for part in key.split("|")]
    best, best_rank = None, None
    for other, ent in sorted(table.items()):
        have = [int(part.lstrip("MNK")) for part in other.split("|")]
        dist = sum(abs(math.log2(a) - math.log2(b)) for a, b in zip(want, have))
        rank = (dist, -have[0] * have[1] * have[2])
        if best_rank is None or rank < best_rank:
            best, best_rank = ent, rank
    return best


_ranked: dict[int, tuple[dict, list]] = {}  # of the table's entries: parsing one took 40 us, three times a call


def _gemm_ranked_tiles(entry: dict) -> list[tuple[tuple[int, ...], int]]:
    """(tile, group_m) of a GEMM table entry, fastest first: the entry's winner, then every other
    timed (tile, GROUP_M) in order of its time."""
    known = _ranked.get(id(entry))
    if known is not None and known[0] is entry:
        return known[1]
    ranked = [(tuple(entry["tile"]), int(entry.get("group_m", GEMM_DEFAULT_GROUP_M)))]
    timed = {**entry.get("timed", {}), **entry.get("refined", {})}
    for name in sorted(timed, key=timed.get):
        tile_part, _, gm_part = name.partition("g")
        try:
            item = (tuple(int(x) for x in tile_part.split("x")), int(gm_part))
        except ValueError:
            continue
        if item not in ranked:
            ranked.append(item)
    _ranked[id(entry)] = (entry, ranked)
    return ranked


PERSISTENT_TILE = (256, 64, 8, 9)
FULL_TILE_ROWS = 128  # query rows from which a launch is prefill-shaped (the smaller block_m)
KEY_GROUP_TILE = (128, 64, 8, 10)
# Where a prefill-shaped launch splits, and a split is at most this many keys, the four-wave kernel: the
# key groups' merge through LDS costs more than the steps it saves (bf16 B1 H1 500x5000 D128 in 20
# splits 16.2 us against 17.7, B1 H2 128x700 in 5 12.6 against 15.4; 1024x8192 in 8 of 1024 keys: 37.7
# against 37.3).
SPLIT_TILE = (128, 64, 4, 5)
SPLIT_TILE_KEYS = 512

# Time of a grid with each kernel: its steps by the simulated schedule (hip_lib.grid_steps) at us per serial
# step. Per kernel the schedule's form, (tiles per step, order, {D: blocks a CU holds}), and per (D,
# causal) the fitted us per step, launch us, steps a block costs beside its own, time of a block alone
# on a CU in that of two sharing one, and f16's step in bf16 ones. Fitted to every kernel's times at 2700
# shapes of both types (1 to 160 heads, 40 to 20000 rows, 5 to 4000 us; mean error 3-7%; on 700 others
# 3-6%, at worst 30%).
GRID_FORM = {
    (256, 64, 8, 8): (1, hip_lib.GRID_HEAD_MAJOR, {64: 1, 128: 1}),
    (256, 64, 8, 9): (1, hip_lib.GRID_PERSISTENT, {64: 1, 128: 1}),
    (128, 64, 8, 10): (2, hip_lib.GRID_HEAVIEST_FIRST, {64: 1, 128: 1}),
    (128, 64, 4, 6): (1, hip_lib.GRID_HEAD_MAJOR, {64: 4, 128: 2}),
    (128, 64, 4, 7): (1, hip_lib.GRID_HEAD_MAJOR, {64: 2, 128: 2}),
}
GRID_STEP_US = {
    (256, 64, 8, 8): {(64, True): (0.865, 0.6, 6.0, 1, 0.96), (64, False): (0.867, 0.2, 6.7, 1, 0.96),
                      (128, True): (1.302, 0.0, 5.5, 1, 0.97), (128, False): (1.325, 0.0, 5.9, 1, 0.96)},
    (256, 64, 8, 9): {(64, True): (0.876, 1.4, 5.8, 1, 0.93), (64, False): (0.892, 1.3, 6.0, 1, 0.92),
                      (128, True): (1.263, 0.9, 5.6, 1, 0.98), (128, False): (1.315, 0.1, 6.2, 1, 0.98)},
    (128, 64, 8, 10): {(64, True): (1.062, 0.5, 5.2, 1, 0.93), (64, False): (1.087, 1.0, 4.4, 1, 0.91),
                       (128, True): (1.867, 0.0, 3.8, 1, 0.98), (128, False): (1.867, 0.4, 3.4, 1, 0.98)},
    (128, 64, 4, 6): {(64, True): (0.993, 2.5, 3.0, 0.66, 1.03), (64, False): (1.070, 3.0, 2.1, 0.60, 1.02),
                      (128, True): (1.786, 2.5, 2.6, 0.63, 1.03), (128, False): (1.809, 2.6, 2.6, 0.61, 1.04)},
}
# The basic variant's bodies: the tile's own (stages 1 of 256 rows is the persistent kernel), and the
# dispatched ping-pong kernel behind the same tile (stages 8).
GRID_BASIC_BODY = {(256, 64, 8, 1): (256, 64, 8, 9), (256, 64, 8, 8): (256, 64, 8, 8), (128, 64, 4, 1): (128, 64, 4, 7)}
GRID_BASIC_STEP_US = {
    (128, 64, 4, 7): {(64, True): (1.004, 2.7, 3.1, 0.69, 0.98), (64, False): (1.001, 2.5, 3.3, 0.68, 0.98),
                      (128, True): (1.537, 1.5, 4.0, 0.71, 1.00), (128, False): (1.631, 1.8, 3.7, 0.66, 0.99)},
}
# A grid of blocks that are no multiple of the XCDs spreads every head over all L2s: its steps take longer.
GRID_UNALIGNED = 1.05
GRID_MAX_BLOCKS = 4096  # of hip_lib.grid_steps
# What a kernel must be ahead of the table's by to displace it. The model's errors are mostly common to
# the kernels (clocks, caches): at 700 shapes it was not fitted to, the choice is 1.5% slower than the
# fastest of eight timed kernels on average, at worst 27% (the nearest bucket's tile with one rule for
# key groups and one for full grids: 5.8%, at worst 65%).
GRID_MODEL_MARGIN = 1.0  # a nearest bucket's tile: no other margin up to 1.02 did better
GRID_BUCKET_MARGIN = 1.03  # the shape's own bucket's, and the preference order's
GRID_UNTIMED_MARGIN = 1.15  # the persistent kernel's, where no bucket of the kind was timed


def _grid_us(body: tuple[int, int, int, int], f16: bool, D: int, causal: bool, BH: int, M: int, N: int) -> float:
    """Modelled time of a grid with a kernel; negative where the model does not reach."""
    per_step, order, per_cu = GRID_FORM[body]
    step, launch, block_steps, alone, f16_step = (GRID_STEP_US.get(body) or GRID_BASIC_STEP_US[body])[D, causal]
    steps = hip_lib.grid_steps(body[0], per_step, order, per_cu[D], block_steps, alone, BH, M, N, causal)
    blocks = math.ceil(M / body[0]) * BH
    if steps < 0:
        return -1.0
    if blocks > 64 and blocks % 8:
        steps *= GRID_UNALIGNED
    return launch + steps * step * (f16_step if f16 else 1)


@functools.lru_cache(maxsize=4096)
def choose_full_grid_tile(f16: bool, D: int, causal: bool, BH: int, M: int, N: int, best: tuple[int, int, int, int],
                          margin: float = GRID_MODEL_MARGIN,
                          tiles: tuple[tuple[int, int, int, int], ...] = tuple(GRID_STEP_US)) -> tuple[int, int, int, int]:
    """Tile of a whole-grid launch by the simulated schedules, of the given ones; best where none is ahead
    of it by the margin, or where the model does not reach."""
    if D not in (64, 128) or BH <= 0 or M <= 0 or best not in tiles:
        return best
    heads = GRID_MAX_BLOCKS // math.ceil(M / 128)
    if BH > heads >= 16:  # in many rounds the kernels compare as with fewer heads, as many over the XCDs
        BH = heads - 8 + (BH - heads) % 8
    us = {t: _grid_us(GRID_BASIC_BODY.get(t, t), f16, D, causal, BH, M, N) for t in tiles}
    if min(us.values()) < 0:
        return best
    fastest = min(us, key=us.get)
    return fastest if us[fastest] * margin < us[best] else best


def _near_own_corner(table: dict, key: str, BH: int, M: int, N: int) -> bool:
    """The shape is within a sixteenth of its swept bucket's upper corner: that timing is its own."""
    return key in table and all(16 * x > 15 * _bucket(x) for x in (BH, M, N))


def choose_fa_tile(variant: int, dtype, D: int, causal: bool, B: int, H: int, M: int, N: int,
                   candidates: list[FaTileChoice]) -> FaTileChoice:
    """Timed-table winner among candidates (the shape's bucket, else its nearest swept bucket of the
    same variant, dtype, head dim and causality), else the first candidate (preference order); but for the
    size a bucket was timed at, the kernel that the simulated schedules put ahead of it
    (choose_full_grid_tile). A bucket spans a factor of two in each size, and a grid's rounds, its longest
    block and the blocks that share a CU change within it: f16 D128 causal B1 H66 N=4200 in the bucket of
    H128 N=8192 takes 422 us with its persistent kernel and 325 dispatched. Split-KV launches
    differ: few rows fill the chip by splitting and keep the table's tile; full query tiles that split
    (prefill_splits) take the key-group kernel, or SPLIT_TILE for short splits."""
    table, key = load_tune_table()["fa"], fa_table_key(variant, dtype, D, causal, B, H, M, N)
    entry = _nearest_fa_entry(table, key)
    by_tile = {(c.block_m, c.block_n, c.waves, c.stages): c for c in reversed(candidates)}
    best = candidates[0]
    if entry is not None:
        want = tuple(entry["tile"])
        best = next((c for t, c in reversed(by_tile.items()) if t[:len(want)] == want), best)
    if _near_own_corner(table, key, B * H, M, N):
        return best
    if variant == hip_lib.FA_VARIANT_SLICED:
        if M < FULL_TILE_ROWS:
            return best
        splits = prefill_splits(B * H * math.ceil(M / 128), M, N, 128, 64, causal, D) if KEY_GROUP_TILE in by_tile else 1
        if splits > 1:
            return by_tile.get(SPLIT_TILE, best) if N <= splits * SPLIT_TILE_KEYS else by_tile[KEY_GROUP_TILE]
    known = GRID_BASIC_BODY if variant == hip_lib.FA_VARIANT_BASIC else GRID_STEP_US
    tiles = tuple(t for t in known if t in by_tile)
    f16, tile = "bfloat16" not in str(dtype), (best.block_m, best.block_n, best.waves, best.stages)
    if tile not in tiles:  # a kernel the model does not know (a caller's hint, a table's choice)
        return best
    margin = GRID_BUCKET_MARGIN if entry is None or key in table else GRID_MODEL_MARGIN
    if entry is None:
        others = tuple(t for t in tiles if t != PERSISTENT_TILE)
        tile = choose_full_grid_tile(f16, D, causal, B * H, M, N, tile, margin, others)
        tiles, margin = (tile, *(t for t in tiles if t == PERSISTENT_TILE)), GRID_UNTIMED_MARGIN
    return by_tile.get(choose_full_grid_tile(f16, D, causal, B * H, M, N, tile, margin, tiles), best)


@functools.lru_cache(maxsize=256)
def split_residency(dtype, D: int, block_m: int, block_n: int, waves: int, stages: int) -> int:
    """Workgroups of the sliced variant's split kernel one CU holds at once: the lower of the
    register bound (waves per SIMD x 4 SIMDs / waves per workgroup) and the LDS bound, from the
    compiler's resource table; RESIDENT_DEFAULT when the kernel is not in it."""
    tile = hip_lib.FaTile(block_m, block_n, waves, stages, 2)
    try:
        res = hip_lib.compiled_resources().get(hip_lib.fwd_kernel_symbol(hip_lib.FA_VARIANT_SLICED, dtype, D, tile))
    except (hip_lib.FaLibraryError, KeyError):
        res = None
    if not res:
        return RESIDENT_DEFAULT
    by_regs = max(1, int(res["Occupancy [waves/SIMD]"]) * 4 // waves)
    lds = int(res["LDS Size [bytes/block]"])
    by_lds = LDS_PER_CU // lds if lds else by_regs
    return max(1, min(by_regs, by_lds))


def _prefill_us(base: int, M: int, N: int, block_m: int, causal: bool, splits: int, D: int) -> float:
    """Modelled time of a prefill-shaped grid of base workgroups (with their splits, one or less per CU),
    but for what does not depend on the splits. A causal block sees M keys at most, however long N is."""
    tiles = math.ceil(math.ceil(N / 64) / splits)  # of a split
    us = min(math.ceil((min(M, N) if causal else N) / 64), tiles) * PREFILL_STEP_US[D] * (1.5 if block_m > 128 else 1)
    if splits > 1:
        rows = base * M / math.ceil(M / block_m)
        us += PREFILL_SPLIT_US + splits * rows * D * 8 / PREFILL_SPLIT_BYTES_PER_US
    return us


def prefill_splits(base: int, M: int, N: int, block_m: int, block_n: int, causal: bool, D: int = 128) -> int:
    """Splits that give each CU a workgroup, halved while half as many are clearly cheaper; 1 when no
    split pays. No split is left without keys."""
    n_tiles = max(1, math.ceil(N / block_n))
    splits = max(1, min(PREFILL_SPLIT_CUS // max(1, base), n_tiles // 2, MAX_SPLITS))
    us = _prefill_us(base, M, N, block_m, causal, splits, D)
    while splits > 3:
        half = _prefill_us(base, M, N, block_m, causal, splits // 2, D)
        if half > 0.9 * us:
            break
        splits, us = splits // 2, half
    if us * PREFILL_SPLIT_MARGIN >= _prefill_us(base, M, N, block_m, causal, 1, D):
        return 1
    return math.ceil(n_tiles / math.ceil(n_tiles / splits))


@functools.lru_cache(maxsize=4096)
def choose_splits(B: int, H: int, M: int, N: int, block_m: int, block_n: int, H_kv: int | None = None,
                  causal: bool = False, resident_per_cu: int = RESIDENT_DEFAULT, D: int = 128) -> int:
    """KV splits for the sliced variant, keeping at least two KV tiles per split.

    Decode-shaped grids (M < block_m: a few query rows per tile, K/V streaming dominates) split
    until NUM_CUS x resident_per_cu workgroups (the split kernel's resident capacity,
    split_residency) are in flight; their fp32 partials are a few rows each. Prefill-shaped grids
    (full query tiles) write partials as large as the output and read them back in the merge, so
    they split up to PREFILL_SPLIT_CUS workgroups and only where that pays (prefill_splits). Split
    launches of decode shapes pack the query heads of a GQA group into one tile (hip_lib.pack_group), so they
    count workgroups per kv head."""
    n_tiles = max(1, math.ceil(N / block_n))
    if n_tiles < 4:
        return 1
    if M >= block_m:
        if block_m > 128 and prefill_splits(math.ceil(M / 128) * B * H, M, N, 128, block_n, causal, D) == 1:
            return 1  # the rule the tile was chosen by (choose_fa_tile)
        return prefill_splits(math.ceil(M / block_m) * B * H, M, N, block_m, block_n, causal, D)
    target = NUM_CUS * max(1, resident_per_cu)

    def splits_for(base: int) -> int:
        if base >= target:
            return 1
        return max(1, min(math.ceil(target / base), n_tiles // 2, MAX_SPLITS))

    H_kv = H if H_kv is None else H_kv
    group = hip_lib.pack_group(H, H_kv, M, causal, block_m, 2)
    if group > 1:
        packed = splits_for(max(1, math.ceil(M * group / block_m) * B * H_kv))
        if packed > 1:
            return packed
    return splits_for(max(1, math.ceil(M / block_m) * B * H))


def gemm_cost(tile: tuple[int, int, int, int], M: int, N: int, K: int, ksplits: int = 1) -> float:
    """Modelled time (us) of a product with a tile, its K split over ksplits workgroups per tile."""
    c, lat, thr, ends = GEMM_COST[tile]
    tiles = math.ceil(M / tile[0]) * math.ceil(N / tile[1])
    slabs = max(1, math.ceil(K / tile[2]))  # K = 0 is the launch's to refuse
    per = math.ceil(slabs / ksplits)
    parts = math.ceil(slabs / per)
    steps = math.ceil(per / GEMM_GROUPS.get(tile, 1))
    us = c + (steps + ends) * math.hypot(lat * math.ceil(tiles * parts / NUM_CUS), thr * tiles * parts / NUM_CUS)
    if ksplits > 1:
        us += GEMM_SPLIT_US + parts * M * N * 8 / GEMM_SPLIT_BYTES_PER_US
    return us


def _octaves_to_bucket(M: int, N: int, K: int) -> float:
    """Distance of the sizes' bucket from the nearest swept one, as _nearest_gemm_entry measures it."""
    want = [math.log2(_bucket(x)) for x in (M, N, K)]
    return min(sum(abs(w - math.log2(int(part.lstrip("MNK")))) for w, part in zip(want, key.split("|")))
               for key in load_tune_table()["gemm"])


def _swept_size(M: int, N: int, K: int) -> bool:
    """The sizes are within a quarter of a swept bucket's own (its upper corner): its timing holds."""
    return gemm_table_key(M, N, K) in load_tune_table()["gemm"] and all(4 * x > 3 * _bucket(x) for x in (M, N, K))


def _runs_persistent(tile: tuple[int, int, int, int], M: int, N: int, K: int) -> bool:
    """The launch takes the persistent short-K kernel of the 256x128x64 tile, which the model does not know."""
    return (tile == (256, 128, 64, 8) and M % 256 == 0 and N % 128 == 0 and K % 64 == 0 and 256 <= K <= 1024
            and (M // 256) * (N // 128) % 8 == 0)


def _by_model(choice: tuple[int, int, int, int, int], entry: dict, candidates, M: int, N: int, K: int):
    """The timed choice, or the timed candidate of the entry that the model puts clearly ahead of it."""
    if choice[:4] not in GEMM_COST or _swept_size(M, N, K) or _runs_persistent(choice[:4], M, N, K):
        return choice
    timed = {t for t, _ in _gemm_ranked_tiles(entry)}
    best = min((t for t in candidates if t in GEMM_COST and t in timed), key=lambda t: gemm_cost(t, M, N, K),
               default=choice[:4])
    us, best_us = gemm_cost(choice[:4], M, N, K), gemm_cost(best, M, N, K)
    if us > GEMM_NEAR_MARGIN * best_us or us > GEMM_MODEL_MARGIN * best_us and _octaves_to_bucket(M, N, K) > 2:
        return (*best, GEMM_DEFAULT_GROUP_M)
    return choice


def choose_gemm_splits(M: int, N: int, K: int, tile: tuple[int, int, int, int]) -> tuple[tuple[int, int, int, int], int]:
    """(tile, ksplits): the given tile unsplit, or a split-K tile the model puts clearly ahead of it."""
    if tile not in GEMM_COST or _runs_persistent(tile, M, N, K):
        return tile, 1
    best = min((gemm_cost(t, M, N, K, s), t, s) for t in GEMM_SPLIT_TILES for s in GEMM_SPLITS)
    if best[0] * GEMM_SPLIT_MARGIN < gemm_cost(tile, M, N, K):
        return best[1], best[2]
    return tile, 1


def choose_gemm_tile(M: int, N: int, K: int, hint: tuple[int, int, int] | None = None) -> tuple[int, int, int, int, int]:
    """(block_m, block_n, block_k, waves, group_m) for a GEMM; ValueError when no built tile divides.

    Acceptance matches the reference selector (mma.py:63-81): K % 32 == 0 and either
    (M % 128 == 0 and N % 64 == 0) or (M % 64 == 0 and N % 256 == 0)."""
    if K % 32 != 0:
        raise ValueError("fast 2D contiguous matmul requires K % 32 == 0")
    # the reference's rule, stated here rather than left to the built tile set (a 64x64 tile
    # divides shapes the reference rejects)
    reference_ok = (M % 128 == 0 and N % 64 == 0) or (M % 64 == 0 and N % 256 == 0)
    cands = [t for t in gemm_candidates() if M % t[0] == 0 and N % t[1] == 0 and K % t[2] == 0] if reference_ok else []
    if not cands:
        raise ValueError(
            "fast 2D contiguous matmul requires a supported divisible tile: "
            "(M % 128 == 0 and N % 64 == 0), "
            "(M % 128 == 0 and N % 128 == 0), or "
            "(M % 64 == 0 and N % 256 == 0), with K % 32 == 0"
        )
    if hint is not None:
        # (block_m, block_n, block_k[, waves]) hints narrow the candidates; the table still ranks them
        hint = tuple(hint)
        hinted = [t for t in cands if t[:len(hint)] == hint]
        if not hinted and len(hint) > 3:  # no built tile with that wave count: keep the sizes
            hinted = [t for t in cands if t[:3] == hint[:3]]
        cands = hinted or cands
    # the bucket's (or nearest swept bucket's) winner when it divides, else its fastest timed tile
    # that does, unless the time model puts another clearly ahead; the preference order only without a
    # table
    entry = _nearest_gemm_entry(load_tune_table()["gemm"], gemm_table_key(M, N, K))
    if entry is not None:
        for tile, group_m in _gemm_ranked_tiles(entry):
            if tile in cands:
                return _by_model((*tile, group_m), entry, cands, M, N, K)
    t = cands[0]
    return (*t, _gemm_group_m(M, N, K, t))


def choose_gemm_tile_any(M: int, N: int, K: int) -> tuple[int, int, int, int, int]:
    """(block_m, block_n, block_k, waves, group_m) for any shape the kernel accepts (K % 8 == 0,
    N % 4 == 0; partial tiles in M, N and K are masked in the kernel): the divisible choice when
    there is one, else the tuned tile of the shape's bucket, else the first built tile no larger
    than the problem (rounded up to 64); the time model's choice where that is clearly ahead."""
    if K % 8 != 0 or N % 4 != 0:
        raise ValueError(f"gfx950 GEMM needs K % 8 == 0 and N % 4 == 0 (got M={M} N={N} K={K})")
    cands = gemm_candidates()
    entry = _nearest_gemm_entry(load_tune_table()["gemm"], gemm_table_key(M, N, K))
    try:
        choice = choose_gemm_tile(M, N, K)
        return _by_model(choice, entry, cands, M, N, K) if entry is not None else choice
    except ValueError:
        pass
    if entry is not None:
        for tile, group_m in _gemm_ranked_tiles(entry):
            if tile in cands:
                return _by_model((*tile, group_m), entry, cands, M, N, K)
    fit = [t for t in cands if t[0] <= -(-M // 64) * 64 and t[1] <= -(-N // 64) * 64]
    t = (fit or [min(cands, key=lambda t: t[0] * t[1])])[0]
    return (*t, GEMM_DEFAULT_GROUP_M)


def _gemm_group_m(M: int, N: int, K: int, tile) -> int:
    entry = load_tune_table()["gemm"].get(gemm_table_key(M, N, K))
    if entry is not None and list(entry["tile"]) == list(tile):
        return int(entry.get("group_m", GEMM_DEFAULT_GROUP_M))
    return GEMM_DEFAULT_GROUP_M


# ---- compiled resources ---------------------------------------------------------------------------

def fa_resources(variant: int, dtype, D: int, choice: FaTileChoice) -> dict[str, int] | None:
    sym = hip_lib.fwd_kernel_symbol(variant, dtype, D, choice.to_c())
    return _resources(sym)


def gemm_resources(tile: tuple[int, int, int, int]) -> dict[str, int] | None:
    sym = hip_lib.gemm_kernel_symbol(hip_lib.GemmTile(tile[0], tile[1], tile[2], tile[3], 1))
    return _resources(sym)


def _resources(sym: str) -> dict[str, int] | None:
    raw = hip_lib.compiled_resources().get(sym)
    if raw is None:
        return None
    return {
        "vgprs": int(raw.get("VGPRs", 0)),
        "agprs": int(raw.get("AGPRs", 0)),
        "sgprs": int(raw.get("TotalSGPRs", 0)),
        "lds_bytes": int(raw.get("LDS Size [bytes/block]", 0)),
        "scratch_bytes_per_lane": int(raw.get("ScratchSize [bytes/lane]", 0)),
        "waves_per_simd": int(raw.get("Occupancy [waves/SIMD]", 0)),
    }
