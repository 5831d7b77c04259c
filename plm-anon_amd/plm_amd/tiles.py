"""Tile selection for shapes without a tuned table entry, and the candidate set the tuner sweeps.

A tile is ``{"wave_frags", "k_waves", "split_k", "unroll"}`` (``struct plm_tile`` in
``include/plm_amd.h``). For the packed-weight GEMM behind ``fast_gemm`` (plm_gemm_packed), each
wavefront of a workgroup streams ``16*wave_frags`` weight rows, and either
``k_waves`` = 4, 8 or 16: that many wavefronts split the K range of one ``16*wave_frags``-row tile
(summed in LDS), or ``k_waves`` = 1: four wavefronts take adjacent rows of a ``64*wave_frags``-row
tile over the whole K range and share one copy of X through LDS. ``split_k`` workgroups split K further (fp32 partials summed
in split order); ``unroll`` (2, 4, 6 or 8) K steps of loads are in flight per wavefront. Items
(tile x split) = ``ceil(ceil(N/16) / tile_frags) * split_k`` over a persistent grid.

The chained round (plm_gemm_chain) uses the streaming kernel's tiles: ``64*wave_frags`` rows,
``unroll`` = 2 (``chain_tile``, ``chain_split`` below).
"""

from __future__ import annotations

import math

CU_COUNT = 256          # MI355X compute units
K_WAVES = 4             # wavefronts per workgroup of the row-split layout
LAYOUTS = (4, 8, 16, 1)  # k_waves: K split across 4, 8 or 16 wavefronts, or rows split across 4
LDS_LIMIT = 160 * 1024
FRAG = 1024             # bytes of one packed fragment
X_TILE = 16 * 80        # LDS transpose tile of one X fragment
WAVE_FRAGS = (1, 2, 4)
DEPTHS = (2, 4, 6, 8)
SPLITS = (1, 2, 3, 4, 6, 8, 12, 16)


def _regs(mt: int, nf: int, d: int, kw: int) -> int:
    xn = (mt + 3) // 4 if kw == 1 else mt
    return (d * (nf + xn) + nf * mt + (mt if kw == 1 else 0)) * 4


def pair_x(mt: int, kw: int) -> bool:
    """Whether X is staged two K steps at a time (mirrors ``packed_pair_x``)."""
    return kw == 1 or (kw == 8 and mt >= 4 and 2 * kw * mt * X_TILE + FRAG <= LDS_LIMIT)


def lds_body(mt: int, nf: int, kw: int) -> int:
    """LDS bytes before the warm-up sink (mirrors ``packed_lds_body``)."""
    red, xts = kw * nf * mt * FRAG, kw * mt * X_TILE * (2 if kw != 1 and pair_x(mt, kw) else 1)
    if kw == 1:
        return 4 * mt * X_TILE
    return red + xts if kw == 4 else max(red, xts)


def two_per_cu(M: int, cfg: dict) -> bool:
    """Whether two workgroups of this tile share a CU (mirrors ``packed_two_per_cu``)."""
    mt, nf, d, kw = math.ceil(M / 16), cfg["wave_frags"], cfg["unroll"], cfg["k_waves"]
    r = _regs(mt, nf, d, kw)
    if kw == 1:
        return r <= 100
    if kw > 4:
        return False
    return r <= 128 and (mt <= 6 or r <= 104)


def compiled(M: int, cfg: dict) -> bool:
    """Whether the library has a packed-GEMM kernel for this tile at width M (mirrors
    ``packed_compiled`` in csrc/packed_gemm.h: at most 20 accumulator fragments, and two
    workgroups per CU, or one with the pipeline within 320 registers)."""
    mt, nf, d, kw = math.ceil(M / 16), cfg["wave_frags"], cfg["unroll"], cfg["k_waves"]
    if not (1 <= mt <= 8 and nf in WAVE_FRAGS and d in DEPTHS and kw in LAYOUTS) or nf * mt > 20:
        return False
    if kw > 4:
        return lds_body(mt, nf, kw) + FRAG <= LDS_LIMIT and _regs(mt, nf, d, kw) <= (144 if kw == 8 else 60)
    return two_per_cu(M, cfg) or _regs(mt, nf, d, kw) <= 320


def tile_frags(cfg: dict) -> int:
    """16-row weight fragments of one workgroup tile."""
    return cfg["wave_frags"] * (K_WAVES if cfg["k_waves"] == 1 else 1)


def items(N: int, cfg: dict) -> int:
    return math.ceil(math.ceil(N / 16) / tile_frags(cfg)) * cfg["split_k"]


def steps_per_wave(K: int, cfg: dict) -> int:
    """32-wide K steps each wavefront streams per item (K-split layouts: the shortest share)."""
    return math.ceil(K / 32) // cfg["split_k"] // (1 if cfg["k_waves"] == 1 else cfg["k_waves"])


def candidates(M: int, N: int, K: int, supported=None) -> list[dict]:
    """Every sensible tile for ``(M, N, K)``; ``supported(cfg) -> bool`` filters to compiled kernels."""
    out = []
    for kw in LAYOUTS:
        for nf in WAVE_FRAGS:
            for d in DEPTHS:
                for split in SPLITS:
                    cfg = {"wave_frags": nf, "k_waves": kw, "split_k": split, "unroll": d}
                    if not compiled(M, cfg) or items(N, cfg) > 64 * CU_COUNT:
                        continue
                    if split > 1 and (steps_per_wave(K, cfg) < 2 or
                                      items(N, dict(cfg, split_k=max(1, split // 2))) >= 4 * CU_COUNT):
                        continue  # too little K per wavefront, or plenty of items with half the splitting
                    if supported is not None and not supported(cfg):
                        continue
                    out.append(cfg)
    return out


def _first_compiled(M: int, nf: int, layouts, supported) -> dict | None:
    for kw in layouts:
        for d in DEPTHS:
            cfg = {"wave_frags": nf, "k_waves": kw, "split_k": 1, "unroll": d}
            if compiled(M, cfg) and (supported is None or supported(cfg)):
                return cfg
    return None


# The wide kernel (csrc/wide_gemm.hip), which runs single linears on row-split tiles: its tiles as
# (64-row weight blocks, 16-row X fragments). From this packed size on, with more 128-row tiles than compute
# units and up to 64 rows, they run on the row-split kernel proper (``wide_preferred`` in csrc/packed_api.hip).
WIDE_TILES = ((1, 1), (1, 2), (1, 3), (1, 4), (1, 5), (1, 8), (2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (2, 6), (2, 8),
              (2, 10), (4, 8))
WIDE_WEIGHT_BYTES = 128 << 20
ROW_SPLIT_SPLITS = (1, 2, 3, 4, 6)


def runs_wide(M: int, N: int, K: int) -> bool:
    return (M > 64 or N <= 128 * CU_COUNT or
            math.ceil(N / 256) * 16 * math.ceil(K / 256) * 8 * FRAG < WIDE_WEIGHT_BYTES)


def row_split_splits(M: int, N: int, K: int) -> int:
    """K splits of a row-split tile on the wide kernel with the least modelled time (us): a CU's K steps at
    0.075 us or its loads' 82 KiB per us, whichever is longer, and for the partial sums' round trip 0.8 us,
    0.3 per split and 0.87 per MB. Measured at M = 56: 2048x2048 7.8 / 7.5 us with 1 / 2 splits,
    6144x2048 9.6 / 11.1, 2048x8192 23.6 / 16.8 / 14.1 / 16.1 with 1 / 2 / 4 / 6. Fewer than 32 rows take
    32 rows' splits: the join's latency does not fall with them as the modelled bytes do (6144x2048 at 2 to
    30 rows 9.6 us with 1, 11.0 with 2; 7680x2560 11.1 with 1, 12.6 with 2, 13.9 with 4)."""
    M, steps = max(M, 32), math.ceil(K / 32)

    def cost(split: int) -> float:
        work = min(math.ceil(math.ceil(N / (64 * nf)) * math.ceil(M / (16 * mt)) * split / CU_COUNT)
                   * max(0.075, (4 * nf + mt) / 82) for nf, mt in WIDE_TILES)
        join = 0.8 + 0.3 * split + 0.87e-6 * 4 * split * M * N if split > 1 else 0.0
        return math.ceil(steps / split) * work + join

    return min((s for s in ROW_SPLIT_SPLITS if s == 1 or steps // s >= 16), key=cost)


def _keeps_k_split(M: int, N: int, K: int, cfg: dict) -> bool:
    """Whether a long K over few columns keeps its K-split tile ``cfg``, whose items fit the CUs one each:
    their join is a sum in LDS and fewer partials, or none, while a row-split tile's items each walk a sixth
    of K at best. Row-split against K-split, us:

    * up to 16 rows: 1024x4096 8.6 / 7.7, 2048x8192 12.6 / 11.4, 2048x5632 10.5 / 9.6, 6144x2048 9.2 / 8.2,
      8192x2048 9.8 / 9.4, 7168x1536 8.3 / 7.9, 160x2504 6.0 / 5.5, 160x3368 6.7 / 5.9, 2048x3368 8.8 / 8.5;
      but 4096x3368 10.3 / 10.5, 2048x2048, which needs four splits, 7.2 / 7.5, 7168x1280 the same, 3072x1024
      4.8 / 6.7 and 2560x10240, whose 320 items take two rounds, 15.4 / 18.1;
    * 17 to 32: 160x3368 6.9 / 6.6, 512x4096 7.7 / 7.5, 768x6456 8.9 / 8.2, 1024x8192 11.0 / 9.6, 1024x12936
      13.3 / 12.4; but 768x4096 7.2 / 7.6, 1536x6456 10.9 / 11.9, 1536x12936 16.3 / 18.8;
    * 33 to 64: 160x4096 7.3 / 6.9 and 256x12936 9.9 / 9.6 at 48, 64x8192 8.3 / 7.3 at 56; but 512x6456
      8.9 / 9.2 at 42, 160x8192 at 56 the same."""
    if items(N, cfg) > CU_COUNT:
        return False
    if M <= 16:
        return K >= 4096 or cfg["split_k"] == 1 or (K >= 3072 and N <= 2048) or (K > 2048 and N <= 256)
    if M <= 32:
        return (K >= 4096 and N <= min(1024, K // 6)) or (K >= 3328 and N <= 256)
    return K >= 4096 and N <= (256 if M <= 48 else 64)


def heuristic_tile(M: int, N: int, K: int, supported=None) -> dict:
    """A reasonable tile without measurement: rows split across the wavefronts (the wide kernel's
    linears, with ``row_split_splits``'s K splits; the row-split kernel itself where not ``runs_wide``),
    else, and up to 64 rows where ``_keeps_k_split``, ``k_split_tile``. K splits only where
    ``k_split_tile`` has them too: a weight whose items fill the CUs needs no workspace, so that a call on it
    can be captured first thing, and run beside one on another stream (us unsplit / split: 6144x4096 at
    M = 30 14.1 / 15.5, 8192x8192 at 42 32.9 / 29.5, 6144x14336 at 42 49.3 / 39.3; K-split tiles 15.5, 42.3,
    62.7)."""
    if M <= 64 and K >= 1536 and _first_compiled(M, 2, (8, 4), supported):
        cfg = k_split_tile(M, N, K, supported)
        if _keeps_k_split(M, N, K, cfg):
            return cfg
    for nf in (2, 1, 4):
        cfg = _first_compiled(M, nf, (1,), supported)
        if cfg is None:
            continue
        if runs_wide(M, N, K):
            split = k_split_tile(M, N, K)["split_k"] > 1
            return dict(cfg, split_k=row_split_splits(M, N, K) if split else 1)
        if math.ceil(N / 16) // (K_WAVES * nf) >= CU_COUNT:
            return cfg
    return k_split_tile(M, N, K, supported)


def k_split_tile(M: int, N: int, K: int, supported=None) -> dict:
    """A tile of the K-split layouts without measurement: 32 rows per wavefront with a two-stage pipeline,
    K split across 8 wavefronts (4 where 8 is not compiled), and K splitting until about three quarters
    of the compute units have an item, keeping at least two K steps per wavefront."""
    for nf in (2, 4, 1):
        cfg = _first_compiled(M, nf, (8, 4), supported)
        if cfg is None:
            continue
        split = 1
        while (items(N, dict(cfg, split_k=split)) < CU_COUNT * 3 // 4 and
               steps_per_wave(K, dict(cfg, split_k=2 * split)) >= 2 and split < 16):
            split *= 2
        return dict(cfg, split_k=split)
    raise ValueError(f"no compiled tile fits (M={M}, N={N}, K={K})")


def packed_chain_split(N: int, K: int, cfg: dict, workgroups: int) -> int:
    """K split of one linear of a packed chain (every linear ends at a grid barrier, so its time
    is that of the busiest workgroup): the split with the least estimated busiest-workgroup time,
    counting each item's K steps per wavefront plus a fixed cost of a few steps for the item's end
    (reduction, stores; with split > 1 the partial round trip)."""
    if cfg["k_waves"] == 1:   # linear by linear on the wide kernel; its splits hardly depend on the width
        return row_split_splits(64, N, K)
    tiles_ = math.ceil(math.ceil(N / 16) / tile_frags(cfg))
    ks = math.ceil(K / 32)
    kw = cfg["k_waves"]
    best, best_cost = 1, None
    for split in SPLITS:
        if split > 1 and ks // split // kw < 2:
            break
        per_wg = math.ceil(tiles_ * split / workgroups)
        steps = max(cfg["unroll"], math.ceil(ks / split / kw))
        cost = per_wg * (steps + (3 if split == 1 else 8))
        if best_cost is None or cost < best_cost:
            best, best_cost = split, cost
    return best


# ---------------------------------------------------------------- streaming kernel (chains)

STREAM_UNROLL = 2
LDS_BYTES = 160 * 1024 - 256
TABLE_RESERVE = 16 * 1024
LOADERS = 4             # loader wavefronts per workgroup (PLM_STREAM_LOADERS in csrc/stream_gemm.h)


def _slot(M: int, nf: int) -> int:
    """Ring slot bytes of csrc/stream_gemm.h: one chunk (two K steps) of the X rows and of the
    tile's 64*nf weight rows."""
    mt = math.ceil(M / 16)
    x_groups = -(-2 * mt // LOADERS) * LOADERS     # X row groups, padded to the loader count
    return x_groups * 1024 + K_WAVES * nf * 16 * 128


def ring_slots(M: int, cfg: dict, table_bytes: int = TABLE_RESERVE) -> int:
    """Chunk slots of the streaming kernel's LDS ring (mirrors ``ring_for_table`` in
    csrc/stream_gemm.h): what fits beside the descriptor table, at most 8; 0 if under two."""
    slot = _slot(M, cfg["wave_frags"])
    free = LDS_BYTES - table_bytes
    if free <= 0:
        return 0
    r = min(free // slot, 8)
    return r if r >= 2 else 0


def stream_compiled(M: int, cfg: dict) -> bool:
    """Whether the streaming kernel (plm_gemm, plm_gemm_chain) is compiled for this tile at width M
    (mirrors ``stream_compiled`` in csrc/stream_gemm.h)."""
    mt, nf = math.ceil(M / 16), cfg["wave_frags"]
    if not (1 <= mt <= 8 and nf in WAVE_FRAGS and cfg["unroll"] == STREAM_UNROLL and cfg["k_waves"] == K_WAVES):
        return False
    if ring_slots(M, cfg) < 2:
        return False
    return nf * mt <= 16


def chunks_per_item(K: int, cfg: dict) -> int:
    return math.ceil(math.ceil(K / 32) / cfg["split_k"] / STREAM_UNROLL)


# Tile of a chained round (plm_gemm_chain): 64-row tiles.
CHAIN_TILE = {"wave_frags": 1, "k_waves": K_WAVES, "split_k": 1, "unroll": STREAM_UNROLL}


def chain_tile(M: int) -> dict:
    """CHAIN_TILE at width M (64-row tiles are compiled at every width up to 128)."""
    if not stream_compiled(M, CHAIN_TILE):
        raise ValueError(f"no chain tile is compiled at M={M}")
    return dict(CHAIN_TILE)


def packed_chain_tile(M: int) -> dict:
    """Tile of a packed chained round at width M. At M <= 48, 32-row tiles of eight wavefronts
    splitting K on a four-stage pipeline, one workgroup per CU (the two-stage kernel's smaller
    register count admits two, which measured slower: 1167 against 1025 us for the 1.3B-shape round
    at M = 42). Wider rounds take a row-split tile, whose linears run one after the other on the wide
    kernel: the eight wavefronts each load every X fragment of their K range, seven of them at
    M = 110, while the wide kernel stages X once per workgroup. Per linear, row-split against
    eight-way: hidden 1024 6.4 / 6.9 us at M = 56 and 6.5 / 9.6 at 110 (but 6.4 / 5.6 at M = 30),
    hidden 2048 10.2 / 10.5 and 12.0 / 15.3, hidden 2560 13.9 / 17.0 and 16.5 / 23.9."""
    if M > 48:
        return {"wave_frags": 2, "k_waves": 1, "split_k": 1, "unroll": 2}
    return {"wave_frags": 2, "k_waves": 8, "split_k": 1, "unroll": 4}


def chain_split(N: int, K: int, cfg: dict = CHAIN_TILE, workgroups: int = CU_COUNT) -> int:
    """K split of one linear inside a chain: the smallest power of two that gives about one item
    per resident workgroup, keeping at least two chunks per item."""
    tiles = math.ceil(N / (64 * cfg["wave_frags"]))
    split = 1
    while (tiles * split < workgroups * 3 // 4 and chunks_per_item(K, dict(cfg, split_k=2 * split)) >= 2
           and split < 16):
        split *= 2
    return split
