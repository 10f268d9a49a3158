"""Which GEMM runs a linear of a step: md_linear (hand-written weight-streaming skinny GEMM, csrc/gemm.hip) or the
library GEMM (hipBLASLt through F.linear, with the TunableOp table of magicdec_amd/tuned/).

The rules below are the outcome of the same-box, graph-captured A/B of profiles/r02_gemm_ab.txt (tools/gemm_bench.py:
every decode / verify shape of the 8B and 1B models timed on both, weights cycled to defeat the Infinity Cache):

  * md_linear over the STREAMING weight layout (ops.PackedWeight) wins where the product is a long weight stream --
    M <= 64: w1|w3 (+ fused SiLU*mul), w2 and the lm head of the 8B model, w1|w3 and the lm head of the 1B model
    (4.5-6.0 TB/s against 3.0-5.1); M <= 128: w1|w3 and w2; M = 256: w2 only (K = 14336);
  * the library wins the short streams (qkv / wo of both models, every TP8 shard: the whole call is 10-20 us and the
    split-K combine of md_linear costs a second launch) and everything at M = 256 with K <= 4096 (there the product is
    MFMA / LDS bound, not HBM bound: a 256-row activation slab has to be re-read per 128 output columns).

  * the LAUNCH-BOUND small products (every linear of the 1B draft model, every tensor-parallel shard, the
    narrow projections of an 8B step) go to md_linear_fused (csrc/tilegemm.hip): one launch for the product AND the op
    behind it (rope+append, residual add, SiLU*mul), no split-K combine, no partial sums in HBM.

  * the 129..256-ROW products of a verify step whose column count fills the chip without splitting K, and the
    K = 14336 down projection, go to md_linear_block (csrc/blockgemm.hip: 256 x 128 block tiles, LDS-DMA rings, loader +
    MFMA waves) -- profiles/r04_block_ab_final.txt, same process, graph-captured, weights cycled (us; "lib" includes the
    elementwise kernel behind it, "skinny" its combine launch):
        8B w1|w3 + SiLU*mul  M = 256: lib 85-89 (68.8 + 6.2 inside the cfg3 trace), skinny 108-119, block 67-72
        8B w2 + add + norm   M = 256: lib 66-68, skinny 53.5-55, block 48.6-49.9
        8B lm head           M = 256: lib 293-297, skinny 345-350, block 274-278
        8B w1|w3             M = 128: lib 58-65, skinny 61.6-63.8, block 52.3-57
    and NOT the narrow projections, where splitting K over ~256 workgroups costs a partial-sum round trip the product is
    too small to pay for (wqkv 30-32 vs lib 27 + 6.3 for rope/append: a wash; wo 34-35 vs 25; every TP8 shard slower).

  * the rows of a PROMPT (more than 256) go to md_linear_prompt (csrc/promptgemm.hip), which reads the streaming layout too: prompt_rows.

A weight a hand-written kernel will serve is re-packed once at setup_caches (Transformer._pack_weights); the row-major
copy stays for the products that are left to the library.  MAGICDEC_GEMM=hip forces md_linear wherever it supports the shape,
MAGICDEC_GEMM=lib forces the library, MAGICDEC_FUSED=0/1 switches md_linear_fused off / on everywhere (the A/B
switches)."""
import functools
import os
import re

_MODE = os.environ.get("MAGICDEC_GEMM", "auto")
_FUSED = os.environ.get("MAGICDEC_FUSED", "auto")     # "0": never md_linear_fused, "1": wherever it supports the shape
MIN_STREAM_BYTES = 60e6        # bf16 weight bytes of one call above which the streaming kernel wins at M <= 64
MIN_STREAM_BYTES_M128 = 100e6
# md_linear_fused reads a weight tile once per 32-row M tile (through L2) and a 32-row slab of the activations once per
# weight tile: it is the launch-bound regime's kernel.  Rules from the A/B of tools/fused_bench.py
# (profiles/r03_fused_ab.txt; "unfused" there = hipBLASLt + the small kernel behind it, graph-captured, weights cycled):
#   * M <= 128 (draft steps, autoregressive target steps): fused while m_tiles x weight bytes <= 70 MB and K <= 4096 --
#     the 1B model's wqkv 8.0 vs 15.6 us, wo 10.3 vs 12.2, every TP4 shard of it (6.1-9.8 vs 10.0-15.0), every TP8
#     shard of the 8B model at M = 64 (8.9-12.9 vs 10.8-15.7).  Above that the x slab (M x K, one hot MB) is re-read by
#     every column tile through the same L2 channels and the kernel falls behind (1B w2, K = 8192: 23.6 vs 19.0;
#     1B w1|w3, 1024 tiles: 22.2 vs 20.4) -- those stay on md_linear / the library;
#   * M = 256 (verify): only the qkv projection with its rope+append epilogue (8B/8: 9.2 vs 14.0 us, 8B/4: 18.5 vs
#     19.8); wo / w1|w3 / w2 shards are served faster by the library (14.4 vs 14.1, 30.2 vs 22.9, 23.0 vs 16.6).
FUSED_MAX_L2_BYTES = 70e6
FUSED_MAX_L2_BYTES_T22 = 120e6
FUSED_DEEP_SWIGLU_T22_MAX_L2_BYTES = float(os.environ.get("MAGICDEC_DEEP_SWIGLU_L2", "150e6"))   # (env: A/B switch)
_SHARD70B = os.environ.get("MAGICDEC_SHARD70B", "1")     # "0": without the two rules for the 70B shards (A/B switch)
FUSED_MAX_K = 4096
FUSED_QKV_M256_MAX_L2_BYTES = 110e6
# the bounds of _measured(): tile traffic (M tiles x weight bytes) of a qkv projection (K <= 4096, deeper), and the weight bytes up to
# which 5..32 rows of a gated projection prefer the tile kernel
FUSED_QKV_MAX_L2_BYTES = 270e6
FUSED_QKV_DEEP_MAX_L2_BYTES = 230e6
SWIGLU_ONE_TILE_MAX_BYTES = 210e6
# (profiles/r05_fused_tp8_shard_tiles.txt, M = 256): two more TP8 shards of the 8B verify pass go to the fused kernel --
# w1|w3 (29.4 MB; 2 x 2 tiles: 21.1-22.3 us against 24.1 for the library + the SiLU*mul launch) and wo (4.2 MB, K = 512:
# 12.0 against 14.1 incl. the add + norm behind it); w2 (14.7 MB: 17.1 vs 16.9) and everything wider stay on the library
FUSED_M256_SWIGLU_MAX_BYTES = 32e6
FUSED_M256_NARROW_MAX_BYTES = 5e6
FUSED_M256_RESID_T22_MAX_BYTES = 34e6
_WO256 = os.environ.get("MAGICDEC_WO256", "1")        # "0": the 8B wo at 256 rows stays on the library (A/B switch)
# a linear that can ALSO absorb the RMSNorm in front of it (deferred norm: its input is the un-normalised h of a fused
# residual epilogue) saves that launch (~5 us + a boundary): the 1B w1|w3 at M = 64 (134 MB of tile traffic, 22.2 us
# against md_linear's 21.9) then wins on the fused kernel
FUSED_MAX_L2_BYTES_WITH_NORM = 140e6


# md_linear (the streaming kernel) can absorb the same deferred norm (md_linear_normed): a slab is normalised once
# per workgroup on its way to LDS.  Free while the kernel waits for weights anyway (<= 64 rows); at 128 / 256 rows the
# staging of a slab is as much vector work as its MFMAs and the launch it saves is cheaper (tools/fused_bench.py --pro 1:
# 1B w1|w3 at 128 rows 35.4 vs 30.1 us with the norm as its own launch, 8B at 256 rows 179 vs 105).
SKINNY_NORM_MAX_M = 64
_SKINNY_NORM = os.environ.get("MAGICDEC_SKINNY_NORM", "auto")     # "0": always materialise the norm in front of md_linear


def skinny_absorbs_norm(M: int) -> bool:
    return _SKINNY_NORM != "0" and M <= SKINNY_NORM_MAX_M


def _changed():
    """A switch or the table of tuned solutions is another one."""
    _measured.cache_clear()
    prompt_rows.cache_clear()


def set_mode(mode: str):
    global _MODE
    assert mode in ("auto", "hip", "lib")
    _MODE = mode
    _changed()


def set_fused(mode: str):
    global _FUSED
    assert mode in ("auto", "0", "1")
    _FUSED = mode
    _changed()


def mode() -> str:
    return _MODE


def fused_mode() -> str:
    return _FUSED


def joint_launches() -> bool:
    """May a product share a launch with what is in front of it, or do the switches above say which kernel (or none) it runs on?"""
    return _MODE == "auto" and _FUSED == "auto"


_PACKED = os.environ.get("MAGICDEC_PACKED_COPIES", "auto")   # "0": no streaming-layout copies at all (every linear on the
                                                             # library / the row-major md_linear): saves their HBM


def set_packed_copies(mode: str):
    global _PACKED
    assert mode in ("auto", "0")
    _PACKED = mode


def want_packed(N: int, K: int, swiglu: bool = False, int8: bool = False, rows=None) -> bool:
    """Re-pack this weight into the streaming layout at load time?  Only when a hand-written kernel may actually be
    chosen for it at some row count of a decode / verify step: `rows` = the counts the engine will run (the back-end knows
    them: batch x {1, 2, dec_len}), or None = any of 1..256 (not every bf16 weight with
    K % 128 == 0: the 8B wqkv, served by the library at 64 and 256 rows, is not packed for the 32-row
    steps that a batch of 64 never runs)."""
    if _MODE == "lib" or _PACKED == "0" or K % 64:
        return False
    if int8:
        return K % 128 == 0            # int8 rows are only streamed by md_linear, at every row count
    if _MODE == "hip" or _BLOCK == "1" or _FUSED == "1" or _SPLIT == "1":
        return True
    kinds = ("swiglu",) if swiglu else ("plain", "resid", "qkv")
    for M in ((1,) + tuple(range(32, 257, 32)) if rows is None else tuple(m for m in rows if m <= 256)):
        # (default: every 32-row tile count a rule can depend on)
        for kind in kinds:
            if use_skinny(M, N, K, swiglu, False, True, kind):
                return True
            if use_block(M, N, K, kind) or use_fused(M, N, K, kind, absorbs_norm=True) or use_split(M, N, K, kind):
                return True
    return False


def want_packed_prompt(N: int, K: int) -> bool:
    """Re-pack a weight that only the rows of prompts are multiplied by?"""
    return _MODE != "lib" and _PACKED != "0" and K % 64 == 0 and prompt_rows(8192, N, K) > 0


# Shapes the library holds a tuned solution for (tuned/gemm_gfx950.csv, "tn_N_M_K_...": lines that name one; "Default" says that the
# tuning found none better than the library's own choice).  Some rules below leave these alone: 8B wqkv (6144 x 4096) at 256 rows 32.1 us
# with it, 37.5 on the block kernel; 4096 x 3584 + residual at 128 rows 19.8 against 21.6.
_TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tuned", "gemm_gfx950.csv")
_TUNED = None


def tuned_table(path):
    """The table of tuned solutions that PyTorch took (Engine.utils.enable_tuned_gemms), None: it refused it (other library versions),
    so that none of its solutions is in use."""
    global _TABLE, _TUNED
    _TABLE, _TUNED = path, None
    _changed()


def _tuned(M: int, N: int, K: int) -> bool:
    global _TUNED
    if _TUNED is None:
        rows = set()
        if _TABLE is not None and os.path.exists(_TABLE):
            with open(_TABLE) as f:
                for line in f:
                    m = re.match(r"GemmTunableOp_BFloat16_TN,tn_(\d+)_(\d+)_(\d+)_[^,]*,(?!Default,)", line)
                    if m:
                        rows.add((int(m.group(2)), int(m.group(1)), int(m.group(3))))
        _TUNED = rows
    return (M, N, K) in _TUNED


CUS = 256


def _last_round(workgroups: int) -> float:
    """Rounds of the chip that so many workgroups take, over the rounds they fill: 1.0 = the last one is full."""
    return -(-workgroups // CUS) * CUS / workgroups


def _last_chunk(K: int) -> float:
    """The same of the tile kernel's eight waves, which stage K in chunks of 128 each: 1.0 = the last chunk is whole."""
    return -(-K // 1024) * 1024 / K


@functools.lru_cache(maxsize=4096)
def _slices(kind: str, N: int, K: int) -> int:
    """K slices of md_linear ("skinny") or md_linear_fused_split ("tile") at up to 32 rows; 0: not this shape."""
    from .. import ops
    return ops.linear_planes_count(kind, 1, N, K)


def _skinny_one_round(N: int, K: int) -> bool:
    """Are md_linear's workgroups (128 columns of one K slice) one nearly full round of the chip?"""
    return 0.8 * CUS < -(-N // 128) * _slices("skinny", N, K) <= CUS


@functools.lru_cache(maxsize=16384)      # (asked three times for every linear of a step that is not captured; _changed clears it)
def _measured(M, N, K, kind, absorbs_norm):
    """The kernel for the shapes where the general rules below (drawn for the 1B and 8B models at 32, 64, 128 and 256 rows) were
    measured to pick a slower one of the framework's own kernels, or the library where one of them is faster: "fused" | "block" |
    "skinny" | "split", None: the general rules.  Times in us, the whole sub-step (with the add + norm, the rope or the SiLU*mul
    behind it), graph-captured, weights cycled; every kernel at 13 row counts of 180 shapes a kind, the zoo's among them.  `kind`
    "planes": an output projection whose combine is the residual add + norm launch of a model that keeps its residual in float32 (the
    tile kernel's residual epilogue is no choice there).
    The library's own choice above 128 rows is even but for exact multiples of 32, where it takes a slow kernel (6144 x 4096: 25.7..26.6
    at 161..255 rows, but 33.3 at 192 and 36.8 at 224; 5120 x 5120: 29.7 at 193, 41.5 at 192, 49.6 at 256): `nice` below."""
    if M > 256 or K % 128 or N % 32:
        return None
    nbytes, m_tiles, n_tiles, tiles = N * K * 2, (M + 31) // 32, N // 32, N // 128
    nice = M % 32 == 0
    if kind == "plain":
        # a head in one round of block workgroups (128 columns each: 160..256), 33..128 rows.  Below the streaming kernel's sizes K = 768
        # x 32 000 19.4 / 30.9 on the tile kernel -> 15.3 / 16.4 (64 / 128 rows); against the library above 64 rows from 200 workgroups
        # on (29 952 x 1280 23.8 -> 22.8, but 21 504 x 2048 26.5 against 29.1), against the streaming kernel above 64 rows if the round
        # is full (32 000 x 4096 56.6 -> 52.5, 30 208 x 4096 53.1 against 57.9).  Up to 64 rows that one stays ahead: 32 000 x 2048 27.0 /
        # 30.6, x 4096 49.2 / 52.1 (if K does not fall into many slices: 30 848 x 2944, 23 of them, 67.8 -> 41.6 at 39 rows)
        least = BLOCK_MIN_TILES if nbytes < MIN_STREAM_BYTES or M <= 64 else 200 if nbytes < MIN_STREAM_BYTES_M128 else 240
        if (32 < M <= 128 and N % 128 == 0 and least <= tiles <= CUS
                and (M > 64 or nbytes < MIN_STREAM_BYTES or _slices("skinny", N, K) > 8)):
            return "block"
        # one M tile over a long stream of columns: the tile kernel's workgroups each finish their columns, nothing to combine -- in
        # fewer than two rounds, or where the last round and the last chunk of K are nearly full.  128 256 x 4096 at one row 172 -> 158,
        # x 2048 92 -> 81; 32 000 x 4096 47.6 -> 45.5; but 16 896 x 4224 (2.06 rounds, 4.1 chunks) 27.5 against 32.4, 37 120 x 3200 (4.5,
        # 3.1) 39.5 against 42.4 and 115 328 x 1280 (14.1, 1.25) 49.8 against 56.6.  To 32 rows only within four rounds (32 000 x 4096
        # 49.9 -> 49.4 at 26 rows, 14 336 x 4096 26.2 -> 24.8; 54 912 x 2560 17 % slower); deep and wide to 8 (73 472 x 4736 at 16: 109
        # against 115)
        if (N >= 14336 and nbytes >= MIN_STREAM_BYTES and K >= 1024
                and (n_tiles < 2 * CUS or (_last_round(n_tiles) <= 1.09 and _last_chunk(K) <= 1.15))
                and M <= (8 if K > FUSED_MAX_K and n_tiles > 4 * CUS else 16 if K > FUSED_MAX_K or n_tiles > 4 * CUS else 32)):
            return "fused"
    if kind == "swiglu":
        # up to four rows the tile kernel stages four, also with a norm to absorb: 28 672 x 4096 43.9 -> 42.2, 37 888 x 3584 52.0 ->
        # 47.4, 55 296 x 5120 92.6 -> 88.0; at 16 rows 44.9 / 51.7 / 92.0 on the skinny kernel against 44.7 / 52.4 / 95.6
        # (not 61 312 x 1152, its second chunk of K nearly empty: 28.3 against 34.2)
        whole = n_tiles < 2 * CUS or _last_chunk(K) <= 1.15
        if M <= 4 and N >= 14336 and nbytes >= MIN_STREAM_BYTES and whole:
            return "fused"
        # without a norm: to 16 rows 24 576 x 4096 38.4 -> 35.5, 22 016 x 4096 34.5 -> 31.8 (26 624 x 4864, 259 MB: 5 % slower); to 32
        # rows within three rounds, the last one nearly full: 24 576 x 4096 41.3 -> 38.6, 22 016 x 4096 36.5 -> 35.8, but 18 432 x 5120
        # (2.25 rounds) 35.5 against 39.6 and 27 648 x 3584 (3.4) 40.4 against 42.5
        if (not absorbs_norm and N >= 14336 and MIN_STREAM_BYTES <= nbytes <= SWIGLU_ONE_TILE_MAX_BYTES and whole
                and (M <= 16 or (M <= 32 and n_tiles <= 3 * CUS and _last_round(n_tiles) <= 1.19))):
            return "fused"
        # 65..128 rows, more than one round of block workgroups (296 or 432: the last round nearly empty): 37 888 x 3584
        # 84.6 -> 63.2 on the skinny kernel, 55 296 x 5120 133 -> 102 (128 rows), 124 -> 99 (96)
        if 64 < M <= 128 and N % 128 == 0 and tiles > CUS:
            return "skinny"
    if kind in ("resid", "planes") and N <= 8192:
        # the deep projections at one M tile: the tile kernel's K split where its workgroups (64 columns of one slice) are one nearly
        # full round.  3584 x 18 944 30.8 / 32.5 -> 28.5 / 31.9 (1 / 31 rows), 4096 x 14 336 27.1 -> 25.7, 4096 x 18 432 32.4 -> 30.3;
        # with half a round (4096 x 11 008) 23.1 against 26.8, with a second (5120 x 13 824) 32.3 against 36.7
        if (kind == "resid" and K >= 8192 and nbytes >= MIN_STREAM_BYTES and M <= 32 and N % 64 == 0
                and 0.8 * CUS < N // 64 * _slices("tile", N, K) <= CUS):
            return "split"
        if FUSED_MAX_K < K < 8192:
            if kind == "planes":
                # 2048 x 7680: 16.0 / 20.3 / 26.5 / 24.6 / 32.2 in the library -> 12.9 / 14.5 / 16.9 / 21.4 / 28.3 (1 / 32 / 64 / 128 / 256
                # rows); the tile kernel's K split 14.8 / 17.1 / 24.2 / 22.8 / 35.0.  More slices are more planes to write and add, the
                # more so the more rows: 896 x 7680 (60) 15.5 against 19.8 at 41 rows, 2048 x 4864 (19) 18.2 against 20.7 at 101,
                # 2176 x 5120 (14) 24.4 against 27.8 at 144 but 30.4 -> 25.8 at 256; and a second round costs (6784 x 4992, 689
                # workgroups, 34.0 against 38.3 at 75; 3072 x 7040, 264, 40.1 against 48.7 at 256)
                slices, one = _slices("skinny", N, K), _skinny_one_round(N, K)
                workgroups = -(-N // 128) * slices
                if M <= 64:
                    return "skinny" if slices <= 50 else None
                if M <= 128:
                    return "skinny" if (one and slices <= 30) or (slices <= 15 and workgroups <= 1.7 * CUS) else None
                return "skinny" if (one and K >= 6000) or (nice and slices <= 15 and workgroups <= CUS) else None
            if K <= 5632 and M <= 128:
                if M <= 32 and nbytes < 30e6:
                    return "skinny"   # 2048 x 5632: 14.3 / 13.4 / 18.4 in the library -> 11.4 / 11.7 / 13.2 (1 / 8 / 32 rows)
                # one round of the tile kernel: 2048 x 5632 21.1 / 19.4 -> 15.2 / 14.5 (64 / 128), 5120 x 5120 22.8 -> 16.5 (32);
                # 4608 x 4352 at 64 (288 workgroups) 23.6 against 30.8
                if n_tiles * m_tiles <= CUS:
                    return "fused"
        # 3584..5632 deep and wide, more than one round of tile workgroups: the library against the skinny kernel (up to 128 rows):
        # 3584 x 3584 23.8 / 26.5 -> 22.4 / 23.3 (96 / 128), 5120 x 5120 26.1 / 36.6 -> 22.8 / 27.9 (64 / 128), 4096 x 4096 25.9 -> 21.9
        # (96); or the block kernel, at multiples of 32 rows and for the deeper ones: 3584 x 3584 33.8 -> 25.5 (192; at 170 24.3 against
        # 27.1), 5120 x 5120 54.8 -> 32.6 (256), 38.6 -> 33.0 (247)
        if (kind == "resid" and 3584 <= K <= 5632 and N >= 3584 and N % 128 == 0 and M > (32 if K > FUSED_MAX_K else 64)
                and not (M > 128 and _WO256 != "0" and K <= FUSED_MAX_K and nbytes <= FUSED_M256_RESID_T22_MAX_BYTES
                         and (N // 64) * ((m_tiles + 1) // 2) >= 192) and not _tuned(M, N, K)):
            # (6912 x 3968, 31 slices: 28.6 against 47.6; 6784 x 4992, 689 workgroups, 32.5 against 37.9)
            if M <= 128 and _slices("skinny", N, K) <= 15 and -(-N // 128) * _slices("skinny", N, K) <= 1.6 * CUS:
                return "skinny"
            if M > 128 and (nice or (K >= 5120 and N >= 4608)):
                return "block"
    # 4096 x 4096 on the tile kernel's K split 36.3 / 33.8 -> 27.5 / 28.8 (192 / 256 rows), 3456 x 1664 94 -> 32 (213); the wide ones
    # only in one round (5632 x 768, 264 workgroups, 22.7 against 30.8)
    if (kind == "planes" and K <= FUSED_MAX_K and M > 128 and use_fused(M, N, K, "resid")
            and (N <= 4608 or -(-N // 128) * _slices("skinny", N, K) <= CUS)):
        return "skinny"
    if kind == "qkv" and K <= 5632 and N >= 4096 and n_tiles * m_tiles >= 100:
        # the tile kernel ends in rope + append; the library needs a launch for that: 4608 x 3584 25.0 / 27.8 -> 18.0 / 22.8 (96 / 128
        # rows), 6144 x 4096 28.5 -> 25.0 (96), 26.4 -> 25.0 (128), 7168 x 5120 31.5 / 34.7 -> 26.0 / 32.2 (64 / 96).  The 8B one is
        # level at exactly 64 rows (22.8 / 22.2; 23.1 / 21.1 at 47): the library, so that 64- and 256-row steps need no second copy
        lim = FUSED_QKV_MAX_L2_BYTES if K <= FUSED_MAX_K else FUSED_QKV_DEEP_MAX_L2_BYTES
        level = M == 64 and 3584 < K <= FUSED_MAX_K and 1.25 < _last_round(n_tiles * m_tiles) < 1.5
        if M <= 128 and m_tiles * nbytes <= lim:
            return None if level else "fused"
        # above 128 rows where the library is slow: multiples of 32 (4608 x 3584 35.2 / 40.5 -> 27.3 / 32.0 at 192 / 256), 129..159
        # (6144 x 4096 44.8 -> 29.5; not the wide ones: 8192 x 3200 28.1 against 36.2) and 193..223 narrow (4608 x 3584 38.0 -> 28.1,
        # 4224 x 4224 40.2 -> 33.7; 5504 x 3584 29.7 against 33.2)
        if M > 128 and m_tiles * nbytes <= lim and not _tuned(M, N, K):
            if n_tiles * m_tiles <= (6.5 if nice else 4.5 if M < 160 else 4.05 if m_tiles == 7 else 0) * CUS:
                return "fused"
    # ... and where its budget ends, the block kernel ahead of the rope launch: 7168 x 5120 39.3 / 48.5 / 57.4 -> 36.6 / 40.3 / 43.8
    # (128 / 192 / 256), 6144 x 4096 39.0 -> 35.6 (192), 36.8 -> 33.7 (224)
    if kind == "plain" and 96 < M and 4096 <= K <= 5632 and N % 128 == 0 and 40 <= tiles <= 64 and not _tuned(M, N, K):
        # (other row counts than multiples of 32 where it is deep, 7168 x 5120 38.5 -> 36.5 at 103; 5120 x 4096 is level, 22.9 at 97)
        if (K >= 4608 or M >= 192) if nice else tiles <= 56 and (K >= 5120 or (tiles == 40 and M <= 128)):
            return "block"
    return None


def use_fused(M: int, N: int, K: int, kind: str = "plain", absorbs_norm: bool = False) -> bool:
    """kind: "qkv" (rope+append epilogue), "resid", "swiglu" or "plain"; absorbs_norm: the call would also apply a
    deferred RMSNorm to its input."""
    if _MODE == "lib" or _FUSED == "0" or M > 256 or K % 128 or N % 32:
        return False
    if _FUSED == "1":
        return True
    own = _measured(M, N, K, kind, absorbs_norm)
    if own is not None:
        return own == "fused"
    kind = "resid" if kind == "planes" else kind
    m_tiles = (M + 31) // 32
    # a product the kernel runs with 2 x 2 tiles (csrc/tilegemm.hip launch_tile_pro: two M tiles, an even number of column
    # tiles, >= 192 tile groups; with the deferred-norm prologue, K <= 4096) re-reads the weights once per
    # PAIR of M tiles: the 1B w1|w3 -- 18.4-18.9 us at 64 rows against md_linear's 22.8-23.2, and with the norm absorbed
    # 20.3 (profiles/r06_fused_pro22_ab.txt); at 128 rows (the two-token draft step) 32.0 with the norm against the library
    # + rmsnorm + SiLU*mul launches (20.5 + 5.1 + 5.4 in the trace), which also frees that weight's row-major copy
    t22 = (kind in ("swiglu", "plain", "resid") and m_tiles >= 2 and (N // 32) % 2 == 0
           and (N // 64) * ((m_tiles + 1) // 2) >= 192 and (not absorbs_norm or (kind == "swiglu" and K <= 4096)))
    l2_bytes = ((m_tiles + 1) // 2 if t22 else m_tiles) * N * K * 2
    if M <= 128:
        # the 70B model's TP-8 shards at the 128 rows of their verify step (tools/shard_bench.py,
        # profiles/r06_shard70b_ab.txt): w2 (8192 x 3584, 2 x 2 tiles) 22.0 us against 24.4 for the library -- wide products
        # on 2 x 2 tiles may re-read up to 120 MB; wqkv (1280 x 8192) 16.7 against 21.1 + the rope/append launch -- a deep
        # NARROW qkv shard is fused up to K = 8192 once >= 128 tile workgroups exist (at 32 rows, 40 workgroups, the
        # library wins: 15.1 vs 18.2)
        wide = t22 and _SHARD70B != "0"
        lim = FUSED_MAX_L2_BYTES_WITH_NORM if absorbs_norm else (FUSED_MAX_L2_BYTES_T22 if wide else FUSED_MAX_L2_BYTES)
        if l2_bytes <= lim and K <= FUSED_MAX_K:
            return True
        if _SHARD70B == "0" or not (FUSED_MAX_K < K <= 2 * FUSED_MAX_K):
            return False
        # deep (4096 < K <= 8192) shards -- the 70B model's and Qwen2.5-32B's (dim 5120) at TP-8, tools/shard_bench.py:
        #   qkv: 70B 1280 x 8192 at 128 rows 16.7 us against 21.1 + rope/append; Qwen 896 x 5120 11.5-12.1 against 13.7 + 5
        #        (112 tile workgroups); with 40 workgroups (70B at 32 rows) the library wins, 15.1 vs 18.2;
        #   w1|w3 on 2 x 2 tiles: Qwen 6912 x 5120 at 128 rows 27.0-27.2 against 36.5 for library + SiLU*mul (34.5 md_linear)
        if kind == "qkv":
            return l2_bytes <= FUSED_QKV_M256_MAX_L2_BYTES and (N // 32) * m_tiles >= 100
        return kind == "swiglu" and t22 and not absorbs_norm and l2_bytes <= FUSED_DEEP_SWIGLU_T22_MAX_L2_BYTES
    if kind == "swiglu":
        return N * K * 2 <= FUSED_M256_SWIGLU_MAX_BYTES and K <= FUSED_MAX_K
    if kind in ("plain", "resid"):
        if N * K * 2 <= FUSED_M256_NARROW_MAX_BYTES and K <= FUSED_MAX_K:         # measured at K = 512 only
            return True
        # the 8B wo at 256 rows on 2 x 2 tiles (4 x 64 tile groups = 256 workgroups) WITH its residual add is a
        # measured tie with the library + add/norm launch (25.2-25.9 vs 24.9-25.0 us, profiles/r06_fused_pro22_ab.txt;
        # in-trace A/B profiles/r06_ab_wo256_*): taking it leaves NO weight of the 8B / 1B pair at batch 64 held in two layouts during
        # decode (the library read the row-major tensor) and one library kernel fewer in the verify pass
        return (_WO256 != "0" and kind == "resid" and t22 and K <= FUSED_MAX_K
                and N * K * 2 <= FUSED_M256_RESID_T22_MAX_BYTES)
    return kind == "qkv" and l2_bytes <= FUSED_QKV_M256_MAX_L2_BYTES and K <= FUSED_MAX_K


def use_skinny(M: int, N: int, K: int, swiglu: bool, int8: bool, packed: bool, kind: str = None, absorbs_norm: bool = False) -> bool:
    if _MODE == "lib" or M > 256:
        return False
    if _MODE == "hip" or int8:          # int8 rows are only streamed by md_linear (the library path dequantises)
        return True
    if not packed:
        return False
    if _measured(M, N, K, kind or ("swiglu" if swiglu else "plain"), absorbs_norm) == "skinny":
        return True
    nbytes = N * K * 2
    if M <= 64:
        return nbytes >= MIN_STREAM_BYTES
    if M <= 128:
        return nbytes >= MIN_STREAM_BYTES_M128
    return K >= 8192 and nbytes >= MIN_STREAM_BYTES_M128


# md_linear_fused_split (csrc/tilegemm.hip, FL_PARTIAL) -- the tile kernel with K ALSO split over workgroups, for the
# deep narrow output projections of a <= 128-row step whose combine launch is the residual add + RMSNorm launch anyway: the 1B
# model's w2 (N = 2048, K = 8192, 33.5 MB), which every single-launch decomposition leaves per-CU-ingest-bound (fused tile
# kernel 22-24 us, library 15.7 + 5 for the add + norm, md_linear 17 + 5).  Rule from tools/split_bench.py
# (profiles/r06_split_ab.txt).
SPLIT_MIN_K = 8192
SPLIT_MAX_M = 128
_SPLIT = os.environ.get("MAGICDEC_SPLIT", "auto")      # "0": never, "1": every output projection it supports


def set_split(mode: str):
    global _SPLIT
    assert mode in ("auto", "0", "1")
    _SPLIT = mode


def use_split(M: int, N: int, K: int, kind: str) -> bool:
    """md_linear_fused_split_add_rmsnorm for this output projection (kind "resid")?"""
    if _MODE == "lib" or _SPLIT == "0" or kind not in ("resid", "planes") or M > 256 or K % 128 or N % 32 or N > 8192:
        return False
    if _SPLIT == "1":
        return True
    own = _measured(M, N, K, kind, False)
    if own is not None:
        return own == "split"
    return M <= SPLIT_MAX_M and K >= SPLIT_MIN_K and N * K * 2 < MIN_STREAM_BYTES


def use_few(M: int, N: int, K: int) -> bool:
    """md_linear_few in the place of what `choose` (and use_split) gives one of the framework's own kernels, for at most 16 rows?  Its tiles
    are of 16 columns: where those are one round of the chip at most, twice the CUs load the weight.  us, md_linear_fused / here, 1 and 16
    rows, 40 random products of 512 to 4 096 columns: 608 x 2 816 7.4 -> 5.6, 8.9 -> 6.5; 3 136 x 4 864 12.9 -> 9.4, 13.8 -> 11.0;
    2 048 x 2 048 5.6 -> 5.3, 6.2 -> 5.8; level at K = 1 280 and 7 % slower below 1 024.  Wider ones lose (4 352 x 4 352 12.9 / 14.5), and
    so do 128 columns and fewer, a handful of workgroups in either form (64 x 1 536 1.11 times, 128 x 1 280 1.08; 160 to 256 level or ahead).
    Deep ones (asked for with a row to four) against the K split and the weight-streaming kernel, with the norm behind them, which here
    the next product absorbs: 4 096 x 14 336 26.4 -> 22.9, 2 048 x 8 192 11.4 -> 10.4, 2 464 x 13 056 20.4 -> 17.7, but 608 x 14 592 (38
    workgroups) 10.1 / 15.3."""
    if not joint_launches() or not 1 <= M <= 16 or not 128 < N <= 16 * CUS or N % 32 or K % 256 or K < 1024:
        return False
    return K < SPLIT_MIN_K or N >= 1024


BLOCK_MIN_TILES = 160          # 128-column tiles that fill the chip without a K split (w1|w3: 224, lm head: 1002)
_BLOCK = os.environ.get("MAGICDEC_BLOCK", "auto")      # "0": never md_linear_block, "1": wherever it supports the shape


def set_block(mode: str):
    global _BLOCK
    assert mode in ("auto", "0", "1")
    _BLOCK = mode


def block_mode() -> str:
    return _BLOCK


def use_block(M: int, N: int, K: int, kind: str, absorbs_norm: bool = False) -> bool:
    """md_linear_block for this linear?  kind: "swiglu", "resid" (output projection + residual add + RMSNorm: the split-K
    combine launch does both) or "plain"."""
    if _MODE == "lib" or _BLOCK == "0" or M > 256 or N % 128 or K % 64:
        return False
    if _BLOCK == "1":
        return True
    own = _measured(M, N, K, kind, absorbs_norm)
    if own is not None:
        return own == "block"
    kind = "resid" if kind == "planes" else kind
    tiles = N // 128
    if M > 128:
        if kind == "resid":
            return K >= 8192 and N <= 8192 and N * K * 2 >= MIN_STREAM_BYTES_M128   # the 8B w2 (K = 14336); wo and
                                                                                    # the TP shards stay on the library
        return tiles >= BLOCK_MIN_TILES and kind in ("swiglu", "plain")
    return M > 64 and kind == "swiglu" and tiles >= BLOCK_MIN_TILES      # cfg2's 128-row verify: w1|w3 only


def choose(M: int, N: int, K: int, swiglu: bool, int8: bool, packed: bool, kind: str = None,
           absorbs_norm: bool = False) -> str:
    """"fused" (md_linear_fused), "block" (md_linear_block), "skinny" (md_linear) or "lib" (hipBLASLt) for one linear
    of a step."""
    kind = kind or ("swiglu" if swiglu else "plain")
    if packed and not int8 and _BLOCK == "1" and use_block(M, N, K, kind, absorbs_norm):
        return "block"
    if packed and not int8 and use_fused(M, N, K, kind, absorbs_norm):
        return "fused"
    if packed and not int8 and use_block(M, N, K, kind, absorbs_norm):
        return "block"
    return "skinny" if use_skinny(M, N, K, swiglu, int8, packed, kind, absorbs_norm) else "lib"


def prompt_over_block(M: int, N: int, K: int, swiglu: bool = False) -> bool:
    """Do 129 to 256 rows that `choose` gives to md_linear_block run on md_linear_prompt instead?  It takes 256 columns a workgroup, the block
    kernel 128: twice the columns in one round of the chip, which takes it 1.5 to 1.6 times as long at up to 192 rows, 1.68 to 1.74 times
    beyond.  Gate | up of 55 296 x 5 120 at 130 / 192 / 256 rows 143 / 163 / 174 -> 125 / 136 / 147 us, 37 888 x 3 584 93 / 102 / 113 -> 76 / 80
    / 86, a head of 128 256 x 4 096 241 / 259 / 275 -> 207 / 223 / 245; in one round of both (28 672 x 4 096: 54 / 59 / 65 and 53 / 59 / 72)
    or where its last round is the emptier one (152 064 x 3 584, 256 rows: 302 and 313) the block kernel stays."""
    from .. import ops
    if _MODE != "auto" or _BLOCK == "1" or not 128 < M <= 256:
        return False
    wide, narrow = -(-N // (256 * CUS)), -(-N // (128 * CUS))
    return (1.6 if M <= 192 else 1.74) * wide < narrow and ops.linear_prompt_us(M, N, K, swiglu) >= 0


@functools.lru_cache(maxsize=4096)
def prompt_rows(M: int, N: int, K: int, swiglu: bool = False, rows_stay: bool = False) -> int:
    """How many of a prompt's M rows (more than a step has; weight in the streaming layout) go to md_linear_prompt in one call: none (the
    library), all, or whole row tiles with fewer than 129 left for md_linear.
    Against the library, 435 random products of 257 to 16 384 rows: 0.77 of its time with the activation behind it, 0.61 with the weight's
    rows brought back in front; 1.11 at the worst (12 719 x 2 048 x 8 192, 341 us).  Its workgroups take all of K, so that a few hundred
    rows of a narrow and deep product leave most CUs idle: 374 x 2 048 x 10 240 in 58 us where the library's split of K takes 41, or 61
    with the rows to bring back; the line is where those cross over the same products.  rows_stay: the weight is one whose row-major
    tensor is never released (a pool's, or one that steps of more than 256 rows read), so that the library has nothing to bring back; over
    330 products of 257 to 2 600 rows the two cross at 1.45 times the ideal (1.10 of the library's time at the worst; beyond it 449 x
    2 048 x 5 632 in 38 us for 27, 301 x 4 096 x 14 336 in 91 for 74), those of less than a round of small tiles alone: 8 196 x 8 192 x 512
    takes 74 us for the library's 137, far from an ideal that counts neither's first steps.
    Rows just behind whole rounds of tiles are a round more: 8 196 x 4 096 x 18 432 in 950 us, 8 192 in 760 and the other four in 40 on the
    weight-streaming kernel, whose time the last line bounds from above (49 / 55 us for 28 672 x 4 096 at 64 / 128 rows, 16 / 21 for 4 096
    x 4 096, 54 / 64 for 5 120 x 27 648)."""
    from .. import ops
    us = ops.linear_prompt_us(M, N, K, swiglu) if _MODE != "lib" and M > 256 else -1.0
    few = rows_stay and M * N < CUS * 128 * 128
    if us < 0 or us > (1.45 if few else 2.4) * (2e-6 * M * N / 1400 * K + 12):
        return 0
    rest = M % 256
    if 0 < rest <= 128 and M - rest > 256 and ops.linear_supported(rest, N, K, swiglu):
        streamed = (12 + N * K * 2 / 5.5e6) * (1.0 if rest <= 64 else 1.2)
        if ops.linear_prompt_us(M - rest, N, K, swiglu) + streamed < 0.97 * us:
            return M - rest
    return M
