"""y = x W^T (+ b) for the parts: picks the matrix product by dtype and shape.

float32: the 32-bit matrix-core kernels (ops.gemm32: multiply-adds in 32-bit, no reduced-precision mode; ops.gemm32_gated), or the
  multiply-add kernel of the vector units where rows are no multiples of 16 bytes.
bfloat16, up to 16 rows of up to 6,144 columns, 17 to 32 rows of up to 4,096, or 33 to 64 rows of up to 2,048:
  ops.gemm_decode, one workgroup per compute unit, with the activation or the rotation and cache store in
  its epilogue; up to 16 rows it also norms its rows on the way in and adds its result to the residual
  rows where the parts ask for that (decode_product, adds_residual_in_epilogue).
bfloat16, few rows otherwise: the hand-written kernel that streams the weight once
  (ops.gemm_stream); it takes up to 64 rows, one workgroup per 16 rows and 16 weight rows, so
  beyond 16 rows the weights are re-read from L2 and it only pays for the smaller matrices.
  A product whose result goes to a norm may be left as 32-bit partial sums over shares of K, which
  the norm kernel adds up (linear_partial_sums): that fills the chip for a short, wide weight; for 17 to
  64 rows it is ops.gemm_decode with K shared out to 2 to 8 sets of workgroups (ops.gemm_slices, which
  keeps a slice of all rows in LDS, where that kernel is switched off).
bfloat16, more rows: ops.gemm_tiles, tiles on the matrix cores with the activation, the rotation and cache store, or the
  partial sums of a product that goes to a norm in the epilogue; the library's matrix product (hipBLASLt through
  torch.mm), which is where the reference's engine uses a library too (nn.Linear, src/llmserve/model/llama.py:64-67), only
  for the sizes where it is still the faster one (tiles_pay) and for K or N that the tiles cannot take.
Operands the matrix-core kernels cannot take (K not a multiple of 8) fall to the 32-bit
multiply-add kernel, which takes anything.

LLMSERVE_GEMM=own in the environment keeps the library out altogether: what neither the streaming kernel nor the tiles
take then goes to this repository's plain tiled kernels (ops.gemm_bf16).
"""

from __future__ import annotations

import os

import torch

from ..ops import library as ops
from .registry import JoinedRows

OWN_KERNELS_ONLY = os.environ.get("LLMSERVE_GEMM", "") == "own"


STREAM_ROWS = 16  # up to here the streaming kernel always wins
STREAM_MAX_ROWS = 64
# beyond STREAM_ROWS: bytes of weight times blocks of 16 rows up to which the streaming kernel still beats
# the library (measured on the TinyLlama shapes at 32 and 64 rows, with the epilogue it saves counted in)
STREAM_REREAD_BYTES = 64e6


# A plain product of up to 8 rows against a weight this large (the vocabulary's): ops.gemm_decode shares it out to the compute units in
# one stretch each and streams it faster than ops.gemm_stream's thousands of small workgroups where all its waves have whole chunks of K
# (two, three, four or six of 128 columns each) or beyond 4 rows.  Microseconds, gemm_decode and gemm_stream: 32000 x 2048 22.1 and 24.2 at 1
# row, 22.5 and 26.2 at 8; 128256 x 2048 78 and 82, 82 and 90; 32000 x 4096 41.4 and 43.4, 42.5 and 46.9; 32064 x 3072 31.0 and 31.9; 100352 x
# 6144 188 and 189, 190 and 206.  Otherwise 50304 x 1024 19.8 and 18.2 at 1 row, 50264 x 1600 28.5 and 26.3, 262144 x 1152 94 and 85, 151936 x
# 896 42.1 and 40.1, 64000 x 2560 50.4 and 49.1, but at 8 rows 20.2 and 19.9, 29.0 and 29.6, 101 and 105, 44.8 and 45.5, 52.3 and 56.6.
STREAM_LARGE_ROWS = 8
STREAM_LARGE_BYTES = 100e6
STREAM_LARGE_ODD_ROWS = 4


def streams_large(m: int, n: int, k: int, cus: int = 256) -> bool:
    """Whether a plain product of `m` rows against a large weight [n, k] that ops.gemm_decode takes is faster by ops.gemm_stream."""
    if m > STREAM_LARGE_ROWS or 2 * n * k < STREAM_LARGE_BYTES:
        return False
    return (m <= STREAM_LARGE_ODD_ROWS and k not in (2048, 3072, 4096, 6144)) or _shares_meet(n, k, cus)


def _shares_meet(n: int, k: int, cus: int) -> bool:
    """Whether the compute units' stretches of a weight [n, k] start on the same channels of memory.  Starts 127 or 129 times a
    power of two apart are slow, their neighbours are not, whatever that power: as if fields of 7 bits of an address, added without carry,
    chose the channel, where such starts cancel out and all units walk the weight side by side on few channels.  TB/s of gemm_decode at 1 row, K = 4096, by rows a compute unit:
    126 6.4, 127 5.2, 128 6.4; 253 6.6, 254 5.5, 255 6.6, 257 6.6, 258 5.7, 260 6.6 (gemm_stream 5.9 and 6.3 to 6.4)."""
    apart = n // cus * k
    return n % cus == 0 and apart > 0 and ((apart & -apart) * 127 == apart or (apart & -apart) * 129 == apart)


DECODE_KERNEL = os.environ.get("LLMSERVE_DECODE_GEMM", "1") != "0"


def decode_product(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether x [M, K] against weight goes to ops.gemm_decode (one workgroup per compute unit)."""
    return DECODE_KERNEL and ops.gemm_decode_supported(x, weight)


def adds_residual_in_epilogue(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether a product whose result is added to the residual rows does that sum itself (ops.gemm_decode's
    residual epilogue), up to GEMM_DECODE_NORM_ROWS rows.  There the norm that follows is the next product's prologue, or,
    with rows too long for that, a kernel which then adds nothing up (`adds_long_rows`).  With more rows that kernel adds up
    partial sums as it reads them, and the product is faster with its K shared out (measured at 32 rows: 1.08 against 1.12 ms
    a step of the TinyLlama shape)."""
    if x.shape[0] > ops.GEMM_DECODE_NORM_ROWS:
        return False
    return decode_product(x, weight) or (
        DECODE_KERNEL and x.dtype == torch.bfloat16 and ops.gemm_decode_adds(*x.shape) and ops.gemm_bf16_supported(x, weight)
        and ops.gemm_decode_reaches(x, weight) and adds_long_rows(weight.shape[0], ops.compute_units(x.device)))


def adds_long_rows(n: int, cus: int = 256) -> bool:
    """Whether a product of rows that are too long for a compute unit is added to the residual rows by ops.gemm_decode, in tiles of 16 weight
    rows that each take the rows of x in again, and not by the norm behind partial sums of ops.gemm_stream.  Not where a share of the weight's
    n rows that takes two tiles or more fills less than two thirds of them: 5120 x 13824, 20 rows in two tiles, 29.3, 30.6 and 36.3 microseconds at 1, 8
    and 16 rows, with the norm still to be done by the next product, where stream and norm take 30.2, 33.5 and 38.7.  Nine other weights of 4096 x
    11008 to 12288 x 6400 at 1 to 16 rows with a norm kernel behind either 1 to 17 % faster, and up to 6,144 columns that kernel is spared as well
    (4096 x 14336 21.7 and 28.3 at 8 rows, 3072 x 8192 10.9 and 16.3).  A single tile is taken however little of it is filled: its rows of x are read once."""
    most = -(-n // min(n, cus))
    return most <= 16 or 2 * (-(-most // 16) * 16) <= 3 * most


def few_rows(m: int, weight: torch.Tensor) -> bool:
    """Whether `m` bfloat16 rows against `weight` go to ops.gemm_stream."""
    if m <= STREAM_ROWS:
        return m > 0
    return m <= STREAM_MAX_ROWS and -(-m // 16) * weight.numel() * 2 <= STREAM_REREAD_BYTES


# Up to how many multiply-adds ops.gemm_tiles is the faster way; larger products go to the library.  Tiles gain by what they
# spare (a kernel behind the product, a pass over its result, a short K walk where K comes in parts); the library gains by sharing
# the last round of tiles out, which the tiles do not, and that weighs more the more rounds there are.  Means over 1,900
# products of 33 to 2,048 rows (tiles' time over the library's with the kernel behind it; below the line, and beyond): plain 0.89
# (1.05), gated 0.93 (1.04), rotation and cache store 0.77 (1.00), parts of K for a norm 0.81 (1.04).  The library's times jump from
# size to size, so single products lie on the wrong side: 1 in 18 below the line is more than 5 percent slower in tiles, at most 19, and 1
# in 6 beyond it more than 5 percent faster.  Single sizes, microseconds, tiles and library:
#   plain   4608 x 2048 15 and 16 at 333 rows; 6144 x 2048 18 and 25 at 333, 52 and 46 at 2,048; 32000 x 2048 60 and 57 at 512
#   gated   11264 x 2048 30 and 37 at 512 rows; 22016 x 4096 59 and 66 at 200, 101 and 87 at 512, 169 and 167 at 1,024; 28672 x 4096
#           398 and 374 at 2,048
#   rotary  2560 x 2048 11 and 19 at 512 rows; 12288 x 4096 60 and 62 at 512, 104 and 92 at 1,024
#   parts   4096 x 11008 51 and 73 at 512 rows; 8192 x 28672 151 and 306 at 200, 430 and 263 at 640 (without the norm)
# The gated line was drawn when such products took 10 to 30 % longer in tiles.  Against a weight below TILES_GATED_SMALL they are the tiles',
# whatever the rows: 8 such weights of 5632 x 1024 to 14336 x 3072 at 72 to 4,096 rows, 192 products, 0.78 in the mean, 1.08 at most (14336 x 3072 at
# 2,500); 11264 x 2048: 36 and 49 at 768 rows, 53 and 58 at 1,024, 66 and 75 at 1,300, 68 and 81 at 1,536, 90 and 99 at 2,048; 17920 x 1536 71
# and 83 at 1,300; 16384 x 2048 85 and 94.  22016 x 4096 and larger weights are the library's at some sizes still (1.06 at 512 rows).
# Gated products of TILES_GATED_WORK and more against a weight below TILES_GATED_WEIGHT (200 MB, which the 256 MB memory-side cache
# holds) are the tiles' again: 27 such products of 17 weights 0.95 in the mean, 0.72 to 1.19, where larger weights are at 1.05; 22016 x
# 4096 at 2,048 rows 299 and 425 (the means, too, from before).
# Plain products of TILES_LONG_K columns and more whose tiles leave half the compute units without one are the library's, which
# shares their K out (one result cannot come in parts, and each tile walks all of K): 65 such products of 9 weights, from 65 rows on,
# 1.17 in the mean.  2048 x 5632 28 and 16 at 128 rows, 25 and 21 at 228, but 28 and 33 at 613; 1024 x 4096 13 and 9 at 96.
# Products whose tiles are one round that three quarters of the compute units have a part in leave the library nothing to share out.  Beyond
# TILES_WORK, 67 plain ones of 14 weights up to 28672 x 4096 and 128 to 4,096 rows, 0.92 in the mean, 0.72 to 1.02 (2048 x 5632 46 and 51 at
# 1,629 rows, 4096 x 4096 54 and 58 at 2,048, 4096 x 11008 145 and 164 at 2,048, 8192 x 8192 96 and 103 at 768), and 40 gated ones, 0.87,
# 0.70 to 0.96 (22016 x 4096 64 and 78 at 330, 12288 x 4096 60 and 67 at 610).  Of columns beyond TILES_ROUND_K and of tiles of 256 x
# 256 (one wave to a SIMD) too many were slower: 2048 x 16384 151 and 141 at 2,048, 6144 x 2048 53 and 48 at 2,500.  Rotations and parts gain
# what they spare behind the product on top: 15360 x 5120 rotated at 512 and 528 rows 0.85 and 0.88, and 9 products that go to a norm, in the parts
# of K that their plan has, 0.90, at most 0.95 (8192 x 8192 at 1,024 rows 0.93, 3072 x 8192 at 3,000 0.91).
TILES_WORK = {"plain": 18e9, "gated": 18e9, "rotary": 40e9, "parts": 60e9}
TILES_GATED_WORK = 130e9
TILES_GATED_WEIGHT = 100e6
TILES_LONG_K = 4096
TILES_GATED_SMALL = 50e6
TILES_ROUND_K = 12288


def tiles_pay(kind: str, m: int, n: int, k: int, cus: int = 256) -> bool:
    """Whether m rows against a weight [n, k] are faster by ops.gemm_tiles ("plain", "gated" or "rotary" with what follows in the
    epilogue, "parts": K in parts for a norm to add up) than by the library: a rule by sizes alone."""
    work = m * n * k
    if kind == "gated" and n * k < TILES_GATED_WEIGHT:
        if work >= TILES_GATED_WORK or n * k < TILES_GATED_SMALL:
            return True
    if m > 64:
        rows, weight_rows = ops.GEMM_TILES[ops.gemm_tiles_plan(m, n, k, 1, cus)[0]][:2]
        tiles = -(-m // rows) * -(-n // weight_rows)
        if kind == "plain" and k >= TILES_LONG_K and 2 * tiles <= cus:
            return False
        if 0.75 * cus <= tiles <= cus and k <= TILES_ROUND_K and rows * weight_rows < 65536:
            return True
    return work < TILES_WORK[kind]


def tiles_fit(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether x [M, K] against weight may go to ops.gemm_tiles, once the kernels for few rows have declined."""
    return x.shape[0] > STREAM_ROWS and ops.gemm_tiles_supported(x, weight)


def tiles_product(x: torch.Tensor, weight: torch.Tensor, kind: str = "plain") -> bool:
    """Whether a product of this kind goes there."""
    return tiles_fit(x, weight) and (OWN_KERNELS_ONLY or tiles_pay(kind, x.shape[0], *weight.shape, ops.compute_units(x.device)))


def brings_near(x: torch.Tensor, weight: torch.Tensor, near: torch.Tensor) -> tuple[int, int]:
    """With how many compute units ops.gemm_tiles, given x against weight with `near` behind it, brings `near` into the memory-side cache,
    and how many bytes: what it is told (`brings`), and where there are any the product of `near` is (`from_cache`)."""
    n, k = weight.shape
    return ops.gemm_tiles_brings(x.shape[0], n, k, near, ops.compute_units(x.device))


# A short, wide weight gives the streaming kernel fewer tiles than the chip has CUs (TinyLlama's o_proj and
# down_proj: 128), and long rows make each workgroup wait for several rounds of loads.  Sharing K out to
# several workgroups per tile fills the chip: measured 4.3 -> 3.2 microseconds of reading for 2048 x 2048 and
# 10.0 -> 6.8 for 2048 x 5632.  The partial sums are added up by the norm kernel that follows.
SPLIT_K = os.environ.get("LLMSERVE_SPLIT_K", "1") != "0"
SPLIT_K_WORKGROUPS = 1024  # aim for about this many workgroups (a CU holds eight of them)
SPLIT_K_MAX = 4


def k_splits_for(m: int, weight: torch.Tensor) -> int:
    n, k = weight.shape
    workgroups = -(-n // 16) * -(-m // 16)
    chunks = -(-k // 512)
    return max(1, min(SPLIT_K_MAX, SPLIT_K_WORKGROUPS // workgroups, chunks // 2))


# 17 to 64 rows against a weight of up to this many bytes: ops.gemm_slices (a slice of all rows in LDS, one
# array of partial sums per 512 of K).  Measured at 64 rows on 2048 x 2048 and 2048 x 5632: 6.3 and 11.5
# microseconds against the library's 11.6 and 18.0; the partial sums are a quarter of the weight's bytes at 64
# rows, written here and read by the norm, which is what a larger weight does not earn back.
SLICES_MAX_WEIGHT_BYTES = 24e6


def slices_pay(m: int, weight: torch.Tensor) -> bool:
    """Whether `m` bfloat16 rows against `weight` are best left as partial sums per slice of K (ops.gemm_slices),
    for a norm to add up."""
    return SPLIT_K and STREAM_ROWS < m <= STREAM_MAX_ROWS and weight.numel() * 2 <= SLICES_MAX_WEIGHT_BYTES


def linear_partial_sums(x: torch.Tensor, weight: torch.Tensor, from_cache: bool = False):
    """x W^T as `PartialSums` (K shared out to several workgroups per tile), or None where that does not
    pay or does not apply; for callers whose result goes to a norm next.  `from_cache`: as for ops.gemm_tiles."""
    from .registry import PartialSums

    m = x.shape[0]
    if not (SPLIT_K and x.dtype == torch.bfloat16 and ops.gemm_bf16_supported(x, weight)):
        return None
    if STREAM_ROWS < m <= STREAM_MAX_ROWS and DECODE_KERNEL and ops.gemm_decode_reaches(x, weight):
        k_parts = ops.gemm_decode_k_parts(m, weight.shape[1])
        if k_parts > 1:  # the rows in registers, K shared out to a few sets of workgroups
            parts = torch.empty((k_parts, m, weight.shape[0]), dtype=torch.float32, device=x.device)
            return PartialSums(ops.gemm_decode(parts, x, weight, k_parts=k_parts), x.dtype)
    if slices_pay(m, weight):
        parts = torch.empty((-(-weight.shape[1] // ops.SLICE_K), m, weight.shape[0]), dtype=torch.float32, device=x.device)
        return PartialSums(ops.gemm_slices(parts, x, weight), x.dtype)
    if not few_rows(m, weight):
        if tiles_product(x, weight, "parts"):
            k_parts = ops.gemm_tiles_plan(m, weight.shape[0], weight.shape[1], 4, ops.compute_units(x.device), from_cache)[1]
            if k_parts > 1:
                parts = torch.empty((k_parts, m, weight.shape[0]), dtype=torch.float32, device=x.device)
                return PartialSums(ops.gemm_tiles(parts, x, weight, from_cache=from_cache), x.dtype)
        return None
    splits = k_splits_for(m, weight)
    if splits < 2:
        return None
    parts = torch.empty((splits, m, weight.shape[0]), dtype=torch.float32, device=x.device)
    ops.gemm_stream(parts, x, weight, k_splits=splits)
    return PartialSums(parts, x.dtype)


def _tiles_take(out: torch.Tensor, bias: torch.Tensor | None, n: int) -> bool:
    """Whether ops.gemm_tiles stores into `out` and adds `bias` (the library's product takes any strides, and a bias of another
    dtype or of one number)."""
    return (out.stride(1) == 1 and out.stride(0) % 4 == 0 and out.data_ptr() % (4 * out.element_size()) == 0 and
            (bias is None or (bias.dtype == torch.bfloat16 and bias.is_contiguous() and bias.shape == (n,))))


def takes_stream(stream: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether the product of few rows against `weight` makes them from a 32-bit stream on its way in (ops.gemm_decode_stream), and not behind
    a kernel that does: a launch less, where the product is ops.gemm_decode's anyway."""
    m, (n, k) = stream.shape[0], weight.shape
    return (DECODE_KERNEL and ops.gemm_decode_stream_supported(stream, weight) and ops.gemm_decode_fits(m, k)
            and not streams_large(m, n, k, ops.compute_units(stream.device)))


def joins_pay(m: int, n: int, k: int, gated: bool, cus: int = 256) -> bool:
    """Whether `m` rows that a stream's open sum makes are closed faster by the product against a weight [n, k] on its way in than by the kernel for
    it.  Every workgroup reads all of the stream and of what joins it, in turns of 4 rows: a second turn of more than 2,048 columns takes longer than
    that kernel where little else is in flight, one tile of 16 weight rows to a workgroup (or 8 gated pairs), and beyond 3,072 columns anywhere.
    Microseconds on the way in and apart, one turn of 4 rows and 8 rows: 2304 x 2304 6.7 and 7.5, 8.0 and 7.6; 2 x 2048 x 2560 gated 8.2 and 8.8, 9.5 and
    9.0; 3072 x 3072 7.7 and 8.4, 9.2 and 8.8; 4096 x 4096 9.3 and 10.5, 11.8 and 11.1; 2 x 10240 x 4096 gated 28.7 and 29.6, 31.3 and 30.2.  Shares of other sizes,
    8 rows: 2 x 3072 x 2560 gated 9.8 and 10.8; 6144 x 3072 11.2 and 11.5; 2048 x 3072 7.6 and 8.0.  Up to 2,048 columns 8 rows are 5 to 20 % faster.
    A norm reads the stream alone: 8 rows of 2,304 to 4,096 columns 6 % faster in the mean, 1 of 36 sizes more than 2 % slower."""
    if m <= 4 or k <= 2048:
        return True
    units = n // 2 if gated else n
    share = -(-units // min(units, cus))
    return k <= 3072 and not (share <= 8 if gated else 8 < share <= 16)


def joined_product(x, weight: torch.Tensor, out: torch.Tensor, bias: torch.Tensor | None = None, **epilogue) -> bool:
    """The product of `JoinedRows` x into `out` (float32, or bfloat16 with the gated `epilogue`) with x's sum closed on the way in, where that is
    the faster way; False, with nothing done, otherwise."""
    if x.dtype != torch.bfloat16 or not takes_stream(x.stream, weight):
        return False
    if not joins_pay(x.shape[0], *weight.shape, epilogue.get("swiglu", False), ops.compute_units(out.device)):
        return False
    stream = torch.empty_like(x.stream)
    ops.gemm_decode_stream(out, x.stream, weight, bias, joins=(x.delta.y, x.delta.weight, x.delta.eps, stream), **epilogue)
    x.resolve(stream)
    return True


def adds_to_stream(rows: int, weight: torch.Tensor) -> bool:
    """Whether the product of `rows` bfloat16 rows against `weight` adds its result, times its gate, to a 32-bit stream in its epilogue
    (`GatedStream.add`): where it is ops.gemm_decode's and the norm behind the sum is no kernel of its own, or one that adds nothing up."""
    return (DECODE_KERNEL and 0 < rows <= ops.GEMM_DECODE_NORM_ROWS and weight.dtype == torch.bfloat16 and weight.is_contiguous()
            and weight.data_ptr() % 16 == 0 and weight.shape[1] % 8 == 0 and 0 < weight.numel() < 1 << 30
            and ops.gemm_decode_fits(rows, weight.shape[1]))


def linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None = None,
           out_dtype: torch.dtype | None = None, out: torch.Tensor | None = None, from_cache: bool = False) -> torch.Tensor:
    """x [M, K] (unit inner stride; or `JoinedRows`), weight [N, K] -> [M, N] in out_dtype (default: x's).  `from_cache`: as for
    ops.gemm_tiles."""
    out_dtype = out_dtype or x.dtype
    m, n = x.shape[0], weight.shape[0]
    if out is None:
        out = torch.empty((m, n), dtype=out_dtype, device=x.device)
    if isinstance(x, JoinedRows):
        if out.dtype == torch.float32 and joined_product(x, weight, out, bias):
            return out
        x = x.materialize()
    if m == 0:
        return out
    if x.dtype == torch.bfloat16 and ops.gemm_bf16_supported(x, weight):
        if decode_product(x, weight) and not streams_large(m, n, weight.shape[1], ops.compute_units(x.device)):
            return ops.gemm_decode(out, x, weight, bias)
        if few_rows(m, weight):
            return ops.gemm_stream(out, x, weight, bias)
        if tiles_product(x, weight) and _tiles_take(out, bias, n):
            return ops.gemm_tiles(out, x, weight, bias, from_cache=from_cache)
        if OWN_KERNELS_ONLY:
            return ops.gemm_bf16(out, x, weight, bias, kernel="skinny" if m <= 64 else "tile")
        if bias is None:
            return torch.mm(x, weight.t(), out_dtype=out.dtype, out=out)
        return torch.addmm(bias.to(out.dtype), x, weight.t(), out_dtype=out.dtype, out=out)
    if out.dtype == torch.float32 and ops.gemm32_supported(x, weight):
        return ops.gemm32(out, x, weight, bias)
    return ops.gemm_fma(out, x, weight, bias)
