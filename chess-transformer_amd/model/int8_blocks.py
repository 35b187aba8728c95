"""Int8 transformer blocks on gfx950: the module API of the reference's model/int8_blocks.py.

Same names, signatures, operator schemas (chess::int8_linear, chess::norm_quant,
chess::mix_norm_quant, chess::rotate_quant) and Int8Block / quantize_blocks behaviour, so that
engine/inference.py (int8_model, reference :267-272) and the MCTS that calls it run unchanged.
Underneath, every operator is one launch of a hand-written HIP kernel from libchess_hip.so
(csrc/): no Triton, no NVRTC, no fallback. A shape the kernels do not take raises ValueError
where the reference fell back to another kernel (reference int8_cuda.py:369-381).
"""
from __future__ import annotations

import json
import math
import os

import torch
from torch import nn

from model import hip_kernels
from model.fused_blocks import FusedBlock, linear, link_input_mixes, template_attention
from model.hip_kernels import aligned, check, library_for, pointer, stream_of

# model/int8_blocks.py:14-17 of the reference: the mlp's hidden is rotated in blocks of 32 (H H^T = 32 I) and
# zero-padded to a multiple of 128 for down
HADAMARD_BLOCK = 32
DOWN_INPUT_MULTIPLE = 128
INT8_DEPTH = 64
# The GEMM's tiles by the rows a compute unit's share is (the reference's table format, int8_blocks.py:19-31), timed on an
# MI355X: 1 is 64 x 64, 2 128 x 128, 3 128 x 64 (rows x outputs, a 4-stage ring), 4 256 x 128, 6 128 x 128 (eight
# wavefronts, a 3-stage ring), 5 128 x 128 (eight wavefronts, a 2-stage ring of 128-byte stages),
# 7 128 x 128, 8 128 x 64 (a 3-stage ring), 9 128 x 64, 10 256 x 64, 11 128 x 128 (a 2-stage ring: three workgroups a
# compute unit, which is what the batch-1024 network runs fastest with), 13 128 x 128 (a 2-stage ring of 128-byte stages:
# down's 2,048-byte rows, read in whole L2 lines), 14 32 x 32 with K split over 4 wavefronts (the reference's small_int8
# for one or two positions, int8_cuda.py:34-183: in a kernel trace 3.6, 4.3 and 6.2 us where tile 1 takes 4.4, 5.2 and 7.6
# for projection, gate_up and down at 70 rows; gate_up's tile 1 is faster again at 140 rows, the others from about 200),
# 15 the depth-512 kernel whose wavefronts hold their weights in registers and stream x in blocks of 32 rows
# (gemm_resident.h): its workgroups load their weights once and then need long streams of row blocks, so gate_up takes
# it past 40 rows a compute unit and projection past 100 (whose 1,600 columns leave 7 of the last column group's 8
# wavefronts without outputs). Forwards alternated on one box, projection / gate_up tiles: batch 128 3.70 / 3.84 / 3.71 ms
# (11 / 10, 15 / 10, 11 / 15), batch 256 6.01 / 6.03 / 5.94, batch 512 11.13 / 10.92 / 10.68 and 10.50 with both on 15;
# batch 1024 19.48-19.55 against 19.77-19.82 ms for projection alone, 19.65-19.67 against 20.41-20.44 for gate_up alone
# (167.5 against 188.8 us a launch in the network's trace).
# down takes tile 16 past 48 rows a compute unit: the depth-2048 kernel whose wavefronts hold a quarter of the depth of 64
# columns each in registers (gemm_deep.h). Forwards alternated on one box, down on the table's tiles before it (11 up to
# 160 rows, 13 past them) against tile 16: batch 128 3.833 against 3.85 ms (tile 5 stays), batch 256 5.955 against 5.826,
# batch 512 10.38 against 9.72, batch 1024 18.76-18.83 against 17.92; batch 64 2.304-2.310 against 2.355-2.358 with tile
# 16 from 16 rows, three runs alternated on one box. From 8 to 32 rows it takes the eight-wavefront
# tile 6 (batch 64: 2.44-2.48 against 2.50-2.53 ms a forward with tile 12, four runs alternated on one box) and up to 48
# tile 5 (batch 128: 3.82-3.89 against 3.92-3.97 with tile 11). Between 4 and 9 rows a compute unit (batches 15 to 32)
# projection takes tile 1 and then 8 (batch 16: 0.06 ms a forward faster than tile 11, batch 32: 0.035), and gate_up takes
# tile 8, now its 2-stage twin 9, up to 18 rows (batch 16 / 32 / 64: 0.05 / 0.03 / 0.045 ms faster than tile 10; 9 against
# 8 at batch 64: 2.411-2.432 against 2.420-2.441 ms a forward, six runs alternated on one box). The 128-byte-stage tiles
# do not pay there: at batch 64 the table's tiles ran 2.304-2.311 ms a forward against 2.394-2.402 with gate_up on tile 12,
# 2.575-2.576 on tile 13, 2.323-2.326 with projection on tile 13 and 2.371-2.379 on tile 12 (three runs alternated on one
# box). Every tile gives the same bits.
INT8_TILES = {"gfx950": {"projection": [(0.55, 14), (5, 1), (9, 8), (100, 11), (math.inf, 15)],
                         "gate_up": [(0.3, 14), (4, 1), (18, 9), (40, 10), (math.inf, 15)],
                         "down": [(0.55, 14), (8, 1), (32, 6), (48, 5), (math.inf, 16)]}}
# projection of rows of 768 or more (768 to 1,152 columns, graphs of launches on an MI355X): 3,570 rows in 8.1 us on tile 6
# and 9.1 on tile 11, 7,000 in 12.1 on tile 13 and 13.8, 17,920 in 26.8 and 29.5; past them tile 0, which takes the weights
# in registers at such depths too (35,000 rows: 40.1 against 44.4 us on tile 4, 69,930 69.3 against 87.3). Where the last
# round of workgroups would be small, tile 11 (long_projection_tile): past 256 of tile 6's (768 to 1,152 at 3,570 rows, 252
# of them, 8.1 against 9.1 us on tile 11, at 3,873, 279, 10.5 and 9.6; 1,024 to 1,600 at 5,100 18.3 and 17.4), and where
# tile 13's last 512 places are less than LEAST_LAST_ROUND full (768 to 960 at 8,785, 552, 16.9 and 14.9; 768 to 768 at
# 13,000, 612, 17.4 and 16.4; 1,024 to 1,600 at 7,000, 715, 20.5 and 19.6; but 768 to 960 at 12,000, 752, 17.7 and 18.2).
# Rows of 640 keep the table (to 640, 960, 1,280 and 1,600 columns tile 13 takes up to 11% more than tile 11: 640 to 1,280
# at 8,785 rows 16.4 and 15.5, 640 to 640 at 14,000 15.8 and 14.2). (for the shipped table only: one put in INT8_TILES in
# its place, or edited there, holds for every depth)
LONG_PROJECTION_DEPTH, LEAST_LAST_ROUND = 768, 0.43
LONG_PROJECTION_TILES = {"gfx950": [(0.55, 14), (5, 1), (9, 8), (20, 6), (75, 13), (math.inf, 0)]}
SHIPPED_PROJECTION_TILES = list(INT8_TILES["gfx950"]["projection"])
# the split-K tile's wavefronts: each reads 1, 2 or 4 steps of 128 bytes of K, and the outputs go 8 columns a lane
SPLIT_WAVES = {14: 4}
# the tiles whose wavefronts hold their weights in registers for the whole depth: 15 (gemm_resident.h) at depth 512, N a
# multiple of 8, no residual or input mix; 16 (gemm_deep.h, down's, the depth split over four wavefronts) at depth 2048, N a
# multiple of 128, not gated, no bias, the residual added (with or without the next block's mix)
RESIDENT_TILE, RESIDENT_DEPTH = 15, 512
DEEP_TILE, DEEP_DEPTH = 16, 2048
# and their launches' limits: outputs under 2 GiB (32-bit offsets of two-byte values), and no more column groups (of 256 gated
# and 512 other columns, and of 128) than the compute units of an XCD
RESIDENT_OUTPUT_BYTES, RESIDENT_GROUPS = 1 << 31, 32
# each tile's (rows, output columns, wavefronts, ring stages), the shapes the kernels are instantiated with
TILE_SHAPES = {1: (64, 64, 4, 4), 2: (128, 128, 4, 4), 3: (128, 64, 4, 4), 4: (256, 128, 8, 3), 5: (128, 128, 8, 2), 6: (128, 128, 8, 3),
               7: (128, 128, 4, 3), 8: (128, 64, 4, 3), 9: (128, 64, 4, 2), 10: (256, 64, 4, 2), 11: (128, 128, 4, 2), 12: (128, 64, 4, 2),
               13: (128, 128, 4, 2), 14: (32, 32, 4, 1)}
# rows a workgroup of the norm kernel (a group of lanes a row); no count changes a bit
NORM_ROWS = 4
# rotate_quant's rows a wavefront by the rows a compute unit's share is (the reference's format, int8_blocks.py:33-50): one
# until the launch fills the chip, then two (at 71,680 rows of 2,048 on an MI355X: 83.6 us against 93.5 for one; at batch
# 64 one row a wavefront ran 2.304-2.310 ms a forward against 2.349-2.350 with two, alternated on one box)
ROTATE_ROWS = {"gfx950": [(128, 1), (math.inf, 2)]}
UNTIMED_ROTATE_ROWS = 0   # the kernel's own choice by size
# down with rotate_quant folded in (chess_rotated_int8_linear) by the rows a compute unit's share is: 0 keeps rotate_quant
# and down as two launches; 1 to 4 are the folded kernel's tiles (1: 128 x 512, 2: 64 x 512, 3: 128 x 256, 4: 64 x 256).
# Two launches everywhere: the network at batch 1024, alternated on one box, ran 20.69 / 20.74 ms a forward so and
# 20.73 / 20.72 ms folded with tile 1 (21.44 / 21.36 with tile 2, 21.32 / 21.24 with tile 3); at batch 256 6.07 ms so
# against 6.74 (tile 4), 6.90 (tile 3) and 7.02 (tile 2), and a 64-board search call 2.363 ms (p50) so against 2.574
# (tile 4): the folded kernel is bound by its data movement at one workgroup a compute unit, and the gated GEMM's block
# maxima cost it 15 us a block.
ROTATED_DOWN_TILES = {"gfx950": [(math.inf, 0)]}
# Experiments override a table without a rebuild: CHESS_INT8_TILES='{"gate_up": [[18, 9], ["inf", 10]]}' replaces the named
# roles' entries of INT8_TILES' gfx950 table, CHESS_ROTATE_ROWS='[["inf", 1]]' ROTATE_ROWS' and CHESS_ROTATED_DOWN='[["inf", 0]]'
# ROTATED_DOWN_TILES' ("inf" for no bound).
TILES_VARIABLE, ROTATE_VARIABLE, ROTATED_VARIABLE = "CHESS_INT8_TILES", "CHESS_ROTATE_ROWS", "CHESS_ROTATED_DOWN"


def _bounded(entries) -> list[tuple[float, int]]:
    table = [(math.inf if most in ("inf", None) else float(most), int(choice)) for most, choice in entries]
    if not table or table[-1][0] != math.inf or any(a[0] >= b[0] for a, b in zip(table, table[1:])):
        raise ValueError(f"a table runs by growing bounds and ends unbounded, not {entries}")
    return table


def apply_overrides(environment=os.environ) -> None:
    """Replaces table entries named by the CHESS_INT8_TILES / CHESS_ROTATE_ROWS / CHESS_ROTATED_DOWN variables (read at
    import; the tests call it again). Forced tiles and rows never change a bit."""
    tiles = environment.get(TILES_VARIABLE)
    if tiles:
        for role, entries in json.loads(tiles).items():
            if role not in INT8_TILES["gfx950"]:
                raise ValueError(f"{TILES_VARIABLE} names {role}: the roles are {sorted(INT8_TILES['gfx950'])}")
            INT8_TILES["gfx950"][role] = _bounded(entries)
    rows = environment.get(ROTATE_VARIABLE)
    if rows:
        ROTATE_ROWS["gfx950"] = _bounded(json.loads(rows))
    rotated = environment.get(ROTATED_VARIABLE)
    if rotated:
        ROTATED_DOWN_TILES["gfx950"] = _bounded(json.loads(rotated))


apply_overrides()


def tile_takes(tile: int, N: int, K: int, gated: bool = False, bias: bool = False, residual: bool = False, M: int = 0) -> bool:
    """Whether tile takes N outputs of depth K with that epilogue (of M rows, where given); the whole-K tiles take every shape
    int8_linear takes, the split-K and register-held ones only some."""
    if tile in (RESIDENT_TILE, DEEP_TILE) and 2 * M * N >= RESIDENT_OUTPUT_BYTES:
        return False
    if tile == RESIDENT_TILE:
        return K == RESIDENT_DEPTH and N % 8 == 0 and not residual and N <= RESIDENT_GROUPS * (256 if gated else 512)
    if tile == DEEP_TILE:
        return K == DEEP_DEPTH and N % 128 == 0 and not gated and not bias and residual and N <= RESIDENT_GROUPS * 128
    waves = SPLIT_WAVES.get(tile)
    return waves is None or (N % 8 == 0 and K % (128 * waves) == 0 and K // (128 * waves) in (1, 2, 4))


def long_projection_tile(tile: int, M: int, N: int, units: int) -> int:
    """LONG_PROJECTION_TILES' tile, or 11 where the last round of its workgroups is too small: tile 6 holds one of 128 x 128 a compute
    unit and pays in its first round alone, tile 13 two, and pays where the last round fills LEAST_LAST_ROUND of them."""
    workgroups = -(-M // 128) * -(-N // 128)
    if tile == 6:
        return tile if workgroups <= units else 11
    if tile == 13:
        return tile if (workgroups - 1) % (2 * units) + 1 >= LEAST_LAST_ROUND * 2 * units else 11
    return tile


def int8_tile(device: torch.device, matmul: str, M: int, N: int = 0, K: int = 0, gated: bool | None = None, bias: bool = False,
              residual: bool | None = None) -> int:
    """The tile of int8_linear for M rows of matmul (reference int8_blocks.py:39-42, keyed by gfx target, not capability):
    the table's entry for the rows a compute unit's share is, or, given N and K, the first entry from there on whose tile
    takes them with that epilogue (gated and residual default to the role's: gate_up gated, down with the residual; none
    takes them: 0, the kernel's own pick of a whole-K tile, which takes every shape)."""
    arch, units = hip_kernels.gpu(device)
    tiles = INT8_TILES.get(arch, INT8_TILES["gfx950"])[matmul]
    if matmul == "projection" and tiles == SHIPPED_PROJECTION_TILES and K >= LONG_PROJECTION_DEPTH and K % 128 == 0:
        tiles = LONG_PROJECTION_TILES.get(arch, LONG_PROJECTION_TILES["gfx950"])
        tiles = [(most, long_projection_tile(tile, M, N, units) if N else tile) for most, tile in tiles]
    share = M / units
    candidates = [tile for most, tile in tiles if share <= most]
    gated = matmul == "gate_up" if gated is None else gated
    residual = matmul == "down" if residual is None else residual
    return next((tile for tile in candidates if not N or tile_takes(tile, N, K, gated, bias, residual, M)), 0)


def config_for(device: torch.device, kind: str, M: int, K: int, N: int = 0) -> int:
    """The tile int8_linear launches for M rows of kind (projection, gate_up or down) at depth K: the reference's config_for
    (int8_cuda.py:347-354), which there names one of its small-batch CUDA kernels, and here always a tile of the table."""
    return int8_tile(device, kind, M, N, K)


def takes_rows(device: torch.device, kinds: tuple[str, ...], M: int, K: int) -> bool:
    """Whether one of kinds' matmuls of M rows and depth K takes the split-K tile, this build's counterpart of the reference's
    small-batch kernels (int8_cuda.py:357-358)."""
    return any(config_for(device, kind, M, K) in SPLIT_WAVES for kind in kinds)


def rotate_rows(device: torch.device, M: int) -> int:
    """rotate_quant's rows a wavefront for M rows (reference int8_blocks.py:45-50): the target's ROTATE_ROWS entry for the rows a
    compute unit's share is; a target without one lets the kernel choose."""
    arch, units = hip_kernels.gpu(device)
    shares = ROTATE_ROWS.get(arch)
    if shares is None:
        return UNTIMED_ROTATE_ROWS
    share = M / units
    return next(rows for most, rows in shares if share <= most)


def rotated_down_tile(device: torch.device, M: int, hidden: int, width: int) -> int:
    """The folded rotation's tile for M rows whose hidden of `hidden` columns is rotated to `width` (0: rotate_quant and down
    as two launches). The folded kernel takes no padding columns and whole blocks of 128."""
    if hidden != width or width % 128 or M == 0:
        return 0
    arch, units = hip_kernels.gpu(device)
    shares = ROTATED_DOWN_TILES.get(arch, [(math.inf, 0)])
    share = M / units
    return next(tile for most, tile in shares if share <= most)


def hadamard(size: int) -> torch.Tensor:
    """Sylvester's Hadamard matrix of +-1, size a power of two: symmetric, its square is size times the identity."""
    if size <= 0 or size & (size - 1):
        raise ValueError(f"a Sylvester Hadamard matrix has a power-of-two size, not {size}")
    index = torch.arange(size)
    ones = torch.bitwise_and(index[:, None], index[None, :])
    parity = torch.zeros_like(ones)
    while bool(ones.any()):
        parity ^= ones & 1
        ones = ones >> 1
    return 1.0 - 2.0 * parity.float()


def down_inputs(hidden: int) -> int:
    return -(-hidden // DOWN_INPUT_MULTIPLE) * DOWN_INPUT_MULTIPLE


def tile_id(tile: int | tuple[int, ...]) -> int:
    """The library's number for a tile. The reference's launch_int8_linear takes a Triton tile (rows, columns, depth, warps,
    stages[, registers]) (int8_blocks.py:105-108); such a tuple names the tile of the same rows and output columns here, the
    one with as many ring stages if there is one, else the first. Depth, warps and registers are the kernel's own."""
    if isinstance(tile, int):
        if tile != 0 and tile not in TILE_SHAPES and tile not in (RESIDENT_TILE, DEEP_TILE):
            raise ValueError(f"int8_linear has tiles {sorted({*TILE_SHAPES, RESIDENT_TILE, DEEP_TILE})} (0 picks by size), not {tile}")
        return tile
    if len(tile) < 5:
        raise ValueError(f"a tile tuple is (rows, columns, depth, warps, stages[, registers]), not {tile}")
    block_m, block_n, _, _, stages = tile[:5]
    same = [number for number, shape in TILE_SHAPES.items() if shape[:2] == (block_m, block_n)]
    if not same:
        shapes = sorted({shape[:2] for shape in TILE_SHAPES.values()})
        raise ValueError(f"int8_linear has no {block_m} x {block_n} tile; its tiles are {shapes} (rows x output columns)")
    return next((number for number in same if TILE_SHAPES[number][3] == stages), same[0])


def _require(tensor: torch.Tensor | None, dtype: torch.dtype, name: str) -> None:
    if tensor is not None and tensor.dtype != dtype:
        raise ValueError(f"{name} is {tensor.dtype}, the kernel takes {dtype}")


def launch_int8_linear(x: torch.Tensor, x_scale: torch.Tensor, weight: torch.Tensor, weight_scale: torch.Tensor, bias: torch.Tensor | None,
                       residual: torch.Tensor | None, gated: bool, original: torch.Tensor | None, residual_scale: torch.Tensor | None,
                       input_scale: torch.Tensor | None, tile: int | tuple[int, ...] = 0, out_dtype: torch.dtype = torch.float16) -> torch.Tensor:
    """out = epilogue(x @ weight^T) (x M x K, weight N x K, gated: the gate's rows then up's); tile 0 picks by size, a tuple
    names a tile by its shape (tile_id)."""
    tile = tile_id(tile)
    rows, K = weight.shape
    N = rows // 2 if gated else rows
    if K % INT8_DEPTH != 0:
        raise ValueError(f"int8_linear reads the {K} inputs {INT8_DEPTH} at a time")
    if x.shape[-1] != K:
        raise ValueError(f"int8_linear: x has {x.shape[-1]} inputs and the weight {K}")
    for tensor, dtype, name in ((x, torch.int8, "x"), (weight, torch.int8, "weight"), (x_scale, torch.float32, "x_scale"),
                                (weight_scale, torch.float32, "weight_scale"), (bias, torch.float16, "bias"), (residual, torch.float16, "residual"),
                                (original, torch.float16, "original"), (residual_scale, torch.float16, "residual_scale"),
                                (input_scale, torch.float16, "input_scale")):
        _require(tensor, dtype, name)
    if out_dtype not in (torch.float16, torch.bfloat16):
        raise ValueError(f"int8_linear writes fp16 or bf16, not {out_dtype}")
    library = library_for(x.device)
    x, weight = aligned(x), aligned(weight)
    M = x.numel() // K
    if x_scale.numel() != M or weight_scale.numel() != rows:
        raise ValueError(f"int8_linear: {x_scale.numel()} row scales for {M} rows, {weight_scale.numel()} weight scales for {rows} rows")
    out = torch.empty(*x.shape[:-1], N, device=x.device, dtype=out_dtype)
    residual, original = aligned(residual), aligned(original)
    for tensor, name in ((residual, "residual"), (original, "original")):
        if tensor is not None and tensor.numel() != M * N:
            raise ValueError(f"int8_linear: {name} has {tensor.numel()} values, not {M} x {N}")
    code = library.chess_int8_linear(pointer(x), pointer(x_scale.contiguous()), pointer(weight), pointer(weight_scale.contiguous()),
                                     pointer(bias.contiguous() if bias is not None else None), pointer(residual), pointer(original),
                                     pointer(residual_scale), pointer(input_scale), pointer(out), M, N, K, int(gated),
                                     hip_kernels.OUT_BF16 if out_dtype == torch.bfloat16 else hip_kernels.OUT_F16, tile, stream_of(x.device))
    check(code, "int8_linear")
    return out


def int8_matmul_i32(x: torch.Tensor, weight: torch.Tensor, tile: int | tuple[int, ...] = 0) -> torch.Tensor:
    """The exact int32 sums x @ weight^T of int8_linear's kernel, before any epilogue."""
    tile = tile_id(tile)
    _require(x, torch.int8, "x")
    _require(weight, torch.int8, "weight")
    N, K = weight.shape
    if K % INT8_DEPTH != 0 or x.shape[-1] != K:
        raise ValueError(f"int8_matmul_i32 takes depth a multiple of {INT8_DEPTH} matching the weight's {K}, not {x.shape[-1]}")
    library = library_for(x.device)
    x, weight = aligned(x), aligned(weight)
    out = torch.empty(*x.shape[:-1], N, device=x.device, dtype=torch.int32)
    check(library.chess_int8_matmul_i32(pointer(x), pointer(weight), pointer(out), x.numel() // K, N, K, tile, stream_of(x.device)),
          "int8_matmul_i32")
    return out


# matmul (projection, gate_up or down) selects the tile table; given original with the two scales, the epilogue also applies the
# next block's input mix
@torch.library.custom_op("chess::int8_linear", mutates_args=())
def int8_linear(x: torch.Tensor, x_scale: torch.Tensor, weight: torch.Tensor, weight_scale: torch.Tensor, bias: torch.Tensor | None,
                residual: torch.Tensor | None, gated: bool, matmul: str, original: torch.Tensor | None = None,
                residual_scale: torch.Tensor | None = None, input_scale: torch.Tensor | None = None) -> torch.Tensor:
    rows, K = weight.shape
    tile = int8_tile(x.device, matmul, x.numel() // K, rows // 2 if gated else rows, K, gated, bias is not None, residual is not None)
    return launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, original, residual_scale, input_scale, tile)


@int8_linear.register_fake
def _(x, x_scale, weight, weight_scale, bias, residual, gated, matmul, original=None, residual_scale=None, input_scale=None):
    return x.new_empty(*x.shape[:-1], weight.shape[0] // 2 if gated else weight.shape[0], dtype=torch.float16)


def launch_norm_quant(x: torch.Tensor, original: torch.Tensor | None, residual_scale: torch.Tensor | None, input_scale: torch.Tensor | None,
                      gain: torch.Tensor, mixed: torch.Tensor | None, eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    for tensor, name in ((x, "x"), (original, "original"), (residual_scale, "residual_scale"), (input_scale, "input_scale"), (gain, "gain")):
        _require(tensor, torch.float16, name)
    library = library_for(x.device)
    D = x.shape[-1]
    M = x.numel() // D
    if gain.numel() != D:
        raise ValueError(f"norm_quant: {gain.numel()} gains for rows of {D}")
    q = torch.empty(x.shape, device=x.device, dtype=torch.int8)
    scale = torch.empty(x.shape[:-1], device=x.device, dtype=torch.float32)
    code = library.chess_norm_quant(pointer(x), pointer(original), pointer(residual_scale), pointer(input_scale), pointer(gain.contiguous()),
                                    pointer(mixed), pointer(q), pointer(scale), M, D, float(eps), stream_of(x.device))
    check(code, "mix_norm_quant" if original is not None else "norm_quant")
    return q, scale


@torch.library.custom_op("chess::norm_quant", mutates_args=())
def norm_quant(x: torch.Tensor, gain: torch.Tensor, eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    return launch_norm_quant(aligned(x), None, None, None, gain, None, eps)


@norm_quant.register_fake
def _(x, gain, eps):
    return x.new_empty(x.shape, dtype=torch.int8), x.new_empty(x.shape[:-1], dtype=torch.float32)


@torch.library.custom_op("chess::mix_norm_quant", mutates_args=())
def mix_norm_quant(x: torch.Tensor, original: torch.Tensor, residual_scale: torch.Tensor, input_scale: torch.Tensor, gain: torch.Tensor,
                   eps: float) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    x = aligned(x)
    original = aligned(original)
    if original.shape != x.shape:
        raise ValueError(f"mix_norm_quant: the input {tuple(original.shape)} does not match the stream {tuple(x.shape)}")
    mixed = torch.empty_like(x, dtype=torch.float16)
    q, scale = launch_norm_quant(x, original, residual_scale, input_scale, gain, mixed, eps)
    return mixed, q, scale


@mix_norm_quant.register_fake
def _(x, original, residual_scale, input_scale, gain, eps):
    return x.new_empty(x.shape, dtype=torch.float16), x.new_empty(x.shape, dtype=torch.int8), x.new_empty(x.shape[:-1], dtype=torch.float32)


# rotation matrices seen to be Sylvester's H32, by data_ptr: (the tensor, its version). The kernel computes that transform by
# butterflies, never reading them; the entry holds the tensor, so that no other tensor takes its memory while the entry
# stands (an inference tensor always reports version 0)
_SYLVESTER: dict[int, tuple[torch.Tensor, int]] = {}
_SYLVESTER_MOST = 64


def _check_signs(signs: torch.Tensor) -> None:
    if tuple(signs.shape) != (HADAMARD_BLOCK, HADAMARD_BLOCK):
        raise ValueError(f"rotate_quant rotates blocks of {HADAMARD_BLOCK}, not {tuple(signs.shape)}")
    version = 0 if signs.is_inference() else signs._version
    found = _SYLVESTER.get(signs.data_ptr())
    if found is not None and found[0] is signs and found[1] == version:
        return
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("rotate_quant's rotation was not seen before the graph recording began (run the block once first)")
    if not torch.equal(signs.detach().float().cpu(), hadamard(HADAMARD_BLOCK)):
        raise ValueError("rotate_quant's kernel rotates by Sylvester's H32; these signs are another matrix")
    _SYLVESTER[signs.data_ptr()] = (signs, version)
    while len(_SYLVESTER) > _SYLVESTER_MOST:
        del _SYLVESTER[next(iter(_SYLVESTER))]


#h's rows times the block-diagonal Hadamard matrix, rounded to int8 width wide
@torch.library.custom_op("chess::rotate_quant", mutates_args=())
def rotate_quant(h: torch.Tensor, hadamard_signs: torch.Tensor, width: int) -> tuple[torch.Tensor, torch.Tensor]:
    _require(h, torch.float16, "h")
    _check_signs(hadamard_signs)
    library = library_for(h.device)
    h = aligned(h)
    N = h.shape[-1]
    M = h.numel() // N
    q = torch.empty(*h.shape[:-1], width, device=h.device, dtype=torch.int8)
    scale = torch.empty(h.shape[:-1], device=h.device, dtype=torch.float32)
    check(library.chess_rotate_quant(pointer(h), pointer(q), pointer(scale), M, N, width, rotate_rows(h.device, M), stream_of(h.device)),
          "rotate_quant")
    return q, scale


@rotate_quant.register_fake
def _(h, hadamard_signs, width):
    return h.new_empty(*h.shape[:-1], width, dtype=torch.int8), h.new_empty(h.shape[:-1], dtype=torch.float32)


@torch.library.custom_op("chess::gated_int8_linear_absmax", mutates_args=())
def gated_int8_linear_absmax(x: torch.Tensor, x_scale: torch.Tensor, weight: torch.Tensor, weight_scale: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """gate_up's int8_linear (silu(gate) * up, fp16) and, for each row and 32-column block of it, the largest magnitude of
    that block times Sylvester's H32, as rotate_quant rotates it (rotated_int8_linear's row maxima)."""
    for tensor, dtype, name in ((x, torch.int8, "x"), (weight, torch.int8, "weight"), (x_scale, torch.float32, "x_scale"),
                                (weight_scale, torch.float32, "weight_scale")):
        _require(tensor, dtype, name)
    rows, K = weight.shape
    N = rows // 2
    if K % INT8_DEPTH != 0 or x.shape[-1] != K:
        raise ValueError(f"gated_int8_linear_absmax reads the {K} inputs {INT8_DEPTH} at a time, x has {x.shape[-1]}")
    library = library_for(x.device)
    x, weight = aligned(x), aligned(weight)
    M = x.numel() // K
    if x_scale.numel() != M or weight_scale.numel() != rows:
        raise ValueError(f"gated_int8_linear_absmax: {x_scale.numel()} row scales for {M} rows, {weight_scale.numel()} weight scales for {rows}")
    out = torch.empty(*x.shape[:-1], N, device=x.device, dtype=torch.float16)
    maxima = torch.empty(*x.shape[:-1], N // HADAMARD_BLOCK, device=x.device, dtype=torch.float32)
    tile = int8_tile(x.device, "gate_up", M)
    if tile in SPLIT_WAVES or tile in (RESIDENT_TILE, DEEP_TILE):
        tile = 0
    check(library.chess_gated_int8_linear_absmax(pointer(x), pointer(x_scale.contiguous()), pointer(weight), pointer(weight_scale.contiguous()),
                                                 pointer(out), pointer(maxima), M, N, K, tile, stream_of(x.device)), "gated_int8_linear_absmax")
    return out, maxima


@gated_int8_linear_absmax.register_fake
def _(x, x_scale, weight, weight_scale):
    N = weight.shape[0] // 2
    return x.new_empty(*x.shape[:-1], N, dtype=torch.float16), x.new_empty(*x.shape[:-1], N // HADAMARD_BLOCK, dtype=torch.float32)


def launch_rotated_int8_linear(h: torch.Tensor, block_absmax: torch.Tensor, weight: torch.Tensor, weight_scale: torch.Tensor, bias: torch.Tensor | None,
                               residual: torch.Tensor | None, original: torch.Tensor | None, residual_scale: torch.Tensor | None,
                               input_scale: torch.Tensor | None, tile: int = 0) -> torch.Tensor:
    """int8_linear(*rotate_quant(h, signs, K), weight, ...) in one launch, from h and its block maxima: the same bits."""
    N, K = weight.shape
    for tensor, dtype, name in ((h, torch.float16, "h"), (block_absmax, torch.float32, "block_absmax"), (weight, torch.int8, "weight"),
                                (weight_scale, torch.float32, "weight_scale"), (bias, torch.float16, "bias"), (residual, torch.float16, "residual"),
                                (original, torch.float16, "original"), (residual_scale, torch.float16, "residual_scale"),
                                (input_scale, torch.float16, "input_scale")):
        _require(tensor, dtype, name)
    if h.shape[-1] != K or K % INT8_DEPTH:
        raise ValueError(f"rotated_int8_linear takes hidden rows as wide as the weight's {K} inputs (a multiple of {INT8_DEPTH}), not {h.shape[-1]}")
    library = library_for(h.device)
    h, weight, residual, original = aligned(h), aligned(weight), aligned(residual), aligned(original)
    M = h.numel() // K
    if block_absmax.numel() != M * (K // HADAMARD_BLOCK) or weight_scale.numel() != N:
        raise ValueError(f"rotated_int8_linear: {block_absmax.numel()} block maxima for {M} rows of {K}, {weight_scale.numel()} weight scales for {N}")
    for tensor, name in ((residual, "residual"), (original, "original")):
        if tensor is not None and tensor.numel() != M * N:
            raise ValueError(f"rotated_int8_linear: {name} has {tensor.numel()} values, not {M} x {N}")
    out = torch.empty(*h.shape[:-1], N, device=h.device, dtype=torch.float16)
    code = library.chess_rotated_int8_linear(pointer(h), pointer(block_absmax.contiguous()), pointer(weight), pointer(weight_scale.contiguous()),
                                             pointer(bias.contiguous() if bias is not None else None), pointer(residual), pointer(original),
                                             pointer(residual_scale), pointer(input_scale), pointer(out), M, N, K, tile, stream_of(h.device))
    check(code, "rotated_int8_linear")
    return out


# down of Int8Block.forward with the rotation of its input folded in (reference int8_blocks.py:285-288 as one launch)
@torch.library.custom_op("chess::rotated_int8_linear", mutates_args=())
def rotated_int8_linear(h: torch.Tensor, block_absmax: torch.Tensor, weight: torch.Tensor, weight_scale: torch.Tensor, bias: torch.Tensor | None,
                        residual: torch.Tensor | None, original: torch.Tensor | None = None, residual_scale: torch.Tensor | None = None,
                        input_scale: torch.Tensor | None = None) -> torch.Tensor:
    tile = rotated_down_tile(h.device, h.numel() // weight.shape[1], h.shape[-1], weight.shape[1]) or 1
    return launch_rotated_int8_linear(h, block_absmax, weight, weight_scale, bias, residual, original, residual_scale, input_scale, tile)


@rotated_int8_linear.register_fake
def _(h, block_absmax, weight, weight_scale, bias, residual, original=None, residual_scale=None, input_scale=None):
    return h.new_empty(*h.shape[:-1], weight.shape[0], dtype=torch.float16)


class Int8Block(nn.Module):
    """model/int8_blocks.py:254-288 of the reference: a FusedBlock whose projection, gate_up and down are int8.
    output_scale multiplies down's scales, as fp16 inference shrinks the residual stream."""

    def __init__(self, block: FusedBlock, weights: dict[str, tuple[torch.Tensor, torch.Tensor]], output_scale: float):
        super().__init__()
        self.heads, self.kv_heads, self.dq, self.dv, self.templates_count = block.heads, block.kv_heads, block.dq, block.dv, block.templates_count
        self.ln1, self.ln2 = block.ln1, block.ln2
        self.residual_scale, self.input_scale = block.residual_scale, block.input_scale
        self.q_gain, self.k_gain, self.eps = block.q_gain, block.k_gain, block.eps
        self.projection_bias = block.projection_bias
        # combine_heads stays an fp16 linear: as int8, its input (the attention output) would take a scale per head
        self.combine_heads, self.combine_heads_bias = block.combine_heads, block.combine_heads_bias
        device = block.projection.device
        for name, (integers, scale) in weights.items():
            self.register_buffer(name, integers.to(device).contiguous())
            self.register_buffer(f"{name}_scale", (scale * output_scale if name == "down" else scale).to(device, torch.float32).contiguous())
        self.register_buffer("hadamard_signs", hadamard(HADAMARD_BLOCK).to(device, torch.float16))
        if self.hadamard_signs.is_cuda:
            _check_signs(self.hadamard_signs)
        # link_input_mixes sets these: next_scales (the following block's two mix scales, for down's epilogue to mix with) and
        # input_mixed (this block's input arrives already mixed)
        self.next_scales: tuple[nn.Parameter, nn.Parameter] | None = None
        self.input_mixed = False

    def forward(self, x: torch.Tensor, templates: torch.Tensor, original_board_embed: torch.Tensor) -> torch.Tensor:
        if self.input_mixed:
            normed, scale = norm_quant(x, self.ln1.weight, self.ln1.eps)
        else:
            x, normed, scale = mix_norm_quant(x, original_board_embed, self.residual_scale, self.input_scale, self.ln1.weight, self.ln1.eps)
        projected = int8_linear(normed, scale, self.projection, self.projection_scale, self.projection_bias, None, False, "projection")
        attended = template_attention(projected, templates, self.q_gain, self.k_gain, self.heads, self.kv_heads, self.dq, self.dv, self.templates_count,
                                      self.eps)
        x = linear(attended, self.combine_heads, self.combine_heads_bias, residual=x)
        normed, scale = norm_quant(x, self.ln2.weight, self.ln2.eps)
        if rotated_down_tile(x.device, normed.numel() // normed.shape[-1], self.gate_up.shape[0] // 2, self.down.shape[1]):
            # rotate_quant folded into down: gate_up also gives the rotated blocks' maxima (the same bits as the three launches)
            _check_signs(self.hadamard_signs)
            hidden, maxima = gated_int8_linear_absmax(normed, scale, self.gate_up, self.gate_up_scale)
            if self.next_scales is None:
                return rotated_int8_linear(hidden, maxima, self.down, self.down_scale, None, x)
            return rotated_int8_linear(hidden, maxima, self.down, self.down_scale, None, x, original_board_embed, *self.next_scales)
        hidden = int8_linear(normed, scale, self.gate_up, self.gate_up_scale, None, None, True, "gate_up")
        rotated, scale = rotate_quant(hidden, self.hadamard_signs, self.down.shape[1])
        if self.next_scales is None:
            return int8_linear(rotated, scale, self.down, self.down_scale, None, x, False, "down")
        return int8_linear(rotated, scale, self.down, self.down_scale, None, x, False, "down", original_board_embed, *self.next_scales)


def kernels(device: torch.device):
    """The kernels for device, loaded and checked now rather than while a graph records (reference int8_cuda.py:334-344)."""
    return library_for(device)


def quantize_blocks(model: nn.Module, weights: dict[int, dict], output_scale: float) -> nn.Module:
    """model's blocks of the layers in weights become Int8Blocks; the input mixes are relinked (reference int8_blocks.py:292-298)."""
    blocks = [Int8Block(block, weights[layer], output_scale) if layer in weights else block for layer, block in enumerate(model.encoder)]
    link_input_mixes(blocks)
    model.encoder = nn.ModuleList(blocks)
    if weights:
        kernels(next(model.parameters()).device)
    return model
