"""fp16 blocks and the template attention on gfx950: the module API of the reference's model/fused_blocks.py
that the int8 path uses -- the operators chess::template_attention and chess::linear, FusedBlock,
link_input_mixes, tile_for -- and FusedTransformer, the network the engine calls.

The operators launch the HIP kernels of libchess_hip.so, the input embedding included (chess::board_embedding, which finds
the square features from the boards as the reference's board_embedding_kernel does) and the heads (chess::answer_heads: the
move logits written into the answer rows, the eval head and the expected score). FusedTransformer returns the move logits and
the value logits, as the reference's does on GPUs without its fused ends (gfx950 among them); the answer rows come from the
same launches when asked for (rows=True), which is what the graph lanes ask.
"""
from __future__ import annotations

import math
import threading

import torch
import torch.nn.functional as F
from torch import nn

from model import hip_kernels
from model.encoding import NUM_SQUARES, TOKENS_PER_BOARD
from model.hip_kernels import aligned, check, gpu, library_for, pointer, stream_of
from model.model import EDGE, KING, KNIGHT, NO_PIECE, PAWN, QUEEN, THEIRS, ChessTransformer, TransformerBlock, value_bin_centres

LINEAR_DEPTH, GROUP_M = 32, 8
FEATURE_SLOTS = 23
# linear's tiles by the rows a compute unit's share is (reference fused_blocks.py:183-185), the GEMM's tile numbers: tiles
# 1 and 3 keep the small batches' launches on more compute units than tile 11's 128 x 128 (the network at batch 16 / 32:
# 0.16 / 0.11 ms a forward faster), and from 9 to 48 rows the eight-wavefront 128 x 128 tile 6 (the network, alternated
# on one box: batch 64 2.455-2.468 against 2.506-2.510 ms a forward with tile 8, batch 128 3.82-3.85 against 3.86 with 11)
LINEAR_TILES = {"gfx950": [(5, 1), (9, 3), (48, 6), (100, 11), (math.inf, 15)]}
# tile 15 holds each wavefront's weights in registers (gemm_resident.h): for fp16 sums it takes depth 512 with the bias,
# the residual added or not, not gated (the attention's output projection: 56.8-59.3 against 64.9-65.5 us on tile 11 at
# 71,680 rows, the network at batch 1024 18.85-18.88 against 18.90-18.93 ms, alternated on one box; the fp16 block's
# projection to 1,600 columns: 155.7 against 200.2 us on tile 0); other linears of the table's share take tile 0, the
# kernel's own pick by size
RESIDENT_TILE, RESIDENT_DEPTH = 15, 512
RESIDENT_OUTPUT_BYTES, RESIDENT_COLUMNS = 1 << 31, 32 * 256   # its outputs' (32-bit offsets) and its column groups' limits
# and from this share on where it has 1,024 columns or more, so that each of its workgroups still has a long stream of row
# blocks (graphs of launches, tile 15 and 11, us: 512 to 1,600 columns at 17,920 rows 40.1 and 46.6, at 12,800 30.6 and 35.6; to
# 1,280 at 12,544 rows 27.6 and 26.8, at 13,312 27.8 and 29.8; to 1,024 at 12,544 24.7 and 26.5, at 16,384 27.4 and 26.1, with the
# residual 28.3 and 31.3), up to the 4,096 it was timed with (12,800 rows 58.3 and 77.6)
RESIDENT_WIDE_SHARE, RESIDENT_WIDE_COLUMNS = 48, range(1024, 4097)
# gated, rows of whole lines (tile 12 stages 128 bytes of a row) from 1 KB on; others keep LINEAR_TILES. Graphs of launches, us:
# 512 to 2 x 2,048 4,480 rows 27.5 on tile 12 and 29.3 on tile 6, 1,024 to 2 x 2,816 63.3 and 69.7, but 256 to 2 x 1,024 12.1 and
# 11.7. Past 100 rows a compute unit the eight-wavefront 256 x 128 tile 4 pays for rows of 1,408 bytes or more (tile 4 and 11; 32,000
# and 71,680 rows): 704 to 2 x 2,048 196 and 204, 443 and 444; 768 to 2 x 992 107 and 115, 236 and 249; 1,024 to 2 x 2,816 361 and 385,
# 797 and 842; but 512 to 2 x 2,048 153 and 151, 345 and 328; 512 to 2 x 512 at 35,840 rows 56.3 and 48.8; 256 to 2 x 1,024 49.2 and
# 44.6, 104 and 95; 640 to 2 x 1,280 either way
LINEAR_GATED_TILES = {"gfx950": [(5, 1), (9, 3), (20, 12), (48, 6), (math.inf, 11)]}
LINEAR_GATED_LONG_ROW_TILES = {"gfx950": [(5, 1), (9, 3), (20, 12), (48, 6), (100, 11), (math.inf, 4)]}
GATED_ROW_BYTES, GATED_LONG_ROW_BYTES = 1024, 1408
# f32 out (accumulate_fp32, the policy head's `a`), graphs of launches on an MI355X, us: rows of whole lines up to 2 KB take
# 128 x 64 with 128-byte stages (512 to 512: 9.3 against 10.8 on tile 7 at 4,480 rows, 24.5 against 33.7 at 17,920, 78.8 against
# 84.7 at 71,680; 768 to 768 11.5 against 13.5 at 3,570, 50.4 against 52.9 at 21,000; 1,024 to 1,024 71.8 against 81.3 there) and
# 64 x 64 up to 9 rows a compute unit (1,120 rows 5.7 against 9.5, 7.1 against 11.8 and 8.9 against 14.3); others the 128 x 128
# with a 3-stage ring
LINEAR_F32_TILES = {"gfx950": [(9, 1), (math.inf, 12)]}
LINEAR_F32_OTHER_TILES = {"gfx950": [(4, 1), (math.inf, 7)]}
F32_ROW_BYTES = 2048
# rows of 1.5 KB or more (the fp16 block's down, combine of a width of 768 or more), not gated: 128 x 128 with 128-byte stages,
# whole L2 lines a step (2,048 inputs: 190 against 226 us at 71,680 rows, 94 against 101 with tile 12 at 35,840; 768 inputs to
# 768: 79.2 against 91.9 with tile 11 at 49,000); 128 x 64 with 128-byte stages up to 100 rows a compute unit (2,048 inputs at
# 17,920 rows 54.7 against 58.2 us, 768 inputs 36.8 against 38.6 with tile 11; batch 64 22.0 against 23.8) and 64 x 64 up to 9
# (batch 16: 11.8 against 20.7 us). Rows shorter than 2 KB leave 64 x 64 for 128 x 64 (tile 3) from 5 rows a compute unit once it
# would be more than SMALL_TILES_A_UNIT workgroups a compute unit (768 inputs, with bias: to 1,152 at 1,792 rows, 504 of them,
# 9.8 and 9.0 us; to 1,600 at 2,048, 800, 14.4 and 12.7; to 768 at 2,048, 384, 8.4 and 8.4; at 1,500, 288, 7.3 and 8.0)
LINEAR_LONG_ROW_TILES = {"gfx950": [(9, 1), (100, 12), (math.inf, 13)]}
LINEAR_MANY_TILES = {"gfx950": [(5, 1), (9, 3), (100, 12), (math.inf, 13)]}
LONG_ROW_BYTES, MANY_TILES_ROW_BYTES, SMALL_TILES_A_UNIT = 1536, 2048, 1.6
# template_attention launches of up to this many tokens, query and value widths up to this, share their pairs out by themselves
# (csrc/attention_wave.h) and take any run of pairs a workgroup; the others take groups_per_workgroup's
ATTENTION_SHARING_TOKENS, ATTENTION_SHARING_WIDTH = 80, 64

# Where tile 12's 128 x 64 workgroups are more than the compute units hold at once (three each: 48 KB of LDS) and 128 x 128
# ones are not (two each), rows of ONE_ROUND_ROW_BYTES or more that a table gives to 12 take 13: one round of workgroups,
# not one and a remainder (768 inputs: to 768 at 9,000 rows 852 and 426 of them, 21.7 and 17.1 us, to 1,152 at 6,453 22.3
# and 17.3, f32 out to 768 at 9,000 27.3 and 23.1; but to 768 at 8,000, 756, 15.6 and 16.5, and at 11,000, 1,032 and 516,
# 23.5 and 26.2. Of 768 to 2,048 inputs everywhere between the two, by 1.17 to 1.36; f32 out of 640 to 1,024 by 0.95 to
# 1.26; of 512 by 1.01 to 1.12 up to half a workgroup more a compute unit, 512 to 512 at 12,900 rows 20.4 and 18.4, and 0.93
# to 0.97 past it; of 256 by 0.80 to 1.04)
ONE_ROUND, ONE_ROUND_ROW_BYTES = {12: (128, 64, 3), 13: (128, 128, 2)}, 1280   # each tile's (rows, columns, workgroups a compute unit)
SMALL_REMAINDER_ROW_BYTES, SMALL_REMAINDER = 1024, 0.5


def in_one_round(tile: int, M: int, N: int, units: int, more: float = 0) -> bool:
    rows, columns, held = ONE_ROUND[tile]
    return -(-M // rows) * -(-N // columns) <= (held + more) * units


# tiles lists (share, tile) pairs by growing share; a launch takes the first whose share bounds M / multiprocessors (the last bounds any)
def tile_for(tiles: list[tuple[float, object]], M: int, multiprocessors: int):
    share = M / multiprocessors
    return next(tile for most, tile in tiles if share <= most)


def linear_takes(tile: int, K: int, N: int, gated: bool, bias: bool, residual: bool, accumulate_fp32: bool, mix: bool = False, M: int = 0) -> bool:
    """Whether linear's tile takes the launch: every tile does but 15, which takes fp16 sums of depth 512 into N a multiple of
    8, at most 8,192, with the bias (and the residual or not), not gated, without the next block's input mix, in fp16, and M rows
    (where given) of less than 2 GiB."""
    return tile != RESIDENT_TILE or (K == RESIDENT_DEPTH and N % 8 == 0 and N <= RESIDENT_COLUMNS and 2 * M * N < RESIDENT_OUTPUT_BYTES
                                     and not gated and bias and not mix and not accumulate_fp32)


def linear_tile(device: torch.device, M: int, accumulate_fp32: bool = False, row_bytes: int = 0, gated: bool = False, N: int = 0) -> int:
    arch, units = gpu(device)
    whole_lines = row_bytes > 0 and row_bytes % 128 == 0   # (0: the rows' length is not known)
    if accumulate_fp32:
        table = LINEAR_F32_TILES if whole_lines and row_bytes <= F32_ROW_BYTES else LINEAR_F32_OTHER_TILES
    elif gated and whole_lines and row_bytes >= GATED_ROW_BYTES:
        table = LINEAR_GATED_TILES if row_bytes < GATED_LONG_ROW_BYTES else LINEAR_GATED_LONG_ROW_TILES
    elif row_bytes >= LONG_ROW_BYTES and whole_lines and not gated:
        many = row_bytes < MANY_TILES_ROW_BYTES and (M + 63) // 64 * ((N + 63) // 64) > SMALL_TILES_A_UNIT * units
        table = LINEAR_MANY_TILES if many else LINEAR_LONG_ROW_TILES
    else:
        table = LINEAR_TILES
    tile = tile_for(table.get(arch, table["gfx950"]), M, units)
    if tile == 12 and not gated and N and not in_one_round(12, M, N, units) and in_one_round(13, M, N, units):
        small = row_bytes >= SMALL_REMAINDER_ROW_BYTES and in_one_round(12, M, N, units, SMALL_REMAINDER)
        return 13 if small or row_bytes >= ONE_ROUND_ROW_BYTES else 12
    return tile


def attention_waves(tokens: int) -> int:
    """The wavefronts of a template_attention workgroup that walks a run of pairs: one a slab of 16 queries."""
    return (tokens + 15) // 16


def groups_per_workgroup(positions: int, kv_heads: int, multiprocessors: int = 256, tokens: int = 70) -> int:
    """The most (position, key/value group) pairs a workgroup takes -- a divisor of all the launch's pairs -- while the launch
    keeps as many workgroups as the compute units hold at once (two wavefronts a SIMD, four SIMDs: one workgroup of five to
    eight wavefronts, two of four), so that a workgroup's start (its template registers and first loads) is paid once for
    its pairs; any choice gives the same bits."""
    pairs = positions * kv_heads
    workgroups = multiprocessors * max(1, 8 // attention_waves(tokens))
    groups = max(1, pairs // workgroups)
    while pairs % groups:
        groups -= 1
    return groups


def launch_template_attention(projected: torch.Tensor, templates: torch.Tensor, q_gain: torch.Tensor, k_gain: torch.Tensor, heads: int, kv_heads: int,
                              dq: int, dv: int, templates_count: int, eps: float, groups_per_block: int | None = None) -> torch.Tensor:
    # rows of fp16 (the network's), or of bf16 (the benchmark's standalone config 2): out in the rows' type; the templates and
    # gains (parameters) in either, taken as fp16
    for tensor, name in ((projected, "projected"), (templates, "templates"), (q_gain, "q_gain"), (k_gain, "k_gain")):
        if tensor.dtype not in (torch.float16, torch.bfloat16):
            raise ValueError(f"template_attention's {name} is {tensor.dtype}, the kernel takes fp16 or bf16")
    bf16 = projected.dtype == torch.bfloat16
    q_gain, k_gain = q_gain.half(), k_gain.half()
    B, T, width = projected.shape
    if width != heads * dq + kv_heads * dq + kv_heads * dv + heads * templates_count:
        raise ValueError(f"template_attention: rows of {width} are not q | k | v | template mix for {heads} heads, {kv_heads} key/value heads, "
                         f"widths {dq} and {dv}, {templates_count} templates")
    if templates.shape[0] < templates_count or tuple(templates.shape[1:]) != (NUM_SQUARES, NUM_SQUARES):
        raise ValueError(f"template_attention takes {templates_count} templates of 64 x 64, not {tuple(templates.shape)}")
    library = library_for(projected.device)
    projected = aligned(projected)
    keyed = keyed_templates(templates, templates_count)
    out = torch.empty(B, T, heads * dv, device=projected.device, dtype=projected.dtype)
    shares = T <= ATTENTION_SHARING_TOKENS and max(dq, dv) <= ATTENTION_SHARING_WIDTH
    groups = groups_per_block or (1 if shares else groups_per_workgroup(B, kv_heads, gpu(projected.device)[1], T))
    entry = library.chess_template_attention_bf16 if bf16 else library.chess_template_attention
    code = entry(pointer(projected), pointer(keyed), pointer(q_gain.contiguous()), pointer(k_gain.contiguous()), pointer(out), B, T, heads,
                 kv_heads, dq, dv, templates_count, groups, float(eps), 1 / math.sqrt(dq), stream_of(projected.device))
    check(code, "template_attention")
    return out


#an opaque op, so that torch.compile does not compile through the kernel calls
@torch.library.custom_op("chess::template_attention", mutates_args=())
def template_attention(projected: torch.Tensor, templates: torch.Tensor, q_gain: torch.Tensor, k_gain: torch.Tensor, heads: int, kv_heads: int,
                       dq: int, dv: int, templates_count: int, eps: float) -> torch.Tensor:
    return launch_template_attention(projected, templates, q_gain, k_gain, heads, kv_heads, dq, dv, templates_count, eps)


@template_attention.register_fake
def _(projected, templates, q_gain, k_gain, heads, kv_heads, dq, dv, templates_count, eps):
    B, T, _ = projected.shape
    return projected.new_empty(B, T, heads * dv)


# by data_ptr: (the templates, their version, the templates used, their key-major copy); the entry holds the templates so that
# their memory is not another's
KEYED: dict[int, tuple[torch.Tensor, int, int, torch.Tensor]] = {}
KEYED_MOST = 64
KEYED_LOCK = threading.Lock()
TEMPLATE_SLOTS = 8


def keyed_templates(templates: torch.Tensor, templates_count: int) -> torch.Tensor:
    """keyed[i, j, t] = templates[t, i, j] for t < templates_count, zero up to 8: the kernel reads a query's templates for 4 keys as 64
    contiguous bytes. Made once per templates and version outside graph recording, as the reference pairs its templates
    (attention_cuda.py:410-440)."""
    version = 0 if templates.is_inference() else templates._version
    found = KEYED.get(templates.data_ptr())
    if found is not None and found[1] == version and found[2] == templates_count and found[0].shape == templates.shape:
        return found[3]
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("template_attention's templates were not seen before the graph recording began (run the model once first)")
    with torch.no_grad():
        keyed = torch.zeros(NUM_SQUARES, NUM_SQUARES, TEMPLATE_SLOTS, device=templates.device, dtype=torch.float16)
        keyed[..., :templates_count] = templates[:templates_count].detach().permute(1, 2, 0)
    with KEYED_LOCK:
        KEYED[templates.data_ptr()] = (templates, version, templates_count, keyed)
        while len(KEYED) > KEYED_MOST:
            del KEYED[next(iter(KEYED))]
    return keyed


# by data_ptr: (the K x N weight, its version, its N x K copy); the entry holds the weight so that its memory is not another's
TRANSPOSED: dict[int, tuple[torch.Tensor, int, torch.Tensor]] = {}
TRANSPOSED_MOST = 512
TRANSPOSED_LOCK = threading.Lock()


def transposed_weight(weight: torch.Tensor) -> torch.Tensor:
    """The N x K copy of a K x N weight that the kernel reads (both its operands are read along K), made once per weight and
    version outside graph recording, as the reference pairs its templates once (attention_cuda.py:410-440)."""
    version = 0 if weight.is_inference() else weight._version
    found = TRANSPOSED.get(weight.data_ptr())
    if found is not None and found[1] == version and found[0].shape == weight.shape:
        return found[2]
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("linear's weight was not seen before the graph recording began (run the model once first)")
    with torch.no_grad():
        copy = weight.detach().t().contiguous()
    with TRANSPOSED_LOCK:
        TRANSPOSED[weight.data_ptr()] = (weight, version, copy)
        while len(TRANSPOSED) > TRANSPOSED_MOST:
            del TRANSPOSED[next(iter(TRANSPOSED))]
    return copy


def launch_linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, residual: torch.Tensor | None, gated: bool,
                  accumulate_fp32: bool, original: torch.Tensor | None, residual_scale: torch.Tensor | None, input_scale: torch.Tensor | None,
                  tile: int = 0) -> torch.Tensor:
    K, width = weight.shape
    N = width // 2 if gated else width
    if K % LINEAR_DEPTH != 0:
        raise ValueError(f"linear reads the {K} inputs {LINEAR_DEPTH} at a time")
    if x.shape[-1] != K:
        raise ValueError(f"linear: x has {x.shape[-1]} inputs and the weight {K}")
    for tensor, name in ((x, "x"), (weight, "weight"), (bias, "bias"), (residual, "residual"), (original, "original"),
                         (residual_scale, "residual_scale"), (input_scale, "input_scale")):
        if tensor is not None and tensor.dtype != torch.float16:
            raise ValueError(f"linear's {name} is {tensor.dtype}, the kernel takes fp16")
    library = library_for(x.device)
    x, residual, original = aligned(x), aligned(residual), aligned(original)
    weight = aligned(transposed_weight(weight))
    M = x.numel() // K
    out = x.new_empty(*x.shape[:-1], N, dtype=torch.float32 if accumulate_fp32 else torch.float16)
    code = library.chess_linear(pointer(x), pointer(weight), pointer(bias.contiguous() if bias is not None else None), pointer(residual),
                                pointer(original), pointer(residual_scale), pointer(input_scale), pointer(out), M, N, K, int(gated),
                                hip_kernels.OUT_F32 if accumulate_fp32 else hip_kernels.OUT_F16, tile, stream_of(x.device))
    check(code, "linear")
    return out


#fp16 inputs, f32 sums; fp16 out, or f32 with accumulate_fp32 (reference fused_blocks.py:307-313)
@torch.library.custom_op("chess::linear", mutates_args=())
def linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None = None, residual: torch.Tensor | None = None,
           gated: bool = False, accumulate_fp32: bool = False, original: torch.Tensor | None = None, residual_scale: torch.Tensor | None = None,
           input_scale: torch.Tensor | None = None) -> torch.Tensor:
    K, width = weight.shape
    M, N = x.numel() // K, width // 2 if gated else width
    tile = linear_tile(x.device, M, accumulate_fp32, K * x.element_size(), gated, N)
    takes = lambda tile: linear_takes(tile, K, N, gated, bias is not None, residual is not None, accumulate_fp32, original is not None, M)
    if N in RESIDENT_WIDE_COLUMNS and M > RESIDENT_WIDE_SHARE * gpu(x.device)[1] and takes(RESIDENT_TILE):
        tile = RESIDENT_TILE
    elif not takes(tile):
        tile = 0
    return launch_linear(x, weight, bias, residual, gated, accumulate_fp32, original, residual_scale, input_scale, tile)


@linear.register_fake
def _(x, weight, bias=None, residual=None, gated=False, accumulate_fp32=False, original=None, residual_scale=None, input_scale=None):
    return x.new_empty(*x.shape[:-1], weight.shape[1] // 2 if gated else weight.shape[1], dtype=torch.float32 if accumulate_fp32 else x.dtype)


def launch_rms_norm(x: torch.Tensor, original: torch.Tensor | None, residual_scale: torch.Tensor | None, input_scale: torch.Tensor | None,
                    gain: torch.Tensor, eps: float) -> tuple[torch.Tensor | None, torch.Tensor]:
    """(mixed or None, f16(RMSNorm(mixed or x) * gain)): the fp16 blocks' norms in norm_quant's f32 order, one launch."""
    for tensor, name in ((x, "x"), (original, "original"), (residual_scale, "residual_scale"), (input_scale, "input_scale"), (gain, "gain")):
        if tensor is not None and tensor.dtype != torch.float16:
            raise ValueError(f"rms_norm's {name} is {tensor.dtype}, the kernel takes fp16")
    library = library_for(x.device)
    x, original = aligned(x), aligned(original)
    D = x.shape[-1]
    if gain.numel() != D:
        raise ValueError(f"rms_norm: {gain.numel()} gains for rows of {D}")
    if original is not None and original.shape != x.shape:
        raise ValueError(f"rms_norm: the input {tuple(original.shape)} does not match the stream {tuple(x.shape)}")
    mixed = torch.empty_like(x) if original is not None else None
    out = torch.empty_like(x)
    code = library.chess_rms_norm(pointer(x), pointer(original), pointer(residual_scale), pointer(input_scale), pointer(gain.contiguous()),
                                  pointer(mixed), pointer(out), x.numel() // D, D, float(eps), stream_of(x.device))
    check(code, "rms_norm")
    return mixed, out


def norm_eps(norm: nn.RMSNorm, x: torch.Tensor) -> float:
    """nn.RMSNorm's eps: its own, or the dtype's machine epsilon when it has none (as torch's rms_norm takes it)."""
    return norm.eps if norm.eps is not None else torch.finfo(x.dtype).eps


#the fp16 blocks' RMSNorm (nn.RMSNorm at reference fused_blocks.py:348, 351, 863), f32 inside, fp16 out
@torch.library.custom_op("chess::rms_norm", mutates_args=())
def rms_norm(x: torch.Tensor, gain: torch.Tensor, eps: float) -> torch.Tensor:
    return launch_rms_norm(x, None, None, None, gain, eps)[1]


@rms_norm.register_fake
def _(x, gain, eps):
    return torch.empty_like(x)


#the fp16 block's own input mix and its ln1 (reference fused_blocks.py:346-348): (mixed, normalised)
@torch.library.custom_op("chess::mix_rms_norm", mutates_args=())
def mix_rms_norm(x: torch.Tensor, original: torch.Tensor, residual_scale: torch.Tensor, input_scale: torch.Tensor, gain: torch.Tensor,
                 eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    return launch_rms_norm(x, original, residual_scale, input_scale, gain, eps)


@mix_rms_norm.register_fake
def _(x, original, residual_scale, input_scale, gain, eps):
    return torch.empty_like(x), torch.empty_like(x)


def transposed(weight: torch.Tensor) -> nn.Parameter:
    return nn.Parameter(weight.detach().t().contiguous())


class FusedBlock(nn.Module):
    """A TransformerBlock's weights as the fused kernels read them (reference fused_blocks.py:325-354):
    projection = [Q | K | V | template_mix] transposed, gate_up = [gate | up] transposed."""

    def __init__(self, block: TransformerBlock):
        super().__init__()
        self.heads, self.kv_heads = block.n_heads, block.kv_heads
        self.dq, self.dv, self.templates_count = block.d_qk_head, block.d_head, block.position_templates
        self.ln1, self.ln2 = block.ln1, block.ln2
        self.residual_scale, self.input_scale = block.residual_scale, block.input_scale
        self.q_gain, self.k_gain = block.q_norm.weight, block.k_norm.weight
        self.eps = block.q_norm.eps
        projections = (block.Q, block.K, block.V, block.template_mix)
        mlp = block.mlp
        self.projection = transposed(torch.cat([projection.weight for projection in projections]))
        self.projection_bias = nn.Parameter(torch.cat([projection.bias for projection in projections]).detach())
        self.combine_heads = transposed(block.combine_heads.weight)
        self.combine_heads_bias = block.combine_heads.bias
        self.gate_up = transposed(torch.cat([mlp.gate_projection.weight, mlp.up_projection.weight]))
        self.down = transposed(mlp.down_projection.weight)
        self.next_scales: tuple[nn.Parameter, nn.Parameter] | None = None
        self.input_mixed = False

    def forward(self, x: torch.Tensor, templates: torch.Tensor, original_board_embed: torch.Tensor) -> torch.Tensor:
        #the input mix, when this block makes it, rounds as the reference's three fp16 ops: f16(f16(rs * x) + f16(is * original))
        if self.input_mixed:
            normed = rms_norm(x, self.ln1.weight, norm_eps(self.ln1, x))
        else:
            x, normed = mix_rms_norm(x, original_board_embed, self.residual_scale, self.input_scale, self.ln1.weight, norm_eps(self.ln1, x))
        attended = template_attention(linear(normed, self.projection, self.projection_bias), templates, self.q_gain, self.k_gain, self.heads,
                                      self.kv_heads, self.dq, self.dv, self.templates_count, self.eps)
        x = linear(attended, self.combine_heads, self.combine_heads_bias, residual=x)
        hidden = linear(rms_norm(x, self.ln2.weight, norm_eps(self.ln2, x)), self.gate_up, gated=True)
        if self.next_scales is None:
            return linear(hidden, self.down, residual=x)
        return linear(hidden, self.down, residual=x, original=original_board_embed, residual_scale=self.next_scales[0], input_scale=self.next_scales[1])


# Two neighbouring blocks of the same kind hand the second's input mix to the first's down epilogue (next_scales set on the
# first, input_mixed on the second); at a change of kind the second block mixes its input itself.
def link_input_mixes(blocks: list[nn.Module]) -> None:
    for block in blocks:
        block.next_scales, block.input_mixed = None, False
    for block, following in zip(blocks, blocks[1:]):
        if type(block) is type(following):
            block.next_scales, following.input_mixed = (following.residual_scale, following.input_scale), True


def prepare(templates: torch.Tensor) -> None:
    """The key-major templates, made now rather than while a graph records (reference attention_cuda.py:437-440)."""
    if templates.is_cuda and templates.dtype == torch.float16 and tuple(templates.shape[1:]) == (NUM_SQUARES, NUM_SQUARES):
        keyed_templates(templates, templates.shape[0])


#boards B x T (codes of 1, 4 or 8 bytes): B x T x D. rays 64 x 8 x 8 (each square's squares out along the 8 directions, nearest
#first, 64 past the edge) and jumps 64 x 8 (its knight jumps), offsets the 23 features' first rows (reference fused_blocks.py:472-491)
@torch.library.custom_op("chess::board_embedding", mutates_args=())
def board_embedding(boards: torch.Tensor, rays: torch.Tensor, jumps: torch.Tensor, offsets: torch.Tensor, embed: torch.Tensor, position: torch.Tensor,
                    table: torch.Tensor) -> torch.Tensor:
    if boards.dtype not in (torch.uint8, torch.int32, torch.int64):
        raise ValueError(f"board_embedding reads codes as uint8, int32 or int64, not {boards.dtype}")
    for tensor, name in ((embed, "embed"), (position, "position"), (table, "table")):
        if tensor.dtype != torch.float16:
            raise ValueError(f"board_embedding's {name} is {tensor.dtype}, the kernel takes fp16")
    for tensor, shape, name in ((rays, (NUM_SQUARES, 8, 8), "rays"), (jumps, (NUM_SQUARES, 8), "jumps"), (offsets, (FEATURE_SLOTS,), "offsets")):
        if tensor.dtype != torch.int32 or tuple(tensor.shape) != shape:
            raise ValueError(f"board_embedding's {name} is {tensor.dtype} {tuple(tensor.shape)}, the kernel takes int32 {shape}")
    boards = boards.contiguous()
    B, T = boards.shape
    D = table.shape[1]
    if embed.shape[1] != D or position.shape[1] != D or position.shape[0] < T:
        raise ValueError(f"board_embedding: embed {tuple(embed.shape)}, position {tuple(position.shape)} and table {tuple(table.shape)} for {T} tokens")
    library = library_for(boards.device)
    embed, position, table = aligned(embed), aligned(position), aligned(table)
    out = torch.empty(B, T, D, device=boards.device, dtype=torch.float16)
    code = library.chess_board_embedding(pointer(boards), boards.element_size(), pointer(rays.contiguous()), pointer(jumps.contiguous()),
                                         pointer(offsets.contiguous()), pointer(embed), pointer(position), pointer(table), pointer(out), B, T, D,
                                         embed.shape[0], table.shape[0], PAWN, KNIGHT, QUEEN, KING, THEIRS, EDGE, NO_PIECE, stream_of(boards.device))
    check(code, "board_embedding")
    return out


@board_embedding.register_fake
def _(boards, rays, jumps, offsets, embed, position, table):
    return table.new_empty(*boards.shape, table.shape[1])


class InputEmbedding(nn.Module):
    """Token + position embedding plus the square features (reference fused_blocks.py:494-510), in one kernel that finds each square's
    feature rows from the board itself: the features' sum rounded to the table's precision first, then all three summed in f32."""

    def __init__(self, model: ChessTransformer):
        super().__init__()
        self.embed, self.position_embed, self.features = model.embed, model.position_embed, model.square_features
        self.register_buffer("rays", F.pad(self.features.rays, (0, 1), value=NUM_SQUARES).int().contiguous(), persistent=False)
        self.register_buffer("jumps", self.features.knight_jumps.int().contiguous(), persistent=False)
        self.register_buffer("offsets", self.features.row_offsets.int().contiguous(), persistent=False)

    def forward(self, board_state: torch.Tensor) -> torch.Tensor:
        return board_embedding(board_state, self.rays, self.jumps, self.offsets, self.embed.weight, self.position_embed, self.features.table)


def _check_head_operands(x, a, a_bias, narrow_weight, narrow_bias, cells, promotions, what: str) -> None:
    B, T, D = x.shape
    for tensor, dtype, name in ((x, torch.float16, "x"), (a, torch.float32, "a"), (a_bias, torch.float32, "a_bias"),
                                (narrow_weight, torch.float32, "narrow_weight"), (narrow_bias, torch.float32, "narrow_bias"),
                                (cells, torch.int32, "cells"), (promotions, torch.int32, "promotions")):
        if tensor.dtype != dtype:
            raise ValueError(f"{what}'s {name} is {tensor.dtype}, the kernel takes {dtype}")
    if a.shape != x.shape or a_bias.numel() != D or narrow_weight.shape[1] != D or narrow_bias.numel() != narrow_weight.shape[0]:
        raise ValueError(f"{what}: x {tuple(x.shape)}, a {tuple(a.shape)}, a_bias {a_bias.numel()}, narrow {tuple(narrow_weight.shape)}")
    if cells.shape != promotions.shape:
        raise ValueError(f"{what}: a cell and a promotion place for every move")


# floats a position of chess_move_logits' workspace: the 64 x 64 logits, then 96 tokens x 32 narrow products
MOVE_LOGITS_WORKSPACE = NUM_SQUARES * NUM_SQUARES + 96 * 32


def _launch_move_logits(x, a, a_bias, narrow_weight, narrow_bias, cells, promotions, down_first, out, out_stride, activate) -> torch.Tensor:
    B, T, D = x.shape
    library = library_for(x.device)
    x, a, a_bias, narrow_weight = aligned(x), aligned(a), aligned(a_bias), aligned(narrow_weight)
    narrow = narrow_weight.shape[0]
    down = torch.empty(B, T, narrow - down_first, device=x.device, dtype=torch.float32)
    workspace = torch.empty(B, MOVE_LOGITS_WORKSPACE, device=x.device, dtype=torch.float32)
    code = library.chess_move_logits(pointer(x), pointer(a), pointer(a_bias), pointer(narrow_weight), pointer(narrow_bias.contiguous()),
                                     pointer(cells.contiguous()), pointer(promotions.contiguous()), pointer(out), pointer(down), pointer(workspace),
                                     workspace.numel() * 4, B, T, D, narrow, down_first, cells.numel(), out_stride, int(activate), stream_of(x.device))
    check(code, "move_logits")
    return down


# The bilinear from/to logit of squares i, j expands to a_i . x_j + s_i, a = x A + a_bias (head_weights), so one d x d matmul
# stands for both projections.
#the policy head's move logits after its `a` matmul and board_down's inputs (reference fused_blocks.py:866-871), one launch
@torch.library.custom_op("chess::move_logits", mutates_args=())
def move_logits(x: torch.Tensor, a: torch.Tensor, a_bias: torch.Tensor, narrow_weight: torch.Tensor, narrow_bias: torch.Tensor, cells: torch.Tensor,
                promotions: torch.Tensor, down_first: int) -> tuple[torch.Tensor, torch.Tensor]:
    _check_head_operands(x, a, a_bias, narrow_weight, narrow_bias, cells, promotions, "move_logits")
    out = torch.empty(x.shape[0], cells.numel(), device=x.device, dtype=torch.float32)
    down = _launch_move_logits(x, a, a_bias, narrow_weight, narrow_bias, cells, promotions, down_first, out, cells.numel(), False)
    return out, down


@move_logits.register_fake
def _(x, a, a_bias, narrow_weight, narrow_bias, cells, promotions, down_first):
    B, T, _ = x.shape
    return x.new_empty(B, cells.numel(), dtype=torch.float32), x.new_empty(B, T, narrow_weight.shape[0] - down_first, dtype=torch.float32)


#the heads from the `a` matmul on: the answer rows (the move logits, then the expected score; reference engine/inference.py:19-23,
#fused_blocks.py:697-728) and the value logits, in three launches: the move logits into the rows with board_down's GELU outputs,
#then the eval head's two layers and the expected score (its hidden layer in a workspace of B x H f32). Not the reference's
#chess::heads (fused_blocks.py:743-746, which takes the stream and returns only the rows): its own name, for its own schema.
@torch.library.custom_op("chess::answer_heads", mutates_args=())
def answer_heads(x: torch.Tensor, a: torch.Tensor, a_bias: torch.Tensor, narrow_weight: torch.Tensor, narrow_bias: torch.Tensor, cells: torch.Tensor,
          promotions: torch.Tensor, down_first: int, hidden_weight: torch.Tensor, hidden_bias: torch.Tensor, out_weight: torch.Tensor,
          out_bias: torch.Tensor, centres: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    _check_head_operands(x, a, a_bias, narrow_weight, narrow_bias, cells, promotions, "answer_heads")
    for tensor, name in ((hidden_weight, "hidden_weight"), (hidden_bias, "hidden_bias"), (out_weight, "out_weight"), (out_bias, "out_bias"),
                         (centres, "centres")):
        if tensor.dtype != torch.float32:
            raise ValueError(f"answer_heads' {name} is {tensor.dtype}, the kernel takes f32")
    B, T, _ = x.shape
    moves = cells.numel()
    H, K = hidden_weight.shape
    bins = out_weight.shape[0]
    if K != T * (narrow_weight.shape[0] - down_first) or out_weight.shape[1] != H or hidden_bias.numel() != H or out_bias.numel() != bins \
            or centres.numel() != bins:
        raise ValueError(f"answer_heads: the eval head {tuple(hidden_weight.shape)} then {tuple(out_weight.shape)} for {T} tokens of "
                         f"{narrow_weight.shape[0] - down_first} board_down values")
    rows = torch.empty(B, moves + 1, device=x.device, dtype=torch.float32)
    value_logits = torch.empty(B, bins, device=x.device, dtype=torch.float32)
    activated = _launch_move_logits(x, a, a_bias, narrow_weight, narrow_bias, cells, promotions, down_first, rows, moves + 1, True)
    workspace = torch.empty(B, H, device=x.device, dtype=torch.float32)
    code = library_for(x.device).chess_value_head(pointer(activated), pointer(aligned(hidden_weight)), pointer(hidden_bias.contiguous()),
                                                  pointer(aligned(out_weight)), pointer(out_bias.contiguous()), pointer(centres.contiguous()),
                                                  pointer(value_logits), pointer(rows), pointer(workspace), workspace.numel() * 4, B, K, H, bins,
                                                  moves + 1, moves, stream_of(x.device))
    check(code, "value_head")
    return rows, value_logits


@answer_heads.register_fake
def _(x, a, a_bias, narrow_weight, narrow_bias, cells, promotions, down_first, hidden_weight, hidden_bias, out_weight, out_bias, centres):
    return x.new_empty(x.shape[0], cells.numel() + 1, dtype=torch.float32), x.new_empty(x.shape[0], out_weight.shape[0], dtype=torch.float32)


def move_places(model: ChessTransformer) -> tuple[torch.Tensor, torch.Tensor]:
    """Per move, from * 64 + to and the place of its promotion logit among the narrow columns, to' * 32 + 1 + piece (-1 for none):
    the gathers of reference fused_blocks.py:869-870 as two int32 tables."""
    cells = (model.from_squares * NUM_SQUARES + model.to_squares).int()
    promotions = torch.full_like(cells, -1)
    promotions[model.promotion_move_ids] = (model.promotion_to_squares * 32 + 1 + model.promotion_pieces).int()
    return cells, promotions


def head_weights(model: ChessTransformer) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    """The policy head's from x to bilinear form, expanded so that the kernels never form the projections. With W_f, b_f and
    W_t, b_t the from and to projections and r = sqrt(d):
        (W_f x_i + b_f) . (W_t x_j + b_t) / r = (x_i A + a) . x_j + x_i . f + c,
        A = W_f^T W_t / r,  a = W_t^T b_f / r,  f = W_f^T b_t / r,  c = b_f . b_t / r.
    Returns A (fp16, the `a` matmul's weight, as the reference keeps it: fused_blocks.py:815-823), a (f32), and the narrow
    projection's rows and biases (f32): [f; the promotion logits; board_down's inputs] and [c; their biases]; all formed
    in float64 first."""
    with torch.no_grad():
        root = math.sqrt(model.d_model)
        from_weight, from_bias = model.from_projection.weight.double(), model.from_projection.bias.double()
        to_weight, to_bias = model.to_projection.weight.double(), model.to_projection.bias.double()
        promotion, down = model.promotion_projection, model.board_down_project[0]
        pairing = from_weight.t() @ to_weight / root
        to_side = to_weight.t() @ from_bias / root
        from_side = from_weight.t() @ to_bias / root
        constant = torch.dot(from_bias, to_bias) / root
        narrow = torch.cat([from_side.unsqueeze(0), promotion.weight.double(), down.weight.double()])
        narrow_bias = torch.cat([constant.reshape(1), promotion.bias.double(), down.bias.double()])
    return pairing.half(), to_side.float(), narrow.float(), narrow_bias.float()


class FusedTransformer(nn.Module):
    """ChessTransformer.forward with FusedBlocks, for inference (reference fused_blocks.py:829-874). The forward returns the move
    logits (B x moves f32) and the value logits (B x bins f32), the contract of the reference's FusedTransformer where its fused
    ends are off (fused_blocks.py:415-419, 861-871), which the MCTS unpacks (mcts.py:56). With rows (or, when rows is None,
    fused_heads) it returns the answer rows instead, B x (moves + 1) f32: the move logits, then the expected score -- what the
    graph lanes copy out. Both come from the same launches: the move logits are the rows' first columns."""

    # the forward takes rows=True for the answer rows (the graph lanes ask for them through this flag)
    gives_answer_rows = True

    def __init__(self, model: ChessTransformer, fused_heads: bool = False):
        super().__init__()
        self.d_model = model.d_model
        self.input_embedding = InputEmbedding(model)
        self.templates, self.ln = model.templates, model.ln
        self.encoder = nn.ModuleList(FusedBlock(block) for block in model.encoder)
        link_input_mixes(list(self.encoder))
        prepare(model.templates)
        self.fused_heads = fused_heads
        for name in ("from_squares", "to_squares", "promotion_move_ids", "promotion_to_squares", "promotion_pieces"):
            self.register_buffer(name, getattr(model, name))
        self.a_weight, self.a_bias, self.narrow_weight, self.narrow_bias = (nn.Parameter(tensor, requires_grad=False) for tensor in head_weights(model))
        promotions = model.promotion_projection.out_features
        self.promotion_columns, self.down_columns = slice(1, 1 + promotions), slice(1 + promotions, None)
        cells, promotion_places = move_places(model)
        self.register_buffer("move_cells", cells)
        self.register_buffer("move_promotions", promotion_places)
        hidden, out = model.eval_head[0], model.eval_head[2]
        value = {"hidden_weight": hidden.weight, "hidden_bias": hidden.bias, "out_weight": out.weight, "out_bias": out.bias,
                 "centres": value_bin_centres(out.out_features, out.weight.device)}
        for name, tensor in value.items():
            self.register_buffer(name, tensor.detach().float().contiguous())

    def forward(self, board_state: torch.Tensor, rows: bool | None = None) -> torch.Tensor | tuple[torch.Tensor, torch.Tensor]:
        embed_state = self.input_embedding(board_state)
        original_board_embed = embed_state
        for block in self.encoder:
            embed_state = block(embed_state, self.templates, original_board_embed)
        answers, value_logits = self.answers(rms_norm(embed_state, self.ln.weight, norm_eps(self.ln, embed_state)))
        return answers if (self.fused_heads if rows is None else rows) else (answers[:, :-1], value_logits)

    def answers(self, model_output: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
        """The answer rows and the value logits of the final norm's rows (fp16): `a` = x @ a_weight with f32 sums, then the heads."""
        with torch.autocast(device_type=model_output.device.type, enabled=False):
            a = linear(model_output, self.a_weight, accumulate_fp32=True)
            return answer_heads(model_output, a, self.a_bias, self.narrow_weight, self.narrow_bias, self.move_cells, self.move_promotions,
                         self.down_columns.start, self.hidden_weight, self.hidden_bias, self.out_weight, self.out_bias, self.centres)
