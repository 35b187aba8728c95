"""Parity of the HIP operators with the CPU oracle, on the GPU.

Integer and quantised outputs are checked to the bit (int32 sums, int8 activations and their scales,
and the fp16/bf16 outputs of every epilogue but the gated one); float outputs at the tolerances the
reference's own tests use (tests/test_int8.py:76-90, 246-281 and tests/test_attention_cuda.py:51-71 of
the reference)."""
import math

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import int8_ops as oracle
from model import fused_blocks, int8_blocks
from model.hip_kernels import check, library_for, pointer, stream_of
from model.int8_blocks import (HADAMARD_BLOCK, INT8_TILES, hadamard, int8_linear, int8_matmul_i32, launch_int8_linear, mix_norm_quant, norm_quant,
                               rotate_quant)
from model.fused_blocks import launch_linear, launch_template_attention, linear, mix_rms_norm, rms_norm, template_attention

pytestmark = pytest.mark.gpu


def cpu(tensor: torch.Tensor) -> np.ndarray:
    return tensor.detach().cpu().numpy()


def bits_equal(found: torch.Tensor, expected: np.ndarray) -> bool:
    found = cpu(found)
    return found.shape == expected.shape and np.array_equal(found.view(np.uint8), np.ascontiguousarray(expected.astype(found.dtype)).view(np.uint8))


@pytest.mark.parametrize("D", [128, 192, 256, 512, 768])
@pytest.mark.parametrize("mix", [False, True])
def test_norm_quant_matches_the_oracle_to_the_bit(device, D, mix):
    torch.manual_seed(D)
    x = (torch.randn(3, 70, D, device=device) * 4).half()
    original = torch.randn(3, 70, D, device=device).half()
    gain = (torch.rand(D, device=device) + 0.5).half()
    rs, is_ = torch.tensor([0.8], device=device).half(), torch.tensor([0.5], device=device).half()
    if mix:
        mixed, q, scale = mix_norm_quant(x, original, rs, is_, gain, 1e-5)
        expected_mixed, expected_q, expected_scale = oracle.mix_norm_quant(cpu(x), cpu(original), cpu(rs), cpu(is_), cpu(gain), 1e-5)
        assert bits_equal(mixed, expected_mixed)
    else:
        q, scale = norm_quant(x, gain, 1e-5)
        expected_q, expected_scale = oracle.norm_quant(cpu(x), cpu(gain), 1e-5)
    assert q.dtype == torch.int8 and scale.dtype == torch.float32
    assert bits_equal(q, expected_q) and bits_equal(scale, expected_scale)


@pytest.mark.parametrize("rows, D", [(210, 128), (210, 192), (210, 512), (210, 768), (40000, 512), (16384, 192), (20000, 96), (33000, 768)])
@pytest.mark.parametrize("mix", [False, True])
def test_rms_norm_matches_the_oracle_to_the_bit(device, rows, D, mix):
    """The fp16 blocks' norm (and their own input mix): the oracle's bits, a wavefront a row (210 rows), 16-lane groups of
    four rows a wavefront (from 16,384 rows, rows up to 512) and two whole-wavefront rows a wavefront (33,000 rows of 768);
    within one fp16 rounding of torch's rms_norm in f32 (the reference's nn.RMSNorm)."""
    torch.manual_seed(rows + D)
    x = (torch.randn(rows, D, device=device) * 4).half()
    original = torch.randn(rows, D, device=device).half()
    gain = (torch.rand(D, device=device) + 0.5).half()
    rs, is_ = torch.tensor([0.8], device=device).half(), torch.tensor([0.5], device=device).half()
    if mix:
        mixed, normed = mix_rms_norm(x, original, rs, is_, gain, 1e-5)
        expected_mixed, expected = oracle.rms_norm(cpu(x), cpu(gain), 1e-5, cpu(original), cpu(rs), cpu(is_))
        assert bits_equal(mixed, expected_mixed)
        assert torch.equal(mixed, rs * x + is_ * original)   # the reference's fp16 expression, run by torch
        rows_in = mixed
    else:
        normed = rms_norm(x, gain, 1e-5)
        expected = oracle.rms_norm(cpu(x), cpu(gain), 1e-5)[1]
        rows_in = x
    assert normed.dtype == torch.float16 and bits_equal(normed, expected)
    torchs = F.rms_norm(rows_in.float(), (D,), gain.float(), 1e-5)
    assert ((normed.float() - torchs).abs() <= torchs.half().abs().float() * 2 ** -10 + 2 ** -24).all()


@pytest.mark.parametrize("rows, D", [(16384, 192), (20000, 96), (16400, 64), (33000, 768), (32768, 2048)])
@pytest.mark.parametrize("mix", [False, True])
def test_norm_quant_of_large_launches_matches_the_oracle_to_the_bit(device, rows, D, mix):
    """From 16,384 rows, rows up to 512 take groups of 16 lanes (four rows a wavefront, chunks strided across the group,
    masked past rows that are no power of two); longer rows a wavefront each, two a wavefront from 32,768 rows. Every
    split adds the same balanced tree, so the bits are the oracle's."""
    generator = torch.Generator(device="cpu").manual_seed(rows + D)
    x = (torch.randn(rows, D, generator=generator) * 4).half()
    original = torch.randn(rows, D, generator=generator).half()
    gain = (torch.rand(D, generator=generator) + 0.5).half()
    rs, is_ = torch.tensor([0.8]).half(), torch.tensor([0.5]).half()
    if mix:
        mixed, q, scale = mix_norm_quant(x.to(device), original.to(device), rs.to(device), is_.to(device), gain.to(device), 1e-5)
        expected_mixed, expected_q, expected_scale = oracle.mix_norm_quant(x.numpy(), original.numpy(), rs.numpy(), is_.numpy(), gain.numpy(), 1e-5)
        assert bits_equal(mixed, expected_mixed)
    else:
        q, scale = norm_quant(x.to(device), gain.to(device), 1e-5)
        expected_q, expected_scale = oracle.norm_quant(x.numpy(), gain.numpy(), 1e-5)
    assert bits_equal(q, expected_q) and bits_equal(scale, expected_scale)


@pytest.mark.parametrize("rows, D", [(1, 768), (31, 768), (33, 384), (16389, 384), (33, 1536), (32769, 1536), (33000, 776)])
def test_norms_of_three_quarter_widths_match_the_oracle_to_the_bit(device, rows, D):
    """Rows of 24 elements a lane, 16 (from 16,384 rows), 32 or 64 lanes to a row, with the ends of a wavefront's rows; and 776
    columns, masked, two rows a whole wavefront from 32,768 rows."""
    generator = torch.Generator(device="cpu").manual_seed(rows + D)
    x = (torch.randn(rows, D, generator=generator) * 4).half()
    original = torch.randn(rows, D, generator=generator).half()
    gain = (torch.rand(D, generator=generator) + 0.5).half()
    rs, is_ = torch.tensor([0.8]).half(), torch.tensor([0.5]).half()
    on_device = [t.to(device) for t in (x, original, rs, is_, gain)]
    for found, expected in zip(mix_norm_quant(*on_device, 1e-5), oracle.mix_norm_quant(*(t.numpy() for t in (x, original, rs, is_, gain)), 1e-5)):
        assert bits_equal(found, expected)
    for found, expected in zip(norm_quant(on_device[0], on_device[-1], 1e-5), oracle.norm_quant(x.numpy(), gain.numpy(), 1e-5)):
        assert bits_equal(found, expected)
    assert bits_equal(rms_norm(on_device[0], on_device[-1], 1e-5), oracle.rms_norm(x.numpy(), gain.numpy(), 1e-5)[1])


def test_empty_batches_give_outputs_of_no_rows(device):
    """No positions: every operator on the path returns outputs of no rows and the right types (the C ABI launches nothing
    for them), the int8 GEMM on the table's tiles and on the register-held ones."""
    gain = torch.ones(512, device=device).half()
    x = torch.empty(0, 70, 512, device=device).half()
    q, scale = norm_quant(x, gain, 1e-5)
    assert q.shape == (0, 70, 512) and q.dtype == torch.int8 and scale.shape == (0, 70) and scale.dtype == torch.float32
    rs, is_ = torch.tensor([0.8], device=device).half(), torch.tensor([0.5], device=device).half()
    mixed, q, scale = mix_norm_quant(x, x, rs, is_, gain, 1e-5)
    assert mixed.shape == (0, 70, 512) and mixed.dtype == torch.float16 and q.shape == (0, 70, 512) and scale.shape == (0, 70)
    for matmul, width, depth, held in (("projection", 1600, 512, 15), ("gate_up", 2048, 512, 15), ("down", 512, 2048, 16),
                                       ("mixing down", 512, 2048, 16)):
        x8, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands(matmul, 0, device, width=width, depth=depth)
        for tile in (0, held):
            out = launch_int8_linear(x8, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
            assert out.shape == (0, width) and out.dtype == torch.float16
        role = "down" if matmul.endswith("down") else matmul
        assert int8_linear(x8, x_scale, weight, weight_scale, bias, residual, gated, role, *mix).shape == (0, width)
    q, scale = rotate_quant(torch.empty(0, 70, 2048, device=device).half(), hadamard(HADAMARD_BLOCK).to(device).half(), 2048)
    assert q.shape == (0, 70, 2048) and q.dtype == torch.int8 and scale.shape == (0, 70)
    assert template_attention(*attention_operands(device, 0, 8, 8, 64, 64)).shape == (0, 70, 8 * 64)
    combined = linear(torch.empty(0, 70, 512, device=device).half(), torch.randn(512, 512, device=device).half(),
                      torch.randn(512, device=device).half(), torch.empty(0, 70, 512, device=device).half())
    assert combined.shape == (0, 70, 512) and combined.dtype == torch.float16


def test_norm_quant_rounds_the_rmsnorm(device):
    """The reference's own check (tests/test_int8.py:246-264): the scale is absmax / 127 of torch's rms_norm, every value
    within 0.501 of a step."""
    torch.manual_seed(0)
    x, original = torch.randn(2, 70, 192, device=device).half() * 4, torch.randn(2, 70, 192, device=device).half()
    gain = (torch.rand(192, device=device) + 0.5).half()
    residual_scale, input_scale = torch.tensor([0.8], device=device).half(), torch.tensor([0.5], device=device).half()
    for mix in (False, True):
        if mix:
            mixed, integers, scale = mix_norm_quant(x, original, residual_scale, input_scale, gain, 1e-5)
            assert mixed.dtype == torch.float16 and torch.allclose(mixed.float(), 0.8 * x.float() + 0.5 * original.float(), atol=4e-3, rtol=1e-3)
            normed = F.rms_norm(mixed.float(), (192,), gain.float(), 1e-5)
        else:
            integers, scale = norm_quant(x, gain, 1e-5)
            normed = F.rms_norm(x.float(), (192,), gain.float(), 1e-5)
        step = normed.abs().amax(dim=-1) / 127
        assert integers.dtype == torch.int8 and torch.allclose(scale, step, rtol=1e-5)
        assert ((integers.float() * scale[..., None] - normed).abs() <= 0.501 * step[..., None]).all()


@pytest.mark.parametrize("hidden, width", [(992, 1024), (320, 384), (2048, 2048), (100, 128), (512, 512), (1024, 1024), (1536, 1536)])
def test_rotate_quant_matches_the_oracle_to_the_bit(device, hidden, width):
    torch.manual_seed(hidden)
    h = torch.randn(3, 70, hidden, device=device).half()
    integers, scale = rotate_quant(h, hadamard(HADAMARD_BLOCK).to(device).half(), width)
    expected_q, expected_scale = oracle.rotate_quant(cpu(h), width)
    # a 32-block of padding alone rotates to zeros; a block that holds real columns spreads them over all 32
    padding = -(-hidden // HADAMARD_BLOCK) * HADAMARD_BLOCK
    assert integers.shape == (3, 70, width) and (integers[..., padding:] == 0).all()
    assert bits_equal(integers, expected_q) and bits_equal(scale, expected_scale)


# the network's batch-1024 rows: 1,024 positions of 70 tokens. From 32,768 rows the row kernels take their wide launches
# (two rows a wavefront, full rows without masks), which only the d512 network's batch-256-and-up shapes reach.
WIDE_ROWS = 71680


@pytest.mark.parametrize("mix", [False, True])
def test_norm_quant_at_the_batch_1024_rows_is_the_oracles(device, mix):
    """norm_quant's wide launch (71,680 rows of 512: two rows a wavefront, no masks) against the oracle, to the bit."""
    generator = torch.Generator(device="cpu").manual_seed(17 + mix)
    x = (torch.randn(WIDE_ROWS, 512, generator=generator) * 4).half()
    original = torch.randn(WIDE_ROWS, 512, generator=generator).half()
    gain = (torch.rand(512, generator=generator) + 0.5).half()
    rs, is_ = torch.tensor([0.8]).half(), torch.tensor([0.5]).half()
    if mix:
        mixed, q, scale = mix_norm_quant(x.to(device), original.to(device), rs.to(device), is_.to(device), gain.to(device), 1e-5)
        expected_mixed, expected_q, expected_scale = oracle.mix_norm_quant(x.numpy(), original.numpy(), rs.numpy(), is_.numpy(), gain.numpy(), 1e-5)
        assert bits_equal(mixed, expected_mixed)
    else:
        q, scale = norm_quant(x.to(device), gain.to(device), 1e-5)
        expected_q, expected_scale = oracle.norm_quant(x.numpy(), gain.numpy(), 1e-5)
    assert bits_equal(q, expected_q) and bits_equal(scale, expected_scale)


def test_rotate_quant_at_the_batch_1024_rows_is_the_oracles(device):
    """rotate_quant's wide launch (71,680 rows of 2,048, the network's down input: two rows a wavefront, full rows without
    masks, the cross-lane butterflies as signed FMAs) against the oracle, to the bit."""
    generator = torch.Generator(device="cpu").manual_seed(19)
    h = torch.randn(WIDE_ROWS, 2048, generator=generator).half()
    integers, scale = rotate_quant(h.to(device), hadamard(HADAMARD_BLOCK).to(device).half(), 2048)
    expected_q, expected_scale = oracle.rotate_quant(h.numpy(), 2048)
    assert bits_equal(integers, expected_q) and bits_equal(scale, expected_scale)


@pytest.mark.parametrize("hidden, width", [(992, 1024), (320, 384)])
def test_rotate_quant_rounds_the_rotated_rows(device, hidden, width):
    """The reference's check (tests/test_int8.py:267-281) against the fp32 block-diagonal rotation."""
    torch.manual_seed(0)
    h = torch.randn(3, 70, hidden, device=device).half()
    integers, scale = rotate_quant(h, hadamard(HADAMARD_BLOCK).to(device).half(), width)
    rotation = torch.block_diag(*[hadamard(HADAMARD_BLOCK)] * (width // HADAMARD_BLOCK)).to(device)
    rotated = F.pad(h.float(), (0, width - hidden)) @ rotation
    step = rotated.abs().amax(dim=-1) / 127
    assert torch.allclose(scale, step, rtol=1e-5)
    assert ((integers.float() * scale[..., None] - rotated).abs() <= 0.501 * step[..., None]).all()


def test_rotate_quant_refuses_another_rotation(device):
    h = torch.randn(70, 128, device=device).half()
    with pytest.raises(ValueError):
        rotate_quant(h, -hadamard(HADAMARD_BLOCK).to(device).half(), 128)


@pytest.mark.parametrize("M, N, K", [(1, 196, 256), (70, 200, 1024), (140, 1600, 512), (4480, 1536, 512), (4480, 512, 2048), (333, 64, 64)])
@pytest.mark.parametrize("tile", [1, 2])
def test_int8_sums_are_exact(device, M, N, K, tile):
    generator = torch.Generator(device="cpu").manual_seed(M + N + K)
    x = torch.randint(-127, 128, (M, K), generator=generator, dtype=torch.int8)
    w = torch.randint(-127, 128, (N, K), generator=generator, dtype=torch.int8)
    found = int8_matmul_i32(x.to(device), w.to(device), tile)
    expected = x.long() @ w.long().T
    assert found.dtype == torch.int32 and torch.equal(found.cpu().long(), expected)


@pytest.mark.parametrize("M, N, K", [(1, 200, 512), (70, 1600, 512), (140, 512, 2048), (1120, 512, 2048), (333, 64, 1024), (4480, 2048, 512),
                                     (70, 96, 256)])
@pytest.mark.parametrize("tile", [14])
def test_the_split_k_sums_are_exact(device, M, N, K, tile):
    """The split-K tile's int32 sums, the partial tiles of 4 wavefronts added in LDS, at one to 4,480 rows (ragged last
    row and column tiles); a depth its wavefronts cannot split in 1, 2 or 4 steps of 128 bytes is refused."""
    generator = torch.Generator(device="cpu").manual_seed(M + N + K + tile)
    x = torch.randint(-127, 128, (M, K), generator=generator, dtype=torch.int8)
    w = torch.randint(-127, 128, (N, K), generator=generator, dtype=torch.int8)
    if not int8_blocks.tile_takes(tile, N, K):
        with pytest.raises(ValueError):
            int8_matmul_i32(x.to(device), w.to(device), tile)
        return
    found = int8_matmul_i32(x.to(device), w.to(device), tile)
    assert found.dtype == torch.int32 and torch.equal(found.cpu().long(), x.long() @ w.long().T)


def test_the_split_k_tiles_refuse_what_they_cannot_take(device):
    """The split tile writes 8 columns a lane and takes int8 only: N % 8 != 0 and the fp16 instance are refused."""
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("projection", 70, device, width=196)
    launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 1)
    for tile in SPLIT_TILES:
        with pytest.raises(ValueError):
            launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
        with pytest.raises(ValueError):
            launch_linear(x.half(), (weight.float().t() / 128).half().contiguous(), bias, None, False, False, None, None, None, tile)


def int8_operands(matmul: str, rows: int, device, width: int = 200, depth: int | None = None):
    torch.manual_seed(rows + width)
    down, gated = matmul.endswith("down"), matmul == "gate_up"
    depth = depth or (1024 if down else 512)
    x = torch.randint(-127, 128, (rows, depth), device=device, dtype=torch.int8)
    x_scale = torch.rand(rows, device=device) / 100
    weight = torch.randint(-127, 128, (2 * width if gated else width, depth), device=device, dtype=torch.int8)
    weight_scale = torch.rand(len(weight), device=device) / 100
    bias = torch.randn(width, device=device).half() if matmul == "projection" else None
    residual = torch.randn(rows, width, device=device).half() if down else None
    mix = (torch.randn(rows, width, device=device).half(), torch.tensor([0.9], device=device).half(),
           torch.tensor([0.3], device=device).half()) if matmul == "mixing down" else (None, None, None)
    return x, x_scale, weight, weight_scale, bias, residual, gated, mix


def oracle_int8_linear(operands, out_dtype=np.float16):
    x, x_scale, weight, weight_scale, bias, residual, gated, (original, rs, is_) = operands
    arrays = [None if t is None else cpu(t) for t in (x, x_scale, weight, weight_scale, bias, residual, original, rs, is_)]
    x, x_scale, weight, weight_scale, bias, residual, original, rs, is_ = arrays
    return oracle.int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, original, rs, is_, out_dtype)


@pytest.mark.parametrize("matmul", ["projection", "down", "mixing down"])
@pytest.mark.parametrize("rows", [70, 210, 4480])
def test_int8_linear_epilogues_match_the_oracle_to_the_bit(device, matmul, rows):
    operands = int8_operands(matmul, rows, device)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = operands
    expected = oracle_int8_linear(operands)
    table = (tile for tiles in INT8_TILES.values() for _, tile in tiles["down" if matmul.endswith("down") else matmul])
    for tile in dict.fromkeys((1, 2, *table)):
        if not int8_blocks.tile_takes(tile, expected.shape[-1], x.shape[-1], gated, bias is not None, residual is not None):
            continue   # a register-held tile of another depth or epilogue: its own tests cover it
        out = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
        assert out.dtype == torch.float16 and bits_equal(out, expected), tile


@pytest.mark.parametrize("rows", [70, 4480])
def test_the_gated_epilogue_is_silu_times_up(device, rows):
    operands = int8_operands("gate_up", rows, device)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = operands
    expected = oracle_int8_linear(operands).astype(np.float64)
    first = None
    for tile in (1, 2):
        out = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
        assert np.allclose(cpu(out).astype(np.float64), expected, atol=1e-3, rtol=2e-3), tile
        first = out if first is None else first
        assert torch.equal(out, first)


def same_bits(found: torch.Tensor, expected: torch.Tensor) -> bool:
    as_integers = {torch.float16: torch.int16, torch.bfloat16: torch.int16, torch.float32: torch.int32}
    return found.shape == expected.shape and found.dtype == expected.dtype and torch.equal(
        found.view(as_integers.get(found.dtype, found.dtype)), expected.view(as_integers.get(expected.dtype, expected.dtype)))


def dequantised(integers: torch.Tensor, scale: torch.Tensor) -> torch.Tensor:
    return integers.double() * scale.double()[:, None]


@pytest.mark.parametrize("matmul", ["projection", "gate_up", "down", "mixing down"])
@pytest.mark.parametrize("boards", [1, 3])
def test_int8_linear_is_the_dequantised_matmul(device, matmul, boards):
    """The reference's check (tests/test_int8.py:59-90): every tile, rows and columns leaving tiles part empty."""
    torch.manual_seed(0)
    down, gated = matmul.endswith("down"), matmul == "gate_up"
    width, depth = 200, 1024 if down else 512
    x = torch.randint(-127, 128, (boards, 70, depth), device=device, dtype=torch.int8)
    x_scale = torch.rand(boards, 70, device=device) / 100
    weight = torch.randint(-127, 128, (2 * width if gated else width, depth), device=device, dtype=torch.int8)
    weight_scale = torch.rand(len(weight), device=device) / 100
    bias = torch.randn(width, device=device).half() if matmul == "projection" else None
    residual = torch.randn(boards, 70, width, device=device).half() if down else None
    mix = (torch.randn(boards, 70, width, device=device).half(), torch.tensor(0.9, device=device).half(),
           torch.tensor(0.3, device=device).half()) if matmul == "mixing down" else ()
    projected = dequantised(x.reshape(-1, depth), x_scale.reshape(-1)) @ dequantised(weight, weight_scale).t()
    if matmul == "projection":
        expected = projected + bias.double()
    elif matmul == "gate_up":
        gate, up = projected.chunk(2, dim=-1)
        expected = F.silu(gate) * up
    else:
        expected = projected + residual.reshape(-1, width).double()
    if mix:
        original, residual_scale, input_scale = mix
        expected = residual_scale.double() * expected.half().double() + input_scale.double() * original.reshape(-1, width).double()
    for tile in dict.fromkeys(tile for tiles in INT8_TILES.values() for _, tile in tiles["down" if down else matmul]):
        if not int8_blocks.tile_takes(tile, width, depth, gated, bias is not None, residual is not None):
            continue   # a register-held tile of another depth or epilogue: its own tests cover it
        out = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *(mix or (None, None, None)), tile)
        assert out.dtype == torch.float16 and out.shape == (boards, 70, width)
        assert torch.allclose(out.reshape(-1, width).double(), expected, atol=1e-3, rtol=2e-3), tile


def test_int8_linear_writes_bf16(device):
    operands = int8_operands("projection", 4096, device, width=1536, depth=512)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = operands
    out = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 0, torch.bfloat16)
    expected = oracle_int8_linear(operands, "bf16")
    assert out.dtype == torch.bfloat16
    assert np.array_equal(cpu(out.float()), expected)


@pytest.mark.parametrize("matmul", ["projection", "gate_up", "down", "mixing down"])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16])
def test_the_split_k_tiles_give_the_whole_k_tiles_bits(device, matmul, out_dtype):
    """Split-K against whole-K tiles at 70 rows (one position), every epilogue (the gated one too) in fp16 and bf16."""
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands(matmul, 70, device, width=1600 if matmul == "projection" else 512)
    expected = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 1, out_dtype)
    for tile in SPLIT_TILES:
        if int8_blocks.tile_takes(tile, expected.shape[-1], x.shape[-1]):
            assert same_bits(launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile, out_dtype), expected), tile


def config1_case(M: int, K: int, N: int, device):
    """benchmark config 1: A int8 uniform in [-127, 127], W int8 rounded from N(0, 0.02) (a scale a row), f32 row scales,
    bias N(0, 0.02), bf16 out."""
    from engine.quantization import nearest
    generator = torch.Generator(device="cpu").manual_seed(M + K + N)
    x = torch.randint(-127, 128, (M, K), generator=generator, dtype=torch.int8)
    x_scale = torch.rand(M, generator=generator) / 100
    weight, weight_scale = nearest(torch.randn(N, K, generator=generator) * 0.02)
    bias = (torch.randn(N, generator=generator) * 0.02).half()
    return x, x_scale, weight, weight_scale, bias


CONFIG1_SHAPES = [(512, 1536), (512, 512), (512, 2048), (2048, 512)]   # QKV, attention-out, FFN-up, FFN-down (K to N)


@pytest.mark.parametrize("K, N", CONFIG1_SHAPES, ids=["qkv", "attention_out", "ffn_up", "ffn_down"])
@pytest.mark.parametrize("M", [4096, 16384, 65536])
def test_the_config1_gemms_are_the_oracles_in_bf16(device, M, K, N):
    """The four per-layer shapes of benchmark config 1 with the bias epilogue and bf16 out, the tile the size picks: every row
    against the oracle at M = 4,096; at M = 16,384 and 65,536 the rows of the first, a middle and the last row tile and 256
    rows drawn across the rest (the oracle's integer product of all the rows takes minutes)."""
    x, x_scale, weight, weight_scale, bias = config1_case(M, K, N, device)
    out = launch_int8_linear(x.to(device), x_scale.to(device), weight.to(device), weight_scale.to(device), bias.to(device), None, False,
                             None, None, None, 0, torch.bfloat16)
    assert out.dtype == torch.bfloat16 and out.shape == (M, N)
    rows = np.arange(M) if M <= 4096 else np.unique(np.concatenate([np.arange(256), np.arange(M // 2 - 128, M // 2 + 128), np.arange(M - 256, M),
                                                                       np.random.default_rng(M + N).integers(0, M, 256)]))
    expected = oracle.int8_linear(x.numpy()[rows], x_scale.numpy()[rows], weight.numpy(), weight_scale.numpy(), bias.numpy(), out_dtype="bf16")
    assert np.array_equal(cpu(out.float())[rows], expected)


ALL_TILES = tuple(range(1, 14))   # 5, 12 and 13 take 128-byte stages, 4 to 6 eight wavefronts
SPLIT_TILES = (14,)              # int8 only


@pytest.mark.parametrize("matmul", ["projection", "gate_up", "down", "mixing down"])
def test_every_tile_gives_the_same_bits(device, matmul):
    """Every tile of the int8 GEMM (the split-K ones included) and of its fp16 instance, partial last tiles in rows (210) and
    columns (200): one set of bits."""
    operands = int8_operands(matmul, 210, device)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = operands
    outputs = [launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile) for tile in (*ALL_TILES, *SPLIT_TILES)]
    assert all(same_bits(out, outputs[0]) for out in outputs[1:])
    halves = x.half()
    w16 = (weight.float().t() / 128).half().contiguous()
    fp16 = [launch_linear(halves, w16, bias, residual, gated, False, *mix, tile) for tile in ALL_TILES]
    assert all(same_bits(out, fp16[0]) for out in fp16[1:])


def test_a_reference_tile_tuple_launches_the_tile_of_its_shape(device):
    """launch_int8_linear given the reference's Triton tile (rows, columns, depth, warps, stages[, registers]) runs this
    library's tile of that shape (reference int8_blocks.py:105-108): the reference's sm_120 gate_up tile is tile 9, its
    large down tile tile 6; a shape the library has no tile for is refused."""
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("gate_up", 210, device)
    assert torch.equal(launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, (128, 64, 64, 4, 2)),
                       launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 9))
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("down", 210, device)
    assert torch.equal(launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, (128, 128, 64, 8, 3, 128)),
                       launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 6))
    with pytest.raises(ValueError, match="no 32 x 64 tile"):
        launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, (32, 64, 64, 4, 4))


@pytest.mark.parametrize("matmul, width", [("gate_up", 200), ("gate_up", 2048), ("projection", 200), ("projection", 1600)])
@pytest.mark.parametrize("rows", [1, 31, 33, 210, 4480])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16])
def test_the_register_tile_gives_the_whole_k_tiles_bits(device, matmul, width, rows, out_dtype):
    """Tile 15 (each wavefront's weights held in registers, x streamed in blocks of 32 rows) against tile 1: one row to
    4,480, ragged last blocks, the gated epilogue and the bias one (200 columns: a column group part past N), fp16 and
    bf16; the bias epilogue also against the oracle to the bit."""
    operands = int8_operands(matmul, rows, device, width=width, depth=512)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = operands
    found = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, int8_blocks.RESIDENT_TILE, out_dtype)
    expected = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 1, out_dtype)
    assert same_bits(found, expected)
    if not gated:
        oracle_out = oracle_int8_linear(operands, "bf16" if out_dtype == torch.bfloat16 else np.float16)
        assert np.array_equal(cpu(found.float()), oracle_out.astype(np.float32))


def test_the_register_tile_at_the_batch_1024_rows(device):
    """gate_up at the network's batch-1024 shape (71,680 rows, 512 -> 2 x 2,048): tile 15 and the whole-K tile 10 give the
    same bits, twice in a row on the same output buffer's size (a second launch finds nothing of the first)."""
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("gate_up", 71680, device, width=2048, depth=512)
    expected = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 10)
    for _ in range(2):
        assert same_bits(launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, int8_blocks.RESIDENT_TILE), expected)


@pytest.mark.parametrize("matmul, depth, width", [("projection", 256, 520), ("projection", 512, 520), ("projection", 768, 1032),
                                                  ("projection", 1024, 264), ("gate_up", 256, 264), ("gate_up", 768, 136),
                                                  ("down", 1024, 264), ("mixing down", 1024, 264), ("projection", 768, 1152),
                                                  ("projection", 1024, 1600), ("gate_up", 256, 1408)])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16])
def test_large_launches_of_tile_0_give_the_whole_k_tiles_bits(device, matmul, depth, width, out_dtype):
    """Tile 0 holds the weights in registers where a workgroup's stream of row blocks is long: 41,007 rows (past each
    epilogue's line; a ragged last block and a column group part past N) against tile 1, at every depth it has; five to seven
    column groups, the last part past N and with more streams than each of the others."""
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands(matmul, 41007, device, width=width, depth=depth)
    found = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 0, out_dtype)
    assert same_bits(found, launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 1, out_dtype))


@pytest.mark.parametrize("depth", [256, 512])
@pytest.mark.parametrize("with_residual", [True, False])
def test_large_launches_of_tile_0_give_fp16_sums_the_whole_k_tiles_bits(device, depth, with_residual):
    x, weight, bias, residual = output_projection_operands(41007, 264, device)
    x, weight, residual = x[:, :depth].contiguous(), weight[:depth].contiguous(), residual if with_residual else None
    found = launch_linear(x, weight, bias, residual, False, False, None, None, None, 0)
    assert same_bits(found, launch_linear(x, weight, bias, residual, False, False, None, None, None, 1))


def test_the_register_tile_refuses_what_it_cannot_take(device):
    """Tile 15 holds depth 512 in registers, stores 4 columns a lane and adds no residual or input mix: other depths,
    widths not a multiple of 8 and the down epilogues are refused."""
    tile = int8_blocks.RESIDENT_TILE
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("projection", 70, device, width=256, depth=1024)
    with pytest.raises(ValueError, match="depth"):
        launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("gate_up", 70, device, width=196, depth=512)
    with pytest.raises(ValueError, match="multiple of 8"):
        launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("down", 70, device, width=256, depth=512)
    with pytest.raises(ValueError, match="residual"):
        launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
    assert not int8_blocks.tile_takes(tile, 196, 512) and not int8_blocks.tile_takes(tile, 200, 1024) and int8_blocks.tile_takes(tile, 200, 512)


@pytest.mark.parametrize("matmul", ["down", "mixing down"])
@pytest.mark.parametrize("rows", [1, 17, 210, 2048, 3072, 4480])
@pytest.mark.parametrize("width", [128, 512])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16])
def test_the_deep_register_tile_gives_the_whole_k_tiles_bits(device, matmul, rows, width, out_dtype):
    """Tile 16 (down's depth of 2,048 split over four wavefronts, each holding its quarter of 64 columns in registers, x
    streamed in blocks of 16 rows, the quarters' int32 partials handed over through LDS) against tile 1: one row to 4,480
    (every stream of blocks empty or one block long at one row, two and three blocks long at 2,048 and 3,072, ragged last
    blocks), one and four column groups, the residual with and without the next block's mix, fp16 and bf16; up to 210 rows
    also against the oracle to the bit."""
    operands = int8_operands(matmul, rows, device, width=width, depth=2048)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = operands
    found = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, int8_blocks.DEEP_TILE, out_dtype)
    expected = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 1, out_dtype)
    assert same_bits(found, expected)
    if rows <= 210:
        oracle_out = oracle_int8_linear(operands, "bf16" if out_dtype == torch.bfloat16 else np.float16)
        assert np.array_equal(cpu(found.float()), oracle_out.astype(np.float32))


def test_the_deep_register_tile_at_the_batch_1024_rows(device):
    """down with the next block's mix at the network's batch-1024 shape (71,680 rows, 2,048 -> 512): tile 16 and the
    whole-K tile 13 give the same bits, twice in a row (a second launch finds nothing of the first)."""
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("mixing down", 71680, device, width=512, depth=2048)
    expected = launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 13)
    for _ in range(2):
        assert same_bits(launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, int8_blocks.DEEP_TILE), expected)


def test_the_deep_register_tile_refuses_what_it_cannot_take(device):
    """Tile 16 holds depth 2,048 in registers in column groups of 128 and runs down's epilogue only: other depths, widths
    not a multiple of 128, the bias epilogue without a residual and the gated one are refused."""
    tile = int8_blocks.DEEP_TILE
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("down", 70, device, width=256, depth=1024)
    with pytest.raises(ValueError, match="depth"):
        launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("down", 70, device, width=200, depth=2048)
    with pytest.raises(ValueError, match="multiple of 128"):
        launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("projection", 70, device, width=256, depth=2048)
    with pytest.raises(ValueError, match="epilogue"):
        launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("gate_up", 70, device, width=256, depth=2048)
    with pytest.raises(ValueError, match="not gated"):
        launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)
    assert int8_blocks.tile_takes(tile, 512, 2048, residual=True)
    assert not any((int8_blocks.tile_takes(tile, 512, 1024, residual=True), int8_blocks.tile_takes(tile, 200, 2048, residual=True),
                    int8_blocks.tile_takes(tile, 512, 2048), int8_blocks.tile_takes(tile, 512, 2048, bias=True, residual=True),
                    int8_blocks.tile_takes(tile, 512, 2048, gated=True, residual=True)))


def output_projection_operands(rows: int, width: int, device):
    """the attention's output projection: fp16 x [rows, 512] @ W [512, width], bias and residual"""
    generator = torch.Generator(device="cpu").manual_seed(rows + width)
    x = torch.randn(rows, 512, generator=generator).half().to(device)
    weight = (torch.randn(512, width, generator=generator) / 16).half().to(device)
    return x, weight, torch.randn(width, generator=generator).half().to(device), torch.randn(rows, width, generator=generator).half().to(device)


@pytest.mark.parametrize("rows", [1, 33, 210, 4480])
@pytest.mark.parametrize("width", [200, 512, 1600])
@pytest.mark.parametrize("with_residual", [True, False])
def test_the_register_tile_gives_fp16_sums_the_whole_k_tiles_bits(device, rows, width, with_residual):
    """Tile 15 for fp16 operands (f32 sums taken in the whole-K tiles' k order, fp16 out) against tiles 11 and 1, with the
    bias and the residual (the attention's output projection) and with the bias alone (the fp16 block's projection, 1,600
    columns): one row to 4,480, ragged last blocks, column groups part past N."""
    x, weight, bias, residual = output_projection_operands(rows, width, device)
    residual = residual if with_residual else None
    found = launch_linear(x, weight, bias, residual, False, False, None, None, None, int8_blocks.RESIDENT_TILE)
    for tile in (11, 1):
        assert same_bits(found, launch_linear(x, weight, bias, residual, False, False, None, None, None, tile)), tile


def test_the_register_tile_gives_the_output_projection_at_the_batch_1024_rows(device):
    """The attention's output projection at the network's batch-1024 shape (71,680 rows, 512 -> 512), twice in a row: tile 15
    and tile 11 give the same bits."""
    x, weight, bias, residual = output_projection_operands(71680, 512, device)
    expected = launch_linear(x, weight, bias, residual, False, False, None, None, None, 11)
    for _ in range(2):
        assert same_bits(launch_linear(x, weight, bias, residual, False, False, None, None, None, int8_blocks.RESIDENT_TILE), expected)


def test_the_register_tile_takes_fp16_sums_with_the_bias_only(device):
    """For fp16 operands tile 15 takes the bias epilogue, with or without the residual (fp16 out), at depth 512: without the
    bias, gated, f32 out or at another depth it is refused, and the linear operator falls back to tile 0."""
    from model.fused_blocks import linear_takes
    tile = int8_blocks.RESIDENT_TILE
    x, weight, bias, residual = output_projection_operands(70, 256, device)
    with pytest.raises(ValueError, match="the bias"):
        launch_linear(x, weight, None, residual, False, False, None, None, None, tile)
    with pytest.raises(ValueError, match="the bias"):
        launch_linear(x, torch.cat([weight, weight], 1), None, None, True, False, None, None, None, tile)
    with pytest.raises(ValueError, match="fp16"):
        launch_linear(x, weight, bias, residual, False, True, None, None, None, tile)
    with pytest.raises(ValueError, match="depth"):
        launch_linear(x[:, :256].contiguous(), weight[:256].contiguous(), bias, residual, False, False, None, None, None, tile)
    assert linear_takes(tile, 512, 256, False, True, True, False) and linear_takes(tile, 512, 256, False, True, False, False)
    assert not any((linear_takes(tile, 512, 256, False, False, True, False), linear_takes(tile, 512, 256, True, True, True, False),
                    linear_takes(tile, 256, 256, False, True, True, False), linear_takes(tile, 512, 256, False, True, True, True),
                    linear_takes(tile, 512, 256, False, True, True, False, True)))


def test_128_byte_stages_refuse_rows_of_64(device):
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("projection", 70, device, width=128, depth=192)
    launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 1)   # 64-byte stages take it
    for tile in (5, 12, 13):
        with pytest.raises(ValueError):
            launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, tile)


def test_the_op_picks_a_tile_and_keeps_the_bits(device):
    operands = int8_operands("down", 140, device)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = operands
    assert torch.equal(int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, "down"),
                       launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, gated, *mix, 2))


def test_int8_linear_refuses_what_it_cannot_take(device):
    x, x_scale, weight, weight_scale, bias, *_ = int8_operands("projection", 70, device)
    with pytest.raises(ValueError):
        launch_int8_linear(x[:, :96].contiguous(), x_scale, weight[:, :96].contiguous(), weight_scale, bias, None, False, None, None, None)
    with pytest.raises(ValueError):
        launch_int8_linear(x.float(), x_scale, weight, weight_scale, bias, None, False, None, None, None)


HEADS, KV_HEADS, DV, TEMPLATES, TOKENS, EPS = 24, 12, 32, 8, 70, 1e-5


def attention_operands(device, positions, heads, kv_heads, dq, dv, seed=0, tokens=TOKENS, templates_count=TEMPLATES):
    torch.manual_seed(seed)
    projected = torch.randn(positions, tokens, heads * dq + kv_heads * dq + kv_heads * dv + heads * templates_count, device=device).half()
    templates = (torch.randn(templates_count, 64, 64, device=device) / 2).half()
    q_gain, k_gain = (1 + torch.randn(2, dq, device=device) / 10).half()
    return projected, templates, q_gain, k_gain, heads, kv_heads, dq, dv, templates_count, EPS


def reference_attention(arguments):
    """The reference's fp32 formula (tests/test_attention_cuda.py:51-60)."""
    projected, templates, q_gain, k_gain, heads, kv_heads, dq, dv, templates_count, eps = arguments
    B, T, _ = projected.shape
    q, k, v, c = projected.float().split([heads * dq, kv_heads * dq, kv_heads * dv, heads * templates_count], dim=-1)
    q = F.rms_norm(q.reshape(B, T, heads, dq), (dq,), q_gain.float(), eps).transpose(1, 2)
    k = F.rms_norm(k.reshape(B, T, kv_heads, dq), (dq,), k_gain.float(), eps).transpose(1, 2).repeat_interleave(heads // kv_heads, 1)
    v = v.reshape(B, T, kv_heads, dv).transpose(1, 2).repeat_interleave(heads // kv_heads, 1)
    bias = torch.einsum("biht,tij->bhij", c[:, :64].reshape(B, 64, heads, templates_count), templates.float())
    scores = q @ k.transpose(-2, -1).contiguous() / math.sqrt(dq) + F.pad(bias, (0, T - 64, 0, T - 64))
    return (torch.softmax(scores, -1) @ v).transpose(1, 2).reshape(B, T, heads * dv)


ATTENTION_SHAPES = [(24, 12, 8, 32), (24, 12, 16, 32), (24, 12, 24, 32), (8, 8, 64, 64), (4, 2, 16, 32), (8, 8, 32, 32)]


@pytest.mark.parametrize("heads, kv_heads, dq, dv", ATTENTION_SHAPES)
@pytest.mark.parametrize("positions", [1, 5, 37])
def test_template_attention_is_the_attention_in_fp32(device, heads, kv_heads, dq, dv, positions):
    arguments = attention_operands(device, positions, heads, kv_heads, dq, dv)
    out = template_attention(*arguments)
    expected = reference_attention(arguments)
    assert out.dtype == torch.float16 and out.shape == expected.shape
    assert torch.allclose(out.float(), expected, atol=1e-2)
    rounded = oracle.template_attention(*(cpu(t) if isinstance(t, torch.Tensor) else t for t in arguments))
    assert np.abs(cpu(out.float()) - rounded).max() < 4e-3


@pytest.mark.parametrize("heads, kv_heads, dq, dv", [(8, 8, 64, 128), (8, 4, 32, 16), (4, 4, 64, 64)])
@pytest.mark.parametrize("tokens", [70, 100, 128])
def test_template_attention_at_every_value_width_and_token_count(device, heads, kv_heads, dq, dv, tokens):
    """The value rows read transposed for the P V products: value widths 16 to 128 (2 to 16 chunks a row), 5 to 8 tiles of 16
    tokens, against the reference's fp32 formula."""
    arguments = attention_operands(device, 3, heads, kv_heads, dq, dv, seed=tokens + dv, tokens=tokens)
    out = template_attention(*arguments)
    expected = reference_attention(arguments)
    assert out.shape == expected.shape and torch.allclose(out.float(), expected, atol=1e-2)
    rounded = oracle.template_attention(*(cpu(t) if isinstance(t, torch.Tensor) else t for t in arguments))
    assert np.abs(cpu(out.float()) - rounded).max() < 4e-3


def test_template_attention_at_64_tokens_with_a_bias_per_head(device):
    """benchmark config 2's case, per-head bias: templates_count = heads and one-hot coefficients."""
    projected, templates, q_gain, k_gain, heads, kv_heads, dq, dv, count, eps = attention_operands(device, 16, 8, 8, 64, 64, tokens=64)
    c = projected[..., -heads * count:].reshape(16, 64, heads, count)
    c.zero_()
    c[..., torch.arange(heads), torch.arange(heads)] = 1.0
    arguments = (projected, templates, q_gain, k_gain, heads, kv_heads, dq, dv, count, eps)
    out = template_attention(*arguments)
    assert torch.allclose(out.float(), reference_attention(arguments), atol=1e-2)


def test_template_attention_reads_the_templates_and_their_coefficients(device):
    """The reference's check (tests/test_attention_cuda.py:100-107)."""
    projected, templates, *rest = attention_operands(device, 8, 24, 12, 16, 32)
    without_bias = template_attention(projected, torch.zeros_like(templates), *rest)
    mixed = projected.clone()
    mixed[..., -HEADS * TEMPLATES:] = 0
    assert torch.equal(without_bias, template_attention(mixed, templates, *rest))
    assert (template_attention(projected, templates, *rest).float() - without_bias.float()).abs().max() > 0.05


@pytest.mark.parametrize("heads, kv_heads, dq, dv, tokens, count, dtype", [
    (8, 4, 32, 32, 100, 8, torch.float16), (8, 4, 32, 32, 100, 6, torch.bfloat16), (8, 4, 64, 64, 128, 8, torch.float16),
    (8, 8, 64, 64, 128, 8, torch.bfloat16), (4, 4, 64, 128, 70, 8, torch.float16), (6, 3, 24, 128, 96, 8, torch.float16),
    (4, 4, 128, 64, 70, 8, torch.float16), (2, 2, 104, 128, 80, 8, torch.float16)])
def test_groups_a_workgroup_change_no_bit(device, heads, kv_heads, dq, dv, tokens, count, dtype):
    """Any run of (position, key/value group) pairs a workgroup takes gives the same bits, and the fp32 formula's answer, runs
    across positions and all nine positions in one workgroup too: the kernel of more than 80 tokens or widths past 64, which walks
    the runs through two buffers, its outputs staged over the queries (value widths up to the queries') or stored from the
    registers. (The other kernel shares the pairs out by itself.)"""
    projected, *rest = attention_operands(device, 9, heads, kv_heads, dq, dv, seed=tokens + dv, tokens=tokens, templates_count=count)
    arguments, pairs = (projected.to(dtype), *rest), 9 * kv_heads
    one = launch_template_attention(*arguments, groups_per_block=1)
    assert (one.float() - reference_attention(arguments)).abs().max() < 1e-2
    for groups in [groups for groups in range(2, pairs + 1) if pairs % groups == 0]:
        assert torch.equal(launch_template_attention(*arguments, groups_per_block=groups), one), groups
    with pytest.raises(ValueError):
        launch_template_attention(*arguments, groups_per_block=5)   # not a divisor of the pairs


def whole_pair_positions(device, kv_heads):
    """A few positions more than the most that the kernel of widths up to 64 shares over four wavefronts a pair: six pairs a compute
    unit, of several narrow heads each, over 65 to 80 tokens."""
    units = torch.cuda.get_device_properties(device).multi_processor_count
    return 6 * units // kv_heads + 5


@pytest.mark.parametrize("heads, kv_heads, dq, dv, tokens", [(8, 8, 64, 64, 70), (8, 4, 32, 32, 80), (4, 4, 16, 64, 65), (6, 3, 64, 16, 66)])
def test_large_attention_launches_give_the_small_launchs_bits(device, heads, kv_heads, dq, dv, tokens):
    """65 to 80 tokens: in a large launch a wavefront takes whole (position, key/value group) pairs; every position's rows are the
    same bits as in launches of seven positions (four wavefronts a pair), and the answer is the fp32 formula's. The grouped case
    with two heads a group (6 on 3) once differed on the tokens past the squares of a few positions in the middle of the
    launch."""
    positions = whole_pair_positions(device, kv_heads)
    arguments = attention_operands(device, positions, heads, kv_heads, dq, dv, seed=tokens, tokens=tokens)
    large = template_attention(*arguments)
    assert torch.allclose(large.float(), reference_attention(arguments), atol=1e-2)
    few = torch.cat([template_attention(arguments[0][start:start + 7].contiguous(), *arguments[1:]) for start in range(0, positions, 7)])
    assert torch.equal(few, large)


@pytest.mark.parametrize("heads, kv_heads, dq, dv, tokens, count, positions", [
    (8, 8, 64, 64, 70, 8, 129), (8, 8, 64, 64, 64, 8, 65), (4, 4, 40, 64, 66, 6, 257), (24, 12, 24, 32, 70, 8, 129), (8, 4, 8, 16, 80, 3, 385),
    (2, 1, 32, 32, 65, 8, 1537), (8, 4, 32, 32, 64, 8, 193), (12, 4, 32, 32, 64, 8, 257), (4, 4, 32, 64, 70, 8, 193)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_both_sharings_of_the_pairs_give_the_same_bits(device, heads, kv_heads, dq, dv, tokens, count, positions, dtype):
    """Widths up to 64 and up to 80 tokens: a launch of some pairs a compute unit (more than two of one head each; four, or seven of
    narrow widths over 65 tokens and more, of several; not five of three: the last shape but one) gives its wavefronts whole pairs, and one
    of a few positions shares a pair over four. The same bits, the fp32 formula's answer, at the smallest and largest token counts, query widths that do not fill their chunks and fewer than
    eight templates; a position of infinities and NaNs stays its own."""
    projected, *rest = attention_operands(device, positions, heads, kv_heads, dq, dv, seed=tokens + dq, tokens=tokens, templates_count=count)
    projected = projected.to(dtype)
    arguments = (projected, *rest)
    whole, expected = template_attention(*arguments), reference_attention(arguments)
    # 1e-2, and for bf16 outputs their own rounding, up to half a step of 8 bits: 2^-9 of the value (outputs reach 4 here)
    assert ((whole.float() - expected).abs() <= 1e-2 + (2 ** -9 * expected.abs() if dtype == torch.bfloat16 else 0)).all()
    some = [0, 1, 2, positions // 2, positions - 2, positions - 1]
    assert torch.equal(template_attention(projected[some].contiguous(), *arguments[1:]), whole[some])
    spoilt = projected.clone()
    spoilt[1] = float("nan")
    spoilt[positions - 2, :, ::3] = float("inf")
    clean = [position for position in range(positions) if position not in (1, positions - 2)]
    for boards in (positions, 5):
        rows = list(range(boards - 3)) + list(range(positions - 3, positions))
        kept = [k for k, position in enumerate(rows) if position in set(clean)]
        out = template_attention(spoilt[rows].contiguous(), *arguments[1:])
        assert torch.equal(out[kept], whole[[rows[k] for k in kept]])


@pytest.mark.parametrize("tokens", [64, 65, 70, 72, 73, 80])
@pytest.mark.parametrize("heads, kv_heads, dq, dv, count", [(4, 4, 64, 64, 8), (6, 3, 24, 32, 8), (2, 2, 40, 16, 4)])
def test_attention_reads_and_writes_nothing_past_its_rows(device, tokens, heads, kv_heads, dq, dv, count):
    """Up to 80 tokens, widths up to 64: the last tiles of 16 rows reach past a position's tokens. With NaNs round the input rows
    (and in LDS, left by a launch before) and a sentinel round the outputs, at the C entry: the fp32 formula's answer, the operator's
    bits, and every sentinel as it was, whether the wavefronts take whole pairs (the large launch) or share one."""
    units = torch.cuda.get_device_properties(device).multi_processor_count
    library, guard, sentinel = library_for(device), 128 * 1024, 12345.0
    for positions in (3, 6 * units // kv_heads + 2):
        arguments = attention_operands(device, positions, heads, kv_heads, dq, dv, seed=tokens + dq, tokens=tokens, templates_count=count)
        projected, templates, q_gain, k_gain = arguments[:4]
        rows = torch.full((guard + projected.numel() + guard,), float("nan"), device=device, dtype=torch.float16)
        rows[guard:-guard] = projected.flatten()
        outputs = positions * tokens * heads * dv
        out = torch.full((guard + outputs + guard,), sentinel, device=device, dtype=torch.float16)
        keyed = fused_blocks.keyed_templates(templates, count)
        template_attention(torch.full_like(projected, float("nan")), *arguments[1:])
        at = lambda buffer: pointer(buffer[guard:])
        check(library.chess_template_attention(at(rows), pointer(keyed), pointer(q_gain), pointer(k_gain), at(out), positions, tokens, heads, kv_heads,
                                               dq, dv, count, 1, EPS, 1 / math.sqrt(dq), stream_of(device)), "template_attention")
        found = out[guard:-guard].view(positions, tokens, heads * dv)
        assert torch.allclose(found.float(), reference_attention(arguments), atol=1e-2)
        assert torch.equal(found, template_attention(*arguments))
        assert (out[:guard] == sentinel).all() and (out[-guard:] == sentinel).all()


def bf16_operands(arguments):
    projected, templates, *rest = arguments
    return (projected.bfloat16(), templates, *rest)


@pytest.mark.parametrize("heads, kv_heads, dq, dv", [(8, 8, 64, 64), (24, 12, 16, 32), (4, 2, 16, 32)])
@pytest.mark.parametrize("positions, tokens", [(5, 64), (37, 70), (3, 80)])
def test_bf16_template_attention_is_the_attention_in_fp32(device, heads, kv_heads, dq, dv, positions, tokens):
    """bf16 rows in and out (benchmark config 2's types): the fp32 formula of the reference's test on the same bf16 inputs, at
    config 2's 1e-2; the fp16 kernel's answer on them within 1e-2."""
    arguments = bf16_operands(attention_operands(device, positions, heads, kv_heads, dq, dv, seed=positions + tokens, tokens=tokens))
    out = template_attention(*arguments)
    assert out.dtype == torch.bfloat16
    expected = reference_attention(arguments)
    assert (out.float() - expected).abs().max() < 1e-2
    halves = template_attention(arguments[0].half(), *arguments[1:])
    assert (out.float() - halves.float()).abs().max() < 1e-2


@pytest.mark.parametrize("positions", [16, 4096])
def test_bf16_template_attention_at_64_tokens_with_a_bias_per_head(device, positions):
    """benchmark config 2 in its own types and at its size (4,096 positions x 8 heads x 64 x 64 tokens): bf16 Q/K/V and output,
    a learned 64 x 64 bias per head N(0, 0.5) (one-hot template mix), against the reference's fp32 formula within config 2's
    1e-2 max-abs on every output. P V takes P as a bf16 high and low part, so the output's error is its own bf16 rounding."""
    projected, templates, q_gain, k_gain, heads, kv_heads, dq, dv, count, eps = attention_operands(device, positions, 8, 8, 64, 64, tokens=64)
    c = projected[..., -heads * count:].reshape(positions, 64, heads, count)
    c.zero_()
    c[..., torch.arange(heads), torch.arange(heads)] = 1.0
    arguments = (projected.bfloat16(), templates, q_gain, k_gain, heads, kv_heads, dq, dv, count, eps)
    out = template_attention(*arguments)
    assert out.dtype == torch.bfloat16 and out.shape == (positions, 64, heads * dv)
    assert (out.float() - reference_attention(arguments)).abs().max() < 1e-2


def test_large_bf16_attention_launches_give_the_small_launchs_bits(device):
    """bf16 rows at 70 tokens, a wavefront a pair: a position's rows are a three-position launch's bits."""
    positions = whole_pair_positions(device, 8)
    arguments = bf16_operands(attention_operands(device, positions, 8, 8, 64, 64, seed=70, tokens=70))
    large = template_attention(*arguments)
    assert (large.float() - reference_attention(arguments)).abs().max() < 1e-2
    for rows in (slice(0, 3), slice(positions - 3, positions)):
        assert torch.equal(template_attention(arguments[0][rows].contiguous(), *arguments[1:]), large[rows]), rows


def test_template_attention_refuses_what_it_cannot_take(device):
    projected, templates, q_gain, k_gain, *rest = attention_operands(device, 2, 8, 8, 64, 64)
    with pytest.raises(ValueError):
        template_attention(projected.float(), templates, q_gain, k_gain, *rest)
    with pytest.raises(ValueError):   # bf16 rows take query widths up to 64
        template_attention(*bf16_operands(attention_operands(device, 2, 8, 8, 128, 64)))
    with pytest.raises(ValueError):
        template_attention(projected[:, :, :-8], templates, q_gain, k_gain, *rest)


@pytest.mark.parametrize("M, K, N", [(70, 512, 512), (4480, 512, 512), (210, 768, 1600), (333, 96, 40)])
def test_linear_is_the_matmul(device, M, K, N):
    torch.manual_seed(M)
    x = torch.randn(M, K, device=device).half()
    weight = (torch.randn(K, N, device=device) / math.sqrt(K)).half()
    bias, residual = torch.randn(N, device=device).half(), torch.randn(M, N, device=device).half()
    expected = oracle.linear(cpu(x), cpu(weight), cpu(bias), cpu(residual)).astype(np.float64)
    for tile in (1, 2):
        out = launch_linear(x, weight, bias, residual, False, False, None, None, None, tile)
        assert out.dtype == torch.float16 and np.allclose(cpu(out).astype(np.float64), expected, atol=2e-3, rtol=2e-3), tile


def test_linear_gated_mixed_and_fp32(device):
    torch.manual_seed(1)
    x = torch.randn(280, 256, device=device).half()
    gate_up = (torch.randn(256, 2 * 320, device=device) / 16).half()
    hidden = linear(x, gate_up, gated=True)
    expected = oracle.linear(cpu(x), cpu(gate_up), gated=True).astype(np.float64)
    assert np.allclose(cpu(hidden).astype(np.float64), expected, atol=2e-3, rtol=4e-3)
    down = (torch.randn(320, 256, device=device) / 18).half()
    residual, original = torch.randn(280, 256, device=device).half(), torch.randn(280, 256, device=device).half()
    rs, is_ = torch.tensor([0.8], device=device).half(), torch.tensor([0.5], device=device).half()
    mixed = linear(hidden, down, residual=residual, original=original, residual_scale=rs, input_scale=is_)
    expected = oracle.linear(cpu(hidden), cpu(down), residual=cpu(residual), original=cpu(original), residual_scale=cpu(rs),
                             input_scale=cpu(is_)).astype(np.float64)
    assert np.allclose(cpu(mixed).astype(np.float64), expected, atol=4e-3, rtol=4e-3)
    wide = linear(x, gate_up, accumulate_fp32=True)
    assert wide.dtype == torch.float32
    assert np.allclose(cpu(wide), cpu(x).astype(np.float64) @ cpu(gate_up).astype(np.float64), atol=1e-3, rtol=1e-4)


@pytest.mark.parametrize("M, K, N", [(2560, 96, 72), (5120, 160, 64), (26112, 96, 72)])
def test_gated_linear_takes_rows_of_no_whole_lines(device, M, K, N):
    """Rows of a multiple of 64 bytes but not of 128, at the shares of rows where longer ones take tiles that stage 128 bytes of a
    row; the tolerances of the gated launch above."""
    torch.manual_seed(M + K)
    x = torch.randn(M, K, device=device).half()
    gate_up = (torch.randn(K, 2 * N, device=device) / math.sqrt(K)).half()
    expected = oracle.linear(cpu(x), cpu(gate_up), gated=True).astype(np.float64)
    assert np.allclose(cpu(linear(x, gate_up, gated=True)).astype(np.float64), expected, atol=2e-3, rtol=4e-3)


def test_the_kernels_run_in_graphs_on_two_streams(device):
    """The reference's isolation check (tests/test_int8.py:161-184, tests/test_attention_cuda.py:110-130): two graphs replayed
    together on two streams give the eager bits."""
    operands = int8_operands("mixing down", 140, device)
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = operands
    attention = attention_operands(device, 6, 24, 12, 24, 32, seed=2)
    signs = hadamard(HADAMARD_BLOCK).to(device).half()
    run = lambda first: (int8_linear(first, x_scale, weight, weight_scale, bias, residual, gated, "down", *mix),
                         template_attention(*attention), rotate_quant(residual, signs, 256)[0])
    inputs = [x, x.flip(0).contiguous()]
    expected = [run(first) for first in inputs]
    streams, buffers, graphs, outputs = [torch.cuda.Stream() for _ in range(2)], [first.clone() for first in inputs], [], []
    for stream, buffer in zip(streams, buffers):
        stream.wait_stream(torch.cuda.current_stream())
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=stream):
            outputs.append(run(buffer))
    for replay in range(5):
        torch.cuda.synchronize()
        for stream, graph in zip(streams, graphs):
            with torch.cuda.stream(stream):
                graph.replay()
        torch.cuda.synchronize()
        for found, answer in zip(outputs, expected):
            assert all(torch.equal(a, b) for a, b in zip(found, answer)), replay


def test_outputs_of_two_gib_take_the_kernels_own_pick(device):
    """524,304 rows of 512 to 2 x 2,048 columns write 2 GiB, past what tile 15's 32-bit offsets take: the table's choice gives
    them to tile 0, whose first and last rows are a small launch's bits."""
    M, ends = 524304, 48
    x, x_scale, weight, weight_scale, bias, residual, gated, mix = int8_operands("gate_up", ends, device, width=2048, depth=512)
    many = torch.zeros(M, 512, device=device, dtype=torch.int8)
    scales = torch.ones(M, device=device)
    for at in (slice(0, ends), slice(M - ends, M)):
        many[at], scales[at] = x, x_scale
    out = int8_linear(many, scales, weight, weight_scale, None, None, True, "gate_up")
    expected = launch_int8_linear(x, x_scale, weight, weight_scale, None, None, True, None, None, None, 1)
    assert same_bits(out[:ends], expected) and same_bits(out[-ends:], expected) and not out[ends:-ends].any()
