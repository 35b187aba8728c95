"""The host-side choices around the kernels, on the CPU: tile tables, the attention launch's (position, group) runs and
the policy head's move tables (the reference's tile_for, fused_blocks.py:183-192, and its move gathers, :869-870)."""
import math

import pytest
import torch

from model import fused_blocks, hip_kernels, int8_blocks
from model.encoding import NUM_SQUARES
from model.fused_blocks import groups_per_workgroup, move_places, tile_for
from model.model import ChessTransformer


def test_tile_for_takes_the_first_row_share_that_fits():
    tiles = [(4, 1), (32, 3), (math.inf, 11)]
    assert tile_for(tiles, 4 * 256, 256) == 1
    assert tile_for(tiles, 4 * 256 + 1, 256) == 3
    assert tile_for(tiles, 71680, 256) == 11


def test_a_projection_table_put_in_the_shipped_ones_place_holds_at_every_depth(monkeypatch):
    monkeypatch.setattr(hip_kernels, "gpu", lambda device: ("gfx950", 256))
    chosen = lambda K: int8_blocks.int8_tile(torch.device("cuda"), "projection", 3570, 1152, K, bias=True)
    assert (chosen(512), chosen(640), chosen(768), chosen(832)) == (11, 11, 6, 11)   # 832: no whole 128-byte lines
    monkeypatch.setitem(int8_blocks.INT8_TILES["gfx950"], "projection", [(math.inf, 3)])
    assert (chosen(512), chosen(768)) == (3, 3)
    monkeypatch.setitem(int8_blocks.INT8_TILES["gfx950"], "projection", list(int8_blocks.SHIPPED_PROJECTION_TILES))   # put back
    assert (chosen(512), chosen(768), chosen(832)) == (11, 6, 11)
    int8_blocks.INT8_TILES["gfx950"]["projection"][-2] = (100, 2)                                                    # edited in place
    assert (chosen(512), chosen(768)) == (2, 2)


def test_the_tile_choices_ask_torch_about_what_is_no_gpu(monkeypatch):
    def properties(device):
        raise ValueError(f"asked about {device}")
    monkeypatch.setattr(torch.cuda, "get_device_properties", properties)
    monkeypatch.setattr(hip_kernels, "_gpus", {0: ("gfx950", 256)})
    assert hip_kernels.gpu(torch.device("cuda", 0)) == ("gfx950", 256)
    for device in (torch.device("cpu"), "cpu"):
        with pytest.raises(ValueError, match="asked about cpu"):
            hip_kernels.gpu(device)


def test_no_choice_of_an_int8_block_asks_torch_for_its_properties(monkeypatch):
    """A block's choices of tiles and rows ask for the GPU's target and compute units through hip_kernels.gpu, which asks torch once
    a process."""
    def properties(device):
        raise AssertionError("torch was asked")
    monkeypatch.setattr(torch.cuda, "get_device_properties", properties)
    monkeypatch.setattr(hip_kernels, "_gpus", {0: ("gfx950", 256)})
    device = torch.device("cuda", 0)
    for M in (70, 4480, 71680):
        int8_blocks.rotate_rows(device, M)
        int8_blocks.rotated_down_tile(device, M, 2048, 2048)
        for role in ("projection", "gate_up", "down"):
            int8_blocks.int8_tile(device, role, M, 512, 512)
        for f32, gated in ((False, False), (False, True), (True, False)):
            fused_blocks.linear_tile(device, M, f32, 1024, gated, 512)


@pytest.mark.parametrize("M, N, expected", [(3584, 1152, 6), (3585, 1152, 11), (7000, 1152, 13), (8785, 960, 11), (12000, 960, 13),
                                            (13000, 768, 11), (17920, 1152, 13), (19200, 1152, 13), (19201, 1152, 0)])
def test_long_projections_leave_tiles_whose_last_round_is_small(monkeypatch, M, N, expected):
    monkeypatch.setattr(hip_kernels, "gpu", lambda device: ("gfx950", 256))
    assert int8_blocks.int8_tile(torch.device("cuda"), "projection", M, N, 768, bias=True) == expected


@pytest.mark.parametrize("M, K, N, gated, f32, bias, expected", [
    (8192, 768, 768, False, False, True, 12), (8193, 768, 768, False, False, True, 13), (10880, 768, 768, False, False, True, 13),
    (10881, 768, 768, False, False, True, 12), (8193, 768, 768, False, True, True, 13), (6453, 768, 1152, False, False, True, 13),
    (8193, 512, 768, False, True, True, 13), (9472, 512, 768, False, True, True, 13), (9473, 512, 768, False, True, True, 12),
    (8193, 256, 768, False, True, True, 12),
    (256 * 48, 512, 1600, False, False, True, 6), (256 * 48 + 1, 512, 1600, False, False, True, 15),    # the long streams' first row
    (256 * 49, 512, 1016, False, False, True, 11), (256 * 49, 512, 1024, False, False, True, 15),        # and least columns
    (256 * 49, 512, 1604, False, False, True, 11), (256 * 49, 512, 1600, False, False, False, 11),       # no whole 8 columns; no bias
    (256 * 49, 768, 1600, False, False, True, 12), (256 * 101, 768, 768, False, False, True, 13),        # long rows
    (256 * 7, 768, 1152, False, False, True, 3), (256 * 7, 768, 768, False, False, True, 1), (256 * 7, 1024, 1152, False, False, True, 1),
    (256 * 9, 704, 512, False, False, True, 3), (256 * 101, 512, 512, True, False, False, 11), (256 * 20, 512, 512, True, False, False, 12),
    (256 * 101, 704, 512, True, False, False, 4), (256 * 101, 256, 512, True, False, False, 0), (256 * 20, 256, 512, True, False, False, 6),
    (256 * 9, 512, 512, False, True, False, 1), (256 * 10, 512, 512, False, True, False, 12), (256 * 10, 768, 768, False, True, False, 12),
    (256 * 10, 1088, 768, False, True, False, 7),
    (256 * 10, 32, 512, False, True, False, 7),                                                          # rows of no whole lines
    (256 * 10, 96, 512, True, False, False, 6), (256 * 20, 544, 512, True, False, False, 6), (256 * 101, 96, 512, True, False, False, 0)])
def test_linear_picks_its_tile_by_rows_depth_and_epilogue(monkeypatch, M, K, N, gated, f32, bias, expected):
    chosen = []
    def launched(x, weight, *arguments):
        chosen.append(arguments[-1])
        return x.new_empty(0)
    monkeypatch.setattr(fused_blocks, "gpu", lambda device: ("gfx950", 256))
    monkeypatch.setattr(fused_blocks, "launch_linear", launched)
    width = 2 * N if gated else N
    x, weight = torch.empty(1, dtype=torch.float16).expand(M, K), torch.empty(K, width, dtype=torch.float16)
    fused_blocks.linear(x, weight, torch.empty(width, dtype=torch.float16) if bias else None, None, gated, f32)
    assert chosen == [expected]


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("gated", [False, True])
def test_linear_picks_no_tile_that_refuses_its_rows(monkeypatch, f32, gated):
    """Tiles 5, 12 and 13 stage 128 bytes of a row at a time and refuse rows of no whole 128 bytes; linear takes any multiple of 32
    inputs (64 bytes), at every share of rows."""
    monkeypatch.setattr(fused_blocks, "gpu", lambda device: ("gfx950", 256))
    for K in range(32, 2112, 32):
        for M in (1, 256 * 4, 256 * 5, 256 * 9, 256 * 10, 256 * 20, 256 * 21, 256 * 48, 256 * 49, 256 * 75, 256 * 100, 256 * 101):
            assert K % 64 == 0 or fused_blocks.linear_tile(torch.device("cuda"), M, f32, 2 * K, gated) not in (5, 12, 13), (M, K)


def test_linear_tiles_for_rows_of_unknown_length_take_any_row(monkeypatch):
    """linear_tile asked without the rows' bytes names a tile that takes rows of any length."""
    monkeypatch.setattr(fused_blocks, "gpu", lambda device: ("gfx950", 256))
    for M in (1, 256 * 5, 256 * 10, 256 * 21, 256 * 49, 256 * 101):
        for f32, gated in ((False, False), (False, True), (True, False), (True, True)):
            assert fused_blocks.linear_tile(torch.device("cuda"), M, f32, gated=gated) not in (5, 12, 13), (M, f32, gated)
    assert fused_blocks.linear_tile(torch.device("cuda"), 256 * 10, True) == 7


@pytest.mark.parametrize("positions", [1, 3, 16, 64, 100, 256, 1024, 4096])
@pytest.mark.parametrize("kv_heads", [8, 12])
@pytest.mark.parametrize("tokens", [64, 70, 100])
def test_attention_runs_divide_the_pairs_and_keep_the_chip_busy(positions, kv_heads, tokens):
    pairs = positions * kv_heads
    groups = groups_per_workgroup(positions, kv_heads, 256, tokens)
    workgroups = pairs // groups
    assert pairs % groups == 0
    # at least one workgroup a compute unit when there are enough pairs; when a workgroup takes several pairs, no more
    # workgroups than the compute units hold at once
    assert workgroups >= min(pairs, 256)
    assert groups == 1 or workgroups <= 256 * (8 // fused_blocks.attention_waves(tokens)) * 2


def test_attention_runs_by_tokens():
    """One workgroup a compute unit at five slabs of 16 tokens and more, two at four (8 key/value groups)."""
    assert [groups_per_workgroup(b, 8, 256, 100) for b in (16, 64, 128, 256, 1024)] == [1, 2, 4, 8, 32]
    assert [groups_per_workgroup(b, 8, 256, 64) for b in (16, 64, 128, 256, 1024)] == [1, 1, 2, 4, 16]
    assert [fused_blocks.attention_waves(tokens) for tokens in (64, 65, 80, 81, 128)] == [4, 5, 5, 6, 8]


def test_the_move_tables_are_the_gathers_of_the_heads():
    model = ChessTransformer(d_model=64, num_layers=1, n_heads=2, mlp_hidden=64, value_bins=4)
    cells, promotions = move_places(model)
    assert cells.dtype == torch.int32 and cells.shape == model.from_squares.shape
    assert torch.equal(cells.long() // NUM_SQUARES, model.from_squares) and torch.equal(cells.long() % NUM_SQUARES, model.to_squares)
    promoting = torch.zeros_like(cells, dtype=torch.bool)
    promoting[model.promotion_move_ids] = True
    assert (promotions[~promoting] == -1).all()
    placed = promotions[model.promotion_move_ids].long()
    assert torch.equal(placed // 32, model.promotion_to_squares) and torch.equal(placed % 32, 1 + model.promotion_pieces)
