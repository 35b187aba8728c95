"""The names and contracts the reference's engine reads from this package, on the CPU: every name its engine modules import
from engine.inference and model.int8_blocks, ExactSizeCompiled's dispatch by batch size (reference engine/inference.py:251-263),
FusedTransformer's return contract on gfx950 (reference fused_blocks.py:415-419, 856-871, unpacked by mcts.py:56) and the
tile tables' override for experiments."""
import math

import pytest
import torch
from torch import nn

from engine import inference
from model import int8_blocks
from model.fused_blocks import FusedTransformer
from model.model import ChessTransformer

# what the reference's engine modules import from this package, name for name
IMPORTED = {
    "engine.inference": {
        "engine/engine_search.py:17": ("ExactSizeCompiled", "GraphedBatches", "chunk_positions", "fp16_model", "int8_model", "small_graph_sizes"),
        "engine/uci.py:16": ("cpu_batches",),
        "engine/quantization.py:14": ("FP16_RESIDUAL_SCALE", "answer_rows", "fp16_model"),
    },
    "model.int8_blocks": {
        "engine/quantization.py:18": ("DOWN_INPUT_MULTIPLE", "HADAMARD_BLOCK", "Int8Block", "down_inputs", "hadamard"),
        "tests/test_int8.py:18-21": ("INT8_TILES", "int8_tile", "rotate_rows", "int8_linear", "launch_int8_linear", "norm_quant", "mix_norm_quant",
                                     "rotate_quant", "quantize_blocks"),
    },
    "model.fused_blocks": {"engine/quantization.py:17": ("link_input_mixes",)},
    "engine.quantization": {"engine/engine_search.py:176, engine/inference.py:269": ("int8_weights",)},
}


@pytest.mark.parametrize("module, site", [(module, site) for module, sites in IMPORTED.items() for site in sites])
def test_every_name_the_engine_imports_is_here(module, site):
    imported = __import__(module, fromlist=["_"])
    missing = [name for name in IMPORTED[module][site] if not hasattr(imported, name)]
    assert not missing, f"{site} imports {missing} from {module}"


class Recorder(nn.Module):
    """Answers a batch with its size, and records the options each call got."""
    gives_answer_rows = True
    d_model = 8

    def __init__(self):
        super().__init__()
        self.calls = []

    def forward(self, boards, **options):
        self.calls.append((len(boards), options))
        return boards.float().sum(1, keepdim=True)


def test_exact_size_compiled_runs_the_model_for_every_size():
    model = Recorder()
    compiled = inference.ExactSizeCompiled(model, 16)
    assert compiled.exact is model and compiled.dynamic is model and compiled.exact_size == 16
    assert compiled.gives_answer_rows and compiled.d_model == 8
    for size in (1, 16, 17):
        boards = torch.arange(size * 3).reshape(size, 3)
        assert torch.equal(compiled(boards), model(boards))
    # the lanes' answer rows go through it with the rows switch
    inference.network_rows(compiled, torch.zeros(4, 3))
    assert model.calls[-1] == (4, {"rows": True})


def test_exact_size_compiled_compiles_each_side_with_a_backend():
    model = nn.Linear(3, 2)
    compiled = inference.ExactSizeCompiled(model, 4, backend="eager")
    assert compiled.exact is not model and compiled.dynamic is not compiled.exact
    for size in (4, 5):
        boards = torch.randn(size, 3)
        with torch.no_grad():
            assert torch.allclose(compiled(boards), model(boards))


def test_network_rows_take_answer_rows_of_other_models():
    class Pair(nn.Module):
        def forward(self, boards):
            return boards.float(), torch.zeros(len(boards), 4)
    rows = inference.network_rows(Pair(), torch.ones(2, 5))
    assert rows.shape == (2, 6) and torch.equal(rows[:, :5], torch.ones(2, 5))


def test_the_fused_network_returns_logits_and_value_logits_by_default():
    model = ChessTransformer(d_model=64, num_layers=1, n_heads=2, mlp_hidden=64, value_bins=4)
    fused = FusedTransformer(model)
    assert fused.fused_heads is False and fused.gives_answer_rows
    assert FusedTransformer(model, fused_heads=True).fused_heads
    assert inference.fused_model(ChessTransformer(d_model=64, num_layers=1, n_heads=2, mlp_hidden=64, value_bins=4)).fused_heads is False


@pytest.fixture
def tables():
    saved = ({role: list(entries) for role, entries in int8_blocks.INT8_TILES["gfx950"].items()}, list(int8_blocks.ROTATE_ROWS["gfx950"]))
    yield
    int8_blocks.INT8_TILES["gfx950"].update(saved[0])
    int8_blocks.ROTATE_ROWS["gfx950"] = saved[1]


def test_the_environment_overrides_a_table(tables):
    int8_blocks.apply_overrides({int8_blocks.TILES_VARIABLE: '{"gate_up": [[18, 9], ["inf", 10]], "down": [["inf", 13]]}',
                                 int8_blocks.ROTATE_VARIABLE: '[[4, 1], ["inf", 2]]'})
    assert int8_blocks.INT8_TILES["gfx950"]["gate_up"] == [(18.0, 9), (math.inf, 10)]
    assert int8_blocks.INT8_TILES["gfx950"]["down"] == [(math.inf, 13)]
    assert int8_blocks.ROTATE_ROWS["gfx950"] == [(4.0, 1), (math.inf, 2)]
    with pytest.raises(ValueError, match="roles"):
        int8_blocks.apply_overrides({int8_blocks.TILES_VARIABLE: '{"combine": [["inf", 1]]}'})
    with pytest.raises(ValueError, match="unbounded"):
        int8_blocks.apply_overrides({int8_blocks.ROTATE_VARIABLE: '[[4, 1]]'})
    with pytest.raises(ValueError, match="growing"):
        int8_blocks.apply_overrides({int8_blocks.ROTATE_VARIABLE: '[[4, 1], [2, 1], ["inf", 2]]'})


def test_the_shipped_tables_end_unbounded():
    for entries in (*int8_blocks.INT8_TILES["gfx950"].values(), int8_blocks.ROTATE_ROWS["gfx950"]):
        assert int8_blocks._bounded(entries) == [(float(most), choice) for most, choice in entries]


def test_tile_shapes_are_the_kernels_instantiations():
    """TILE_SHAPES against the launches gemm_tiles.h instantiates (tile 11 is its default case; 14 is the split-K tile)."""
    import re
    from pathlib import Path
    source = (Path(int8_blocks.__file__).parent.parent / "csrc" / "gemm_tiles.h").read_text()
    launches = {int(case) if case else 11: tuple(map(int, shape)) for case, *shape in
                re.findall(r"(?:case (\d+)|default): return launch<In, (\d+), (\d+), (\d+), (\d+), NB, (\d+)", source)}
    assert set(launches) == set(int8_blocks.TILE_SHAPES) - set(int8_blocks.SPLIT_WAVES)
    for tile, (rows, columns, waves_m, waves_n, stages) in launches.items():
        assert int8_blocks.TILE_SHAPES[tile] == (rows, columns, waves_m * waves_n, stages), tile


def test_a_reference_tile_tuple_names_the_tile_of_its_shape():
    """The reference's launch_int8_linear takes Triton tiles (rows, columns, depth, warps, stages[, registers]); the shapes the
    library has map to its tiles, the rest are refused by name."""
    assert int8_blocks.tile_id(0) == 0 and int8_blocks.tile_id(10) == 10
    assert int8_blocks.tile_id((128, 64, 64, 4, 2)) == 9      # reference sm_120 gate_up, batch 1024
    assert int8_blocks.tile_id((128, 64, 64, 4, 3)) == 8      # reference sm_86/89 gate_up
    assert int8_blocks.tile_id((128, 128, 64, 8, 3, 128)) == 6
    assert int8_blocks.tile_id((64, 64, 64, 4, 4)) == 1
    assert int8_blocks.tile_id((128, 128, 128, 4, 5)) == 2    # no 5-stage twin: the first 128 x 128
    with pytest.raises(ValueError, match="no 32 x 64 tile"):
        int8_blocks.tile_id((32, 64, 64, 4, 4))
    assert int8_blocks.tile_id(15) == 15 and int8_blocks.tile_id(16) == 16
    with pytest.raises(ValueError, match="tiles"):
        int8_blocks.tile_id(17)


def test_the_register_held_tiles_take_only_their_launches():
    """Which launches tiles 15 and 16 take (the tables give way to tile 0 for the rest): 15 depth 512 and N a multiple of
    8 without a residual, gated or not; 16 down's depth 2048, N a multiple of 128, not gated, no bias, with the residual;
    the whole-K tiles every launch; and the fp16 linear's tile 15 the bias epilogue without the input mix."""
    from model.fused_blocks import linear_takes
    takes = int8_blocks.tile_takes
    assert takes(15, 1600, 512) and takes(15, 2048, 512, gated=True) and takes(15, 200, 512, bias=True)
    assert not any((takes(15, 196, 512), takes(15, 512, 2048), takes(15, 512, 512, residual=True)))
    assert takes(16, 512, 2048, residual=True) and takes(16, 128, 2048, residual=True)
    assert not any((takes(16, 512, 2048), takes(16, 200, 2048, residual=True), takes(16, 512, 1024, residual=True),
                    takes(16, 512, 2048, bias=True, residual=True), takes(16, 512, 2048, gated=True, residual=True)))
    assert all(takes(tile, 196, 1024, True, True, True) for tile in range(1, 14))
    assert linear_takes(15, 512, 1600, False, True, False, False) and linear_takes(15, 512, 512, False, True, True, False)
    assert not any((linear_takes(15, 512, 512, False, True, True, False, True), linear_takes(15, 512, 512, True, True, False, False),
                    linear_takes(15, 512, 512, False, False, True, False), linear_takes(15, 512, 512, False, True, True, True)))
    assert linear_takes(11, 2048, 512, True, False, True, True, True)


def test_launches_past_the_register_held_tiles_limits_take_tile_0(monkeypatch):
    """Tiles 15 and 16 write outputs under 2 GiB and take at most 32 column groups (a compute unit's XCD has 32 on an MI355X); the
    tables' and linear's choices give larger launches to tile 0, which takes them (8,192 positions of the d512 network: gate_up
    writes 2.3 GB)."""
    from model import fused_blocks, hip_kernels
    monkeypatch.setattr(hip_kernels, "gpu", lambda device: ("gfx950", 256))
    monkeypatch.setattr(fused_blocks, "gpu", lambda device: ("gfx950", 256))
    cuda, chosen = torch.device("cuda"), []
    tile = int8_blocks.int8_tile
    assert [tile(cuda, "gate_up", positions * 70, 2048, 512) for positions in (7489, 7490, 8192)] == [15, 0, 0]
    assert tile(cuda, "gate_up", 524287, 2048, 512) == 15 and tile(cuda, "gate_up", 524288, 2048, 512) == 0
    assert tile(cuda, "projection", 671088, 1600, 512, bias=True) == 15 and tile(cuda, "projection", 671089, 1600, 512, bias=True) == 0
    assert tile(cuda, "down", 2097151, 512, 2048) == 16 and tile(cuda, "down", 2097152, 512, 2048) == 0
    assert tile(cuda, "gate_up", 71680, 8192, 512) == 15 and tile(cuda, "gate_up", 71680, 8200, 512) == 0
    assert tile(cuda, "down", 71680, 4096, 2048) == 16 and tile(cuda, "down", 71680, 4224, 2048) == 0
    monkeypatch.setattr(fused_blocks, "launch_linear", lambda x, weight, *arguments: chosen.append(arguments[-1]) or x.new_empty(0))
    for M, N in ((262143, 4096), (262144, 4096), (71680, 8192), (71680, 8200)):
        x = torch.empty(1, dtype=torch.float16).expand(M, 512)
        fused_blocks.linear(x, torch.empty(1, dtype=torch.float16).expand(512, N), torch.empty(1, dtype=torch.float16).expand(N))
    assert chosen == [15, 0, 15, 0]
