"""Benchmark of Fry's int8 network evaluation on one MI355X.

A step is one forward of the 28-block d512 int8 network (27 int8 blocks + the fp16 last, the reference's semantics at
the benchmark's sizes) over a batch of synthetic positions already on the GPU, replayed as a HIP graph as the engine's lanes
replay theirs. Prints ONE JSON line: positions/s at batch 1024 (value), batch-64 latency, the standalone GEMM and
attention configs, the roofline of the dominant kernel (timed with HIP events on the stream it runs on) and the CPU
baseline (the CPU oracle's fp32 forward, the reference's CPU path, on a bounded sample, on this host's cores).

python bench.py [--gpus 1] [--steps K] [--warmup W] [--batch 1024] [--sweep] [--no-cpu]
python bench.py --kernel-only      the dominant kernel and a plain copy alone, for rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE
python bench.py --pmc-summary DIR  reads those two runs' counter_collection.csv files and prints the HBM bytes per launch
python bench.py --network-only     eager forwards of the network at --batch (no graph, no timing), for rocprofv3 --pmc runs
                                   whose counters are summarised per kernel by --counter-summary DIR
python bench.py --trace-summary DIR  per-kernel durations of the graph replays in a rocprofv3 --kernel-trace run
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
for _path in (ROOT, ROOT / "chess-transformer_amd"):
    if str(_path) not in sys.path:
        sys.path.insert(0, str(_path))

INT8_PEAK_TOPS = 5000.0      # MI355X dense int8 MFMA, TOPS
FP16_PEAK_TFLOPS = 2500.0    # dense fp16/bf16 MFMA
HBM_PEAK_GBS = 8000.0
SETTINGS = {"d_model": 512, "num_layers": 28, "n_heads": 8, "kv_heads": 8, "mlp_hidden": 2048, "value_bins": 128, "position_templates": 8}
TOKENS = 70
# the GEMM's tiles (rows x outputs, waves, ring stages), as chess_int8_linear numbers them
GEMM_TILES = {1: "64x64, 4 waves, 4 stages", 2: "128x128, 4 waves, 4 stages", 3: "128x64, 4 waves, 4 stages", 4: "256x128, 8 waves, 3 stages",
              5: "128x128, 8 waves, 2 stages of 128 bytes", 6: "128x128, 8 waves, 3 stages", 7: "128x128, 4 waves, 3 stages", 8: "128x64, 4 waves, 3 stages",
              9: "128x64, 4 waves, 2 stages", 10: "256x64, 4 waves, 2 stages", 11: "128x128, 4 waves, 2 stages",
              12: "128x64, 4 waves, 2 stages of 128 bytes", 13: "128x128, 4 waves, 2 stages of 128 bytes", 14: "32x32, K split over 4 waves",
              15: "blocks of 32 rows, each wave's weights held in registers, 8 waves",
              16: "blocks of 16 rows, K split over 4 waves, each wave's weights held in registers, 8 waves"}
def gemm_kernel_name(tile: int) -> str:
    return {14: "split_kernel<int8>", 15: "resident_kernel<int8>", 16: "deep_kernel<int8>"}.get(tile, "gemm_kernel<int8>")


# HBM bytes per launch of the dominant kernel, from rocprofv3 FETCH_SIZE / WRITE_SIZE runs scaled by a plain copy's counters
TRAFFIC = ROOT / "profiles" / "gate_up_gemm_batch1024_traffic.json"
# the sources the gate_up kernel is built from: a traffic figure measured on other sources is not the kernel that runs
GEMM_SOURCES = ("chess_common.h", "lds_dma.h", "hadamard.h", "gemm.h", "gemm_tiles.h", "gemm_split.h", "gemm_resident.h", "gemm_deep.h",
                "gemm.hip", "gemm_i8_gated.hip")
COPY_BYTES = 1 << 29
MI355X_CUS = 256


def log(message: str) -> None:
    print(message, file=sys.stderr, flush=True)


def synthetic_model(settings: dict, seed: int = 0):
    """Random-init weights as the benchmark states them: linear weights and biases N(0, 0.02), norm gains 1 + N(0, 0.1), templates
    N(0, 0.5), square-feature table N(0, 0.1), the input mixed in (residual 0.8, input 0.5). Drawn with numpy's generator
    (PCG64, float32 normals), whose stream is the same on every machine, so that the GPU box builds the very network the
    committed expected outputs (tests/golden/) were computed for."""
    import numpy as np
    import torch
    from model.model import ChessTransformer
    rng = np.random.default_rng(seed)
    model = ChessTransformer(**settings).eval()
    normal = lambda parameter, std: torch.from_numpy(rng.standard_normal(tuple(parameter.shape), dtype=np.float32) * np.float32(std))
    with torch.no_grad():
        for name, parameter in model.named_parameters():
            if name.endswith("residual_scale"):
                parameter.fill_(0.8)
            elif name.endswith("input_scale"):
                parameter.fill_(0.5)
            elif name == "templates":
                parameter.copy_(normal(parameter, 0.5))
            elif name == "square_features.table":
                parameter.copy_(normal(parameter, 0.1))
            elif "norm" in name or name.startswith("ln") or ".ln" in name:
                parameter.copy_(1 + normal(parameter, 0.1))
            else:
                parameter.copy_(normal(parameter, 0.02))
    return model


POSITIONS = ROOT / "tests" / "golden" / "positions.npz"


def legal_boards(count: int, first: int = 0):
    """count seeded random legal positions (0-80 random legal plies from the start; tests/golden/positions.npz, 4,096 of them)
    from the first-th on, as int64 tokens [count, 70], wrapping round the fixture past its end."""
    import numpy as np
    import torch
    tokens = np.load(POSITIONS)["tokens"]
    return torch.from_numpy(tokens[(first + np.arange(count)) % len(tokens)].astype(np.int64))


class Graphed:
    """The network recorded as one HIP graph for a batch size, replayed on its own stream."""

    def __init__(self, network, batch: int, device):
        import torch
        self.stream = torch.cuda.Stream(device)
        self.boards = legal_boards(batch).to(device)
        self.stream.wait_stream(torch.cuda.current_stream(device))
        with torch.cuda.stream(self.stream), torch.no_grad():
            for _ in range(2):
                network(self.boards)
        torch.cuda.synchronize(device)
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=self.stream), torch.no_grad():
            self.outputs = network(self.boards)
        torch.cuda.synchronize(device)

    def replay(self):
        import torch
        with torch.cuda.stream(self.stream):
            self.graph.replay()


def time_graph(graphed: Graphed, steps: int, warmup: int) -> tuple[float, list[float]]:
    """(ms per step over the timed region, per-replay ms)."""
    import torch
    for _ in range(warmup):
        graphed.replay()
    torch.cuda.synchronize()
    events = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(steps)]
    start = time.perf_counter()
    for begin, end in events:
        begin.record(graphed.stream)
        graphed.replay()
        end.record(graphed.stream)
    torch.cuda.synchronize()
    total = (time.perf_counter() - start) * 1e3
    return total / steps, [begin.elapsed_time(end) for begin, end in events]


def time_kernel(launch, repeats: int = 30) -> float:
    """Average ms of one launch, by HIP events on the current stream (the one the kernels launch on)."""
    import torch
    for _ in range(3):
        launch()
    stream = torch.cuda.current_stream()
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    begin.record(stream)
    for _ in range(repeats):
        launch()
    end.record(stream)
    torch.cuda.synchronize()
    return begin.elapsed_time(end) / repeats


def time_graphed(launch, repeats: int = 30, replays: int = 5) -> float:
    """Average ms of one launch, from a HIP graph of `repeats` launches replayed `replays` times (HIP events around the
    replays on the capturing stream): the kernel's own time, without the host's launch overhead between eager launches."""
    import torch
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(3):
            launch()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for _ in range(repeats):
            launch()
    torch.cuda.synchronize()
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    with torch.cuda.stream(stream):
        graph.replay()
        begin.record(stream)
        for _ in range(replays):
            graph.replay()
        end.record(stream)
    torch.cuda.synchronize()
    return begin.elapsed_time(end) / (repeats * replays)


def gemm_case(M: int, K: int, N: int, gated: bool, device, out_dtype=None, epilogue="bias"):
    """config 1: A int8 uniform in [-127, 127], W int8 rounded from N(0, 0.02), f32 scales, bias, bf16 (or fp16) out."""
    import torch
    from model.int8_blocks import launch_int8_linear
    from engine.quantization import nearest
    generator = torch.Generator(device=device).manual_seed(M + K + N)
    x = torch.randint(-127, 128, (M, K), device=device, dtype=torch.int8, generator=generator)
    x_scale = torch.rand(M, device=device, generator=generator) / 100
    weight, weight_scale = nearest(torch.randn(2 * N if gated else N, K, device=device, generator=generator) * 0.02)
    weight, weight_scale = weight.to(device), weight_scale.to(device)
    bias = (torch.randn(N, device=device, generator=generator) * 0.02).half() if epilogue == "bias" and not gated else None
    out_dtype = out_dtype or torch.float16
    return lambda: launch_int8_linear(x, x_scale, weight, weight_scale, bias, None, gated, None, None, None, 0, out_dtype)


def gemm_bytes(M: int, K: int, N: int, gated: bool, out_bytes: int = 2) -> int:
    rows = 2 * N if gated else N
    return M * K + rows * K + 4 * M + 4 * rows + 2 * N + out_bytes * M * N


def standalone_gemms(device) -> dict:
    """benchmark config 1: the four per-layer shapes at M = 4096, 16384, 65536 with bf16 out, each a graph of 30 launches."""
    import torch
    results = {}
    for M in (4096, 16384, 65536):
        for name, K, N in (("qkv", 512, 1536), ("attention_out", 512, 512), ("ffn_up", 512, 2048), ("ffn_down", 2048, 512)):
            ms = time_graphed(gemm_case(M, K, N, False, device, torch.bfloat16))
            tops = 2 * M * N * K / ms / 1e9
            gbs = gemm_bytes(M, K, N, False) / ms / 1e6
            attainable = min(INT8_PEAK_TOPS, 2 * M * N * K / gemm_bytes(M, K, N, False) * HBM_PEAK_GBS / 1e3)
            results[f"{name}_M{M}"] = {"ms": round(ms, 4), "tops": round(tops, 1), "frac_of_int8_peak": round(tops / INT8_PEAK_TOPS, 4),
                                       "frac_of_attainable": round(tops / attainable, 4), "gb_per_s": round(gbs, 1)}
    return results


def standalone_attention(device) -> dict:
    """benchmark config 2: 4096 positions x 8 heads x 64 wide over 64 tokens, a learned 64 x 64 bias per head (one-hot template mix),
    bf16 Q/K/V and output as the config asks (and the network's fp16 beside it)."""
    import torch
    from model.fused_blocks import template_attention
    B, T, H, d = 4096, 64, 8, 64
    generator = torch.Generator(device=device).manual_seed(2)
    projected = torch.randn(B, T, 3 * H * d + H * H, device=device, generator=generator).half()
    mix = projected[..., 3 * H * d:].reshape(B, T, H, H)
    mix.zero_()
    mix[..., torch.arange(H), torch.arange(H)] = 1.0
    templates = (torch.randn(H, 64, 64, device=device, generator=generator) * 0.5).half()
    gains = torch.ones(d, device=device).half()
    moved = projected.numel() * 2 + B * T * H * d * 2 + templates.numel() * 2
    rows_bf16 = projected.bfloat16()
    ms = time_graphed(lambda: template_attention(rows_bf16, templates, gains, gains, H, H, d, d, H, 1e-5))
    ms_fp16 = time_graphed(lambda: template_attention(projected, templates, gains, gains, H, H, d, d, H, 1e-5))
    return {"dtype": "bf16", "ms": round(ms, 4), "gb_per_s": round(moved / ms / 1e6, 1), "frac_of_hbm": round(moved / ms / 1e6 / HBM_PEAK_GBS, 4),
            "bytes": moved, "positions": B, "fp16_ms": round(ms_fp16, 4)}


def gate_up_case(device, batch: int, weight=None, weight_scale=None):
    """The dominant kernel at the network's shape: the gated gate_up GEMM of an int8 block (2 x 2048 weight rows, depth 512) over the
    batch's rows, with the tile the network picks; returns (launch, rows, tile)."""
    import torch
    from engine.quantization import nearest
    from model.int8_blocks import int8_tile, launch_int8_linear
    M = batch * TOKENS
    generator = torch.Generator(device=device).manual_seed(5)
    # activations as norm_quant leaves them: a normal row quantised to 127 at its absmax
    y = torch.randn(M, 512, device=device, generator=generator)
    absmax = y.abs().amax(dim=1, keepdim=True)
    x = torch.round(y * (127 / absmax)).to(torch.int8)
    x_scale = (absmax[:, 0] / 127).float()
    if weight is None:
        weight, weight_scale = nearest(torch.randn(2 * 2048, 512, device=device, generator=generator) * 0.02)
        weight, weight_scale = weight.to(device), weight_scale.to(device)
    tile = int8_tile(device, "gate_up", M)
    return (lambda: launch_int8_linear(x, x_scale, weight, weight_scale, None, None, True, None, None, None, tile)), M, tile


def in_network_launches(network, batch: int, device, passes: int = 4) -> list[float]:
    """ms of every gate_up launch inside forwards of the whole network: HIP events recorded on the launching stream just before
    and after each gated int8_linear, over eager forwards (the GPU runs behind the host at this batch, so each pair brackets the
    kernel alone; torch records no timing events into a graph on ROCm)."""
    import torch
    from model import int8_blocks
    original, with_maxima = int8_blocks.launch_int8_linear, int8_blocks.gated_int8_linear_absmax
    pairs = []

    def bracketed(launch, *args, **kwargs):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        out = launch(*args, **kwargs)
        end.record()
        pairs.append((begin, end))
        return out

    def timed(*args, **kwargs):   # int8_linear's gated launches (the blocks that keep rotate_quant apart)
        return bracketed(original, *args, **kwargs) if args[6] else original(*args, **kwargs)

    boards = legal_boards(batch).to(device)
    with torch.no_grad():
        network(boards)
        torch.cuda.synchronize(device)
        int8_blocks.launch_int8_linear = timed
        int8_blocks.gated_int8_linear_absmax = lambda *args: bracketed(with_maxima, *args)   # and the blocks that fold it into down
        try:
            for _ in range(passes):
                network(boards)
        finally:
            int8_blocks.launch_int8_linear, int8_blocks.gated_int8_linear_absmax = original, with_maxima
        torch.cuda.synchronize(device)
    return [begin.elapsed_time(end) for begin, end in pairs]


PARITY_FIXTURE = ROOT / "tests" / "golden" / "network_d512x28.npz"


def fixture_parity(network, device) -> dict | None:
    """The benchmarked network (seed 0, bench.py's own) on the 1,024 legal positions whose float64 oracle outputs the test
    fixture holds: the north star's bars measured in the same run (logits within 2e-2, value within 5e-3, argmax the same on
    at least 99.9% of the positions), as numbers."""
    import numpy as np
    import torch
    from model.model import expected_score
    if not PARITY_FIXTURE.exists():
        return None
    data = np.load(PARITY_FIXTURE)
    boards = torch.from_numpy(data["boards"].astype(np.int64))
    with torch.no_grad():
        rows = network(boards.to(device)).float().cpu()
    expected = torch.from_numpy(data["logits"])
    scores = expected_score(torch.from_numpy(data["value_logits"]))
    flips = int((rows[:, :-1].argmax(-1) != expected.argmax(-1)).sum())
    return {"positions": len(boards), "argmax_agreement": round(1 - flips / len(boards), 5), "flips": flips, "argmax_bar": 0.999,
            "max_logit_difference": float((rows[:, :-1] - expected).abs().max()), "logit_bar": 2e-2,
            "max_value_difference": float((rows[:, -1] - scores).abs().max()), "value_bar": 5e-3}


def dominant_kernel(device, network, batch: int) -> dict:
    """The gated gate_up GEMM, timed where it runs: its launches inside the network's graph replays. The same kernel launched
    alone back to back is timed too ("standalone_launch_ms"); that figure runs slower, as its input is no longer in the
    memory-side cache the preceding norm_quant left it in and 30 heavy launches in a row lower the clock."""
    block = network.encoder[0]
    launch, M, tile = gate_up_case(device, batch, block.gate_up, block.gate_up_scale)
    standalone_ms = time_kernel(launch)
    durations = in_network_launches(network, batch, device)
    ms = sum(durations) / len(durations)
    ops = 2 * M * (2 * 2048) * 512
    achieved = ops / ms / 1e9
    traffic = json.loads(TRAFFIC.read_text()) if TRAFFIC.exists() else None
    if traffic is not None and (traffic.get("rows") != M or traffic.get("tile") != tile or traffic.get("source_sha") != gemm_source_hash()):
        traffic = None   # measured on another kernel
    return {"kernel": f"{gemm_kernel_name(tile)} tile {tile} ({GEMM_TILES[tile]}), gate_up with the gated SiLU epilogue", "bound": "mfma",
            "achieved": round(achieved, 1), "peak": INT8_PEAK_TOPS, "unit": "TOPS", "frac": round(achieved / INT8_PEAK_TOPS, 4),
            "traffic": traffic["hbm_bytes"] if traffic else None, "ops_per_launch": ops, "avg_launch_ms": round(ms, 4),
            "launches_timed": len(durations), "standalone_launch_ms": round(standalone_ms, 4), "rows": M,
            "algorithmic_bytes": M * 512 + 4096 * 512 + 4 * M + 4 * 4096 + 2 * M * 2048}


def gemm_source_hash() -> str:
    """sha256 (first 16 hex digits) of the gate_up kernel's sources, which the traffic figure is keyed on."""
    import hashlib
    digest = hashlib.sha256()
    for name in GEMM_SOURCES:
        digest.update((ROOT / "chess-transformer_amd" / "csrc" / name).read_bytes())
    return digest.hexdigest()[:16]


def kernel_only(batch: int, repeats: int = 20) -> int:
    """The dominant kernel and a copy of COPY_BYTES alone, for counter runs: the copy's FETCH_SIZE / WRITE_SIZE give the
    counters' scale."""
    import torch
    device = torch.device("cuda", 0)
    launch, M, tile = gate_up_case(device, batch)
    source = torch.empty(COPY_BYTES, device=device, dtype=torch.uint8).random_(0, 255)
    target = torch.empty_like(source)
    for _ in range(repeats):
        launch()
        target.copy_(source)
    torch.cuda.synchronize()
    log(f"kernel-only: {repeats} launches of gate_up tile {tile} over {M} rows and {repeats} copies of {COPY_BYTES} bytes")
    return 0


def network_only(batch: int, passes: int = 2) -> int:
    """Eager forwards of the d512 x 28 network at batch (one untimed, then passes), for rocprofv3 --pmc runs: every kernel of a
    forward is a dispatch of its own, so the counters come per kernel. A copy of COPY_BYTES follows, for FETCH_SIZE / WRITE_SIZE's
    scale."""
    import torch
    from engine.inference import int8_network
    from engine.quantization import nearest_int8_weights
    device = torch.device("cuda", 0)
    torch.cuda.set_device(device)
    model = synthetic_model(SETTINGS)
    network = int8_network(model.to(device), nearest_int8_weights(model), fused_heads=True)
    boards = legal_boards(batch).to(device)
    with torch.no_grad():
        for _ in range(1 + passes):
            network(boards)
    source = torch.empty(COPY_BYTES, device=device, dtype=torch.uint8).random_(0, 255)
    torch.empty_like(source).copy_(source)
    torch.cuda.synchronize()
    log(f"network-only: {1 + passes} eager forwards at batch {batch}, then a copy of {COPY_BYTES} bytes")
    return 0


def kernel_role(name: str) -> str:
    """The network's part a kernel plays, from its (mangled) name: the GEMM's template arguments tell the int8 matmuls apart by
    their operand type, weight row groups (2: gated) and epilogue flags."""
    import re
    if "gemm_kernel" in name or "split_kernel" in name:
        found = re.search(r"(?:gemm|split)_kernelI(a|DF16_)?((?:Li\d+E)+)(DF16_|DF16b|f|i)?Lb(\d)ELi(n?\d+)E", name)
        numbers = [int(v) for v in re.findall(r"Li(\d+)E", found.group(2))] if found else []
        if "split_kernel" in name:
            found = re.search(r"split_kernelI((?:Li\d+E)+)(DF16_|DF16b|i)Li(n?\d+)E", name)
            numbers = [int(v) for v in re.findall(r"Li(\d+)E", found.group(1))] if found else []
            nb, epilogue = (numbers[2] if len(numbers) > 2 else 1), (found.group(3) if found else "?")
            return {"2": "down (split-K)", "6": "down (split-K)", "1": "projection (split-K)"}.get(epilogue, "gate_up (split-K)" if nb == 2 else "int8 split-K")
        if not found:
            return "gemm"
        int8 = found.group(1) == "a"
        nb = numbers[4] if len(numbers) > 4 else 1
        epilogue = found.group(5)
        out = found.group(3)
        if int8:
            if nb == 2:
                return "gate_up (int8, gated, rotated block maxima)" if epilogue == "8" else "gate_up (int8, gated)"
            return {"1": "projection (int8)", "2": "down (int8)", "6": "down (int8, mixes the next input)"}.get(epilogue, "int8 gemm")
        if out == "f":
            return "policy head a (fp16, f32 out)"
        if nb == 2:
            return "fp16 block gate_up"
        return {"3": "combine (fp16, bias + residual)", "1": "fp16 block projection", "2": "fp16 block down",
                "6": "fp16 block down (mix)"}.get(epilogue, "fp16 gemm")
    if "resident_kernel" in name:   # template arguments In, NB, OutT, EPI, depth
        found = re.search(r"resident_kernelI(a|DF16_)Li(\d)E(?:DF16_|DF16b)Li(\d)E", name)
        if found and found.group(1) == "DF16_":
            return "fp16 block projection (weights in registers)" if found.group(3) == "1" else "combine (fp16, bias + residual, weights in registers)"
        if found and found.group(2) == "2":
            return "gate_up (int8, gated, weights in registers)"
        return {"2": "down (int8, weights in registers)", "6": "down (int8, mixes the next input, weights in registers)"}.get(
            found.group(3) if found else "", "projection (int8, weights in registers)")
    if "deep_kernel" in name:   # template arguments OutT, EPI
        found = re.search(r"deep_kernelI(?:DF16_|DF16b)Li(\d)E", name)
        return "down (int8, mixes the next input, weights in registers)" if found and found.group(1) == "6" else "down (int8, weights in registers)"
    if "rotated_kernel" in name:
        found = re.search(r"rotated_kernelILi\d+ELi\d+ELi\d+ELi\d+ELi(n?\d+)E", name)
        return "down (int8, rotation folded in, mixes the next input)" if found and found.group(1) == "6" else "down (int8, rotation folded in)"
    found = re.search(r"norm_quant_kernelILi\d+ELi\d+ELi\d+ELb\dELb(\d)", name)
    if found:   # template arguments C, LANES, R, VECTOR, QUANT, FULL: without QUANT it is the fp16 blocks' RMSNorm
        return "norm_quant" if found.group(1) == "1" else "rms_norm (fp16 block, final norm)"
    for key, role in (("norm_quant_kernel", "norm_quant"), ("rotate_quant", "rotate_quant"), ("template_attention", "template_attention"),
                      ("board_embedding", "board_embedding"), ("head_blocks", "move logits: product blocks"), ("head_gather", "move logits: gather"),
                      ("move_logits", "move_logits"), ("value_hidden", "value_hidden"),
                      ("value_score", "value_score"), ("copy", "copy")):
        if key in name:
            return role
    return name.split("<")[0][:60]


def counter_summary(folder: Path) -> int:
    """Per kernel role, the average per dispatch of every counter in the rocprofv3 --pmc runs under folder (their
    counter_collection.csv files), as a markdown table, with derived figures. GRBM_GUI_ACTIVE is summed over the 8 XCDs, so a
    dispatch's cycles are GRBM_GUI_ACTIVE / 8. From those: int8 MFMA % = 512 SQ_INSTS_VALU_MFMA_MOPS_I8 over the dense peak at
    the running clock (256 CUs x 4 SIMDs x 2,048 ops a cycle); MFMA busy % = SQ_VALU_MFMA_BUSY_CYCLES / (cycles x 1,024 SIMDs);
    VALU busy % = 4 SQ_ACTIVE_INST_VALU / (cycles x 1,024) (the SQ's wave counters count 4-cycle units); co-exec % = the MFMA
    busy cycles that VALU work overlaps; L2 requests a cycle a channel (128 channels); per wavefront, its VALU and MFMA
    instructions and its cycles spent waiting."""
    import csv
    values: dict[str, dict[str, list[float]]] = {}
    for path in sorted(folder.rglob("*counter_collection.csv")):
        rows = list(csv.DictReader(path.open()))
        number = "Dispatch_Id" if rows and "Dispatch_Id" in rows[0] else "Correlation_Id"
        # the forwards' dispatches only (from the first input embedding on), not the network's set-up on the GPU
        embeddings = [int(row[number]) for row in rows if kernel_role(row["Kernel_Name"]) == "board_embedding"]
        first = min(embeddings) if embeddings else 0
        for row in rows:
            if int(row[number]) >= first:
                values.setdefault(kernel_role(row["Kernel_Name"]), {}).setdefault(row["Counter_Name"], []).append(float(row["Counter_Value"]))
    columns = ["dispatch cycles", "int8 MFMA % of peak", "MFMA busy %", "VALU busy %", "MFMA co-exec with VALU %",
               "L2 requests /cycle/channel", "L2 hit %", "TA busy %", "VALU instr /wave", "MFMA instr /wave", "transcendental /wave",
               "waiting cycles /wave", "wave cycles /wave", "LDS instr /wave", "LDS bank conflict cycles /wave", "FETCH_SIZE KiB", "WRITE_SIZE KiB"]
    print("| kernel | dispatches | " + " | ".join(columns) + " |")
    print("|---|---|" + "---|" * len(columns))
    for role in sorted(values):
        mean = {counter: sum(v) / len(v) for counter, v in values[role].items()}
        dispatches = max(len(v) for v in values[role].values())
        cycles = mean.get("GRBM_GUI_ACTIVE", 0) / 8
        waves = mean.get("SQ_WAVES")

        def ratio(top, bottom, scale=1.0, digits=1):
            return f"{scale * top / bottom:,.{digits}f}" if top is not None and bottom else ""
        cells = [f"{cycles:,.0f}" if cycles else "",
                 ratio(mean.get("SQ_INSTS_VALU_MFMA_MOPS_I8"), cycles * 2097152, 512 * 100),
                 ratio(mean.get("SQ_VALU_MFMA_BUSY_CYCLES"), cycles * 1024, 100),
                 ratio(mean.get("SQ_ACTIVE_INST_VALU"), cycles * 1024, 400),
                 ratio(mean.get("SQ_VALU_MFMA_COEXEC_CYCLES"), mean.get("SQ_VALU_MFMA_BUSY_CYCLES"), 100),
                 ratio(mean.get("TCC_REQ_sum"), cycles * 128, 1, 2),
                 ratio(mean.get("TCC_HIT_sum"), (mean.get("TCC_HIT_sum") or 0) + (mean.get("TCC_MISS_sum") or 0), 100),
                 ratio(mean.get("TA_BUSY_avr"), cycles, 100),
                 ratio(mean.get("SQ_INSTS_VALU"), waves, 1, 0), ratio(mean.get("SQ_INSTS_MFMA"), waves, 1, 0),
                 ratio(mean.get("SQ_INSTS_VALU_TRANS_F32"), waves, 1, 0), ratio(mean.get("SQ_WAIT_ANY"), waves, 4, 0),
                 ratio(mean.get("SQ_WAVE_CYCLES"), waves, 4, 0), ratio(mean.get("SQ_INSTS_LDS"), waves, 1, 0),
                 ratio(mean.get("SQ_LDS_BANK_CONFLICT"), waves, 1, 0),
                 f"{mean['FETCH_SIZE']:,.0f}" if "FETCH_SIZE" in mean else "", f"{mean['WRITE_SIZE']:,.0f}" if "WRITE_SIZE" in mean else ""]
        print(f"| {role} | {dispatches} | " + " | ".join(cells) + " |")
    return 0


def trace_summary(folder: Path) -> int:
    """Per kernel role, the average duration and the time a forward, over the graph replays in the rocprofv3 --kernel-trace
    run under folder (its kernel_trace.csv): a forward starts at the input embedding's launch, and the replays are the
    forwards that run without gaps (the eager forwards of the roofline timing have host gaps between their launches)."""
    import csv
    rows = []
    for path in sorted(folder.rglob("*kernel_trace.csv")):
        rows += list(csv.DictReader(path.open()))
    rows.sort(key=lambda row: int(row["Start_Timestamp"]))
    starts = [i for i, row in enumerate(rows) if kernel_role(row["Kernel_Name"]) == "board_embedding"] + [len(rows)]
    forwards = []
    for first, end in zip(starts, starts[1:]):
        span = int(rows[end - 1]["End_Timestamp"]) - int(rows[first]["Start_Timestamp"])
        busy = sum(int(row["End_Timestamp"]) - int(row["Start_Timestamp"]) for row in rows[first:end])
        if busy >= 0.95 * span:
            forwards.append(rows[first:end])
    if not forwards:
        print("no graph replays found")
        return 1
    durations: dict[str, list[float]] = {}
    shapes: dict[str, str] = {}
    for forward in forwards:
        for row in forward:
            role = kernel_role(row["Kernel_Name"])
            durations.setdefault(role, []).append((int(row["End_Timestamp"]) - int(row["Start_Timestamp"])) / 1e3)
            shapes[role] = f"{int(row['Grid_Size_X']) // int(row['Workgroup_Size_X'])} x {row['Workgroup_Size_X']}"
    spans = [(int(f[-1]["End_Timestamp"]) - int(f[0]["Start_Timestamp"])) / 1e3 for f in forwards]
    total = sum(spans) / len(spans)
    print(f"{len(forwards)} graph replays, {len(forwards[0])} launches and {total:,.1f} us a forward\n")
    print("| kernel | workgroups x threads | launches a forward | average us | us a forward | share |")
    print("|---|---|---|---|---|---|")
    for role, values in sorted(durations.items(), key=lambda item: -sum(item[1])):
        each = sum(values) / len(values)
        per_forward = sum(values) / len(forwards)
        print(f"| {role} | {shapes[role]} | {len(values) // len(forwards)} | {each:,.1f} | {per_forward:,.1f} | {per_forward / total:.1%} |")
    return 0


def pmc_summary(folder: Path, batch: int) -> int:
    """HBM bytes per launch of the dominant kernel from two rocprofv3 --pmc runs (FETCH_SIZE, WRITE_SIZE, KiB per dispatch), each
    scaled by what the counter reads for the copy of COPY_BYTES."""
    import csv
    from model.fused_blocks import tile_for
    from model.int8_blocks import INT8_TILES
    values: dict[str, dict[str, list[float]]] = {}
    for path in sorted(folder.rglob("*counter_collection.csv")):
        for row in csv.DictReader(path.open()):
            values.setdefault(row["Counter_Name"], {}).setdefault(row["Kernel_Name"], []).append(float(row["Counter_Value"]))
    mean = {}
    for counter, kernels in values.items():
        averages = {name: sum(v) / len(v) for name, v in kernels.items()}
        # the copy of COPY_BYTES is the largest copy the run makes; the GEMM is the only GEMM kernel
        copies = [name for name in averages if "copy" in name.lower()]
        gemms = [name for name in averages if "gemm_kernel" in name or "resident_kernel" in name]
        mean[counter] = {"copy": max(averages[name] for name in copies), "gemm": averages[gemms[0]]}
    fetch_scale = COPY_BYTES / (mean["FETCH_SIZE"]["copy"] * 1024)
    write_scale = COPY_BYTES / (mean["WRITE_SIZE"]["copy"] * 1024)
    fetch = mean["FETCH_SIZE"]["gemm"] * 1024 * fetch_scale
    write = mean["WRITE_SIZE"]["gemm"] * 1024 * write_scale
    M = batch * TOKENS
    tile = tile_for(INT8_TILES["gfx950"]["gate_up"], M, MI355X_CUS)
    result = {"rows": M, "tile": tile, "source_sha": gemm_source_hash(), "hbm_bytes": round(fetch + write), "fetch_bytes": round(fetch), "write_bytes": round(write),
              "fetch_kib_raw": mean["FETCH_SIZE"]["gemm"], "write_kib_raw": mean["WRITE_SIZE"]["gemm"],
              "copy_fetch_kib": mean["FETCH_SIZE"]["copy"], "copy_write_kib": mean["WRITE_SIZE"]["copy"],
              "fetch_scale": round(fetch_scale, 4), "write_scale": round(write_scale, 4),
              "algorithmic_bytes": M * 512 + 4096 * 512 + 4 * M + 4 * 4096 + 2 * M * 2048,
              "kernel": f"{gemm_kernel_name(tile)} tile {tile} ({GEMM_TILES[tile]}), gate_up with the gated SiLU epilogue: {M:,} x 512 int8 by "
                        "4,096 x 512 int8 -> {M:,} x 2,048 fp16".replace("{M:,}", f"{M:,}"),
              "commands": [f"cd /tmp && timeout -s KILL 180 rocprofv3 --pmc {counter} --output-format csv -d $R/gpurun_out/pmc/{counter.lower()} "
                           f"-o {counter.lower()} -- python3 $R/bench.py --kernel-only" for counter in ("FETCH_SIZE", "WRITE_SIZE")]
                          + ["cd $R && python3 bench.py --pmc-summary gpurun_out/pmc"],
              "scaling": f"FETCH_SIZE and WRITE_SIZE are KiB per dispatch; a copy of {COPY_BYTES:,} bytes reads "
                         f"{mean['FETCH_SIZE']['copy']:,.0f} KiB on FETCH_SIZE (x{fetch_scale:.4f} to bytes) and "
                         f"{mean['WRITE_SIZE']['copy']:,.0f} KiB on WRITE_SIZE (x{write_scale:.4f})"}
    print(json.dumps(result, indent=1))
    return 0


CONFIG0 = {"d_model": 256, "num_layers": 4, "n_heads": 8, "kv_heads": 8, "mlp_hidden": 1024, "value_bins": 128, "position_templates": 8}


def usable_cpus() -> int:
    """The CPUs this process may run on: its affinity set, within the container's CPU quota (cgroup v2 cpu.max) if it has one."""
    count = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    try:
        quota, period = Path("/sys/fs/cgroup/cpu.max").read_text().split()[:2]
        if quota != "max":
            count = min(count, max(1, int(quota) // int(period)))
    except (OSError, ValueError):
        pass
    return count


def time_cpu_forward(state: dict, settings: dict, batch: int, threads: int, runs: int, warmups: int) -> dict:
    """p50 / p99 ms of the CPU forward of batch legal positions (oracle/network.py fp32_forward: the reference's CPU path,
    model/model.py:245-270, as engine/inference.py:274-278 serves it) on threads torch threads, over runs after warmups."""
    import torch
    from oracle import network as oracle_network
    torch.set_num_threads(threads)
    boards = legal_boards(batch, 1024)
    for _ in range(warmups):
        oracle_network.fp32_forward(state, settings, boards)
    times = []
    for _ in range(runs):
        start = time.perf_counter()
        oracle_network.fp32_forward(state, settings, boards)
        times.append((time.perf_counter() - start) * 1e3)
    times.sort()
    p50, p99 = times[len(times) // 2], times[min(len(times) - 1, math.ceil(0.99 * len(times)) - 1)]
    return {"batch": batch, "threads": threads, "runs": runs, "warmups": warmups, "p50_ms": round(p50, 2), "p99_ms": round(p99, 2),
            "positions_per_s": round(batch / p50 * 1e3, 2)}


def cpu_baseline(model_state: dict, runs: int = 20, warmups: int = 3) -> dict:
    """The CPU baseline: the fp32 CPU forward of config 0 (d256 x 4, batch 64) and config 3 (the d512 x
    28 network, batch 64), p50 and p99 over runs after warmups, on every CPU this process may use and on one thread (the
    engine's own setting, reference engine/uci.py:557). The one-thread d512 x 28 figure takes batches of 8 (a forward of 64
    takes about 15 s on one core), still 20 runs. value: config 3 on all usable threads, positions/s at the p50."""
    import torch
    threads = usable_cpus()
    config0 = synthetic_model(CONFIG0, 1)
    config0_state = {name: value.clone() for name, value in config0.state_dict().items()}
    results = {"config0_all_threads": time_cpu_forward(config0_state, CONFIG0, 64, threads, runs, warmups),
               "config0_one_thread": time_cpu_forward(config0_state, CONFIG0, 64, 1, runs, warmups),
               "config3_all_threads": time_cpu_forward(model_state, SETTINGS, 64, threads, runs, warmups),
               "config3_one_thread": time_cpu_forward(model_state, SETTINGS, 8, 1, runs, warmups)}
    torch.set_num_threads(threads)
    headline = results["config3_all_threads"]
    return {"value": headline["positions_per_s"], "unit": "positions/s", "cores": threads, "kind": "port",
            "sample": f"config 3: the d512 x 28 network's fp32 CPU forward (oracle/network.py fp32_forward, torch CPU) of 64 seeded legal "
                      f"positions, p50 of {runs} runs after {warmups} warm-ups, {threads} threads",
            "host_cpus": os.cpu_count(), "usable_cpus": threads, **results}


def main() -> int:
    parser = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    parser.add_argument("--gpus", type=int, default=1)
    parser.add_argument("--steps", type=int, default=50)
    parser.add_argument("--warmup", type=int, default=5)
    parser.add_argument("--batch", type=int, default=1024)
    parser.add_argument("--latency-batch", type=int, default=64)
    parser.add_argument("--sweep", action="store_true", help="also time batches 1, 16, 64, 256, 1024, 4096")
    parser.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    parser.add_argument("--cpu-runs", type=int, default=20, help="timed CPU forwards per configuration (after 3 warm-ups)")
    parser.add_argument("--no-standalone", action="store_true", help="skip the standalone GEMM and attention configs")
    parser.add_argument("--kernel-only", action="store_true", help="run only the dominant kernel and a copy, for counter runs")
    parser.add_argument("--pmc-summary", type=Path, help="summarise the FETCH_SIZE / WRITE_SIZE runs under this folder")
    parser.add_argument("--network-only", action="store_true", help="eager forwards of the network at --batch, for counter runs")
    parser.add_argument("--counter-summary", type=Path, help="per-kernel table of the counter runs under this folder")
    parser.add_argument("--trace-summary", type=Path, help="per-kernel table of the graph replays in the kernel trace under this folder")
    arguments = parser.parse_args()
    if arguments.pmc_summary:
        return pmc_summary(arguments.pmc_summary, arguments.batch)
    if arguments.counter_summary:
        return counter_summary(arguments.counter_summary)
    if arguments.trace_summary:
        return trace_summary(arguments.trace_summary)
    if arguments.gpus != 1:
        print(f"bench.py measures one GPU: every box here has one and nothing in this build uses a second (asked for {arguments.gpus})",
              file=sys.stderr)
        return 2
    if arguments.kernel_only:
        return kernel_only(arguments.batch)
    if arguments.network_only:
        return network_only(arguments.batch)

    import torch
    from engine.inference import int8_network
    from engine.quantization import nearest_int8_weights

    device = torch.device("cuda", 0)
    torch.cuda.set_device(device)
    log(f"building the d512 x 28 int8 network on {torch.cuda.get_device_name(device)}")
    model = synthetic_model(SETTINGS)
    state = {name: value.clone() for name, value in model.state_dict().items()}
    weights = nearest_int8_weights(model)
    network = int8_network(model.to(device), weights, fused_heads=True)   # the answer rows the graph lanes copy out

    log(f"batch {arguments.batch}: recording and timing {arguments.steps} steps after {arguments.warmup} warm-up")
    graphed = Graphed(network, arguments.batch, device)
    ms_per_step, per_replay = time_graph(graphed, arguments.steps, arguments.warmup)
    positions_per_s = arguments.batch / (ms_per_step / 1e3)
    log(f"  {ms_per_step:.3f} ms/step, {positions_per_s:,.0f} positions/s")
    del graphed

    latency = None
    if arguments.latency_batch > 0:
        log(f"batch {arguments.latency_batch}: latency over 200 replays")
        small = Graphed(network, arguments.latency_batch, device)
        _, latencies = time_graph(small, 200, 20)
        latencies.sort()
        p50, p99 = latencies[len(latencies) // 2], latencies[int(len(latencies) * 0.99) - 1]
        latency = {"batch": arguments.latency_batch, "p50_ms": round(p50, 4), "p99_ms": round(p99, 4),
                   "positions_per_s": round(arguments.latency_batch / (p50 / 1e3), 1)}
        log(f"  p50 {p50:.3f} ms, p99 {p99:.3f} ms")
        del small

    sweep = {}
    if arguments.sweep:
        for batch in (1, 16, 64, 256, 1024, 4096):
            graphed = Graphed(network, batch, device)
            ms, replays = time_graph(graphed, 200, 10)
            replays.sort()
            p50, p99 = replays[len(replays) // 2], replays[int(len(replays) * 0.99) - 1]
            sweep[batch] = {"ms_per_batch": round(ms, 4), "p50_ms": round(p50, 4), "p99_ms": round(p99, 4),
                            "positions_per_s": round(batch / ms * 1e3, 1)}
            log(f"  sweep batch {batch}: {ms:.3f} ms, p50 {p50:.3f} ms, p99 {p99:.3f} ms, {batch / ms * 1e3:,.0f} positions/s")
            del graphed

    parity = fixture_parity(network, device) if arguments.batch == 1024 else None
    if parity:
        log(f"parity on the {parity['positions']} fixture positions: argmax agreement {parity['argmax_agreement']} ({parity['flips']} flips), "
            f"logits {parity['max_logit_difference']:.2e} max, value {parity['max_value_difference']:.2e} max")

    roofline = dominant_kernel(device, network, arguments.batch)
    log(f"gate_up GEMM in the network: {roofline['avg_launch_ms']:.3f} ms over {roofline['launches_timed']} launches, "
        f"{roofline['achieved']:.0f} TOPS ({roofline['frac']:.1%} of dense int8 peak); alone {roofline['standalone_launch_ms']:.3f} ms")

    standalone = {}
    if not arguments.no_standalone:
        standalone["gemm"] = standalone_gemms(device)
        standalone["attention"] = standalone_attention(device)
        log(f"standalone attention: {standalone['attention']['ms']} ms, {standalone['attention']['gb_per_s']} GB/s")

    baseline = None
    if not arguments.no_cpu:
        log(f"CPU baseline: fp32 forwards of configs 0 and 3, {arguments.cpu_runs} runs each on {usable_cpus()} threads and on one")
        baseline = cpu_baseline(state, arguments.cpu_runs)
        for name in ("config0_all_threads", "config0_one_thread", "config3_all_threads", "config3_one_thread"):
            run = baseline[name]
            log(f"  {name}: batch {run['batch']} on {run['threads']} threads, p50 {run['p50_ms']} ms, {run['positions_per_s']} positions/s")

    result = {"metric": "positions/sec at batch 1024 (28L int8 net)", "value": round(positions_per_s, 1), "unit": "positions/s", "n_gpus": 1,
              "steps": arguments.steps, "warmup": arguments.warmup, "ms_per_step": round(ms_per_step, 4), "higher_is_better": True,
              "scaling": "weak", "vs_baseline": None, "dtype": "int8",
              "data": "synthetic: random-init weights (N(0, 0.02)), round-to-nearest int8 per channel, seeded random legal positions "
                      "(tests/golden/positions.npz)",
              "config": {"workload": f"Fry int8 network d512 x 28 (27 int8 blocks + fp16 last), T=70, batch {arguments.batch}, HIP graph replay",
                         "batch": arguments.batch, "tokens": TOKENS, "d_model": 512, "layers": 28, "heads": 8, "mlp_hidden": 2048},
              "batch64": latency, "roofline": roofline, "cpu_baseline": baseline, "parity": parity, **standalone}
    if sweep:
        result["sweep"] = sweep
    print(json.dumps(result), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
