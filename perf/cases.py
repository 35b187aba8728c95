"""The work that a user has this framework do, as cases to measure: an engine's search calls through the graph lanes, the eager
forward, and the layers that both are made of, each through its public entry point.

Three networks stand for the range: d512 (8 heads of 64, hidden 2,048, 28 blocks, the benchmark's), d768 (24 query heads on 12
key/value heads, query width 16 and value width 32, hidden 992 padded to 1,024, 28 blocks: the attention and row shapes that the
operators' tests are written for) and d256 (8 heads of 32, hidden 1,024, 4 blocks: the benchmark's small network). Weights are
random and fixed; the seed makes the inputs. A network and its graphs are made once a process, as an engine makes them at its
start and keeps them."""
import functools
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "chess-transformer_amd"))

from engine.inference import GraphedBatches, fused_model, int8_network
from model.encoding import START_POSITION_TOKENS
from model.fused_blocks import template_attention
from model.int8_blocks import launch_int8_linear
from model.model import ChessTransformer

NETWORKS = {"d512": {"d_model": 512, "num_layers": 28, "n_heads": 8, "kv_heads": 8, "qk_ratio": 1.0, "mlp_hidden": 2048},
            "d768": {"d_model": 768, "num_layers": 28, "n_heads": 24, "kv_heads": 12, "qk_ratio": 0.5, "mlp_hidden": 992},
            "d256": {"d_model": 256, "num_layers": 4, "n_heads": 8, "kv_heads": 8, "qk_ratio": 1.0, "mlp_hidden": 1024}}
TOKENS, SQUARES, TEMPLATES, BINS, MOVES, VOCABULARY = 70, 64, 8, 128, 1968, 81
STREAM = 1 / 16          # the inference networks' residual stream is scaled by this
EPS = 1e-5
WEIGHT_SEED = 20
# the 23 square features' rows: four piece offsets, eight neighbours, eight lines, knights, two pawns
FEATURE_ROWS = [226] * 4 + [14] * 8 + [85] * 8 + [9] + [15] * 2


def listed():
    return [
        # one leaf, the smallest search call: nothing but latency, 230 launches in a graph
        {"name": "lane_d512_1", "kind": "lane", "network": "d512", "positions": 1},
        # a search's ordinary round of leaves
        {"name": "lane_d512_64", "kind": "lane", "network": "d512", "positions": 64},
        # an odd round on the grouped-query network: rows of 768, a hidden width that is padded
        {"name": "lane_d768_51", "kind": "lane", "network": "d768", "positions": 51},
        # throughput: self-play and scoring in bulk, the benchmark's batch
        {"name": "forward_d512_1024", "kind": "forward", "network": "d512", "positions": 1024},
        # one middle block of the int8 networks at the batch of several rounds, and at odd and large ones
        {"name": "int8_block_d512_256", "kind": "int8_block", "network": "d512", "positions": 256},
        {"name": "int8_block_d768_700", "kind": "int8_block", "network": "d768", "positions": 700},
        {"name": "int8_block_d256_999", "kind": "int8_block", "network": "d256", "positions": 999},
        # the fp16 network's block: the last of every int8 network, and all of those that calibrate one
        {"name": "fp16_block_d512_512", "kind": "fp16_block", "network": "d512", "positions": 512},
        # the benchmark's largest standalone product, bf16 out
        {"name": "linear_bf16_65536", "kind": "linear", "rows": 65536, "depth": 512, "outputs": 2048, "type": "bf16", "epilogue": "bias"},
        # the benchmark's standalone attention: bf16 rows over the 64 squares, a bias a head
        {"name": "attention_bf16_4096", "kind": "attention", "positions": 4096, "tokens": 64, "heads": 8, "kv_heads": 8, "query": 64, "value": 64,
         "type": "bf16"},
        # both ends of the network: the heads on their own, and the boards' embedding
        {"name": "heads_d512_300", "kind": "heads", "network": "d512", "positions": 300},
        {"name": "embedding_d512_1024", "kind": "embedding", "network": "d512", "positions": 1024},
    ]


def draw(rng):
    between = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    network = rng.choice(["d512", "d512", "d768", "d256"])
    kind = rng.choice(["lane", "lane", "forward", "int8_block", "int8_block", "fp16_block", "linear", "attention", "heads", "embedding"])
    if kind == "linear":
        depth, outputs = rng.choice([(512, 1536), (512, 512), (512, 2048), (2048, 512), (768, 1152), (1024, 768), (256, 1024)])
        return {"kind": kind, "rows": between(1000, 65536), "depth": depth, "outputs": outputs, "type": rng.choice(["bf16", "f16"]),
                "epilogue": rng.choice(["bias", "residual"])}
    if kind == "attention":
        heads, kv_heads, query, value = rng.choice([(8, 8, 64, 64), (8, 8, 32, 32), (24, 12, 8, 32), (24, 12, 16, 32), (24, 12, 24, 32), (4, 2, 16, 32)])
        return {"kind": kind, "positions": between(16, 4096), "tokens": rng.choice([64, 70, 70, 80]), "heads": heads, "kv_heads": kv_heads, "query": query,
                "value": value, "type": rng.choice(["bf16", "f16", "f16"])}
    most = {"lane": 256, "forward": 1000, "int8_block": 1500, "fp16_block": 1000, "heads": 1500, "embedding": 4000}[kind]
    least = {"lane": 1, "forward": 16}.get(kind, 64)
    return {"kind": kind, "network": network, "positions": between(least, most)}


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _layers(case):
    """A block's cases take the second of four: its input arrives mixed, and it mixes the next one's."""
    return 4 if case["kind"] in ("int8_block", "fp16_block") else NETWORKS[case["network"]]["num_layers"]


@functools.lru_cache(maxsize=8)
def _state(name, layers):
    """The fp32 network's state dict: N(0, 0.02), gains 1 + N(0, 0.1), templates N(0, 0.5), square features N(0, 0.1), the input mixed in."""
    s, generator, state = NETWORKS[name], _generator(WEIGHT_SEED), {}
    d, heads, kv, h = s["d_model"], s["n_heads"], s["kv_heads"], s["mlp_hidden"]
    value = d // heads
    query = round(s["qk_ratio"] * value)

    def normal(key, *shape, std=0.02, mean=0.0):
        state[key] = mean + std * torch.randn(*shape, device="cuda", generator=generator)

    def dense(key, outputs, inputs, bias=True):
        normal(key + ".weight", outputs, inputs)
        if bias:
            normal(key + ".bias", outputs)

    normal("embed.weight", VOCABULARY, d)
    normal("position_embed", TOKENS, d)
    normal("square_features.table", sum(FEATURE_ROWS), d, std=0.1)
    normal("templates", TEMPLATES, SQUARES, SQUARES, std=0.5)
    for i in range(layers):
        p = "encoder.%d." % i
        dense(p + "Q", heads * query, d)
        dense(p + "K", kv * query, d)
        dense(p + "V", kv * value, d)
        dense(p + "template_mix", TEMPLATES * heads, d)
        dense(p + "combine_heads", d, d)
        dense(p + "mlp.up_projection", h, d, bias=False)
        dense(p + "mlp.gate_projection", h, d, bias=False)
        dense(p + "mlp.down_projection", d, h, bias=False)
        for gain, width in (("q_norm", query), ("k_norm", query), ("ln1", d), ("ln2", d)):
            normal(p + gain + ".weight", width, std=0.1, mean=1.0)
        state[p + "residual_scale"] = torch.full((1,), 0.8, device="cuda")
        state[p + "input_scale"] = torch.full((1,), 0.5, device="cuda")
    normal("ln.weight", d, std=0.1, mean=1.0)
    for key, outputs, inputs in (("from_projection", d, d), ("to_projection", d, d), ("promotion_projection", 4, d), ("board_down_project.0", 16, d),
                                 ("eval_head.0", d, TOKENS * 16), ("eval_head.2", BINS, d)):
        dense(key, outputs, inputs)
    return state


def _nearest(weight):
    scale = weight.double().abs().amax(1) / 127
    return torch.round(weight.double() / scale[:, None]).to(torch.int8), scale.float()


def _hadamard(size=32):
    H = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    while len(H) < size:
        H = torch.cat([torch.cat([H, H], 1), torch.cat([H, -H], 1)])
    return H


@functools.lru_cache(maxsize=8)
def _int8_weights(name, layers):
    """Every block's but the last's three products, rounded to nearest: down's inputs are rotated in blocks of 32 (H / 32 undoes the
    rotation of the activations) and padded to a multiple of 128."""
    state, H, weights = _state(name, layers), _hadamard() / 32, {}
    for i in range(layers - 1):
        w = lambda key: state["encoder.%d.%s.weight" % (i, key)].double()
        down = w("mlp.down_projection")
        outputs, hidden = down.shape
        rotated = torch.zeros(outputs, -(-hidden // 128) * 128, dtype=torch.float64, device="cuda")
        rotated[:, :hidden] = (down.view(outputs, -1, 32) @ H).reshape(outputs, hidden)
        weights[i] = {"projection": _nearest(torch.cat([w("Q"), w("K"), w("V"), w("template_mix")])),
                      "gate_up": _nearest(torch.cat([w("mlp.gate_projection"), w("mlp.up_projection")])), "down": _nearest(rotated)}
    return weights


@functools.lru_cache(maxsize=8)
def _network(name, layers, int8=True):
    settings = dict(NETWORKS[name], num_layers=layers, value_bins=BINS, position_templates=TEMPLATES)
    with torch.device("cuda"):
        model = ChessTransformer(**settings).eval()
    model.load_state_dict({key: value.clone() for key, value in _state(name, layers).items()}, strict=False)
    model.requires_grad_(False)
    return int8_network(model, _int8_weights(name, layers)) if int8 else fused_model(model)


@functools.lru_cache(maxsize=16)
def _lanes(name, layers, positions):
    return GraphedBatches(_network(name, layers), [positions], in_flight=1)


def _boards(count, seed):
    """Positions as a game passes through them: some of the 32 men taken, the others on any free square, pawns off the end ranks."""
    rng, men = np.random.default_rng(seed), np.array(START_POSITION_TOKENS)
    boards = np.zeros((count, TOKENS), dtype=np.int64)
    for board in boards:
        left = [code for code in men[:SQUARES] if code in (6, 12) or (code and rng.random() < 0.75)]
        squares = rng.permutation(SQUARES)
        middle, ends = [s for s in squares if 8 <= s < 56], [s for s in squares if s < 8 or s >= 56]
        pawns = [code for code in left if code in (1, 7)]
        others = [code for code in left if code not in (1, 7)]
        for code in pawns:
            board[middle.pop()] = code
        free = rng.permutation(middle + ends)
        board[free[:len(others)]] = others
        board[SQUARES:TOKENS - 1] = men[SQUARES:TOKENS - 1] - rng.integers(0, 2, TOKENS - 1 - SQUARES)
        board[TOKENS - 1] = men[TOKENS - 1] + (rng.integers(0, SQUARES) if rng.random() < 0.1 else 0)
    return boards


def _stream(case, seed):
    """A block's two inputs: the residual stream and the input embedding, at the scaled stream's size."""
    d, generator = NETWORKS[case["network"]]["d_model"], _generator(seed)
    shape = (case["positions"], TOKENS, d)
    return [(torch.randn(shape, device="cuda", generator=generator) * size).half() for size in (0.05, 0.03)]


def _linear_inputs(case, seed):
    """int8 rows as norm_quant leaves them (a normal row on the grid of its largest value), weights rounded from N(0, 0.02)."""
    generator, depth, outputs = _generator(seed), case["depth"], case["outputs"]
    x, x_scale = _nearest_rows(torch.randn(case["rows"], depth, device="cuda", generator=generator))
    weight, weight_scale = _nearest(torch.randn(outputs, depth, device="cuda", generator=generator) * 0.02)
    if case["epilogue"] == "bias":
        return x, x_scale, weight, weight_scale, (torch.randn(outputs, device="cuda", generator=generator) * 0.02).half(), None
    return x, x_scale, weight, weight_scale, None, torch.randn(case["rows"], outputs, device="cuda", generator=generator).half()


def _nearest_rows(x):
    absmax = x.abs().amax(1)
    return torch.round(x * (127 / absmax)[:, None]).to(torch.int8), absmax / 127


def _attention_inputs(case, seed):
    generator, heads, kv, query, value = _generator(seed), case["heads"], case["kv_heads"], case["query"], case["value"]
    width = heads * query + kv * query + kv * value + heads * TEMPLATES
    projected = torch.randn(case["positions"], case["tokens"], width, device="cuda", generator=generator)
    projected[..., -heads * TEMPLATES:] *= 0.4
    gains = [(1 + 0.1 * torch.randn(query, device="cuda", generator=generator)).half() for _ in range(2)]
    templates = (0.5 * torch.randn(TEMPLATES, SQUARES, SQUARES, device="cuda", generator=generator)).half()
    return projected.to(torch.bfloat16 if case["type"] == "bf16" else torch.float16), templates, *gains


def _normed(case, seed):
    d = NETWORKS[case["network"]]["d_model"]
    return torch.randn(case["positions"], TOKENS, d, device="cuda", generator=_generator(seed)).half()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        return kind, case, _linear_inputs(case, seed)
    if kind == "attention":
        return kind, case, _attention_inputs(case, seed)
    layers = _layers(case)
    if kind == "lane":
        return kind, _lanes(case["network"], layers, case["positions"]), _boards(case["positions"], seed)
    network = _network(case["network"], layers, kind != "fp16_block")
    if kind in ("int8_block", "fp16_block"):
        return kind, (network.encoder[1], network.templates), _stream(case, seed)
    if kind == "heads":
        return kind, network, _normed(case, seed)
    return kind, network, torch.from_numpy(_boards(case["positions"], seed)).cuda()


@torch.no_grad()
def run(state):
    kind, handle, inputs = state
    if kind == "lane":
        return handle.collect(handle.launch(inputs))
    if kind == "forward":
        return handle(inputs)
    if kind in ("int8_block", "fp16_block"):
        block, templates = handle
        return block(inputs[0], templates, inputs[1])
    if kind == "linear":
        x, x_scale, weight, weight_scale, bias, residual = inputs
        return launch_int8_linear(x, x_scale, weight, weight_scale, bias, residual, False, None, None, None,
                                  out_dtype=torch.bfloat16 if handle["type"] == "bf16" else torch.float16)
    if kind == "attention":
        return template_attention(*inputs, handle["heads"], handle["kv_heads"], handle["query"], handle["value"], TEMPLATES, EPS)
    if kind == "heads":
        return handle.answers(inputs)
    return handle.input_embedding(inputs)


def work(case):
    """Bytes: the weights, the inputs and the outputs, once each. Operations: the products', two a multiply-add."""
    kind = case["kind"]
    if kind == "linear":
        rows, depth, outputs = case["rows"], case["depth"], case["outputs"]
        added = 2 * outputs if case["epilogue"] == "bias" else 2 * rows * outputs
        return {"bytes": rows * depth + outputs * depth + 4 * (rows + outputs) + added + 2 * rows * outputs, "flops": 2 * rows * depth * outputs}
    B = case["positions"]
    if kind == "attention":
        T, heads, kv, query, value = (case[key] for key in ("tokens", "heads", "kv_heads", "query", "value"))
        width = heads * query + kv * (query + value) + heads * TEMPLATES
        return {"bytes": 2 * B * T * (width + heads * value) + 2 * TEMPLATES * SQUARES * SQUARES,
                "flops": 2 * B * heads * (T * T * (query + value) + SQUARES * SQUARES * TEMPLATES)}
    s = NETWORKS[case["network"]]
    d, heads, kv, h = s["d_model"], s["n_heads"], s["kv_heads"], s["mlp_hidden"]
    value = d // heads
    query = round(s["qk_ratio"] * value)
    width = heads * query + kv * (query + value) + heads * TEMPLATES
    products = d * width + 3 * d * h
    block_flops = 2 * B * (TOKENS * (products + d * d) + heads * (TOKENS * TOKENS * (query + value) + SQUARES * SQUARES * TEMPLATES))
    head_flops = 2 * B * (TOKENS * d * d + SQUARES * SQUARES * d + TOKENS * 21 * d + TOKENS * 16 * d + d * BINS)
    head_weights = 2 * d * d + 4 * (21 * d + TOKENS * 16 * d + d * BINS)
    answers = 4 * B * (MOVES + BINS)
    embedding = 2 * d * (VOCABULARY + TOKENS + sum(FEATURE_ROWS))
    if kind == "int8_block":
        return {"bytes": 3 * 2 * B * TOKENS * d + products + 2 * d * d, "flops": block_flops}
    if kind == "fp16_block":
        return {"bytes": 3 * 2 * B * TOKENS * d + 2 * (products + d * d), "flops": block_flops}
    if kind == "heads":
        return {"bytes": 2 * B * TOKENS * d + head_weights + answers, "flops": head_flops}
    if kind == "embedding":
        return {"bytes": 8 * B * TOKENS + embedding + 2 * B * TOKENS * d, "flops": B * d * (TOKENS * 2 + SQUARES * 23)}
    layers = s["num_layers"]
    weights = (layers - 1) * (products + 2 * d * d) + 2 * (products + d * d)
    return {"bytes": weights + 8 * B * TOKENS + embedding + head_weights + answers, "flops": layers * block_flops + head_flops}


def tolerance(case):
    """About four times what the kernels differ by from exact() here: a whole network 0.0027 to 0.0056 (a rounding in one block moves
    int8 steps in all that follow), an int8 block 0.0005 to 0.0012, an fp16 block 0.00035, the rounding of bf16 outputs 0.0017 and
    of fp16 ones 0.0003, the heads 0.0002 (the fp16 product of their two projections)."""
    kind = case["kind"]
    if kind in ("linear", "attention"):
        return {"rel": 0.007 if case["type"] == "bf16" else 0.0015}
    return {"rel": {"lane": 0.02, "forward": 0.02, "int8_block": 0.0045, "fp16_block": 0.0014, "heads": 0.0008, "embedding": 0.0012}[kind]}


def _rms(x, gain):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain


def _quantised(x):
    """Rows as the int8 products read them: on the grid of the row's largest magnitude / 127."""
    step = x.abs().amax(-1, keepdim=True).clamp(min=1e-20) / 127
    return torch.round(x / step) * step


def _attend(projected, templates, q_gain, k_gain, heads, kv, query, value):
    B, T, _ = projected.shape
    q, k, v, mix = projected.split([heads * query, kv * query, kv * value, heads * TEMPLATES], -1)
    q = _rms(q.reshape(B, T, heads, query), q_gain).transpose(1, 2)
    k = _rms(k.reshape(B, T, kv, query), k_gain).transpose(1, 2).repeat_interleave(heads // kv, 1).contiguous()
    v = v.reshape(B, T, kv, value).transpose(1, 2).repeat_interleave(heads // kv, 1).contiguous()
    scores = torch.matmul(q.contiguous(), k.transpose(2, 3).contiguous()) / math.sqrt(query)
    mix = mix[:, :SQUARES].reshape(B, SQUARES, heads, TEMPLATES)
    for t in range(TEMPLATES):
        scores[:, :, :SQUARES, :SQUARES] += mix[..., t].transpose(1, 2).unsqueeze(-1) * templates[t]
    return torch.matmul(torch.softmax(scores, -1), v).transpose(1, 2).reshape(B, T, heads * value)


def _half_state(name, layers):
    """The state in 64 bits as the inference networks hold it: the stream scaled, everything but the heads' weights in fp16."""
    scaled = ("combine_heads.weight", "combine_heads.bias", "down_projection.weight", "embed.weight", "position_embed", "square_features.table")
    kept = ("from_projection", "to_projection", "promotion_projection", "board_down_project", "eval_head")
    state = {}
    for key, value in _state(name, layers).items():
        value = value * STREAM if key.endswith(scaled) else value
        state[key] = value.double() if key.startswith(kept) else value.half().double()
    return state


def _exact_block(state, i, name, x, original, weights, templates, mixed, mixes):
    s, p = NETWORKS[name], "encoder.%d." % i
    heads, kv = s["n_heads"], s["kv_heads"]
    value = s["d_model"] // heads
    query = round(s["qk_ratio"] * value)
    if not mixed:
        x = state[p + "residual_scale"] * x + state[p + "input_scale"] * original
    if weights is None:
        dense = {"projection": torch.cat([state[p + key + ".weight"] for key in ("Q", "K", "V", "template_mix")]),
                 "gate_up": torch.cat([state[p + "mlp.gate_projection.weight"], state[p + "mlp.up_projection.weight"]]),
                 "down": state[p + "mlp.down_projection.weight"]}
        rounded = lambda rows: rows
    else:
        dense = {key: integers.double() * scale.double()[:, None] for key, (integers, scale) in weights.items()}
        dense["down"] = dense["down"] * STREAM
        rounded = _quantised
    bias = torch.cat([state[p + key + ".bias"] for key in ("Q", "K", "V", "template_mix")])
    projected = rounded(_rms(x, state[p + "ln1.weight"])) @ dense["projection"].T + bias
    attended = _attend(projected, templates, state[p + "q_norm.weight"], state[p + "k_norm.weight"], heads, kv, query, value)
    x = x + attended @ state[p + "combine_heads.weight"].T + state[p + "combine_heads.bias"]
    gate, up = (rounded(_rms(x, state[p + "ln2.weight"])) @ dense["gate_up"].T).chunk(2, -1)
    hidden = F.silu(gate) * up
    if weights is not None:
        hidden = rounded((hidden.view(*hidden.shape[:-1], -1, 32) @ _hadamard()).flatten(-2))
        hidden = F.pad(hidden, (0, dense["down"].shape[1] - hidden.shape[-1]))
    x = x + hidden @ dense["down"].T
    if mixes:
        following = "encoder.%d." % (i + 1)
        x = state[following + "residual_scale"] * x + state[following + "input_scale"] * original
    return x


def _feature_rows(boards):
    """B x 64 x 23: each square's row within each feature's rows, found square by square on the 8 x 8 board."""
    B, device = len(boards), boards.device
    edge = 13
    rows = torch.zeros(B, SQUARES, 23, dtype=torch.long, device=device)
    padded = torch.full((B, 8 + 14, 8 + 14), edge, dtype=torch.long, device=device)   # [rank + 7, file + 7]
    padded[:, 7:15, 7:15] = boards[:, :SQUARES].view(B, 8, 8)
    at = lambda file, rank: padded[:, 7 + rank:15 + rank, 7 + file:15 + file].reshape(B, SQUARES)
    place = torch.arange(SQUARES, device=device)
    for slot, code in enumerate((6, 12, 5, 11)):                 # kings and queens: the first of each, or none
        found = torch.where(boards[:, :SQUARES] == code, place, SQUARES).amin(1, keepdim=True)
        offset = (place // 8 - found // 8 + 7) * 15 + place % 8 - found % 8 + 7
        rows[..., slot] = torch.where(found < SQUARES, offset, 225)
    for slot, (file, rank) in enumerate([(0, 1), (0, -1), (1, 0), (-1, 0), (1, 1), (-1, 1), (1, -1), (-1, -1)]):
        rows[..., 4 + slot] = at(file, rank)
        line, pawn = torch.zeros(B, SQUARES, dtype=torch.long, device=device), torch.zeros(B, SQUARES, dtype=torch.long, device=device)
        for distance in range(7, 0, -1):                         # the nearest last, so that it stays
            code = at(file * distance, rank * distance)
            line = torch.where((code > 0) & (code != edge), 1 + (code - 1) * 7 + distance - 1, torch.where(code == edge, 0, line))
            pawn = torch.where((code == 1) | (code == 7), 1 + (code == 7).long() * 7 + distance - 1, torch.where(code == edge, 0, pawn))
        rows[..., 12 + slot] = line
        if file == 0:
            rows[..., 21 + slot] = pawn
    jumps = torch.stack([at(file, rank) for file, rank in ((1, 2), (2, 1), (2, -1), (1, -2), (-1, -2), (-2, -1), (-2, 1), (-1, 2))], -1)
    rows[..., 20] = (jumps == 2).sum(-1).clamp(max=2) * 3 + (jumps == 8).sum(-1).clamp(max=2)
    return rows


def _exact_embedding(state, boards):
    first = torch.tensor([0] + FEATURE_ROWS[:-1], device="cuda").cumsum(0)
    x = state["embed.weight"][boards] + state["position_embed"]
    features = _feature_rows(boards) + first
    for slot in range(23):
        x[:, :SQUARES] += state["square_features.table"][features[..., slot]]
    return x


def _moves():
    """(from, to, promotion piece or -1) in the ids' order: each square's queen and knight moves by target, then the promotions."""
    steps = [(f, r) for f in range(-7, 8) for r in range(-7, 8) if (f or r) and (f == 0 or r == 0 or abs(f) == abs(r) or abs(f * r) == 2)]
    moves = [(s, t, -1) for s in range(64) for t in range(64) if (t % 8 - s % 8, t // 8 - s // 8) in steps]
    for start, end in ((6, 7), (1, 0)):
        moves += [(start * 8 + f, end * 8 + t, piece) for f in range(8) for t in range(max(f - 1, 0), min(f + 2, 8)) for piece in (0, 2, 1, 3)]
    return moves


def _exact_heads(state, x):
    weight, bias = (lambda key: state[key + ".weight"]), (lambda key: state[key + ".bias"])
    dense = lambda key, rows: rows @ weight(key).T + bias(key)
    squares = x[:, :SQUARES]
    products = torch.matmul(dense("from_projection", squares), dense("to_projection", squares).transpose(1, 2).contiguous()) / math.sqrt(x.shape[-1])
    promotions = dense("promotion_projection", squares)
    moves = torch.tensor(_moves(), device="cuda")
    logits = products[:, moves[:, 0], moves[:, 1]]
    promoting = moves[:, 2] >= 0
    logits[:, promoting] += promotions[:, moves[promoting, 1], moves[promoting, 2]]
    values = dense("eval_head.2", F.gelu(dense("eval_head.0", F.gelu(dense("board_down_project.0", x)).flatten(1))))
    return logits, values


def _expected_score(values):
    centres = (torch.arange(BINS, device="cuda", dtype=torch.float64) + 0.5) / BINS
    return torch.softmax(values, -1) @ centres


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, x_scale, weight, weight_scale, bias, residual = _linear_inputs(case, seed)
        out = (x.double() @ weight.double().T) * x_scale.double()[:, None] * weight_scale.double()
        return out + (bias if residual is None else residual).double()
    if kind == "attention":
        projected, templates, q_gain, k_gain = (tensor.double() for tensor in _attention_inputs(case, seed))
        return torch.cat([_attend(part, templates, q_gain, k_gain, case["heads"], case["kv_heads"], case["query"], case["value"])
                          for part in projected.split(256)])
    name, layers = case["network"], _layers(case)
    state = _half_state(name, layers)
    templates, int8 = state["templates"], _int8_weights(name, layers)
    if kind in ("int8_block", "fp16_block"):
        weights = int8[1] if kind == "int8_block" else None
        return torch.cat([_exact_block(state, 1, name, x.double(), original.double(), weights, templates, True, True)
                          for x, original in zip(*(tensor.split(256) for tensor in _stream(case, seed)))])
    if kind == "heads":
        logits, values = _exact_heads(state, _normed(case, seed).double())
        return torch.cat([logits, _expected_score(values)[:, None]], 1), values
    boards = torch.from_numpy(_boards(case["positions"], seed)).cuda()
    if kind == "embedding":
        return torch.cat([_exact_embedding(state, part) for part in boards.split(512)])
    parts = []
    for part in boards.split(128):
        x = original = _exact_embedding(state, part)
        for i in range(layers):
            last = i == layers - 1
            x = _exact_block(state, i, name, x, original, int8.get(i), templates, 0 < i < layers - 1, i < layers - 2)
        parts.append(_exact_heads(state, _rms(x, state["ln.weight"])))
    logits, values = (torch.cat(outputs) for outputs in zip(*parts))
    return torch.cat([logits, _expected_score(values)[:, None]], 1) if kind == "lane" else (logits, values)
