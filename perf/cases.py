"""The workloads that the packed NF4 linear path is timed on.

Each case is work that a program using this package has it do, through the
public functions of `riftco-transformer_amd/device.py`: the decode step of a
7B-shaped decoder-only model (hidden width 4096, feed-forward width 11008), its
small batches, prefill, a training step of a layer with a low-rank adapter, the
input backward, layers whose widths fit no tile, the dense product and the
quantizer.  `listed()` names the fixed cases, `draw()` makes further ones of
the same kinds and ranges.

A case's "kind" says which functions it calls:

  forward   linear_forward, one call
  decode    the seven projections of each layer for `rows` tokens, captured
            once as a HIP graph and replayed for every token, projections that
            share their input grouped (linear_forward_group), every layer with
            its own weights
  adapted   lora_linear_forward_group: query, key and value of one layer,
            adapters on query and value
  train     lora_linear_forward and lora_linear_backward of one layer
  backward  linear_input_backward, one call
  matmul    the dense fp32 product
  quantize  quantize_weight of one layer's weight

Weights are N(0, 0.02) put through the package's own quantizer, activations
N(0, 1), upstream gradients N(0, 0.01), biases N(0, 0.01), adapter factors
N(0, 0.05).
"""
import importlib

import torch

device = importlib.import_module("riftco-transformer_amd.device")

WEIGHT_SIGMA = 0.02
UPSTREAM_SIGMA = 0.01
BIAS_SIGMA = 0.01
ADAPTER_SIGMA = 0.05
ALPHA = 32.0                  # adapter scale = ALPHA / rank
SECOND_LEVEL_BLOCK = 256
LARGEST_WEIGHT = 11008 * 4096
LARGEST_ROWS = 2048


def listed():
    return [
        # One projection of a one-token decode step, called by itself: the
        # smallest call, where the launch and the host path count.
        {"name": "one_projection", "kind": "forward", "rows": 1,
         "output_width": 4096, "input_width": 4096, "block": 64,
         "nested": False, "bias": False},
        # One token through four layers of the model, as a serving loop
        # replays it.
        {"name": "decode_step", "kind": "decode", "rows": 1, "layers": 4,
         "hidden": 4096, "feed_forward": 11008, "nested": False},
        # Four sequences decoded together, nested scales.
        {"name": "decode_step_four_rows", "kind": "decode", "rows": 4,
         "layers": 2, "hidden": 4096, "feed_forward": 11008, "nested": True},
        # A batch of sixteen sequences through the gate projection.
        {"name": "small_batch", "kind": "forward", "rows": 16,
         "output_width": 11008, "input_width": 4096, "block": 64,
         "nested": False, "bias": True},
        # Sixty-four tokens through an attention block's projections while its
        # adapters are not merged.
        {"name": "adapted_projections", "kind": "adapted", "rows": 64,
         "hidden": 4096, "rank": 16, "nested": True},
        # A prompt whose length fits no tile through the down projection.
        {"name": "short_prompt", "kind": "forward", "rows": 300,
         "output_width": 4096, "input_width": 11008, "block": 64,
         "nested": True, "bias": False},
        # Prefill: batch 4 x 512 tokens through the gate projection.
        {"name": "prefill", "kind": "forward", "rows": 2048,
         "output_width": 11008, "input_width": 4096, "block": 64,
         "nested": False, "bias": False},
        # A QLoRA training step of one layer on the same batch, forward and
        # backward, with all its gradients.
        {"name": "training_step", "kind": "train", "rows": 2048,
         "output_width": 11008, "input_width": 4096, "rank": 16,
         "nested": True, "bias": True},
        # Input gradient of a small batch.
        {"name": "small_input_backward", "kind": "backward", "rows": 16,
         "output_width": 11008, "input_width": 4096, "block": 64,
         "nested": True},
        # A layer whose widths are multiples of nothing: blocks straddle rows.
        {"name": "odd_widths", "kind": "forward", "rows": 16,
         "output_width": 4097, "input_width": 4095, "block": 64,
         "nested": False, "bias": True},
        # The dense product at the layer's shape (unpacked projections).
        {"name": "dense_product", "kind": "matmul", "batch": 1, "rows": 2048,
         "shared": 4096, "columns": 4096},
        # Packing one layer's weight when a model is loaded.
        {"name": "quantize", "kind": "quantize", "output_width": 11008,
         "input_width": 4096, "block": 64, "nested": True},
    ]


def log_uniform(rng, low, high):
    """A whole number in [low, high], uniform over its logarithm."""
    return min(high, max(low, round(low * (high / low) ** rng.random())))


def draw_widths(rng, odd_share):
    """(output_width, input_width) of a layer, at most the largest listed
    weight."""
    while True:
        if rng.random() < odd_share:
            output_width = log_uniform(rng, 255, 4200)
            input_width = log_uniform(rng, 255, 4200)
        else:
            output_width = 64 * log_uniform(rng, 4, 172)
            input_width = rng.choice([
                64 * log_uniform(rng, 4, 172), 1024, 2048, 4096, 11008])
        if output_width * input_width <= LARGEST_WEIGHT:
            return output_width, input_width


def draw_one(rng):
    kind = rng.choice(["forward", "forward", "forward", "decode", "adapted",
                       "train", "train", "backward", "backward", "matmul",
                       "quantize"])
    nested = rng.random() < 0.5
    if kind == "decode":
        return {"kind": kind, "rows": rng.randint(1, 4),
                "layers": rng.randint(1, 4),
                "hidden": 64 * rng.randint(16, 64),
                "feed_forward": 64 * rng.randint(43, 172), "nested": nested}
    if kind == "adapted":
        return {"kind": kind, "rows": log_uniform(rng, 1, 512),
                "hidden": 64 * rng.randint(16, 64),
                "rank": rng.choice([4, 8, 16, 32, 64]), "nested": nested}
    if kind == "matmul":
        return {"kind": kind, "batch": rng.choice([1, 1, 2, 8]),
                "rows": log_uniform(rng, 16, LARGEST_ROWS),
                "shared": log_uniform(rng, 16, 4096),
                "columns": log_uniform(rng, 16, 11008)}
    output_width, input_width = draw_widths(
        rng, 0.2 if kind in ("forward", "backward", "quantize") else 0.0)
    case = {"kind": kind, "output_width": output_width,
            "input_width": input_width, "nested": nested}
    if kind != "quantize":
        case["rows"] = log_uniform(rng, 1, LARGEST_ROWS)
    if kind == "train":
        case["rank"] = rng.choice([4, 8, 16, 32, 64])
    else:
        case["block"] = rng.choice([64, 64, 64, 32, 128])
    if kind in ("forward", "train"):
        case["bias"] = rng.random() < 0.5
    return case


def draw(rng):
    """One more case of the same kinds and ranges, no larger than the largest
    listed one."""
    costs = [work(case) for case in listed()]
    most_bytes = max(cost["bytes"] for cost in costs)
    most_flops = max(cost["flops"] for cost in costs)
    while True:
        case = draw_one(rng)
        cost = work(case)
        if cost["bytes"] <= most_bytes and cost["flops"] <= most_flops:
            return case


# ---- inputs ------------------------------------------------------------------

def normal(generator, shape, sigma):
    return torch.randn(shape, generator=generator, device="cuda",
                       dtype=torch.float32).mul_(sigma)


def packed(generator, output_width, input_width, block, nested):
    return device.quantize_weight(
        normal(generator, (output_width, input_width), WEIGHT_SIGMA), block,
        nested, SECOND_LEVEL_BLOCK)


def adapter(generator, output_width, input_width, rank):
    """(A, B, scale) of a low-rank adapter."""
    return (normal(generator, (rank, input_width), ADAPTER_SIGMA),
            normal(generator, (output_width, rank), ADAPTER_SIGMA),
            ALPHA / rank)


def prepare_decode(case, generator):
    """The serving loop's graph: it reads `hidden_state` and the feed-forward
    activation where they lie and writes the same outputs for every token."""
    rows, hidden, wide = case["rows"], case["hidden"], case["feed_forward"]
    layers = []
    for _ in range(case["layers"]):
        layers.append({
            "attention": [packed(generator, hidden, hidden, 64,
                                 case["nested"]) for _ in range(3)],
            "output": packed(generator, hidden, hidden, 64, case["nested"]),
            "gated": [packed(generator, wide, hidden, 64, case["nested"])
                      for _ in range(2)],
            "down": packed(generator, hidden, wide, 64, case["nested"]),
        })
    hidden_state = normal(generator, (rows, hidden), 1.0)
    wide_state = normal(generator, (rows, wide), 1.0)

    def step():
        outputs = []
        for layer in layers:
            outputs += device.linear_forward_group(hidden_state,
                                                   layer["attention"])
            outputs.append(device.linear_forward(hidden_state,
                                                 layer["output"]))
            outputs += device.linear_forward_group(hidden_state,
                                                   layer["gated"])
            outputs.append(device.linear_forward(wide_state, layer["down"]))
        return outputs

    step()  # first use outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = step()
    return {"graph": graph, "outputs": outputs, "layers": layers,
            "inputs": (hidden_state, wide_state)}


def prepare(case, seed):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    kind = case["kind"]
    if kind == "decode":
        state = prepare_decode(case, generator)
    elif kind == "adapted":
        hidden = case["hidden"]
        state = {
            "x": normal(generator, (case["rows"], hidden), 1.0),
            "weights": [packed(generator, hidden, hidden, 64, case["nested"])
                        for _ in range(3)],
            "adapters": [adapter(generator, hidden, hidden, case["rank"]),
                         None,
                         adapter(generator, hidden, hidden, case["rank"])],
        }
    elif kind == "matmul":
        state = {
            "left": normal(generator, (case["batch"], case["rows"],
                                       case["shared"]), 1.0),
            "right": normal(generator, (case["batch"], case["shared"],
                                        case["columns"]), WEIGHT_SIGMA),
        }
    elif kind == "quantize":
        state = {"dense": normal(generator, (case["output_width"],
                                             case["input_width"]),
                                 WEIGHT_SIGMA)}
    else:
        output_width, input_width = case["output_width"], case["input_width"]
        state = {"weight": packed(generator, output_width, input_width,
                                  case.get("block", 64), case["nested"])}
        if kind in ("forward", "train"):
            state["x"] = normal(generator, (case["rows"], input_width), 1.0)
            state["bias"] = (normal(generator, (output_width,), BIAS_SIGMA)
                             if case["bias"] else None)
        if kind in ("backward", "train"):
            state["dy"] = normal(generator, (case["rows"], output_width),
                                 UPSTREAM_SIGMA)
        if kind == "train":
            state["adapter"] = adapter(generator, output_width, input_width,
                                       case["rank"])
    state["case"] = case
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        return device.linear_forward(state["x"], state["weight"],
                                     state["bias"])
    if kind == "decode":
        state["graph"].replay()
        return state["outputs"]
    if kind == "adapted":
        outputs, reduced = device.lora_linear_forward_group(
            state["x"], state["weights"], state["adapters"])
        return outputs + [product for product in reduced
                          if product is not None]
    if kind == "train":
        lora_a, lora_b, scale = state["adapter"]
        y, reduced = device.lora_linear_forward(
            state["x"], state["weight"], lora_a, lora_b, scale, state["bias"])
        dx, d_a, d_b = device.lora_linear_backward(
            state["dy"], state["x"], state["weight"], lora_a, lora_b, scale,
            reduced)
        return {"y": y, "reduced": reduced, "dx": dx, "d_a": d_a, "d_b": d_b}
    if kind == "backward":
        return device.linear_input_backward(state["dy"], state["weight"])
    if kind == "matmul":
        return device.matmul(state["left"], state["right"])
    weight = device.quantize_weight(state["dense"], case["block"],
                                    case["nested"], SECOND_LEVEL_BLOCK)
    outputs = {"codes": weight.codes, "scales": weight.primary_scales}
    if case["nested"]:
        outputs["second_level"] = weight.secondary_scales
        outputs["offset"] = weight.offset
    return outputs


# ---- what a pass cannot do without -------------------------------------------

def payload_bytes(output_width, input_width, block, nested):
    """Packed codes and scales of one weight."""
    count = output_width * input_width
    blocks = -(-count // block)
    scales = (blocks + 4 * (-(-blocks // SECOND_LEVEL_BLOCK)) if nested
              else 4 * blocks)
    return (count + 1) // 2 + scales


def work(case):
    kind = case["kind"]
    if kind == "decode":
        rows, hidden, wide = case["rows"], case["hidden"], case["feed_forward"]
        payload = (4 * payload_bytes(hidden, hidden, 64, case["nested"]) +
                   2 * payload_bytes(wide, hidden, 64, case["nested"]) +
                   payload_bytes(hidden, wide, 64, case["nested"]))
        weights = 4 * hidden * hidden + 3 * wide * hidden
        outputs = 4 * rows * (5 * hidden + 2 * wide)
        inputs = 4 * rows * (hidden + wide)
        return {"bytes": case["layers"] * (payload + outputs) + inputs,
                "flops": 2 * case["layers"] * rows * weights}
    if kind == "adapted":
        rows, hidden, rank = case["rows"], case["hidden"], case["rank"]
        return {
            "bytes": 3 * payload_bytes(hidden, hidden, 64, case["nested"]) +
            4 * (4 * rows * hidden + 4 * rank * hidden + 2 * rows * rank),
            "flops": 2 * rows * (3 * hidden * hidden + 4 * hidden * rank)}
    if kind == "matmul":
        batch, rows = case["batch"], case["rows"]
        shared, columns = case["shared"], case["columns"]
        return {"bytes": 4 * batch * (rows * shared + shared * columns +
                                      rows * columns),
                "flops": 2 * batch * rows * shared * columns}
    output_width, input_width = case["output_width"], case["input_width"]
    weights = output_width * input_width
    payload = payload_bytes(output_width, input_width, case.get("block", 64),
                            case["nested"])
    if kind == "quantize":
        return {"bytes": 4 * weights + payload, "flops": weights}
    rows = case["rows"]
    bias = 4 * output_width if case.get("bias") else 0
    activations = 4 * rows * (input_width + output_width)
    if kind in ("forward", "backward"):
        return {"bytes": payload + activations + bias,
                "flops": 2 * rows * weights}
    # train: the weight, x and the adapter are inputs of both halves
    rank = case["rank"]
    return {
        "bytes": payload + 2 * activations + bias +
        8 * rank * (input_width + output_width) + 4 * rows * rank,
        "flops": 2 * rows * (2 * weights + 3 * rank * (input_width +
                                                       output_width))}


def tolerance(case):
    """Relative errors of fp32 products, about four times what the same path
    shows against sums in 64 bits over the widths above (2-norm: up to 5e-7,
    dense products whose widths fit no tile up to 1e-6).  The quantizer's
    outputs are whole numbers and the scales they belong to."""
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] == "matmul":
        return {"rel": 4.0e-6, "max": 3.0e-5}
    return {"rel": 2.0e-6, "max": 1.2e-5}
