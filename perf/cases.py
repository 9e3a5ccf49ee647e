"""The work a program has this framework do, as cases that can be timed: the quantised linears of a decoder layer
during decode, batched decode and prefill, with and without adapters, and the two ways weights get into the packed
form when a model is loaded.

A layer here has the widths the benchmark and the tests use: hidden 2560, MLP 9216, q / k / v of 8192 / 1024 / 1024
columns in a full-attention layer, in_proj_qkv / in_proj_z of 8192 / 4096 in a linear-attention one, 4096 -> 2560 out of
either; `draw` varies the widths, the row counts and the options around them.  Every state owns its weights, so passes
over several states stream them from memory as a model of many layers does.
"""
from __future__ import annotations

import torch

from kiln_amd import layer_pack, lora, marlin_gemm, marlin_proj
from kiln_amd.layer_pack import LayerProjections, PackKind

FULL = (PackKind.QProj, PackKind.KProj, PackKind.VProj)
LINEAR = (PackKind.InProjQkv, PackKind.InProjZ)


def listed():
    return [
        # one projection of one token: the smallest call there is (an attention block's output projection)
        {"name": "proj_m1", "path": "proj", "m": 1, "k": 4096, "n": 2560, "groupsize": 128},
        # a single stream decoding: one token through four layers, three linear-attention and one full-attention,
        # called eagerly, layer by layer
        {"name": "layers_m1", "path": "layers", "m": 1, "layers": 4, "hidden": 2560, "inter": 9216, "rank": 0, "groupsize": 128},
        # a batch of 16 decoding: the MLP of a layer as one call (the benchmark's headline sizes)
        {"name": "mlp_m16", "path": "mlp", "m": 16, "hidden": 2560, "inter": 9216, "groupsize": 128},
        # the same batch in a serving loop that captured its decode step into a HIP graph and replays it per token
        {"name": "graph_m16", "path": "graph", "m": 16, "layers": 4, "hidden": 2560, "inter": 9216, "groupsize": 128},
        # a small batch with two adapters on every projection of a layer
        {"name": "lora_layer_m11", "path": "layers", "m": 11, "layers": 1, "hidden": 2560, "inter": 9216, "rank": 8, "groupsize": 128},
        # a large decode batch (or a short prompt) on weights quantised per column
        {"name": "layers_m50_percol", "path": "layers", "m": 50, "layers": 2, "hidden": 2560, "inter": 9216, "rank": 0, "groupsize": -1},
        # a prefill chunk of 512 tokens with two adapters, ranks 16 + 32, on gate and up side by side
        {"name": "lora_m512", "path": "lora", "m": 512, "k": 2560, "n": 18432, "rank_a": 16, "rank_b": 32, "groupsize": 128},
        # a ragged prompt through one layer
        {"name": "layers_m777", "path": "layers", "m": 777, "layers": 1, "hidden": 2560, "inter": 9216, "rank": 0, "groupsize": 128},
        # chunked prefill: 2048 tokens through an MLP
        {"name": "mlp_m2048", "path": "mlp", "m": 2048, "hidden": 2560, "inter": 9216, "groupsize": 128},
        # the largest chunk the scheduler hands out
        {"name": "mlp_m8192", "path": "mlp", "m": 8192, "hidden": 2560, "inter": 9216, "groupsize": 128},
        # loading a model: the bf16 weights of a layer, quantised and packed, with the fused packs built
        {"name": "pack_layer", "path": "pack", "hidden": 2560, "inter": 9216, "full": True, "groupsize": 128},
        # loading a GPTQ checkpoint: one projection's tensors in host memory, repacked onto the card
        {"name": "load_gptq", "path": "gptq", "k": 2560, "n": 9216, "zeros": True, "groupsize": 128},
    ]


def _rows(rng, least, most):
    """Row counts, evenly over their logarithm; most of them off every tile's edge."""
    return min(most, max(least, round(least * (most / least) ** rng.random())))


def _width(rng, least, most, step):
    return max(least, round(least * (most / least) ** rng.random() / step) * step)


def draw(rng):
    path = rng.choice(["proj", "layers", "layers", "mlp", "mlp", "graph", "lora", "pack", "gptq"])
    groupsize = rng.choice([128, 128, 128, -1])
    hidden, inter = _width(rng, 1024, 4096, 256), _width(rng, 2816, 12288, 256)
    k, n = _width(rng, 1024, 9216, 128), _width(rng, 1024, 18432, 256)
    if path == "proj":
        return {"path": path, "m": _rows(rng, 1, 4096), "k": k, "n": n, "groupsize": groupsize}
    if path == "layers":
        m = _rows(rng, 1, 2048)
        return {"path": path, "m": m, "layers": rng.randint(1, 4) if m <= 64 else 1, "hidden": hidden, "inter": inter,
                "rank": rng.choice([0, 0, 4, 8]), "groupsize": groupsize}
    if path == "mlp":
        return {"path": path, "m": _rows(rng, 1, 4096), "hidden": hidden, "inter": inter, "groupsize": groupsize}
    if path == "graph":
        return {"path": path, "m": _rows(rng, 1, 64), "layers": rng.randint(1, 4), "hidden": hidden, "inter": inter,
                "groupsize": groupsize}
    if path == "lora":
        return {"path": path, "m": _rows(rng, 1, 2048), "k": k, "n": n, "rank_a": rng.choice([8, 16]),
                "rank_b": rng.choice([4, 16, 32]), "groupsize": groupsize}
    if path == "pack":
        return {"path": path, "hidden": hidden, "inter": inter, "full": rng.random() < 0.5, "groupsize": groupsize}
    return {"path": path, "k": k, "n": n, "zeros": rng.random() < 0.5, "groupsize": groupsize}


class _Source:
    """Seeded values on the card."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, dtype=torch.bfloat16, device="cuda", generator=self.gen) * std

    def weight(self, k, n):
        # [in, out], as checkpoints of this kind hold them: normal, about 1 / sqrt(in)
        return self.normal(k, n, std=k ** -0.5)

    def packed(self, k, n, groupsize):
        return marlin_proj.pack_from_bf16(self.weight(k, n), groupsize)

    def adapters(self, k, n, rank):
        two = [lora.LoraProjectionWeights(self.normal(rank, k, std=k ** -0.5), self.normal(n, rank, std=0.1)) for _ in range(2)]
        return lora.stack_adapters(two, (0.5, 1.0))


def _attention_width(hidden):
    """Columns of the wide attention projections: 8192 at hidden 2560."""
    return max(1024, hidden * 16 // 5 // 512 * 512)


def _layer_shapes(hidden, inter, full):
    wide = _attention_width(hidden)
    if full:
        attn = {PackKind.QProj: (hidden, wide), PackKind.KProj: (hidden, 1024), PackKind.VProj: (hidden, 1024),
                PackKind.OProj: (wide // 2, hidden)}
    else:
        attn = {PackKind.InProjQkv: (hidden, wide), PackKind.InProjZ: (hidden, wide // 2), PackKind.OutProj: (wide // 2, hidden)}
    return {**attn, PackKind.GateProj: (hidden, inter), PackKind.UpProj: (hidden, inter), PackKind.DownProj: (inter, hidden)}


def _layers(src, case, count):
    """`count` layers as a loader leaves them: every projection packed, the fused packs built, the bf16 copies dropped.
    Every fourth is a full-attention layer (the only one, where there is one)."""
    layers = []
    for i in range(count):
        full = count == 1 or i % 4 == 3
        layer = LayerProjections({kind: src.weight(k, n) for kind, (k, n) in _layer_shapes(case["hidden"], case["inter"], full).items()})
        layer_pack.pack_layers([layer], groupsize=case["groupsize"], drop_bf16=True, fuse_gate_up=True, fuse_same_input_groups=True)
        layers.append((layer, FULL if full else LINEAR, PackKind.OProj if full else PackKind.OutProj))
    return layers


def _layer_step(layer, kinds, out_kind, x, attn, loras):
    """The quantised linears of one layer: the projections of the layer's input, the attention block's output
    projection, and the MLP.  (Norms and attention itself are another library's.)"""
    outs = list(layer.forward_same_input(kinds, x, {k: loras.get(k) for k in kinds}))
    outs.append(layer.forward(out_kind, attn, loras.get(out_kind)))
    h = layer.swiglu(x, loras.get(PackKind.GateProj), loras.get(PackKind.UpProj))
    outs.append(h)
    outs.append(layer.forward(PackKind.DownProj, h, loras.get(PackKind.DownProj)))
    return outs


def _all_steps(state):
    outs = []
    for (layer, kinds, out_kind), loras in zip(state["layers"], state["loras"]):
        outs += _layer_step(layer, kinds, out_kind, state["x"], state["attn"], loras)
    return outs


def prepare(case, seed):
    src, path = _Source(seed), case["path"]
    g = case["groupsize"]
    state = {"path": path, "groupsize": g}
    if path == "proj":
        state["x"] = src.normal(1, case["m"], case["k"])
        state["w"] = src.packed(case["k"], case["n"], g)
    elif path in ("layers", "graph"):
        hidden = case["hidden"]
        state["layers"] = _layers(src, case, case["layers"])
        state["x"] = src.normal(case["m"], hidden)
        state["attn"] = src.normal(case["m"], _attention_width(hidden) // 2, std=0.5)
        state["loras"] = [{} for _ in state["layers"]]
        if case.get("rank"):
            state["loras"] = [{kind: src.adapters(p.k, p.n, case["rank"]) for kind, p in layer.packed.items()}
                              for layer, _, _ in state["layers"]]
        if path == "graph":
            # what a serving loop does once per batch size: a pass on the capture stream, then the capture
            stream = torch.cuda.Stream()
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                _all_steps(state)
            torch.cuda.current_stream().wait_stream(stream)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                outs = _all_steps(state)
            state["graph"], state["outs"] = graph, outs
    elif path == "mlp":
        hidden, inter = case["hidden"], case["inter"]
        gate, up = src.packed(hidden, inter, g), src.packed(hidden, inter, g)
        state["gate_up"] = marlin_gemm.interleave_gate_up_device(gate.b_packed, gate.scales, up.b_packed, up.scales, g)
        state["down"] = src.packed(inter, hidden, g)
        state["x"] = src.normal(case["m"], hidden)
    elif path == "lora":
        k, n = case["k"], case["n"]
        state["w"] = src.packed(k, n, g)
        state["x"] = src.normal(case["m"], k)
        two = [lora.LoraProjectionWeights(src.normal(r, k, std=k ** -0.5), src.normal(n, r, std=0.1)) for r in (case["rank_a"], case["rank_b"])]
        state["lora"] = lora.stack_adapters(two, (0.5, 1.0))
    elif path == "pack":
        state["weights"] = {kind: src.weight(k, n) for kind, (k, n) in _layer_shapes(case["hidden"], case["inter"], case["full"]).items()}
    else:
        k, n = case["k"], case["n"]
        groups = 1 if g == -1 else k // g
        state["qweight"] = torch.randint(-2**31, 2**31, (k // 8, n), dtype=torch.int64, device="cuda", generator=src.gen).to(torch.int32).cpu()
        state["scales"] = (torch.rand(groups, n, device="cuda", generator=src.gen) * 0.018 + 0.002).half().cpu()
        # every zero-point of these checkpoints is 8
        state["qzeros"] = torch.full((groups, n // 8), 0x88888888 - 2**32, dtype=torch.int32) if case["zeros"] else None
    return state


def run(state):
    path, g = state["path"], state["groupsize"]
    if path == "proj":
        return marlin_proj.matmul_bf16(state["x"], state["w"])
    if path == "layers":
        return _all_steps(state)
    if path == "graph":
        state["graph"].replay()
        return state["outs"]
    if path == "mlp":
        return marlin_gemm.marlin_w4a16_mlp(state["x"], *state["gate_up"], state["down"].b_packed, state["down"].scales, g)
    if path == "lora":
        return lora.proj_forward(state["x"], state["w"], state["lora"])
    if path == "pack":
        layer = LayerProjections(dict(state["weights"]))
        layer_pack.pack_layers([layer], groupsize=g, drop_bf16=True, fuse_gate_up=True, fuse_same_input_groups=True)
        packs = list(layer.packed.values()) + [layer.gate_up_fused] + list(layer.same_input_fused.values())
        return [t for p in packs for t in (p.b_packed, p.scales)]
    w = marlin_proj.pack_from_gptq(state["qweight"], state["scales"], state["qzeros"], g, torch.device("cuda", torch.cuda.current_device()))
    return w.b_packed, w.scales


def _weight_bytes(k, n, g):
    return k * n // 2 + (1 if g == -1 else k // g) * n * 2


def work(case):
    g, path = case["groupsize"], case["path"]
    flops = nbytes = 0
    if path in ("proj", "lora"):
        m, k, n = case["m"], case["k"], case["n"]
        r = case["rank_a"] + case["rank_b"] if path == "lora" else 0
        nbytes = _weight_bytes(k, n, g) + 2 * m * (k + n) + 2 * r * (k + n)
        flops = 2 * m * k * n + 2 * m * r * (k + n)
    elif path == "mlp":
        m, hidden, inter = case["m"], case["hidden"], case["inter"]
        nbytes = _weight_bytes(hidden, 2 * inter, g) + _weight_bytes(inter, hidden, g) + 4 * m * hidden
        flops = 6 * m * hidden * inter
    elif path in ("layers", "graph"):
        m, hidden, inter, r = case["m"], case["hidden"], case["inter"], 2 * (case.get("rank") or 0)
        nbytes = 2 * m * (hidden + _attention_width(hidden) // 2)
        for i in range(case["layers"]):
            for k, n in _layer_shapes(hidden, inter, case["layers"] == 1 or i % 4 == 3).values():
                nbytes += _weight_bytes(k, n, g) + 2 * m * n + 2 * r * (k + n)
                flops += 2 * m * k * n + 2 * m * r * (k + n)
            nbytes -= 2 * m * inter          # gate and up leave as their product
    elif path == "pack":
        hidden, inter = case["hidden"], case["inter"]
        same = {kind for group in (FULL, LINEAR) for kind in group} | {PackKind.GateProj, PackKind.UpProj}
        for kind, (k, n) in _layer_shapes(hidden, inter, case["full"]).items():
            # read once; written packed, and again in the fused pack where the projection is part of one
            nbytes += 2 * k * n + _weight_bytes(k, n, g) * (2 if kind in same else 1)
    else:
        k, n = case["k"], case["n"]
        nbytes = 2 * _weight_bytes(k, n, g) + ((1 if g == -1 else k // g) * n // 2 if case["zeros"] else 0)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # loading moves and forms integers; everything else is f32 sums rounded to bf16 once or twice (8 bits: a half ulp is
    # 2e-3 to 4e-3 of a value, and a value next to a rounding boundary may land on either side of it)
    return "exact" if case["path"] in ("pack", "gptq") else {"rel": 5e-3, "max": 5e-2}
