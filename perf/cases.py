"""The workloads that this library's speed is judged by.

Every case is one of four uses of the public interface (stk_amd.ops), and each of them covers a range of sizes:

  infer     a mixture-of-experts layer without gradients, tokens in and tokens out: route, topology, first product with
            its activation on the gathered token rows, second product scattered back to the tokens
  train     the same layer forward and backward, with the gradients of the tokens, of both weights and of the router's
            weights
  products  the three block-sparse products on a topology that the caller keeps: a mixture-of-experts pattern or a
            uniformly random one, forward only or with all gradients
  convert   a dense matrix to the blocked format and back

A layer gets new expert choices with every batch, so `infer` and `train` route and build their topology on each pass;
`products` keeps its topology as the holder of a fixed sparsity pattern does.
"""
import math

import torch

import stk_amd as stk

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _layer(name, use, tokens, experts, top_k, hidden, ffn, routing="uniform", blocking=128, dtype="bf16", w1="in_out"):
    """w1: "in_out" [hidden, experts * ffn], or "out_in" [experts * ffn, hidden] used through its .t() view."""
    return {"name": name, "use": use, "tokens": tokens, "experts": experts, "top_k": top_k, "hidden": hidden, "ffn": ffn,
            "routing": routing, "blocking": blocking, "dtype": dtype, "w1": w1}


def _moe_products(name, direction, tokens, experts, top_k, hidden, ffn, routing="uniform", blocking=128, dtype="bf16"):
    return {"name": name, "use": "products", "pattern": "moe", "direction": direction, "tokens": tokens, "experts": experts, "top_k": top_k,
            "hidden": hidden, "ffn": ffn, "routing": routing, "blocking": blocking, "dtype": dtype}


def _random_products(name, direction, rows, cols, inner, density, blocking=128, dtype="bf16", views=False):
    """views: the dense operands arrive as .t() views where the product takes them either way."""
    return {"name": name, "use": "products", "pattern": "random", "direction": direction, "rows": rows, "cols": cols, "inner": inner,
            "density": density, "blocking": blocking, "dtype": dtype, "views": views}


def _convert(name, rows, cols, density, blocking=128, dtype="bf16"):
    return {"name": name, "use": "convert", "rows": rows, "cols": cols, "density": density, "blocking": blocking, "dtype": dtype}


def listed():
    return [
        # one decoding step of a serving batch: every expert that is hit has its weights read for a handful of rows
        _layer("decode", "infer", 64, 64, 2, 1024, 4096),
        # the prompts of a serving batch (8 x 2048 tokens) through the layer of the forward benchmark
        _layer("prefill", "infer", 16384, 64, 1, 1024, 4096),
        # one training step of the same layer
        _layer("train", "train", 16384, 64, 1, 1024, 4096),
        # the large training step: top-2 over experts of Zipf-distributed popularity
        _layer("train_large_skewed", "train", 32768, 64, 2, 2048, 8192, routing="zipf"),
        # small blocks in fp16, one expert with half of the tokens
        _layer("train_small_blocks", "train", 16384, 64, 1, 1024, 4096, routing="half", blocking=64, dtype="fp16"),
        # sizes that are multiples of the block and of nothing else, few experts, weights stored one row per output feature
        _layer("train_odd_sizes", "train", 5003, 16, 2, 1152, 2944, w1="out_in"),
        # the forward benchmark: the three products on a kept mixture-of-experts topology
        _moe_products("moe_products", "forward", 16384, 64, 1, 1024, 4096),
        # a quarter of the blocks of a square matrix at random, each product and each transpose of the sparse operand
        _random_products("random_products", "forward", 4096, 4096, 4096, 0.25, views=True),
        # a small pruned layer with its gradients: a few blocks, the time of the calls themselves
        _random_products("small_products", "train", 512, 1024, 512, 0.5, dtype="fp16"),
        # float32 values
        _random_products("float32_products", "forward", 1024, 1024, 1024, 0.5, dtype="fp32"),
        # format conversion of a pruned weight matrix, both ways, transpose metadata included
        _convert("convert", 8192, 8192, 0.25),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _blocks(rng, low, high, blocking):
    """A size between low and high (in units of 128) that is a multiple of the block."""
    return max(1, _log_uniform(rng, low * 128, high * 128) // blocking) * blocking


def draw(rng):
    use = rng.choice(["infer", "infer", "train", "train", "products_moe", "products_random", "products_random", "convert"])
    blocking = rng.choice([128, 128, 128, 64])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if use in ("infer", "train", "products_moe"):
        sizes = (_log_uniform(rng, 16, 32768), rng.choice([4, 8, 16, 32, 64]), rng.choice([1, 2]), _blocks(rng, 2, 16, blocking), _blocks(rng, 4, 64, blocking))
        routing = rng.choice(["uniform", "uniform", "zipf", "half"])
        if use == "products_moe":
            case = _moe_products("", rng.choice(["forward", "train"]), *sizes, routing=routing, blocking=blocking, dtype=dtype)
        else:
            case = _layer("", use, *sizes, routing=routing, blocking=blocking, dtype=dtype, w1=rng.choice(["in_out", "out_in"]))
    else:
        dtype = rng.choice([dtype, dtype, "fp32"])
        most = 16 if dtype == "fp32" else 64
        rows, cols = _blocks(rng, 2, most, blocking), _blocks(rng, 2, most, blocking)
        density = round(rng.choice([0.1, 0.2, 0.25, 0.5]) * rng.uniform(0.8, 1.25), 3)
        if use == "convert":
            case = _convert("", rows, cols, density, blocking=rng.choice([blocking, 32]), dtype=dtype)
        else:
            case = _random_products("", rng.choice(["forward", "train"]), rows, cols, _blocks(rng, 2, min(most, 32), blocking), density, blocking=blocking,
                                    dtype=dtype, views=rng.random() < 0.5)
    del case["name"]
    return case


# ---------------------------------------------------------------------------------------------------- inputs
def _normal(shape, std, dtype, gen):
    """N(0, std) values, a slice of rows at a time so that no fp32 copy of a large weight is made."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    rows = max(1, (1 << 26) // max(1, out[0].numel()))
    for r in range(0, shape[0], rows):
        part = out[r:r + rows]
        part.copy_(torch.randn(part.shape, device="cuda", generator=gen) * std)
    return out


def _expert_probabilities(case):
    """Popularity of the experts (by which they are drawn without replacement for a token)."""
    n = case["experts"]
    if case["routing"] == "zipf":        # s = 1.2
        p = [(e + 1) ** -1.2 for e in range(n)]
    elif case["routing"] == "half":      # expert 0 with as much as all the others
        p = [n - 1.0] + [1.0] * (n - 1)
    else:
        p = [1.0] * n
    return [v / sum(p) for v in p]


def _choices(case, gen):
    """[tokens, top_k] int32: the most likely experts under Gumbel noise, as a softmax router with noise picks them."""
    logp = torch.tensor(_expert_probabilities(case), device="cuda").log()
    noise = torch.rand(case["tokens"], case["experts"], device="cuda", generator=gen).clamp_(1e-20, 1 - 1e-7)
    return (logp - torch.log(-torch.log(noise))).topk(case["top_k"], dim=1).indices.to(torch.int32)


def _random_pattern(rows, cols, density, blocking, dtype, gen):
    """A dense matrix of which the given share of blocks, chosen uniformly, holds N(0, 1) values and the rest zeros."""
    br, bc = rows // blocking, cols // blocking
    keep = torch.zeros(br * bc, device="cuda")
    keep[torch.randperm(br * bc, device="cuda", generator=gen)[:max(1, round(density * br * bc))]] = 1.0
    dense = torch.randn(br, blocking, bc, blocking, device="cuda", generator=gen) * keep.view(br, 1, bc, 1)
    return dense.reshape(rows, cols).to(dtype)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, b = _DTYPES[case["dtype"]], case["blocking"]
    s = {"case": case}
    if case["use"] == "convert":
        s["dense"] = _random_pattern(case["rows"], case["cols"], case["density"], b, dtype, gen)
        return s
    if case["use"] == "products" and case["pattern"] == "random":
        m, n, k = case["rows"], case["cols"], case["inner"]
        s["s"] = stk.ops.to_sparse(_random_pattern(m, n, case["density"], b, dtype, gen), b)
        s["s"].data.mul_(0.02)
        operand = lambda rows, cols: _normal((cols, rows), 1.0, dtype, gen).t() if case["views"] else _normal((rows, cols), 1.0, dtype, gen)
        s["a"], s["w"], s["v"], s["u"] = operand(m, k), operand(k, n), operand(n, k), operand(k, m)
        outs = {"g_sdd": s["s"].data.shape, "g_dsd": (m, k), "g_dds": (k, n)}
    else:
        tokens, experts, hidden, ffn = case["tokens"], case["experts"], case["hidden"], case["ffn"]
        # (a kept topology is part of the case: its expert choices are the same ones for every seed)
        top = _choices(case, gen if case["use"] != "products" else torch.Generator(device="cuda").manual_seed(0))
        w1 = _normal((experts * ffn, hidden) if case.get("w1") == "out_in" else (hidden, experts * ffn), hidden ** -0.5, dtype, gen)
        s["w1"], s["w2"] = w1, _normal((experts * ffn, hidden), ffn ** -0.5, dtype, gen)
        x = _normal((tokens, hidden), 1.0, dtype, gen)
        if case["use"] == "products":
            r = stk.ops.route(top, experts, b)
            rows = r.row_slots.numel()
            s["x"] = stk.ops.padded_gather(x, r)     # padding rows are zero, as in a layer
            s["topo"] = stk.ops.dmoe_topology(r.padded_bins, b, rows // b, ffn // b, dtype=dtype)
            outs = {"g_sdd": s["topo"].data.shape, "g_dsd": (rows, hidden), "g_dds": (hidden, experts * ffn)}
        else:
            s["top"], s["x"] = top, x
            s["weights"] = torch.rand(tokens, case["top_k"], device="cuda", generator=gen)
            outs = {"g": (tokens, hidden)}
    if case["use"] == "train" or case.get("direction") == "train":
        for name, shape in outs.items():
            s[name] = _normal(shape, 1.0, dtype, gen)
        for name in ("x", "w1", "w2", "weights", "a", "w", "v", "u"):
            if name in s:
                s[name].requires_grad_(True)
        if "s" in s:
            s["s"].requires_grad_(True)
    return s


# ---------------------------------------------------------------------------------------------------- one pass
def _route_and_topology(s):
    c = s["case"]
    r = stk.ops.route(s["top"], c["experts"], c["blocking"])
    topo = stk.ops.dmoe_topology(r.padded_bins, c["blocking"], r.row_slots.numel() // c["blocking"], c["ffn"] // c["blocking"], dtype=s["x"].dtype)
    return r, topo


def _infer(s):
    w1 = s["w1"].t() if s["case"]["w1"] == "out_in" else s["w1"]
    with torch.no_grad():
        r, topo = _route_and_topology(s)
        h = stk.ops.gather_sdd(s["x"], r, w1, topo, "gelu_tanh")
        return {"y": stk.ops.dsd_scatter(h, s["w2"], r, s["weights"])}


def _train(s):
    w1 = s["w1"].t() if s["case"]["w1"] == "out_in" else s["w1"]
    r, topo = _route_and_topology(s)
    h = stk.ops.sdd_fused(stk.ops.padded_gather(s["x"], r), w1, topo, "gelu_tanh", save_sums=True)
    y = stk.ops.padded_scatter(stk.ops.dsd(h, s["w2"]), r, s["weights"])
    dx, dw1, dw2, dweights = torch.autograd.grad(y, (s["x"], s["w1"], s["w2"], s["weights"]), s["g"])
    return {"y": y.detach(), "dx": dx, "dw1": dw1, "dw2": dw2, "dweights": dweights}


def _products_moe(s):
    x, w1, w2, topo = s["x"], s["w1"], s["w2"], s["topo"]
    h = stk.ops.sdd(x, w1, topo)
    y = stk.ops.dsd(h, w2)
    z = stk.ops.dds(x.t(), h)
    out = {"h": h.data.detach(), "y": y.detach(), "z": z.detach()}
    if s["case"]["direction"] == "train":
        grads = torch.autograd.grad((h.data, y, z), (x, w1, w2), (s["g_sdd"], s["g_dsd"], s["g_dds"]))
        out.update(zip(("dx", "dw1", "dw2"), grads))
    return out


def _products_random(s):
    m = s["s"]
    if s["case"]["direction"] == "train":
        leaves = [s["a"], s["w"], m.data, s["v"], s["u"]]
        h, y, z = stk.ops.sdd(s["a"], s["w"], m), stk.ops.dsd(m, s["v"]), stk.ops.dds(s["u"], m)
        grads = torch.autograd.grad((h.data, y, z), leaves, (s["g_sdd"], s["g_dsd"], s["g_dds"]))
        out = {"h": h.data.detach(), "y": y.detach(), "z": z.detach()}
        out.update(zip(("da", "dw", "ds", "dv", "du"), grads))
        return out
    return {"h": stk.ops.sdd(s["a"], s["w"], m).data, "y": stk.ops.dsd(m, s["v"]), "z": stk.ops.dds(s["u"], m),
            "yt": stk.ops.dsd(m.t(), s["a"]), "zt": stk.ops.dds(s["w"], m.t())}


def _convert_both_ways(s):
    m = stk.ops.to_sparse(s["dense"], s["case"]["blocking"])
    return {"data": m.data, "row_indices": m.row_indices, "column_indices": m.column_indices, "offsets": m.offsets,
            "column_indices_t": m.column_indices_t, "offsets_t": m.offsets_t, "block_offsets_t": m.block_offsets_t, "dense": stk.ops.to_dense(m)}


def run(state):
    case = state["case"]
    if case["use"] == "infer":
        return _infer(state)
    if case["use"] == "train":
        return _train(state)
    if case["use"] == "convert":
        return _convert_both_ways(state)
    return _products_moe(state) if case["pattern"] == "moe" else _products_random(state)


# ---------------------------------------------------------------------------------------------------- work
def work(case):
    e = 4 if case["dtype"] == "fp32" else 2
    b, train = case["blocking"], case["use"] == "train" or case.get("direction") == "train"
    if case["use"] == "convert":
        total = case["rows"] // b * (case["cols"] // b)
        nnz = max(1, round(case["density"] * total))
        # the dense matrix in, the values out; the values in, the dense matrix out
        return {"bytes": 2 * (case["rows"] * case["cols"] + nnz * b * b) * e + 14 * nnz, "flops": 0}
    if case["use"] == "products" and case["pattern"] == "random":
        m, n, k = case["rows"], case["cols"], case["inner"]
        nnz = max(1, round(case["density"] * (m // b) * (n // b)))
        values, dense = nnz * b * b, m * k + k * n
        flops = 2.0 * values * k
        if not train:       # five products; in: values and four dense operands, out: the values of one and four dense results
            return {"bytes": (2 * values + 4 * dense) * e, "flops": 5 * flops}
        # three products and six gradient products; in: values, four operands, three gradients, out: three results, five gradients
        return {"bytes": (4 * values + 6 * dense) * e, "flops": 9 * flops}
    tokens, experts, hidden, ffn, slots = case["tokens"], case["experts"], case["hidden"], case["ffn"], case["tokens"] * case["top_k"]
    # experts that get tokens, and the rows that their blocks hold without any padding
    hit = sum(1.0 - (1.0 - min(1.0, case["top_k"] * p)) ** tokens for p in _expert_probabilities(case))
    weight, all_weights = hit * hidden * ffn, experts * hidden * ffn
    flops = 2.0 * slots * hidden * ffn
    if case["use"] == "infer":
        return {"bytes": (2 * weight + 2 * tokens * hidden) * e, "flops": 2 * flops}
    if case["use"] == "train":
        return {"bytes": (2 * weight + 2 * all_weights + 4 * tokens * hidden) * e, "flops": 6 * flops}
    values, rows = slots * ffn, slots * hidden
    if not train:           # x, both weights in; h, y and the dense weight gradient out
        return {"bytes": (2 * weight + 2 * rows + values + all_weights) * e, "flops": 3 * flops}
    # gradients of three products: two each, the one with respect to h twice
    return {"bytes": (2 * weight + 4 * rows + 2 * values + 4 * all_weights) * e, "flops": 9 * flops}


def tolerance(case):
    if case["use"] == "convert":
        return "exact"
    # The gradients of a layer pass through four roundings to the value type.  Against a dense layer in fp32 they are off by up
    # to 3.8e-3 (largest element 7e-2) in bf16 and 4.2e-4 (1.1e-2) in fp16, the float32 products against fp64 by 4e-7 (4e-6)
    # at an inner size of 512 and with its root beyond.
    return {"bf16": {"rel": 1e-2, "max": 0.2}, "fp16": {"rel": 1.5e-3, "max": 0.03}, "fp32": {"rel": 4e-6, "max": 4e-5}}[case["dtype"]]
