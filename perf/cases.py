"""The work that a DPA4/SeZM program has the operators do, as measurable cases.

One pass of a case is what such a program asks for through the public entry
points: a forward alone where only energies or features are needed
(``"step": False``), or a forward and the gradients that the forces need
(``"step": True``).  Eight kinds of work:

``sum``      ``kernels.segment_sum``: the envelope-weighted aggregation of the
             edge messages.  DeepMD's seam hands over rows of
             ``(lmax + 1)^2 * channels`` floats with an edge and a node scale;
             the standalone operator is used on narrower rows.
``softmax``  ``kernels.segment_softmax``: attention weights per destination,
             one channel per head (4 to 16 in the attention seam), or per
             feature channel (64 and 256 in the operators' latency runs).
``gie``      ``kernels.zonal_scatter``: the geometric initial embedding for
             lmax 1 to 4, with DeepMD's map (one radial slot per degree l) or
             one radial slot per row.
``gie_norm`` ``gie_zonal_scatter_rmsnorm``: the same followed by the RMSNorm
             over each node's row, at inference.
``rmsnorm``  ``kernels.rmsnorm`` over node or edge rows.
``force``    ``kernels.force_assembly``: force and virial of a water-like
             periodic box, every MD step.
``csr``      ``kernels.group_by_source``: run whenever the neighbour list is
             rebuilt.
``chain``    ``edge_stream_combine``: one fused elementwise chain over the
             edge features.

Graphs, features and degrees follow ``bysj_amd/workloads.py``.  The CSR, the
source grouping and the radial slot map belong to the neighbour graph and are
kept by the program from call to call, so ``prepare`` makes them.
"""
from __future__ import annotations

import numpy as np
import torch

from bysj_amd import kernels, workloads
from bysj_amd.kernels.edge_stream import edge_stream_combine
from bysj_amd.kernels.gie import gie_zonal_scatter_rmsnorm

WATER_DEGREE = 90.5      # neighbours within 6 A at 0.1 atoms / A^3
LARGEST_BYTES = 4.0e9    # no drawn case moves more than the largest listed ones
HUB_DEGREE = 512


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # The smallest call: 1,024 destinations, plain sum over 128 channels, with its gradient.
        {"name": "sum_small_step", "kind": "sum", "nodes": 1024, "degree": 40.0, "channels": 128, "scales": False,
         "ordered": False, "step": True},
        # DeepMD's envelope seam at lmax 3 with 64 channels: rows of 16 * 64 floats, edge and node scales, edges not
        # sorted by destination, in a force evaluation of a 3,000-atom box.
        {"name": "sum_message_step", "kind": "sum", "nodes": 3000, "degree": 90.5, "channels": 1024, "scales": True,
         "ordered": True, "step": True},
        # Attention weights of 8 heads over 16,384 destinations, 1% of them hubs of degree 512.
        {"name": "softmax_heads", "kind": "softmax", "nodes": 16384, "degree": 48.0, "hubs": 0.01, "channels": 8,
         "null": True, "ordered": False, "step": False},
        # Per-channel attention, 64 channels, 3,000 atoms with about 60 neighbours, in a force evaluation.
        {"name": "softmax_c64_step", "kind": "softmax", "nodes": 3000, "degree": 60.6, "hubs": 0.0, "channels": 64,
         "null": True, "ordered": False, "step": True},
        # The same at 256 channels on an 8,192-atom water box.
        {"name": "softmax_c256_step", "kind": "softmax", "nodes": 8192, "degree": 90.5, "hubs": 0.0, "channels": 256,
         "null": True, "ordered": False, "step": True},
        # The geometric initial embedding with DeepMD's map, lmax 3, 64 channels, 24,576 atoms, force evaluation.
        {"name": "gie_lmax3_step", "kind": "gie", "nodes": 24576, "degree": 90.5, "lmax": 3, "channels": 64,
         "slot_per_row": False, "ordered": False, "step": True},
        # Embedding and norm at inference with one radial slot per row, 8,192 atoms.
        {"name": "gie_norm_lmax3", "kind": "gie_norm", "nodes": 8192, "degree": 90.5, "lmax": 3, "channels": 64,
         "slot_per_row": True, "ordered": False, "step": False},
        # RMSNorm of 24,576 node rows of 16 * 64 floats with the gradients of input and scale.
        {"name": "rmsnorm_rows_step", "kind": "rmsnorm", "rows": 24576, "width": 1024, "step": True},
        # Force and virial of 65,536 atoms (5.9M edges) in float32, atoms in no spatial order.
        {"name": "force_f32", "kind": "force", "nodes": 65536, "dtype": "float32", "spatial": False},
        # The same in float64 for a small box, atoms in no spatial order.
        {"name": "force_f64_small", "kind": "force", "nodes": 3000, "dtype": "float64", "spatial": False},
        # Source grouping of that large box when its neighbour list is rebuilt.
        {"name": "csr_sources", "kind": "csr", "nodes": 65536, "degree": 90.5, "sorted": False},
        # silu(x + a * s + b) over edge features of 10 rows of 64 channels, 3,000 atoms.
        {"name": "chain_silu", "kind": "chain", "edges": 271500, "rows": 10, "channels": 64, "activation": "silu"},
    ]


def _log(rng, low, high):
    """An integer spread over the logarithm of [low, high]."""
    return int(round(float(np.exp(rng.uniform(np.log(low), np.log(high))))))


def _draw(rng):
    kind = rng.choice(["sum", "softmax", "softmax", "gie", "gie", "gie_norm", "rmsnorm", "force", "csr", "chain"])
    degree = round(rng.uniform(20.0, 100.0), 1)
    if kind == "sum":
        # per-head features, lmax 1 to 4 messages of 32 to 128 channels, and any other row
        channels = rng.choice([64, 128, 4 * 64, 9 * 64, 16 * 64, 16 * 32, 25 * 32, _log(rng, 5, 1024)])
        return {"kind": kind, "nodes": _log(rng, 256, 65536), "degree": degree, "channels": channels,
                "scales": rng.random() < 0.7, "ordered": rng.random() < 0.5, "step": rng.random() < 0.6}
    if kind == "softmax":
        channels = rng.choice([4, 8, 16, 32, 64, 128, 256, _log(rng, 3, 256)])
        return {"kind": kind, "nodes": _log(rng, 256, 65536), "degree": degree,
                "hubs": rng.choice([0.0, 0.0, 0.01]), "channels": channels, "null": rng.random() < 0.7,
                "ordered": rng.random() < 0.4, "step": rng.random() < 0.6}
    if kind in ("gie", "gie_norm"):
        return {"kind": kind, "nodes": _log(rng, 256, 24576), "degree": degree, "lmax": rng.choice([1, 2, 3, 3, 4]),
                "channels": rng.choice([32, 64, 64, 128]), "slot_per_row": rng.random() < 0.3,
                "ordered": rng.random() < 0.4, "step": kind == "gie" and rng.random() < 0.6}
    if kind == "rmsnorm":
        width = rng.choice([64, 128, 256, 512, 1024, 25 * 64, 2048, _log(rng, 33, 4096)])
        return {"kind": kind, "rows": _log(rng, 1, 262144), "width": width, "step": rng.random() < 0.5}
    if kind == "force":
        return {"kind": kind, "nodes": _log(rng, 640, 65536), "dtype": rng.choice(["float32", "float64"]),
                "spatial": rng.random() < 0.4}
    if kind == "csr":
        return {"kind": kind, "nodes": _log(rng, 256, 65536), "degree": degree, "sorted": rng.random() < 0.25}
    return {"kind": kind, "edges": _log(rng, 5000, 300000), "rows": rng.choice([1, 4, 9, 10, 16, 25]),
            "channels": rng.choice([32, 64, 64, 128, _log(rng, 5, 128)]),
            "activation": rng.choice(["none", "silu", "gate"])}


def draw(rng):
    while True:
        case = _draw(rng)
        if work(case)["bytes"] <= LARGEST_BYTES:
            return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    return generator


def _randn(generator, *shape):
    return torch.randn(shape, generator=generator, device="cuda")


def _uniform(generator, low, high, *shape):
    return torch.rand(shape, generator=generator, device="cuda") * (high - low) + low


def _edges(case):
    """``(edges, hubs)``: the mean degree holds over the nodes that are no hubs."""
    hubs = int(round(case["nodes"] * case.get("hubs", 0.0)))
    return int(round((case["nodes"] - hubs) * case["degree"])) + hubs * HUB_DEGREE, hubs


def _graph(case, seed, generator):
    """``(dst, offsets, order)``: in-degrees at least 1, Poisson around the mean for a fixed edge count, with hubs."""
    nodes, (edges, hubs) = case["nodes"], _edges(case)
    host = workloads.rng(seed)
    degrees = np.ones(nodes, dtype=np.int64)
    plain = nodes - hubs
    degrees[hubs:] += host.multinomial(edges - hubs * HUB_DEGREE - plain, np.full(plain, 1.0 / plain))
    degrees[:hubs] = HUB_DEGREE
    counts = torch.from_numpy(host.permutation(degrees)).cuda()
    dst = torch.repeat_interleave(torch.arange(case["nodes"], device="cuda"), counts)
    if not case["ordered"]:
        return dst, kernels.segment_offsets(dst, case["nodes"]), None
    dst = dst[torch.randperm(dst.numel(), generator=generator, device="cuda")].contiguous()
    order, offsets = kernels.group_by_source(dst, case["nodes"])
    return dst, offsets, order


def _rows(lmax):
    return (lmax + 1) ** 2 - 1


def _slots(case):
    """``(slot of each zonal row, number of radial slots)``: one slot per row (slot 0 is the scalar's), or DeepMD's."""
    if case["slot_per_row"]:
        return list(range(1, _rows(case["lmax"]) + 1)), _rows(case["lmax"]) + 1
    return [l - 1 for l in range(1, case["lmax"] + 1) for _ in range(2 * l + 1)], case["lmax"]


def _gate_rows(rows):
    """SeZM's gate map: row 0 takes SiLU, the rows of degree l take gate l - 1."""
    return [-1 if r == 0 else int(np.sqrt(r)) - 1 for r in range(rows)]


def prepare(case, seed):
    generator = _generator(seed)
    return {"case": case, **globals()[f"_prepare_{case['kind']}"](case, seed, generator)}


def _prepare_sum(case, seed, generator):
    dst, offsets, order = _graph(case, seed, generator)
    edges, step = dst.numel(), case["step"]
    state = {"src": _randn(generator, edges, case["channels"]).requires_grad_(step), "dst": dst, "offsets": offsets,
             "order": order, "edge_scale": None, "node_scale": None}
    if case["scales"]:
        state["edge_scale"] = _uniform(generator, 0.05, 1.0, edges).requires_grad_(step)
        state["node_scale"] = torch.rsqrt((offsets[1:] - offsets[:-1]).float() + 1.0)
    if step:
        state["upstream"] = _randn(generator, case["nodes"], case["channels"])
    return state


def _prepare_softmax(case, seed, generator):
    dst, offsets, order = _graph(case, seed, generator)
    step = case["step"]
    features = workloads.segment_softmax_features(dst.numel(), case["nodes"], case["channels"], seed, "cuda",
                                                  null=case["null"], masked_fraction=0.02)
    state = {"dst": dst, "offsets": offsets, "order": order, "logit": features["logit"].requires_grad_(step),
             "env": features["env"].requires_grad_(step), "null_logit": None}
    if case["null"]:
        state["null_logit"] = features["null_logit"].requires_grad_(step)
    if step:
        state["upstream"] = _randn(generator, dst.numel(), case["channels"])
        state["null_upstream"] = _randn(generator, case["nodes"], case["channels"]) if case["null"] else None
    return state


def _prepare_gie(case, seed, generator):
    dst, offsets, _ = _graph(case, seed, generator)
    slots, n_radial = _slots(case)
    edges, step, rows = dst.numel(), case["step"], len(slots)
    inverse = torch.rsqrt((offsets[1:] - offsets[:-1]).float() + 1.0)
    state = {"zonal": _randn(generator, edges, rows).requires_grad_(step),
             "radial": _randn(generator, edges, n_radial, case["channels"]).requires_grad_(step), "dst": dst,
             "radial_slot": torch.tensor(slots, dtype=torch.int64, device="cuda"),
             "inv_sqrt_deg": inverse.requires_grad_(step)}
    if step:
        state["upstream"] = _randn(generator, case["nodes"], rows + 1, case["channels"])
    return state


def _prepare_gie_norm(case, seed, generator):
    state = _prepare_gie(case, seed, generator)
    state["scale"] = _uniform(generator, 0.5, 1.5, (_rows(case["lmax"]) + 1) * case["channels"])
    return state


def _prepare_rmsnorm(case, seed, generator):
    step = case["step"]
    state = {"x": _randn(generator, case["rows"], case["width"]).requires_grad_(step),
             "scale": _uniform(generator, 0.5, 1.5, case["width"]).requires_grad_(step)}
    if step:
        state["upstream"] = _randn(generator, case["rows"], case["width"])
    return state


def _prepare_force(case, seed, generator):
    graph = workloads.water_graph(case["nodes"], seed, spatial_order=case["spatial"], device="cuda")
    dtype = getattr(torch, case["dtype"])
    src, dst = torch.from_numpy(graph.src).cuda(), torch.from_numpy(graph.dst).cuda()
    src_order, src_offsets = kernels.group_by_source(src, case["nodes"])
    gradient = torch.randn((graph.n_edges, 3), generator=generator, device="cuda", dtype=torch.float64)
    return {"grad_edge": (gradient * np.sqrt(0.5)).to(dtype),
            "edge_vec": torch.from_numpy(graph.edge_vec).cuda().to(dtype), "src": src, "dst": dst,
            "dst_offsets": kernels.segment_offsets(dst, case["nodes"]), "src_offsets": src_offsets,
            "src_order": src_order}


def _prepare_csr(case, seed, generator):
    edges = int(case["nodes"] * case["degree"])
    sources = torch.randint(0, case["nodes"], (edges,), generator=generator, device="cuda")
    return {"sources": torch.sort(sources).values if case["sorted"] else sources}


def _prepare_chain(case, seed, generator):
    edges, rows, channels = case["edges"], case["rows"], case["channels"]
    state = {"x": _randn(generator, edges, rows, channels), "a": _randn(generator, edges, rows, channels),
             "s": _uniform(generator, 0.05, 1.0, edges, 1, 1), "b": _randn(generator, edges, rows, channels),
             "gate": None, "gate_rows": None}
    if case["activation"] == "gate":
        state["gate_rows"] = _gate_rows(rows)
        if max(state["gate_rows"]) >= 0:
            state["gate"] = _randn(generator, edges, max(state["gate_rows"]) + 1, channels)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    case = state["case"]
    call = globals()[f"_run_{case['kind']}"]
    if case.get("step"):
        return call(state)
    with torch.no_grad():
        return call(state)


def _gradients(outputs, leaves, upstream):
    return torch.autograd.grad(outputs, leaves, upstream)


def _run_sum(state):
    out = kernels.segment_sum(state["src"], state["dst"], state["offsets"], state["edge_scale"],
                              state["node_scale"], order=state["order"])
    if not state["case"]["step"]:
        return [out]
    leaves = [state["src"]] + ([state["edge_scale"]] if state["case"]["scales"] else [])
    return [out.detach(), *_gradients([out], leaves, [state["upstream"]])]


def _run_softmax(state):
    result = kernels.segment_softmax(state["logit"], state["env"], state["offsets"], state["null_logit"],
                                     order=state["order"])
    outputs = list(result) if state["case"]["null"] else [result]
    if not state["case"]["step"]:
        return outputs
    leaves, upstream = [state["logit"], state["env"]], [state["upstream"]]
    if state["case"]["null"]:
        leaves.append(state["null_logit"])
        upstream.append(state["null_upstream"])
    return [*(out.detach() for out in outputs), *_gradients(outputs, leaves, upstream)]


def _run_gie(state):
    out = kernels.zonal_scatter(state["zonal"], state["radial"], state["dst"], state["radial_slot"],
                                state["inv_sqrt_deg"])
    if not state["case"]["step"]:
        return [out]
    leaves = [state["zonal"], state["radial"], state["inv_sqrt_deg"]]
    return [out.detach(), *_gradients([out], leaves, [state["upstream"]])]


def _run_gie_norm(state):
    return [gie_zonal_scatter_rmsnorm(state["zonal"], state["radial"], state["dst"], state["radial_slot"],
                                      state["inv_sqrt_deg"], state["scale"])]


def _run_rmsnorm(state):
    out = kernels.rmsnorm(state["x"], state["scale"])
    if not state["case"]["step"]:
        return [out]
    return [out.detach(), *_gradients([out], [state["x"], state["scale"]], [state["upstream"]])]


def _run_force(state):
    return list(kernels.force_assembly(state["grad_edge"], state["edge_vec"], state["src"], state["dst"],
                                       state["dst_offsets"], state["src_offsets"], state["src_order"]))


def _run_csr(state):
    return list(kernels.group_by_source(state["sources"], state["case"]["nodes"]))


def _run_chain(state):
    terms = [(1.0, state["x"]), (1.0, state["a"], state["s"]), (1.0, state["b"])]
    return [edge_stream_combine(terms, activation=state["case"]["activation"], gate=state["gate"],
                                gate_rows=state["gate_rows"])]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """Each input read once and each output written once, per direction; a multiply-add counts as two."""
    kind, step = case["kind"], case.get("step", False)
    if kind == "rmsnorm":
        values = case["rows"] * case["width"]
        size = 8 * values + 4 * case["width"] + 4 * case["rows"]
        flops = 4 * values
        if step:
            size += 12 * values + 8 * case["width"] + 4 * case["rows"]
            flops += 10 * values
        return {"bytes": size, "flops": flops}
    if kind == "force":
        edges, value = case["nodes"] * WATER_DEGREE, 4 if case["dtype"] == "float32" else 8
        return {"bytes": edges * (6 * value + 8) + case["nodes"] * (16 + 12 * value), "flops": 24 * edges}
    if kind == "csr":
        return {"bytes": 16 * int(case["nodes"] * case["degree"]) + 8 * (case["nodes"] + 1), "flops": 0}
    if kind == "chain":
        values = case["edges"] * case["rows"] * case["channels"]
        gates = max([g + 1 for g in _gate_rows(case["rows"])]) if case["activation"] == "gate" else 0
        return {"bytes": 16 * values + 4 * case["edges"] * (1 + gates * case["channels"]), "flops": 8 * values}

    nodes, channels = case["nodes"], case["channels"]
    edges, _ = _edges(case)
    csr = 8 * (nodes + 1) + (8 * edges if case["ordered"] else 0)
    if kind == "sum":
        scales = 4 * edges + 4 * nodes if case["scales"] else 0
        size = 4 * edges * channels + 4 * nodes * channels + csr + scales
        flops = (2 if case["scales"] else 1) * edges * channels
        if step:
            dot = case["scales"]  # the rows are read again for the edge scale's gradient only
            size += (8 if dot else 4) * edges * channels + 4 * nodes * channels + csr + scales + (4 * edges if dot else 0)
            flops += (3 if dot else 1) * edges * channels
        return {"bytes": size, "flops": flops}
    if kind == "softmax":
        null = 4 * nodes * channels if case["null"] else 0
        size = 8 * edges * channels + 4 * edges + 2 * null + csr
        flops = 6 * edges * channels
        if step:
            size += 12 * edges * channels + 8 * edges + 3 * null + csr
            flops += 5 * edges * channels
        return {"bytes": size, "flops": flops}
    slots, n_radial = _slots(case)
    rows, used = len(slots), len(set(slots))
    inputs = 4 * edges * (rows + used * channels) + csr + 4 * nodes + 8 * rows
    outputs = 4 * nodes * (rows + 1) * channels
    flops = 2 * edges * rows * channels
    if step:
        inputs += 4 * edges * (rows + used * channels) + csr + 4 * nodes + 8 * rows + 4 * nodes * rows * channels
        outputs += 4 * edges * (rows + n_radial * channels) + 4 * nodes
        flops += 4 * edges * rows * channels
    if kind == "gie_norm":
        inputs += 4 * (rows + 1) * channels
        outputs += 4 * nodes
        flops += 4 * nodes * (rows + 1) * channels
    return {"bytes": inputs + outputs, "flops": flops}


# ---------------------------------------------------------------------------
# tolerances and 64-bit results
# ---------------------------------------------------------------------------

# About four times the largest difference measured between the operators and the
# same sums in 64 bits, over the listed and 45 drawn cases: sum 1.8e-7, softmax
# 3.3e-7 (its gradients), gie and gie_norm 1.9e-7, rmsnorm 1.8e-7 (the scale's
# gradient), force 6.7e-8 in float32 and 3.6e-16 in float64, chain 6.2e-8.
_TOLERANCE = {"sum": 8e-7, "softmax": 1.4e-6, "gie": 8e-7, "gie_norm": 8e-7, "rmsnorm": 8e-7, "chain": 2.5e-7}
_FORCE_TOLERANCE = {"float32": 3e-7, "float64": 1.5e-15}


def tolerance(case):
    if case["kind"] == "csr":
        return "exact"
    if case["kind"] == "force":
        return {"rel": _FORCE_TOLERANCE[case["dtype"]]}
    return {"rel": _TOLERANCE[case["kind"]]}


def exact(case, seed):
    state = prepare(case, seed)
    with torch.no_grad():
        return globals()[f"_exact_{case['kind']}"](case, state)


def _double(tensor):
    return tensor.detach().double()


def _scatter(values, dst, nodes):
    return torch.zeros((nodes,) + values.shape[1:], dtype=torch.float64, device="cuda").index_add_(0, dst, values)


def _exact_sum(case, state):
    src, dst, scales = _double(state["src"]), state["dst"], case["scales"]
    edge_scale = _double(state["edge_scale"])[:, None] if scales else None
    node_scale = _double(state["node_scale"])[:, None] if scales else None
    out = _scatter(src * edge_scale if scales else src, dst, case["nodes"])
    out = out * node_scale if scales else out
    if not case["step"]:
        return [out]
    rows = (_double(state["upstream"]) * node_scale if scales else _double(state["upstream"]))[dst]
    if not scales:
        return [out, rows]
    return [out, rows * edge_scale, (rows * src).sum(1)]


def _exact_softmax(case, state):
    logit, env, dst, nodes = _double(state["logit"]), _double(state["env"]), state["dst"], case["nodes"]
    open_edge = env > 0
    value = logit + 2.0 * torch.log(env.clamp_min(1e-30))[:, None]
    value = torch.where(open_edge[:, None], value, torch.full_like(value, -torch.inf))
    peak = torch.full((nodes, case["channels"]), -torch.inf, dtype=torch.float64, device="cuda")
    peak = peak.scatter_reduce(0, dst[:, None].expand_as(value), value, "amax")
    null = _double(state["null_logit"]) if case["null"] else None
    peak = torch.maximum(peak, null) if case["null"] else peak
    peak = torch.where(torch.isfinite(peak), peak, torch.zeros_like(peak))
    weight = torch.exp(value - peak[dst])
    total = _scatter(weight, dst, nodes)
    null_weight = torch.exp(null - peak) if case["null"] else None
    total = total + null_weight if case["null"] else total
    total = torch.where(total > 0, total, torch.ones_like(total))
    alpha = weight / total[dst]
    null_alpha = null_weight / total if case["null"] else None
    outputs = [alpha, null_alpha] if case["null"] else [alpha]
    if not case["step"]:
        return outputs
    upstream = _double(state["upstream"])
    expect = _scatter(alpha * upstream, dst, nodes)
    if case["null"]:
        null_upstream = _double(state["null_upstream"])
        expect = expect + null_alpha * null_upstream
    grad_logit = alpha * (upstream - expect[dst])
    grad_env = torch.where(open_edge, 2.0 * grad_logit.sum(1) / torch.where(open_edge, env, torch.ones_like(env)),
                           torch.zeros_like(env))
    outputs += [grad_logit, grad_env]
    if case["null"]:
        outputs.append(null_alpha * (null_upstream - expect))
    return outputs


def _exact_gie(case, state):
    zonal, dst, nodes = _double(state["zonal"]), state["dst"], case["nodes"]
    inverse = _double(state["inv_sqrt_deg"])
    slots, n_radial = _slots(case)
    rows = len(slots)
    summed = torch.zeros((nodes, rows + 1, case["channels"]), dtype=torch.float64, device="cuda")
    for r, slot in enumerate(slots):
        summed[:, r + 1] = _scatter(zonal[:, r, None] * _double(state["radial"][:, slot]), dst, nodes)
    out = summed * inverse[:, None, None]
    if not case["step"]:
        return [out]
    upstream = _double(state["upstream"])
    grad_zonal = torch.zeros_like(zonal)
    grad_radial = torch.zeros((dst.numel(), n_radial, case["channels"]), dtype=torch.float64, device="cuda")
    for r, slot in enumerate(slots):
        rows_up = (upstream[:, r + 1] * inverse[:, None])[dst]
        grad_zonal[:, r] = (rows_up * _double(state["radial"][:, slot])).sum(1)
        grad_radial[:, slot] += rows_up * zonal[:, r, None]
    return [out, grad_zonal, grad_radial, (upstream * summed).sum((1, 2))]


def _exact_gie_norm(case, state):
    rows = _exact_gie(case, state)[0]
    flat = rows.reshape(case["nodes"], -1)
    normed = flat * torch.rsqrt(flat.square().mean(1, keepdim=True) + 1e-6) * _double(state["scale"])
    return [normed.reshape(rows.shape)]


def _exact_rmsnorm(case, state):
    x, scale = _double(state["x"]), _double(state["scale"])
    inverse = torch.rsqrt(x.square().mean(1, keepdim=True) + 1e-6)
    out = x * inverse * scale
    if not case["step"]:
        return [out]
    upstream = _double(state["upstream"])
    scaled = upstream * scale
    grad_x = inverse * scaled - x * inverse ** 3 * (x * scaled).mean(1, keepdim=True)
    return [out, grad_x, (upstream * x * inverse).sum(0)]


def _exact_force(case, state):
    gradient, vector, nodes = _double(state["grad_edge"]), _double(state["edge_vec"]), case["nodes"]
    force = _scatter(gradient, state["dst"], nodes) - _scatter(gradient, state["src"], nodes)
    outer = (gradient[:, :, None] * vector[:, None, :]).reshape(-1, 9)
    return [force, -_scatter(outer, state["src"], nodes)]


def _exact_csr(case, state):
    sources, nodes = state["sources"], case["nodes"]
    counts = torch.bincount(sources, minlength=nodes)
    return [torch.argsort(sources, stable=True), torch.cat([counts.new_zeros(1), torch.cumsum(counts, 0)])]


def _exact_chain(case, state):
    total = _double(state["x"]) + _double(state["a"]) * _double(state["s"]) + _double(state["b"])
    if case["activation"] == "none":
        return [total]
    key = total
    if case["activation"] == "gate" and state["gate"] is not None:
        gate = _double(state["gate"])
        key = torch.stack([total[:, r] if g < 0 else gate[:, g] for r, g in enumerate(state["gate_rows"])], 1)
    return [total * torch.sigmoid(key)]
