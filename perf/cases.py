"""What the framework's users have it do, as timed cases.

The kinds, each through the entry points that a program calls:

- ``core``: one layer's attention kernels alone, forward then backward
  (``attn_fwd``, ``attn_bwd``);
- ``op``: the attention with its linears (``attention``, ``attention_bwd``);
- ``layer``: the attention block of a PET layer from its tokens (norm, QKV,
  attention, output linear) and its backward;
- ``mlp``: a SwiGLU MLP on fused dense layers with its input adjoint, the
  weights split once (below 256 columns the short-contraction layers, from
  there the norm's pair rows and block pairs, as the evaluation chains them);
- ``forces``: edge gradients, forces and virials from the cutoff adjoints;
- ``model``: a whole energy, forces and virial evaluation;
- ``md``: a molecular dynamics engine's step, positions in on the host and
  energy, forces and virial out on the host.

Structures are diamond (a 3.567, jittered), water at 1 g/cm^3 and uniformly
random positions at 0.1 atoms per cubic Angstrom (ragged neighbour counts),
all periodic; cutoffs 4 to 8 Angstrom with the cosine factor over the last 0.5.
"""
import math

import numpy as np
import torch

from pet_kokkos_amd import attention as att
from pet_kokkos_amd import forces as frc
from pet_kokkos_amd import layer as lay
from pet_kokkos_amd import linear as lin
from pet_kokkos_amd import model as mdl
from pet_kokkos_amd import systems, weights

WIDTH = 0.5  # of the cutoff factor
DENSITY = 0.1  # atoms per cubic Angstrom of a random box


def listed():
    return [
        # the smallest call: a 64-atom cell's attention, where launches count (d 128, 4 heads of 32)
        {"name": "core-diamond-64", "kind": "core", "structure": "diamond", "atoms": 64, "cutoff": 4.5, "heads": 4,
         "head_dim": 32},
        # the headline workload: 1728 atoms with 70 neighbours each, d 256, 8 heads of 32
        {"name": "core-diamond-1728", "kind": "core", "structure": "diamond", "atoms": 1728, "cutoff": 4.5, "heads": 8,
         "head_dim": 32},
        # ragged neighbourhoods under narrow heads (d 128 in 8 heads of 16), an odd atom count
        {"name": "core-ragged-hd16", "kind": "core", "structure": "random", "atoms": 2047, "cutoff": 4.5, "heads": 8,
         "head_dim": 16},
        # a long cutoff: about 180 neighbours an atom
        {"name": "core-long-cutoff", "kind": "core", "structure": "random", "atoms": 640, "cutoff": 7.5, "heads": 8,
         "head_dim": 32},
        # the ragged stress box through the operator with its linears, d 256
        {"name": "op-ragged-4096", "kind": "op", "structure": "random", "atoms": 4096, "cutoff": 5.0, "heads": 8,
         "head_dim": 32},
        # one attention block of the 128-wide model on 648 atoms of water
        {"name": "layer-water-648", "kind": "layer", "structure": "water", "atoms": 648, "cutoff": 4.5, "heads": 4,
         "head_dim": 32},
        # the edge MLPs of the 128-wide model on that water and of a 512-wide one on a small batch, rows ragged
        {"name": "mlp-128", "kind": "mlp", "rows": 26670, "width": 128, "hidden": 512},
        {"name": "mlp-512", "kind": "mlp", "rows": 62291, "width": 512, "hidden": 1024},
        # the forces' edge term of 1728 atoms
        {"name": "forces-diamond-1728", "kind": "forces", "structure": "diamond", "atoms": 1728, "cutoff": 4.5},
        # energy and forces of 648-atom water, the feedforward family at d 128
        {"name": "model-water-648", "kind": "model", "family": "feedforward", "width": 128, "heads": 4, "hidden": 512,
         "waters": 1, "side": 6, "diamonds": 0},
        # one step of an MD engine on 192 atoms of water, the residual family at d 128
        {"name": "md-water-192", "kind": "md", "family": "residual", "width": 128, "heads": 4, "hidden": 512,
         "side": 4},
        # a batch of structures in one call, the feedforward family at d 512 (head_dim 64)
        {"name": "model-batch-512", "kind": "model", "family": "feedforward", "width": 512, "heads": 8, "hidden": 1024,
         "waters": 2, "side": 6, "diamonds": 2},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["core", "core", "core", "op", "layer", "mlp", "mlp", "forces", "model", "md"])
    if kind in ("core", "op", "layer", "forces"):
        structure = rng.choice(["diamond", "random", "random", "water"])
        cutoff = 4.5
        if structure == "diamond":
            atoms = 8 * rng.randint(2, 6) ** 3
        elif structure == "water":
            atoms = 3 * rng.randint(2, 7) ** 3
        else:
            atoms = _log_int(rng, 24, 4096)
            cutoff = round(rng.uniform(4.0, 8.0 if atoms <= 1024 else 5.0), 2)
        case = {"kind": kind, "structure": structure, "atoms": atoms, "cutoff": cutoff}
        if kind != "forces":
            case["heads"], case["head_dim"] = rng.choice([(4, 16), (8, 16), (4, 32), (8, 32), (8, 32), (4, 64), (8, 64),
                                                          (4, 128)])
        return case
    if kind == "mlp":
        width = rng.choice([64, 96, 128, 256, 384, 512])
        rows = _log_int(rng, 300, 120000 if width <= 128 else 62291)
        return {"kind": kind, "rows": rows, "width": width, "hidden": width * (rng.choice([2, 4]) if width < 512 else 2)}
    width, heads = rng.choice([(64, 4), (128, 4), (128, 8), (256, 8)])
    case = {"kind": kind, "family": rng.choice(["feedforward", "residual"]), "width": width, "heads": heads,
            "hidden": width * rng.choice([2, 4])}
    if kind == "md":
        return dict(case, side=rng.randint(2, 5))
    return dict(case, waters=rng.randint(1, 4), side=rng.randint(2, 6), diamonds=rng.randint(0, 3))


# ---- structures and token layouts ---------------------------------------------------


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _positions(case):
    """(positions [N, 3], box length), on the host. The atoms are the case's own,
    so that the rows and slots of its outputs are too; the seed makes the values."""
    n = seed = case["atoms"]
    if case["structure"] == "diamond":
        s = systems.diamond(round((n / 8) ** (1 / 3)), jitter=0.02, seed=seed)
    elif case["structure"] == "water":
        side = round((n / 3) ** (1 / 3))
        s = systems.water_box(side, 3.1 * side, seed=seed)
    else:
        s = systems.random_box(n, DENSITY, seed=seed)
    return s.positions, float(s.cell[0, 0])


def _edges(case):
    """The full directed neighbour list of the periodic cube, grouped by centre:
    off [N + 1], center, reverse (int64) and vec, dist (float64), on the GPU."""
    dev, rc = _device(), case["cutoff"]
    pos, box = _positions(case)
    x = torch.as_tensor(pos, dtype=torch.float64, device=dev)
    n = x.shape[0]
    reach = 0 if box > 2.0 * rc else math.ceil(rc / box) + 1
    side = 2 * reach + 1
    found = []
    for s in range(side ** 3):
        t = (s // (side * side) - reach, s // side % side - reach, s % side - reach)
        v = x[None, :, :] - x[:, None, :]
        if reach == 0:  # the nearest image of each pair
            v -= box * torch.round(v / box)
        else:
            v += box * torch.tensor(t, dtype=torch.float64, device=dev)
        d = (v * v).sum(-1).sqrt_()
        i, j = torch.nonzero((d > 1e-12) & (d <= rc), as_tuple=True)
        found.append(((i * n + j) * side ** 3 + s, (j * n + i) * side ** 3 + (side ** 3 - 1 - s), v[i, j], d[i, j]))
    key, back, vec, dist = (torch.cat([f[q] for f in found]) for q in range(4))
    key, order = torch.sort(key)
    center = key // (n * side ** 3)
    off = torch.zeros(n + 1, dtype=torch.int64, device=dev)
    off[1:] = torch.cumsum(torch.bincount(center, minlength=n), 0)
    reverse = torch.searchsorted(key, back[order]).clamp_(max=max(0, key.numel() - 1))
    reverse = torch.where(key[reverse] == back[order], reverse, torch.full_like(reverse, -1))
    return off, center, reverse, vec[order].contiguous(), dist[order].contiguous()


def _cosine(dist, rc):
    x = ((dist - (rc - WIDTH)) / WIDTH).clamp(0.0, 1.0)
    return 0.5 * (1.0 + torch.cos(math.pi * x))


def _tokens(case):
    """(off int32, slots, cf_seq [N, S], rows, edges): the attention's layout."""
    off, center, _, _, dist = _edges(case)
    n, e = case["atoms"], int(off[-1])
    slots = int((off[1:] - off[:-1]).max()) + 1
    cf = torch.zeros(n, slots, dtype=torch.float32, device=off.device)
    cf[:, 0] = 1.0
    cf[center, 1 + torch.arange(e, device=off.device) - off[center]] = _cosine(dist, case["cutoff"]).float()
    return off.int(), slots, cf, n + e


def _randn(gen, *shape, scale=1.0):
    return torch.randn(*shape, generator=gen, device=gen.device, dtype=torch.float32) * scale


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(seed)


def _linear_init(gen, out, inp):
    return _randn(gen, out, inp, scale=inp ** -0.5), _randn(gen, out, scale=0.1)


# ---- preparation ---------------------------------------------------------------------


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _prepare_core(case, seed):
    off, slots, cf, rows = _tokens(case)
    gen = _generator(seed)
    h, d = case["heads"], case["heads"] * case["head_dim"]
    n, dev = case["atoms"], off.device
    w_in, b_in = _linear_init(gen, 3 * d, d)
    new = lambda *s: torch.empty(*s, dtype=torch.float32, device=dev)
    return {"case": case, "off": off, "cf": cf, "qkv": _randn(gen, rows, d) @ w_in.T + b_in,
            "dmerged": _randn(gen, rows, d), "merged": new(rows, d), "ml": new(n * h * slots, 2),
            "qkv_adj": new(rows, 3 * d), "cfh": new(n, h, slots), "cf_adj": new(n, slots)}


def _run_core(s):
    h, hd = s["case"]["heads"], s["case"]["head_dim"]
    att.attn_fwd(s["qkv"], s["off"], s["cf"], h, hd, merged=s["merged"], ml=s["ml"])
    s["cf_adj"].zero_()
    att.attn_bwd(s["qkv"], s["off"], s["dmerged"], s["merged"], s["ml"], s["cf"], h, hd, cf_seq_adj=s["cf_adj"],
                 qkv_adj=s["qkv_adj"], cfh=s["cfh"])
    return {"merged": s["merged"], "ml": s["ml"], "qkv_adj": s["qkv_adj"], "cf_adj": s["cf_adj"]}


def _prepare_op(case, seed):
    off, slots, cf, rows = _tokens(case)
    gen = _generator(seed)
    d, n = case["heads"] * case["head_dim"], case["atoms"]
    w_in, b_in = _linear_init(gen, 3 * d, d)
    w_out, b_out = _linear_init(gen, d, d)
    new = lambda *s: torch.empty(*s, dtype=torch.float32, device=off.device)
    return {"case": case, "off": off, "cf": cf, "slots": slots, "w_in": w_in, "w_out": w_out, "b_out": b_out,
            "qkv": _randn(gen, rows, d) @ w_in.T + b_in, "out_adj": _randn(gen, rows, d), "out": new(rows, d),
            "in_adj": new(rows, d), "cf_adj": new(n, slots), "ws": att.Workspace(off.device),
            "tokens": att.Tokens(off, n)}


def _run_op(s):
    c = s["case"]
    args = (s["tokens"], s["slots"], c["heads"], c["head_dim"], 1.0)
    att.attention(s["ws"], "layer", s["out"], s["qkv"], s["cf"], s["w_out"], s["b_out"], *args, True)
    s["cf_adj"].zero_()
    att.attention_bwd(s["ws"], "layer", s["in_adj"], s["cf_adj"], s["out_adj"], s["qkv"], s["cf"], s["w_in"],
                      s["w_out"], *args, 0.0)
    return {"out": s["out"], "in_adj": s["in_adj"], "cf_adj": s["cf_adj"]}


def _prepare_layer(case, seed):
    s = _prepare_op(case, seed)
    gen = _generator(seed + 1)
    rows, d = s["qkv"].shape[0], case["heads"] * case["head_dim"]
    del s["qkv"], s["in_adj"]
    s["x"] = _randn(gen, rows, d)
    s["norm_w"] = 1.0 + _randn(gen, d, scale=0.1)
    s["b_in"] = _randn(gen, 3 * d, scale=0.1)
    s["x_adj"] = torch.empty_like(s["x"])
    return s


def _run_layer(s):
    c = s["case"]
    args = (s["tokens"], s["slots"], c["heads"], c["head_dim"], 1.0)
    lay.attention_layer(s["ws"], "layer", s["out"], s["x"], s["norm_w"], None, s["w_in"], s["b_in"], s["cf"],
                        s["w_out"], s["b_out"], *args)
    s["cf_adj"].zero_()
    s["x_adj"].copy_(s["out_adj"])  # the residual stream's share, onto which the edge rows' adjoint accumulates
    lay.attention_layer_bwd(s["ws"], "layer", s["x_adj"], s["cf_adj"], s["out_adj"], s["x"], s["norm_w"], None,
                            s["w_in"], s["b_in"], s["cf"], s["w_out"], *args)
    return {"out": s["out"], "x_adj": s["x_adj"], "cf_adj": s["cf_adj"]}


def _chained(width, hidden):
    """Whether the MLP's activations pass between its products as block pairs."""
    return width >= 256 and hidden >= 512


def _prepare_mlp(case, seed):
    gen = _generator(seed)
    m, d, f = case["rows"], case["width"], case["hidden"]
    w_in, b_in = _linear_init(gen, 2 * f, d)  # rows interleaved (value, gate)
    w_out, b_out = _linear_init(gen, d, f)
    new = lambda *s: torch.empty(*s, dtype=torch.float32, device=gen.device)
    s = {"case": case, "x": _randn(gen, m, d), "norm_w": 1.0 + _randn(gen, d, scale=0.1), "w_in": w_in, "b_in": b_in,
         "w_out": w_out, "b_out": b_out, "y_adj": _randn(gen, m, d), "pre": new(m, 2 * f), "y": new(m, d),
         "z_adj": new(m, d)}
    split = lambda w, transposed=False: (lin.SplitWeights(w, transposed) if (w.shape[0] if transposed else w.shape[1]) > 128
                                         else lin.PairWeights(w.T.contiguous() if transposed else w))
    s["in"], s["out"] = split(w_in), split(w_out)
    s["out_t"], s["in_t"] = split(w_out, True), split(w_in, True)
    if _chained(d, f):
        s["h"], s["pre_adj"] = lin.BlockPairs(m, f, gen.device), lin.BlockPairs(m, 2 * f, gen.device)
        s["scratch"] = torch.empty((m + 128) * (4 * d + 4), dtype=torch.uint8, device=gen.device)
    else:
        s["z"], s["h"], s["pre_adj"] = new(m, d), new(m, f), new(m, 2 * f)
    return s


def _run_mlp(s):
    """y = x + W_out swiglu(W_in norm(x) + b_in) + b_out, then the adjoint of the normed input."""
    if _chained(s["case"]["width"], s["case"]["hidden"]):
        lay.norm_rows(s["z_adj"], s["x"], s["norm_w"], None)  # the normed rows, until the backward's adjoint takes their place
        lin.fused_to_blocks(s["z_adj"], s["in"], s["h"], bias=s["b_in"], pre=s["pre"], act=2, scratch=s["scratch"])
        lin.fused(s["h"], s["out"], s["y"], bias=s["b_out"], cin=s["x"], beta=1.0)
        lin.fused_to_blocks(s["y_adj"], s["out_t"], s["pre_adj"], cin=s["pre"], act=4, scratch=s["scratch"])
    else:
        lay.norm_rows(s["z"], s["x"], s["norm_w"], None)
        lin.swiglu_in_fused(s["pre"], s["h"], s["z"], s["in"], s["b_in"])
        lin.fused(s["h"], s["out"], s["y"], bias=s["b_out"], cin=s["x"], beta=1.0)
        lin.fused(s["y_adj"], s["out_t"], s["pre_adj"], cin=s["pre"], act=4)
    lin.fused(s["pre_adj"], s["in_t"], s["z_adj"])
    return {"y": s["y"], "pre": s["pre"], "z_adj": s["z_adj"]}


def _prepare_forces(case, seed):
    off, center, reverse, vec, dist = _edges(case)
    gen = _generator(seed)
    n, e = case["atoms"], center.numel()
    slots = int((off[1:] - off[:-1]).max()) + 1
    pk = frc.PackedEdges(off.int(), center.int(), reverse.int(), vec, dist, torch.full_like(dist, case["cutoff"]))
    return {"case": case, "pk": pk, "soff": torch.tensor([0, n], dtype=torch.int32, device=off.device),
            "x4_adj": _randn(gen, e, 4), "cutoff_adj": _randn(gen, e), "cf_adj": _randn(gen, n, slots)}


def _run_forces(s):
    f, v, g = frc.forces_and_virial(s["pk"], s["case"]["atoms"], s["soff"], s["x4_adj"], s["cutoff_adj"], s["cf_adj"],
                                    WIDTH, "cosine")
    return {"forces": f, "virial": v, "edge_grad": g}


def _hypers(case):
    w = case["width"]
    res = case["family"] == "residual"
    return weights.Hypers(d_pet=w, d_node=w if res else 2 * w, d_head=128, d_feedforward=case["hidden"],
                          num_heads=case["heads"], featurizer=case["family"])


def _model_inputs(case, seed):
    """(hypers, weights, composition, structures): per-species energies all of
    one sign and some eV, as a fitted composition model's are."""
    h = _hypers(case)
    st = [systems.water_box(case["side"], 3.1 * case["side"], seed=seed + k) for k in range(case.get("waters", 1))]
    st += [systems.diamond(2, jitter=0.01, seed=seed + k) for k in range(case.get("diamonds", 0))]
    comp = -2.0 - 10.0 * np.random.default_rng(seed).random(h.n_species)
    return h, weights.random_weights(h, seed), comp, st


def _prepare_model(case, seed):
    h, w, comp, st = _model_inputs(case, seed)
    return {"case": case, "model": mdl.PetModel(h, w, comp), "x": mdl.structures_input(h, st, _device()), "out": None}


def _run_model(s):
    s["out"] = s["model"].compute(s["x"], out=s["out"])
    return s["out"]


def _prepare_md(case, seed):
    h, w, comp, (st,) = _model_inputs(case, seed)
    calc = mdl.Calculator(mdl.PetModel(h, w, comp), _device())
    e = systems.neighbor_list(st, h.cutoff)
    offsets = np.concatenate([[0], np.cumsum(np.bincount(e.centre, minlength=len(st.positions)))])
    calc.set_neighbors(st.numbers, offsets, e.neigh, e.shift)
    return {"case": case, "calc": calc, "positions": st.positions, "cell": st.cell}


def _run_md(s):
    return s["calc"].compute_step(s["positions"], s["cell"])


# ---- what a pass cannot do without -----------------------------------------------------


def _counts(case):
    """(mean edges an atom, mean squared tokens an atom) of a case's structure."""
    if case["structure"] == "diamond":
        return 70.0, 71.0 ** 2
    m = DENSITY * 4.0 / 3.0 * math.pi * case["cutoff"] ** 3
    return m, (1.0 + m) ** 2 + m


def work(case):
    kind = case["kind"]
    if kind in ("core", "op", "layer"):
        m, c2 = _counts(case)
        n, h, d = case["atoms"], case["heads"], case["heads"] * case["head_dim"]
        t, s = n * (1.0 + m), 1.0 + m
        flops = 14.0 * n * c2 * d
        if kind == "core":  # qkv, the adjoint of merged; merged, its saves, the adjoint of qkv, cf and its adjoint
            return {"bytes": 4 * (8 * t * d + 2 * n * h * s + 2 * n * s), "flops": flops}
        if kind == "op":  # qkv, out_adj, W_in, W_out; out, in_adj
            return {"bytes": 4 * (6 * t * d + 2 * n * s + 4 * d * d), "flops": flops + 2.0 * t * d * d * 5}
        return {"bytes": 4 * (4 * t * d + 2 * n * s + 4 * d * d), "flops": flops + 2.0 * t * d * d * 8}
    if kind == "mlp":
        m, d, f = case["rows"], case["width"], case["hidden"]
        return {"bytes": 4 * (m * (4 * d + 2 * f) + 6 * d * f), "flops": 2.0 * m * 6 * d * f}
    if kind == "forces":
        m, _ = _counts(case)
        n = case["atoms"]
        return {"bytes": n * m * (4 * 5 + 4 * 2 + 8 * 5 + 4 + 8 * 3) + n * (8 * 3 + 8), "flops": n * m * 40.0}
    h = _hypers(case)
    water, diamond = case.get("waters", 1), case.get("diamonds", 0)
    n = water * 3 * case["side"] ** 3 + diamond * 64
    mw = DENSITY * 4.0 / 3.0 * math.pi * h.cutoff ** 3
    e = water * 3 * case["side"] ** 3 * mw + diamond * 64 * 70
    c2 = water * 3 * case["side"] ** 3 * (1 + mw) ** 2 + diamond * 64 * 71 ** 2
    flops = 4.0 * sum(a * b * c for a, b, c in _products(h, n, e))
    flops += h.num_gnn_layers * h.num_attention_layers * 14.0 * c2 * h.d_pet
    params = sum(b * c for _, b, c in _products(h, n, e))
    return {"bytes": 4.0 * params + e * (8 * 5 + 4 * 4) + n * 8 * 4, "flops": flops}


def _products(h, n, e):
    """The dense layers of one forward as (rows, out, in)."""
    d, dn, dh, t, f = h.d_pet, h.d_node, h.d_head, n + e, h.d_feedforward
    head = [(n, dh, dn), (n, dh, dh), (n, 1, dh), (e, dh, d), (e, dh, dh), (e, 1, dh)]
    out = []
    for g in range(h.num_gnn_layers):
        out += [(e, d, d)] * (2 if g else 1)
        block = [(t, 3 * d, d), (t, d, d)]
        if h.residual:
            out += h.num_attention_layers * (block + [(t, f, d), (t, d, f)]) + head
        else:
            out += h.num_attention_layers * (block + [(n, d, dn), (n, dn, d), (n, 4 * dn, dn), (n, dn, 2 * dn),
                                                      (e, 2 * f, d), (e, d, f)])
            out += [(e, 2 * d, 2 * d), (e, d, 2 * d)]
    return out if h.residual else out + head


# (rel, max) of fp32 arithmetic at these lengths: about four times the worst seen
# against exact() over the listed cases and some drawn ones -- core 3.5e-7 (max
# 1.2e-5, where a weight's adjoint cancels), op and layer 6e-7, mlp 3.9e-7, forces
# 8e-8 (32-bit cutoff slopes), whole evaluations 1.5e-6 through all their layers.
TOLERANCE = {"core": (1.5e-6, 6e-5), "op": (2.5e-6, 6e-5), "layer": (2.5e-6, 6e-5), "mlp": (1.6e-6, 3e-5),
             "forces": (3e-7, 1e-5), "model": (6e-6, 6e-5), "md": (6e-6, 6e-5)}


def tolerance(case):
    rel, most = TOLERANCE[case["kind"]]
    return {"rel": rel, "max": most}


# ---- the same in 64 bits -----------------------------------------------------------------


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


class _Slots:
    """Rows of each (atom, slot), padded to the widest atom."""

    def __init__(self, off, n, slots):
        off = off.long()
        s = torch.arange(slots, device=off.device)[None, :]
        self.valid = s <= (off[1:] - off[:-1])[:, None]
        rows = torch.where(s == 0, torch.arange(n, device=off.device)[:, None], n + off[:-1, None] + s - 1)
        self.rows = torch.where(self.valid, rows, torch.zeros_like(rows))


def _scores(qkv, cf, sl, heads):
    """(scores [N, H, S, S], v [N, H, S, hd], live [N, S])."""
    n, s = sl.valid.shape
    d = qkv.shape[1] // 3
    q, k, v = (x.contiguous() for x in qkv[sl.rows.reshape(-1)].reshape(n, s, 3, heads, d // heads).permute(2, 0, 3, 1, 4))
    live = sl.valid & (cf > 0)
    log = torch.log(torch.where(live, cf, torch.ones_like(cf)))
    x = (q @ k.transpose(-1, -2).contiguous()) / math.sqrt(d // heads) + log[:, None, None, :]
    return x.masked_fill(~live[:, None, None, :], -math.inf), v, live


def _attend(qkv, cf, sl, heads):
    """merged [T, D] of qkv [T, 3D]."""
    x, v, live = _scores(qkv, cf, sl, heads)
    out = (torch.softmax(x, -1) @ v).transpose(1, 2) * live[:, :, None, None]
    n, s = sl.valid.shape
    ok = sl.valid.reshape(-1)
    return qkv.new_zeros(qkv.shape[0], qkv.shape[1] // 3).index_copy(
        0, sl.rows.reshape(-1)[ok], out.reshape(n * s, -1)[ok])


def _double(state, *names):
    return [state[k].double() for k in names]


def _exact_core(case, seed):
    s = _prepare_core(case, seed)
    h = case["heads"]
    qkv, cf, g = _double(s, "qkv", "cf", "dmerged")
    sl = _Slots(s["off"], case["atoms"], cf.shape[1])
    qkv.requires_grad_(), cf.requires_grad_()
    merged = _attend(qkv, cf, sl, h)
    qkv_adj, cf_adj = torch.autograd.grad(merged, [qkv, cf], g)
    with torch.no_grad():
        x, _, live = _scores(qkv, cf, sl, h)
        top = x.amax(-1)
        inv = 1.0 / torch.exp(x - top[..., None]).sum(-1)
        keep = live[:, None, :].expand_as(top)
        ml = torch.stack([torch.where(keep, top, torch.full_like(top, float(np.float32(-1e30)))),
                          torch.where(keep, inv, torch.zeros_like(inv))], -1)
    return {"merged": merged.detach(), "ml": ml.reshape(-1, 2), "qkv_adj": qkv_adj, "cf_adj": cf_adj}


def _exact_op(case, seed):
    s = _prepare_op(case, seed)
    qkv, cf, w_in, w_out, b_out, g = _double(s, "qkv", "cf", "w_in", "w_out", "b_out", "out_adj")
    sl = _Slots(s["off"], case["atoms"], cf.shape[1])
    qkv.requires_grad_(), cf.requires_grad_()
    out = _attend(qkv, cf, sl, case["heads"]) @ w_out.T + b_out
    qkv_adj, cf_adj = torch.autograd.grad(out, [qkv, cf], g)
    return {"out": out.detach(), "in_adj": qkv_adj @ w_in, "cf_adj": cf_adj}


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 2.0 ** -23) * w


def _layer_norm(x, w, b):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w + b


def _exact_layer(case, seed):
    s = _prepare_layer(case, seed)
    x, cf, nw, w_in, b_in, w_out, b_out, g = _double(s, "x", "cf", "norm_w", "w_in", "b_in", "w_out", "b_out",
                                                     "out_adj")
    sl = _Slots(s["off"], case["atoms"], cf.shape[1])
    x.requires_grad_(), cf.requires_grad_()
    out = _attend(_rms(x, nw) @ w_in.T + b_in, cf, sl, case["heads"]) @ w_out.T + b_out
    x_adj, cf_adj = torch.autograd.grad(out, [x, cf], g)
    x_adj[case["atoms"]:] += g[case["atoms"]:]  # the atoms' rows are set, the edges' accumulated
    return {"out": out.detach(), "x_adj": x_adj, "cf_adj": cf_adj}


def _exact_mlp(case, seed):
    s = _prepare_mlp(case, seed)
    x, nw, w_in, b_in, w_out, b_out, g = _double(s, "x", "norm_w", "w_in", "b_in", "w_out", "b_out", "y_adj")
    z = _rms(x, nw)
    pre = z @ w_in.T + b_in
    value, gate = pre[:, 0::2], torch.sigmoid(pre[:, 1::2])
    y = x + (value * gate) @ w_out.T + b_out
    h_adj = g @ w_out
    pre_adj = torch.stack([h_adj * gate, h_adj * value * gate * (1.0 - gate)], -1).reshape(pre.shape)
    return {"y": y, "pre": pre, "z_adj": pre_adj @ w_in}


def _exact_forces(case, seed):
    s = _prepare_forces(case, seed)
    pk, rc, n = s["pk"], case["cutoff"], case["atoms"]
    center, e = pk.center.long(), pk.n_edges
    slot = 1 + torch.arange(e, device=center.device) - pk.off.long()[center]
    x4, cut = _double(s, "x4_adj", "cutoff_adj")
    cut = cut + s["cf_adj"].double()[center, slot]
    x = (pk.dist - (rc - WIDTH)) / WIDTH
    slope = torch.where((x > 0) & (x < 1), -0.5 * math.pi * torch.sin(math.pi * x) / WIDTH, torch.zeros_like(x))
    g = x4[:, :3] + (x4[:, 3] + cut * slope)[:, None] * pk.vec / pk.dist[:, None]
    rev = pk.reverse.long()
    pull = g - torch.where((rev >= 0)[:, None], g[rev.clamp(min=0)], torch.zeros_like(g))
    forces = torch.zeros(n, 3, dtype=torch.float64, device=g.device).index_add(0, center, pull)
    return {"forces": forces, "virial": (pk.vec.T @ g).reshape(1, 9), "edge_grad": g}


def _exact_model(case, seed):
    h, w, comp, st = _model_inputs(case, seed)
    x = mdl.structures_input(h, st, _device())
    w = {k: torch.as_tensor(v, dtype=torch.float64, device=x.vec.device) for k, v in w.items()}
    comp = torch.as_tensor(comp, device=x.vec.device)
    n, off, sp, nsp, rev = x.n_atoms, x.off.long(), x.species.long(), x.neigh_species.long(), x.reverse.long()
    center = x.center.long()
    vec = x.vec.clone().requires_grad_()
    dist = torch.sqrt((vec * vec).sum(1))
    smooth = _cosine(dist, h.cutoff)
    cut = x.cut.double() + (smooth - smooth.detach())  # the factors as given, their slope in 64 bits
    sl = _Slots(off, n, x.max_neighbors + 1)
    e = center.numel()
    cf = torch.zeros_like(sl.valid, dtype=torch.float64)
    cf[:, 0] = 1.0
    cf = cf.index_put((center, 1 + torch.arange(e, device=off.device) - off[center]), cut)
    x4 = torch.cat([vec, dist[:, None]], 1)
    lin_ = lambda y, k: y @ w[k + ".weight"].T + w[k + ".bias"]
    silu = torch.nn.functional.silu

    def swiglu(y, k):
        v, g = lin_(y, k + ".w_in").chunk(2, 1)
        return lin_(v * torch.sigmoid(g), k + ".w_out")

    def head(y, side, i):
        k = f"{side}_heads.energy.{i}"
        return lin_(silu(lin_(silu(lin_(y, k + ".0")), k + ".2")), f"{side}_last_layers.energy.{i}.energy___0")[:, 0]

    def readout(node, edge, i):
        return head(node, "node", i).index_add(0, center, cut * head(edge, "edge", i))

    def compress(g, edge):
        parts = [lin_(x4, g + ".edge_embedder")]
        if g + ".neighbor_embedder.weight" in w:
            parts.append(w[g + ".neighbor_embedder.weight"][nsp])
        return lin_(silu(lin_(torch.cat(parts + [edge], 1), g + ".compress.0")), g + ".compress.2")

    def message(y):
        return torch.where((rev >= 0)[:, None], y[rev.clamp(min=0)], torch.zeros_like(y))

    def attention(y, t):
        m = _attend(lin_(y, t + ".attention.input_linear"), cf, sl, h.num_heads)
        return lin_(m, t + ".attention.output_linear")

    edge_in = w["edge_embedder.weight"][nsp]
    node = None if h.residual else w["node_embedders.0.weight"][sp]
    net = 0.0
    for i in range(h.num_gnn_layers):
        g = f"gnn_layers.{i}"
        edge = compress(g, edge_in)
        if h.residual:
            tok = torch.cat([w[f"node_embedders.{i}.weight"][sp], edge])
        for a in range(h.num_attention_layers):
            t = f"{g}.trans.layers.{a}"
            nw = lambda k: w[f"{t}.{k}.weight"]
            if h.residual:
                tok = _layer_norm(tok + attention(tok, t), nw("norm_attention"), w[t + ".norm_attention.bias"])
                mlp = lin_(silu(lin_(tok, t + ".mlp.w_in")), t + ".mlp.w_out")
                tok = _layer_norm(tok + mlp, nw("norm_mlp"), w[t + ".norm_mlp.bias"])
            else:
                tok = torch.cat([lin_(node, t + ".center_contraction"), edge])
                out = attention(_rms(tok, nw("norm_attention")), t)
                node = node + lin_(out[:n], t + ".center_expansion")
                edge = edge + out[n:]
                node = node + swiglu(_rms(node, nw("norm_center_features")), t + ".center_mlp")
                edge = edge + swiglu(_rms(edge, nw("norm_mlp")), t + ".mlp")
        if h.residual:
            net = net + readout(tok[:n], tok[n:], i)
            edge_in = 0.5 * (edge_in + message(tok[n:]))
        else:
            c = _layer_norm(torch.cat([edge, message(edge)], 1), w[f"combination_norms.{i}.weight"],
                            w[f"combination_norms.{i}.bias"])
            edge_in = edge_in + edge + lin_(silu(lin_(c, f"combination_mlps.{i}.0")), f"combination_mlps.{i}.2")
    if not h.residual:
        net = readout(node, edge_in, 0)
    per_atom = net + comp[sp]
    (grad,) = torch.autograd.grad(per_atom.sum(), vec)
    grad = grad.detach()
    zero = lambda *s: torch.zeros(*s, dtype=torch.float64, device=grad.device)
    struct = torch.repeat_interleave(torch.arange(x.n_struct, device=grad.device), x.struct_off.long().diff())
    forces = zero(n, 3).index_add(0, center, grad - message(grad))
    virial = zero(x.n_struct, 3, 3).index_add(0, struct[center], x.vec[:, :, None] * grad[:, None, :])
    per_atom = per_atom.detach()
    return {"energy": zero(x.n_struct).index_add(0, struct, per_atom), "per_atom": per_atom, "forces": forces,
            "virial": virial}


def _exact_md(case, seed):
    o = _exact_model(case, seed)
    return dict(o, energy=float(o["energy"][0]), virial=o["virial"][0])
