"""What the speed of this package is judged by: passes through its two modules, over the sizes they are used at.

A case names the module ("conv": ``TensorProductConv``, "tp": ``TensorProduct``), a problem of the zoo in
``openequivariance_amd/core/problems.py``, the data type, the layout and the module's flags, the size, and how far
a pass goes:

* "forward": inference of a quantity that needs no gradient;
* "step": forward and backward, i.e. an energy with its forces or a training step on energies;
* "force": forward, backward and the backward of that backward, i.e. a training step on forces.

Convolutions run on radius graphs: one periodic cell ("molecules" = 0) or a batch of separate molecules. A pass gets
edge tensors of its own, as in a program whose neighbour list or batch is new at every step; forward and backward
of the pass share them.
"""

import math

import numpy as np
import torch

import openequivariance_amd as oeq
from openequivariance_amd.core import problems as zoo
from openequivariance_amd.core.cg import wigner_3j
from openequivariance_amd.core.graph import CoordGraph, periodic_radius_graph

CUTOFF = 5.0


def _problem_makers():
    groups = (zoo.mace_problems, zoo.nequip_problems, zoo.nequix_problems, zoo.seven_net_problems,
              zoo.diffdock_problems, zoo.e3tools_problems)
    makers = {}
    for group in groups:
        for i, p in enumerate(group()):
            makers[p.label] = lambda group=group, i=i: group()[i]
    makers["nequip-uvu"] = zoo.config2_nequip_uvu
    makers["mace-uvu"] = zoo.config3_mace_uvu
    makers["uvw-shared"] = zoo.config4_uvw_shared
    return makers


_MAKERS = _problem_makers()


def _case(op, problem, run, nodes, degree=0, molecules=0, dtype="float32", layout="mul_ir", deterministic=False,
          kahan=False, name=None):
    c = dict(op=op, problem=problem, run=run, nodes=int(nodes), degree=float(degree), molecules=int(molecules),
             dtype=dtype, layout=layout, deterministic=bool(deterministic), kahan=bool(kahan))
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # molecular dynamics of a small cell: one energy + forces evaluation, where latency and launches count
        _case("conv", "mace-medium", "step", 192, 32, name="md-small-cell"),
        # training on forces with a batch of small molecules (21 atoms each), the usual way NequIP models are trained
        _case("conv", "nequip-revmd17-aspirin", "force", 16 * 21, 12, molecules=16, name="force-training-molecules"),
        # molecular dynamics of a crystal of medium size, mixed multiplicities
        _case("conv", "SevenNet_l3i5-main-layers", "step", 2003, 40, name="md-crystal"),
        # energies of a liquid snapshot, component-major layout, caller-sorted edges
        _case("conv", "nequip-lips", "forward", 5000, 28, layout="ir_mul", deterministic=True, name="inference-liquid"),
        # the headline layer: training batch of large cells, bitwise reproducible mode
        _case("conv", "mace-uvu", "step", 20000, 32, deterministic=True, name="train-large"),
        # the same training batch size as most users have, in the default mode (edges in any order)
        _case("conv", "mace-large", "step", 6001, 32, name="train-default-mode"),
        # double precision, as geometry optimisation and phonons want it
        _case("conv", "mace-large", "step", 1500, 32, dtype="float64", deterministic=True, name="relax-double"),
        # training on forces with a batch of cells
        _case("conv", "mace-large", "force", 3000, 32, deterministic=True, name="force-training-cells"),
        # docking score model: fully connected product with weights per edge
        _case("conv", "DiffDock-L=1", "step", 3000, 20, name="docking-score"),
        # the product on its own, gathered rows supplied by the caller: ordinary and small batches
        _case("tp", "mace-uvu", "step", 50000, name="product-channelwise"),
        _case("tp", "nequip-water", "step", 777, name="product-small"),
        # fully connected product with one weight tensor for all rows (self-interaction, readout)
        _case("tp", "uvw-shared", "step", 100003, name="product-shared-weights"),
    ]


# what a drawn case is taken from: (op, problems, directions, data types, size range, degree range)
_CONV_SMALL = ("mace-medium", "nequip-revmd17-aspirin", "nequip-water", "nequip-uvu", "mace-large")
_CONV_WIDE = ("mace-large", "mace-medium", "nequip-lips", "nequip-revmd17-toluene", "nequix-mp-1-main_layers",
              "SevenNet_l3i5-main-layers", "SevenNet_l3i5-first-layer", "SevenNet_l3i5-last-layer", "mace-uvu")
_FAMILIES = (
    ("conv", _CONV_SMALL, ("forward", "step", "force"), ("float32",), (40, 1000), (8, 40)),
    ("conv", _CONV_WIDE, ("forward", "step", "step", "force"), ("float32",), (500, 12000), (16, 48)),
    ("conv", ("mace-medium", "mace-large", "nequip-lips"), ("forward", "step"), ("float64",), (100, 3000), (16, 40)),
    ("conv", ("DiffDock-L=1", "DiffDock-L=2", "e3tools_conv"), ("forward", "step"), ("float32",), (200, 5000), (8, 30)),
    ("tp", ("mace-uvu", "mace-medium", "nequip-lips", "nequip-water", "nequix-mp-1-main_layers"),
     ("forward", "step", "step"), ("float32", "float32", "float64"), (100, 50000), (0, 0)),
    ("tp", ("uvw-shared", "e3tools_transformer"), ("forward", "step"), ("float32",), (500, 150000), (0, 0)),
)


def draw(rng):
    op, problems, runs, dtypes, sizes, degrees = rng.choice(_FAMILIES)
    problem, run, dtype = rng.choice(problems), rng.choice(runs), rng.choice(dtypes)
    n = int(round(math.exp(rng.uniform(math.log(sizes[0]), math.log(sizes[1])))))
    if op == "tp":
        return _case(op, problem, run, n, dtype=dtype)
    degree = round(math.exp(rng.uniform(math.log(degrees[0]), math.log(degrees[1]))), 1)
    channelwise = problem not in ("DiffDock-L=1", "DiffDock-L=2", "e3tools_conv")
    deterministic = rng.random() < 0.5
    kahan = channelwise and deterministic and rng.random() < 0.15
    layout = "ir_mul" if channelwise and rng.random() < 0.2 else "mul_ir"
    molecules = 0
    if sizes[0] < 100:
        degree = min(degree, n / 2.6)
        if rng.random() < 0.5:
            atoms = rng.randint(9, 30)
            molecules, degree = max(2, n // atoms), min(degree, 0.7 * atoms)
            n = molecules * atoms
    case = _case(op, problem, run, n, degree, molecules, dtype, layout, deterministic, kahan)
    limit = _moved(listed()[4])
    while _moved(case) > limit:
        case["nodes"] = case["nodes"] // 2
    return case


def _make_problem(case):
    p = _MAKERS[case["problem"]]()
    dt = {"float32": np.float32, "float64": np.float64}[case["dtype"]]
    p.irrep_dtype = p.weight_dtype = dt
    p.layout = case["layout"]
    return p


def _edge_count(case):
    return 2 * int(case["nodes"] * case["degree"] / 2)


def _graph(case, seed):
    """(coordinates, receivers, senders, edge vectors): the given number of shortest pairs, in both directions, of
    random points in a periodic cell or of separate molecules (random points in a ball each)."""
    rng = np.random.default_rng(seed)
    n, m, pairs = case["nodes"], case["molecules"], _edge_count(case) // 2
    if m:
        atoms = n // m
        v = rng.normal(size=(m, atoms, 3))
        v *= rng.random((m, atoms, 1)) ** (1.0 / 3.0) / np.linalg.norm(v, axis=2, keepdims=True)
        i, j = np.triu_indices(atoms, 1)
        vec = (v[:, i] - v[:, j]).reshape(-1, 3)
        first = np.arange(m)[:, None] * atoms
        rows, cols, coords = (first + i).reshape(-1), (first + j).reshape(-1), v.reshape(-1, 3)
    else:
        coords, rows, cols, vec = periodic_radius_graph(n, 1.25 * case["degree"], CUTOFF, seed)
        half = len(rows) // 2
        rows, cols, vec = rows[:half], cols[:half], vec[:half]
    assert len(rows) >= pairs, "too few pairs within the cutoff"
    keep = np.argsort(np.linalg.norm(vec, axis=1), kind="stable")[:pairs]
    rows, cols, vec = rows[keep], cols[keep], vec[keep]
    return coords, np.concatenate([rows, cols]), np.concatenate([cols, rows]), np.concatenate([vec, -vec])


def _harmonics(irreps, vec):
    """Real spherical harmonics (component normalisation) of edge vectors, one block per irrep of ``irreps``."""
    v = vec / vec.norm(dim=1, keepdim=True)
    ys = [torch.ones_like(v[:, :1]), math.sqrt(3.0) * v]
    lmax = max(mi.ir.l for mi in irreps)
    for l in range(1, lmax):
        c = torch.from_numpy(np.ascontiguousarray(wigner_3j(l, 1, l + 1))).to(v)
        nxt = torch.einsum("ijk,zi,zj->zk", c, ys[l], ys[1])
        ys.append(nxt * math.sqrt(2 * l + 3) / nxt.norm(dim=1, keepdim=True))
    assert all(mi.mul == 1 for mi in irreps)
    return torch.cat([ys[mi.ir.l] for mi in irreps], dim=1)


def prepare(case, seed):
    p = _make_problem(case)
    dt = getattr(torch, case["dtype"])
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    need_grad = case["run"] != "forward"

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=dev, dtype=dt)

    n, st = case["nodes"], {"run": case["run"], "op": case["op"]}
    if case["op"] == "conv":
        coords, rows, cols, vec = _graph(case, int(seed) % (1 << 31))
        g = CoordGraph(coords, rows.astype(np.int64), cols.astype(np.int64))
        order = g.order
        st["module"] = oeq.TensorProductConv(p, deterministic=case["deterministic"], kahan=case["kahan"])
        if case["deterministic"]:
            edges = (g.rows, g.cols, g.transpose_perm)
        else:
            shuffle = np.random.default_rng(int(seed)).permutation(g.nnz)
            edges, order = (g.rows[shuffle], g.cols[shuffle]), order[shuffle]
        st["edges"] = tuple(torch.from_numpy(np.ascontiguousarray(e)).to(dev) for e in edges)
        e = g.nnz
        y = _harmonics(p.irreps_in2, torch.from_numpy(np.ascontiguousarray(vec[order])).to(dev)).to(dt)
    else:
        st["module"] = oeq.TensorProduct(p)
        e = n
        y = _harmonics(p.irreps_in2, torch.randn(e, 3, generator=gen, device=dev, dtype=torch.float64)).to(dt)
    x = normal(n, p.irreps_in1.dim)
    w = normal(p.weight_numel) if p.shared_weights else normal(e, p.weight_numel)
    st["inputs"] = tuple(t.requires_grad_(need_grad) for t in (x, y.contiguous(), w))
    if need_grad:
        st["grad"] = normal(n, p.irreps_out.dim)
    if case["run"] == "force":
        # cotangents of the three first-order gradients (what the loss on the forces sends back)
        st["grad"].requires_grad_(True)
        st["cotangents"] = tuple(normal(*t.shape) for t in st["inputs"])
    return st


def run(state):
    module, inputs = state["module"], state["inputs"]
    if state["op"] == "conv":
        edges = [t.clone() for t in state["edges"]]  # this step's neighbour list
        call = lambda x, y, w: module(x, y, w, *edges)
    else:
        call = module
    if state["run"] == "forward":
        with torch.no_grad():
            return call(*inputs)
    z = call(*inputs)
    if state["run"] == "step":
        return (z.detach(), *torch.autograd.grad(z, inputs, state["grad"]))
    first = torch.autograd.grad(z, inputs, state["grad"], create_graph=True)
    second = torch.autograd.grad(first, (*inputs, state["grad"]), state["cotangents"])
    return (z.detach(), *(t.detach() for t in first), *second)


def _counts(case):
    """(problem, edges or rows, multiply-adds of the product of one of them)"""
    p = _make_problem(case)
    fmas = 0
    for ins in p.instructions:
        l1, l2, l3 = (p.irreps_in1[ins.i_in1].ir.l, p.irreps_in2[ins.i_in2].ir.l, p.irreps_out[ins.i_out].ir.l)
        nnz = int(np.count_nonzero(np.abs(wigner_3j(l1, l2, l3)) > 1e-12))
        mul1, mul2, mul3 = (p.irreps_in1[ins.i_in1].mul, p.irreps_in2[ins.i_in2].mul, p.irreps_out[ins.i_out].mul)
        fmas += nnz * mul1 * mul2 + (2 * l3 + 1) * (mul1 * mul2 if ins.connection_mode == "uvu" else mul1 * mul2 * mul3)
    e = case["nodes"] if case["op"] == "tp" else _edge_count(case)
    return p, e, fmas


def _moved(case):
    return work(case)["bytes"]


def work(case):
    p, e, fmas = _counts(case)
    size = 8 if case["dtype"] == "float64" else 4
    n = case["nodes"]
    x, y, z = n * p.irreps_in1.dim, e * p.irreps_in2.dim, n * p.irreps_out.dim
    w = p.weight_numel * (1 if p.shared_weights else e)
    index = e * 8 * (3 if case["deterministic"] else 2) if case["op"] == "conv" else 0
    words, products = x + y + w + z, 1
    if case["run"] != "forward":
        words, products = words + 2 * (x + y + w) + z, 4  # operands and dZ in, three gradients out
    if case["run"] == "force":
        # operands, dZ and three cotangents in, four gradients out; the four gradients of the three-term sum
        words, products = words + 3 * (x + y + w) + 2 * z, products + 12
    return {"bytes": words * size + index, "flops": 2 * fmas * e * products}


def tolerance(case):
    """Four times the largest error measured over all outputs of the listed cases, against the same pass in double
    precision on the same inputs: 1.5e-7 (sums over a node's edges and over paths) for channelwise products, 6.5e-7
    for fully connected ones (each output is a sum over up to 64 channels per path as well). Double precision:
    the same multiple of its rounding unit."""
    unit = 2.0**-53 if case["dtype"] == "float64" else 2.0**-24
    fully_connected = any(i.connection_mode == "uvw" for i in _make_problem(case).instructions)
    return {"rel": (44 if fully_connected else 10) * unit}
