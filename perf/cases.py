"""Performance cases of the FlashCart path: what its users run, through the public entry points.

Three groups:

* whole evaluations of a potential (``FlashCartPotential.predict``): molecular dynamics of a periodic
  crystal and of liquid water, screening of a batch of molecules, and one force-matching training
  step (second derivatives, gradients of every parameter);
* the equivariant operations that a program builds its own layers from (``o3.TensorProduct`` as a
  convolution and row by row, ``o3.LinearLayer``, the edge basis), forward and backward;
* the neighbour list on the GPU.

``exact`` restates each of them in plain float64 torch, from the formulas: symmetric traceless
projections built numerically, contractions as dense matrices, derivatives by autograd.
"""

import functools
import itertools
import math

import numpy as np
import torch
import torch.utils.checkpoint

from flashcart_amd import o3
from flashcart_amd.data import AtomicGraph, NeighborList, batch_graphs
from flashcart_amd.data.synthetic import fcc_alloy, model_config, molecules, water_box
from flashcart_amd.model import FlashCartPotential
from flashcart_amd.nn import BesselBasis, PolynomialCutoff
from flashcart_amd.o3._graph import build_graph

DEVICE = "cuda:0"
R_MAX = 5.0
FCC = ["Cu", "Ni", "Fe", "Cr"]
ORGANIC = ["H", "C", "N", "O"]


def listed():
    return [
        # MD of a small periodic cell (32 atoms) with the flagship model, replayed as a HIP graph:
        # the smallest call, bound by launches and latency
        dict(name="md_fcc_32", path="model", system="fcc", nx=2, ny=2, nz=2, channels=128, l_max=3, mode="replay"),
        # MD of 512 water molecules with the 64-channel model, replayed: an ordinary MD box
        dict(name="md_water_1536", path="model", system="water", n_mol=512, channels=64, l_max=2, mode="replay"),
        # screening: energies and forces of a batch of 512 molecules of 20 to 50 atoms, a new batch every call
        dict(name="molecules_512", path="model", system="molecules", n_mol=512, channels=64, l_max=2, mode="eager"),
        # large MD: 25,000 atoms with the flagship model, the neighbour list changing from step to step
        dict(name="md_fcc_25k", path="model", system="fcc", nx=25, ny=25, nz=10, channels=128, l_max=3, mode="eager"),
        # one force-matching training step: energies, forces, gradients of all parameters
        dict(name="train_molecules_192", path="train", n_mol=192, channels=128, l_max=3),
        # convolution product of a small layer on a small graph, all three gradients: the smallest product
        dict(name="conv_2x2_2_small", path="conv", rows=512, edges=4096, l1=2, l2=2, lo=2, channels=32),
        # convolution product of the flagship's second layer at the size of an ordinary training batch,
        # weights per edge, all three gradients
        dict(name="conv_2x3_3_batch", path="conv", rows=2048, edges=88466, l1=2, l2=3, lo=3, channels=128),
        # node-wise product of a product layer (shared weights per path) at the size of a training batch
        dict(name="rows_3x3_3", path="rows", rows=6691, l1=3, l2=3, lo=3, channels=128, shared=True, reduced=False),
        # equivariant linear map that mixes the paths of that product, forward, input and weight gradients
        dict(name="linear_paths_25k", path="linear", rows=25000, l_in=3, l_out=3, fin=128, fout=128,
             paths="4,6,7,6", dtype="float32"),
        # the same layer in float64 (reference calculations, gradient checks), one channel block
        dict(name="linear_f64", path="linear", rows=1501, l_in=2, l_out=2, fin=64, fout=64, paths="1,1,1",
             dtype="float64"),
        # angular and radial basis of 200,000 edges with the gradient of the edge vectors
        dict(name="edge_basis_200k", path="basis", edges=200000, l_max=3, n_radial=8),
        # neighbour list of the 25,000-atom crystal at cutoff + skin from positions on the GPU
        dict(name="neighbors_fcc_25k", path="neighbors", nx=25, ny=25, nz=10, cutoff=6.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cells(rng, lo, hi):
    """nx, ny, nz of a box of about exp(U(log lo, log hi)) fcc cells, not cubic."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    side = n ** (1.0 / 3.0)
    nx = max(2, round(side * rng.uniform(0.8, 1.25)))
    ny = max(2, round(side))
    return dict(nx=nx, ny=ny, nz=max(2, round(n / (nx * ny))))


def draw(rng):
    path = rng.choice(["model", "model", "model", "train", "conv", "conv", "rows", "linear", "linear", "basis",
                       "neighbors"])
    if path == "model":
        system = rng.choice(["fcc", "water", "molecules"])
        case = dict(path=path, system=system, channels=rng.choice([32, 64, 64, 128, 128]), l_max=rng.choice([2, 3]),
                    mode=rng.choice(["eager", "replay"]))
        if system == "fcc":
            case.update(_cells(rng, 8, 5000))
        else:
            case.update(n_mol=_log_int(rng, 4, 512))
        return case
    if path == "train":
        return dict(path=path, n_mol=_log_int(rng, 4, 160), channels=rng.choice([32, 64, 128]),
                    l_max=rng.choice([2, 3]))
    if path == "conv":
        l1, l2, lo = rng.choice([(0, 3, 3), (1, 2, 2), (2, 2, 2), (2, 3, 3)])
        rows = _log_int(rng, 40, 6000)
        return dict(path=path, rows=rows, edges=_log_int(rng, 8 * rows, 50 * rows), l1=l1, l2=l2, lo=lo,
                    channels=rng.choice([16, 32, 64, 96, 128]))
    if path == "rows":
        l, lo = rng.choice([(2, 0), (2, 2), (3, 0), (3, 2), (3, 3)])
        return dict(path=path, rows=_log_int(rng, 30, 25000), l1=l, l2=l, lo=lo, channels=rng.choice([16, 32, 64, 128]),
                    shared=rng.random() < 0.75, reduced=rng.random() < 0.35)
    if path == "linear":
        f64 = rng.random() < 0.25
        l_in = rng.choice([0, 1, 2, 3])
        mixed = rng.random() < 0.5
        # float64 weighs in bytes and in operations: its rows stay within the same cost
        return dict(path=path, rows=_log_int(rng, 30, 8000 if f64 else 25000), l_in=l_in,
                    l_out=rng.choice([l_in, rng.randint(0, l_in)]), fin=rng.choice([16, 32, 33, 64, 96, 128]),
                    fout=rng.choice([16, 32, 64, 100, 128]),
                    paths=",".join(str(rng.randint(1, 7) if mixed else 1) for _ in range(l_in + 1)),
                    dtype="float64" if f64 else "float32")
    if path == "basis":
        return dict(path=path, edges=_log_int(rng, 500, 600000), l_max=rng.choice([1, 2, 3]),
                    n_radial=rng.choice([4, 8, 10]))
    return dict(path=path, cutoff=rng.choice([4.0, 4.75, 5.4, 6.0]), **_cells(rng, 27, 6250))


# -- inputs ----------------------------------------------------------------------------------------------------------

def _gen(seed, device=DEVICE):
    return torch.Generator(device=device).manual_seed(0x5EED + 7919 * int(seed))


def _system(case, seed):
    """(elements, graph) of a model case: float32 graph on the host, neighbour list at R_MAX."""
    system = case.get("system", "molecules")
    if system == "molecules":
        # the sizes belong to the case, the molecules to the seed
        sizes = np.random.default_rng(case["n_mol"]).integers(20, 51, size=case["n_mol"])
        mols = [molecules(1, n_min=int(s), n_max=int(s), seed=100003 * seed + k)[0] for k, s in enumerate(sizes)]
        return ORGANIC, batch_graphs([AtomicGraph.from_arrays(z, p, ORGANIC, R_MAX) for z, p in mols])
    if system == "water":
        # at least 18 molecules, so that the box is wider than the smallest distance its builder keeps
        numbers, pos, cell, pbc = water_box(max(18, case["n_mol"]), density=0.9, seed=seed)
        elements = ["H", "O"]
    else:
        numbers, pos, cell, pbc = fcc_alloy(case["nx"], case["ny"], case["nz"], seed=seed)
        elements = FCC
    return elements, AtomicGraph.from_arrays(numbers, pos, elements, R_MAX, cell=cell, pbc=pbc)


def _model(case, seed, elements, graph):
    """A potential with the packaged architecture on the host. A trained model has no weights that are
    all zero or all one, as some of its initial ones are: every parameter is moved a little. And its
    site energies are binding energies, of one sign: those of the random one would cancel in a sum."""
    avg = graph.edge_index.shape[1] / graph.num_nodes
    torch.manual_seed(1234 + seed)
    model = FlashCartPotential.from_config(model_config(elements, case["channels"], case["l_max"], r_max=R_MAX,
                                                        avg_neighbors=avg))
    with torch.no_grad():
        for p in model.parameters():
            p.add_(0.1 * torch.randn_like(p))
        model.readout.readout_mlp[-1].weight.abs_()
    return model


def _targets(graph, seed):
    """Reference energies and forces of a training batch."""
    g = _gen(seed, "cpu")
    n = graph.n_atoms.to(torch.float32)
    return 0.1 * n * torch.randn(n.shape, generator=g), torch.randn(graph.positions.shape, generator=g)


def _edges(case, seed):
    """Receiver-sorted random edge list of a convolution (degrees vary around the mean)."""
    g = _gen(seed, "cpu")
    i = torch.randint(0, case["rows"], (case["edges"],), generator=g).sort().values
    j = torch.randint(0, case["rows"], (case["edges"],), generator=g)
    return torch.stack([i, j]).to(DEVICE)


def _directions(n, g):
    v = torch.randn(n, 3, device=DEVICE, generator=g)
    return v / v.norm(dim=-1, keepdim=True)


def _tp_inputs(case, seed):
    g = _gen(seed)
    rand = lambda *shape: torch.randn(*shape, device=DEVICE, generator=g)
    C, paths = case["channels"], _paths(case["l1"], case["l2"], case["lo"])
    d1, d2 = (case["l1"] + 1) ** 2, (case["l2"] + 1) ** 2
    n_out = sum(2 * lo + 1 for lo in range(case["lo"] + 1)) if case.get("reduced") else sum(2 * p[2] + 1 for p in paths)
    rows = case["rows"]
    if case["path"] == "conv":
        # edge attributes: the angular expansion of a unit vector, about 1 a component
        return dict(in1=rand(rows, d1 * C), in2=rand(case["edges"], d2), w=rand(case["edges"], len(paths) * C),
                    go=rand(rows, n_out * C), edges=_edges(case, seed))
    w = 1.0 + 0.1 * rand(*((len(paths) * C,) if case["shared"] else (rows, len(paths) * C)))
    return dict(in1=rand(rows, d1 * C), in2=rand(rows, d2 * C), w=w, go=rand(rows, n_out * C))


def _linear_inputs(case, seed):
    g = _gen(seed)
    dt = getattr(torch, case["dtype"])
    paths = [int(p) for p in case["paths"].split(",")]
    fin, fout, lc = case["fin"], case["fout"], min(case["l_in"], case["l_out"])
    rand = lambda *shape: torch.randn(*shape, device=DEVICE, generator=g, dtype=dt)
    x = rand(case["rows"], sum((2 * l + 1) * fin * paths[l] for l in range(case["l_in"] + 1)))
    go = rand(case["rows"], (case["l_out"] + 1) ** 2 * fout)
    return x, go, [rand(fout, fin * paths[l]) for l in range(lc + 1)], paths


def _basis_inputs(case, seed):
    g = _gen(seed)
    n = case["edges"]
    d = 0.8 + (R_MAX - 0.8) * torch.rand(n, 1, device=DEVICE, generator=g)
    vec = d * _directions(n, g)
    return (vec, torch.randn(n, (case["l_max"] + 1) ** 2, device=DEVICE, generator=g),
            torch.randn(n, case["n_radial"], device=DEVICE, generator=g))


def _box(case, seed):
    # a crystal so cold that no neighbour shell crosses the cutoff (the number of pairs is the case's),
    # its atoms in the order in which a simulation hands them over: any
    _, pos, cell, pbc = fcc_alloy(case["nx"], case["ny"], case["nz"], jitter=0.02, seed=seed)
    return pos[np.random.default_rng(seed).permutation(len(pos))], cell, pbc


def _buckets(names, grads):
    """The gradients of each block of the model as one flat tensor, as an optimizer or a reduction
    over ranks takes them (parameters that the loss does not reach have none)."""
    blocks = {}
    for name, grad in zip(names, grads):
        if grad is not None:
            parts = name.split(".")
            key = ".".join(parts[:2 if parts[1].isdigit() else 1])
            blocks.setdefault(key, []).append(grad.reshape(-1))
    return {key: torch.cat(parts) for key, parts in blocks.items()}


def prepare(case, seed):
    path = case["path"]
    if path in ("model", "train"):
        elements, graph = _system(case, seed)
        model = _model(case, seed, elements, graph).to(DEVICE)
        state = dict(path=path, mode=case.get("mode", "train"), model=model, graph=graph.to(DEVICE))
        if path == "train":
            energy, forces = _targets(graph, seed)
            state.update(energy=energy.to(DEVICE), forces=forces.to(DEVICE))
        else:
            for p in model.parameters():
                p.requires_grad_(False)
        return state
    if path in ("conv", "rows"):
        t = _tp_inputs(case, seed)
        C = case["channels"]
        state = dict(path=path, tp=o3.TensorProduct(case["l1"], case["l2"], case["lo"], C, 1 if path == "conv" else C,
                                                    shared_weights=case.get("shared", False),
                                                    reduce_paths=case.get("reduced", False)),
                     args=[t[k].requires_grad_(True) for k in ("in1", "in2", "w")], go=t["go"], graph=None)
        if path == "conv":
            state["graph"] = build_graph(t["edges"], case["rows"])
        return state
    if path == "linear":
        x, go, weights, paths = _linear_inputs(case, seed)
        layer = o3.LinearLayer(case["l_in"], case["l_out"], case["fin"], case["fout"], in_paths=paths)
        layer = layer.to(DEVICE, x.dtype)
        with torch.no_grad():
            for p, w in zip(layer.weight, weights):
                p.copy_(w)
        return dict(path=path, layer=layer, x=x.requires_grad_(True), go=go)
    if path == "basis":
        vec, g_attrs, g_feats = _basis_inputs(case, seed)
        return dict(path=path, vec=vec.requires_grad_(True), grads=(g_attrs, g_feats),
                    irreps=o3.Irreps(case["l_max"]), basis=BesselBasis(case["n_radial"], R_MAX).to(DEVICE),
                    cutoff=PolynomialCutoff(R_MAX, 6).to(DEVICE))
    pos, cell, pbc = _box(case, seed)
    return dict(path=path, pos=torch.as_tensor(pos, device=DEVICE), cell=cell, pbc=pbc, cutoff=case["cutoff"])


# -- one pass --------------------------------------------------------------------------------------------------------

def run(state):
    path = state["path"]
    if path == "model":
        if state["mode"] == "replay":
            return state["model"].predict(state["graph"], compute_forces=True, use_compile=True)
        # .to() makes a new graph object: as in a program whose edge list is new at every step, no
        # connectivity that an earlier pass derived is left on it
        return state["model"].predict(state["graph"].to(DEVICE), compute_forces=True)
    if path == "train":
        model, graph = state["model"], state["graph"].to(DEVICE)
        out = model.predict(graph, compute_forces=True, create_graph=True)
        e_err = (out["energy"] - state["energy"]) / graph.n_atoms
        loss = e_err.square().mean() + (out["forces"] - state["forces"]).square().mean()
        names, params = zip(*model.named_parameters())
        return dict(energy=out["energy"].detach(), forces=out["forces"].detach(),
                    **_buckets(names, torch.autograd.grad(loss, params, allow_unused=True)))
    if path in ("conv", "rows"):
        out = state["tp"](*state["args"], graph=state["graph"])
        return (out.detach(),) + torch.autograd.grad(out, state["args"], state["go"])
    if path == "linear":
        out = state["layer"](state["x"])
        return (out.detach(),) + torch.autograd.grad(out, [state["x"], *state["layer"].weight], state["go"])
    if path == "basis":
        vec = state["vec"]
        d = vec.norm(dim=-1)
        attrs = state["irreps"](vec)
        feats = state["basis"](d) * state["cutoff"](d).unsqueeze(-1)
        return (attrs.detach(), feats.detach()) + torch.autograd.grad((attrs, feats), vec, state["grads"])
    nl = NeighborList(state["cutoff"], backend="device").build(state["pos"], state["cell"], state["pbc"])
    return nl.edge_index, nl.unit_shifts


# -- what a pass cannot do without -----------------------------------------------------------------------------------

def _atoms(case):
    if case.get("system") == "fcc" or case["path"] == "neighbors":
        return 4 * case["nx"] * case["ny"] * case["nz"]
    if case.get("system") == "water":
        return 3 * max(18, case["n_mol"])
    return 35 * case["n_mol"]


def _tp_flops(l1, l2, lo, C):
    """Weighting of every path and its contraction counted as one multiply-add per output component."""
    return sum(2 * (2 * p[2] + 1) * C * 2 for p in _paths(l1, l2, lo))


def _model_work(case):
    n, C, L = _atoms(case), case["channels"], case["l_max"]
    degree = {"fcc": 43.7, "water": 46.0}.get(case.get("system"), 20.8)
    e = n * degree
    Lh = 2
    flops, weights = 0.0, 0.0

    def linear(paths, l_out, rows=1.0):
        nonlocal flops, weights
        for l in range(min(len(paths) - 1, l_out) + 1):
            flops += 2.0 * n * rows * (2 * l + 1) * C * paths[l] * C
            weights += C * paths[l] * C

    def counts(l1, l2, lo):
        c = [0] * (lo + 1)
        for p in _paths(l1, l2, lo):
            c[p[2]] += 1
        return c

    for k in range(2):
        lin, prod_out = (0, Lh) if k == 0 else (Lh, 0)
        P = len(_paths(lin, L, L))
        linear([1] * (lin + 1), lin)
        linear([1] * (lin + 1), L)
        flops += 2.0 * (e / 2) * (8 * 64 + 64 * 64 + 64 * P * C) + e * _tp_flops(lin, L, L, C)
        weights += 8 * 64 + 64 * 64 + 64 * P * C
        linear(counts(lin, L, L), L)
        linear([1] * (L + 1), L)
        linear([1] * (L + 1), L)
        flops += 2.0 * n * C * (L + 1) * C
        linear([1] * (L + 1), L)
        for out in (L, prod_out):
            flops += n * _tp_flops(L, L, out, C)
            linear(counts(L, L, out), out)
        linear([1] * (L + 1), prod_out)
    return n, e, flops, 4 * weights


def work(case):
    path = case["path"]
    if path in ("model", "train"):
        n, e, flops, weight_bytes = _model_work(case)
        io = n * (12 + 8 + 8 + 12 + 4) + e * (16 + 24)
        # forward and input gradients; a training step differentiates those again
        return dict(bytes=io + (2 if path == "train" else 1) * weight_bytes, flops=(6 if path == "train" else 2) * flops)
    if path in ("conv", "rows"):
        C, P = case["channels"], _paths(case["l1"], case["l2"], case["lo"])
        d1, d2 = (case["l1"] + 1) ** 2, (case["l2"] + 1) ** 2
        n_out = (case["lo"] + 1) ** 2 if case.get("reduced") else sum(2 * p[2] + 1 for p in P)
        items = case["edges"] if path == "conv" else case["rows"]
        f2 = 1 if path == "conv" else C
        w_rows = 1 if case.get("shared") else items
        # operands and their gradients, the output and its gradient
        floats = 2 * (case["rows"] * d1 * C + items * d2 * f2 + w_rows * len(P) * C + case["rows"] * n_out * C)
        return dict(bytes=4 * floats + (8 * items if path == "conv" else 0),
                    flops=4 * items * _tp_flops(case["l1"], case["l2"], case["lo"], C))
    if path == "linear":
        paths = [int(p) for p in case["paths"].split(",")]
        size = 8 if case["dtype"] == "float64" else 4
        lc = min(case["l_in"], case["l_out"])
        w = sum(case["fout"] * case["fin"] * paths[l] for l in range(lc + 1))
        macs = case["rows"] * sum((2 * l + 1) * case["fout"] * case["fin"] * paths[l] for l in range(lc + 1))
        io = case["rows"] * (sum((2 * l + 1) * case["fin"] * paths[l] for l in range(case["l_in"] + 1))
                             + (case["l_out"] + 1) ** 2 * case["fout"])
        return dict(bytes=2 * size * (io + w), flops=6 * macs)
    if path == "basis":
        per_edge = 2 * 3 + 2 * (case["l_max"] + 1) ** 2 + 2 * case["n_radial"]
        return dict(bytes=4 * case["edges"] * per_edge, flops=6 * case["edges"] * per_edge)
    n = _atoms(case)
    pairs = n * 4.19 * case["cutoff"] ** 3 * 4 / 3.6 ** 3
    return dict(bytes=24 * n + 28 * pairs, flops=10 * pairs)


def tolerance(case):
    """Four times the distance from ``exact`` measured on an MI355X over the listed and some 40 drawn
    cases (the largest output's, in brackets)."""
    path = case["path"]
    if path == "neighbors":
        return "exact"
    if path == "linear" and case["dtype"] == "float64":
        return {"rel": 1.2e-14}  # (3.0e-15, the weight gradients)
    return {"rel": {
        "model": 1.2e-5,  # (3.1e-6, forces)
        "train": 8e-6,    # (2.0e-6, forces)
        "conv": 6e-7,     # (1.4e-7)
        "rows": 7e-6,     # (1.7e-6, the gradient of weights shared by all rows)
        "linear": 4e-6,   # (8.9e-7, the weight gradients)
        "basis": 2e-6,    # (4.5e-7)
    }[path]}


# -- the same in plain float64 ---------------------------------------------------------------------------------------

STORED = {  # the kept components of a symmetric traceless tensor: (number of x, of y, of z)
    0: [(0, 0, 0)],
    1: [(1, 0, 0), (0, 1, 0), (0, 0, 1)],
    2: [(2, 0, 0), (0, 2, 0), (1, 1, 0), (1, 0, 1), (0, 1, 1)],
    3: [(3, 0, 0), (2, 1, 0), (2, 0, 1), (1, 2, 0), (1, 1, 1), (0, 2, 1), (0, 3, 0)],
}


def _kept(l):
    """Flat positions of the stored components among the 3^l full ones."""
    return [int("0" + "0" * a + "1" * b + "2" * c, 3) for a, b, c in STORED[l]]


@functools.lru_cache(maxsize=None)
def _traceless(l):
    """Orthogonal projector onto the symmetric traceless tensors of rank l, (3^l, 3^l)."""
    if l < 2:
        return np.eye(3 ** l)
    idx = list(itertools.product(range(3), repeat=l))
    rows = []  # linear conditions: equal under a swap of neighbours, every trace zero
    for flat, t in enumerate(idx):
        for a in range(l - 1):
            s = t[:a] + (t[a + 1], t[a]) + t[a + 2:]
            if s > t:
                row = np.zeros(3 ** l)
                row[flat], row[idx.index(s)] = 1.0, -1.0
                rows.append(row)
    for rest in itertools.product(range(3), repeat=l - 2):
        row = np.zeros(3 ** l)
        for a in range(3):
            row[idx.index((a, a) + rest)] = 1.0
        rows.append(row)
    _, s, vt = np.linalg.svd(np.array(rows), full_matrices=True)
    null = vt[int((s > 1e-9).sum()):]
    return null.T @ null


@functools.lru_cache(maxsize=None)
def _full(l):
    """(3^l, 2l+1): all components from the stored ones."""
    w, v = np.linalg.eigh(_traceless(l))
    basis = v[:, w > 0.5]
    return basis @ np.linalg.inv(basis[_kept(l)])


def _odd(n):
    return 1 if n <= 0 else n * _odd(n - 2)


@functools.lru_cache(maxsize=None)
def _coupling(l1, l2, lo):
    """(2lo+1, 2l1+1, 2l2+1): the traceless part of the contraction of two tensors over k axes."""
    f = math.factorial
    k, J = (l1 + l2 - lo) // 2, l1 + l2 + lo
    j1, j2, j3 = J - 2 * l1 - 1, J - 2 * l2 - 1, J - 2 * lo - 1
    norm = f(l1) * f(l2) * _odd(2 * lo - 1) * f((j1 + 1) // 2) * f((j2 + 1) // 2)
    norm /= f(l1 - k) * f(l2 - k) * _odd(j1) * _odd(j2) * _odd(j3) * f(J // 2)
    a = _full(l1).reshape(3 ** (l1 - k), 3 ** k, 2 * l1 + 1)
    b = _full(l2).reshape(3 ** k, 3 ** (l2 - k), 2 * l2 + 1)
    c = np.einsum("ikx,kjy->ijxy", a, b).reshape(3 ** lo, 2 * l1 + 1, 2 * l2 + 1)
    return norm * np.tensordot(_traceless(lo)[_kept(lo)], c, axes=1)


def _paths(l1_max, l2_max, lo_max):
    """(l1, l2, lo, exchanged) in weight order: for each lo the pairs l1 >= l2 with l1 from the first
    operand, then those with l1 > l2 and l1 from the second."""
    out = []
    for lo in range(lo_max + 1):
        for exchanged in (False, True):
            m1, m2 = (l2_max, l1_max) if exchanged else (l1_max, l2_max)
            out += [(a, b, lo, exchanged) for a in range(m1 + 1) for b in range(min(m2, a - exchanged) + 1)
                    if a - b <= lo <= a + b and (a + b + lo) % 2 == 0]
    return out


def _tensor(a, like):
    return torch.as_tensor(a, dtype=like.dtype, device=like.device)


def _product(x, y, w, l1_max, l2_max, lo_max, C, reduced=False, receivers=None, rows=None):
    """Weighted product of x (n, (l1+1)^2 C) with y (n, (l2+1)^2 C or (l2+1)^2); w (P, C) or (n, P, C).
    With ``receivers`` every path is summed over the items of a receiver."""
    n = x.shape[0]
    x = x.reshape(n, -1, C)
    single = y.shape[1] == (l2_max + 1) ** 2 and C > 1
    y = y.reshape(n, -1, 1 if single else C)
    blocks = [[] for _ in range(lo_max + 1)]
    for p, (a, b, lo, exchanged) in enumerate(_paths(l1_max, l2_max, lo_max)):
        B = _tensor(_coupling(a, b, lo), x)
        lx, ly = (b, a) if exchanged else (a, b)
        if exchanged:
            B = B.transpose(1, 2)
        xl, yl = x[:, lx * lx:(lx + 1) ** 2], y[:, ly * ly:(ly + 1) ** 2]
        if single:
            m = (yl.reshape(n, -1) @ B.reshape(-1, 2 * ly + 1).t()).reshape(n, 2 * lo + 1, 2 * lx + 1)
            t = m @ xl
        else:
            outer = (xl.unsqueeze(2) * yl.unsqueeze(1)).reshape(n, -1, C)
            t = B.reshape(2 * lo + 1, -1).unsqueeze(0) @ outer
        t = t * (w[:, p].unsqueeze(1) if w.dim() == 3 else w[p])
        if receivers is not None:
            t = x.new_zeros(rows, 2 * lo + 1, C).index_add(0, receivers, t)
        blocks[lo].append(t)
    n = rows if receivers is not None else n
    if reduced:
        return torch.cat([sum(b).reshape(n, -1) for b in blocks if b], dim=1)
    return torch.cat([torch.stack(b, dim=2).reshape(n, -1) for b in blocks if b], dim=1)


def _f32(x):
    """A constant as the layers store it."""
    return float(np.float32(x))


def _map(weights, x, l_in, l_out, fout, paths=None):
    n, off, outs = x.shape[0], 0, []
    paths = paths or [1] * (l_in + 1)
    fin = x.shape[1] // sum((2 * l + 1) * paths[l] for l in range(l_in + 1))
    for l in range(l_in + 1):
        k = fin * paths[l]
        if l <= l_out:
            outs.append((x[:, off:off + (2 * l + 1) * k].reshape(n, 2 * l + 1, k)
                         @ (weights[l].t() * _f32(float(k) ** -0.5))).reshape(n, -1))
        off += (2 * l + 1) * k
    outs += [x.new_zeros(n, (2 * l + 1) * fout) for l in range(l_in + 1, l_out + 1)]
    return torch.cat(outs, dim=1)


def _dense(sd, key, x):
    w, b = sd[f"{key}.weight"], sd.get(f"{key}.bias")
    y = x @ (w.t() * _f32(float(w.shape[1]) ** -0.5))
    return y if b is None else y + b


def _mlp(sd, key, x):
    x = _f32(1.6765324703310907) * torch.nn.functional.silu(_dense(sd, f"{key}.0", x))
    x = _f32(1.6765324703310907) * torch.nn.functional.silu(_dense(sd, f"{key}.2", x))
    return _dense(sd, f"{key}.4", x)


def _expand(vec, l_max):
    """Traceless powers of the direction of ``vec``, normalised to contract with it to 1."""
    r = vec / vec.norm(dim=-1, keepdim=True)
    full, outs = torch.ones_like(r[:, :1]), []
    for l in range(l_max + 1):
        scale = _odd(2 * l - 1) / math.factorial(l)
        outs.append(scale * full @ _tensor(_traceless(l)[_kept(l)].T.copy(), r))
        full = (full.unsqueeze(2) * r.unsqueeze(1)).reshape(r.shape[0], -1)
    return torch.cat(outs, dim=1)


def _cutoff(d):
    t, p = d / R_MAX, 6
    env = 1 - (p + 1) * (p + 2) / 2 * t ** p + p * (p + 2) * t ** (p + 1) - p * (p + 1) / 2 * t ** (p + 2)
    return env * (d < R_MAX)


def _potential(sd, case, g, positions):
    """Site energies of the packaged architecture from a state dict."""
    C, L, Lh = case["channels"], case["l_max"], 2
    i, j = g["edge_index"]
    n = positions.shape[0]
    vec = positions[j] - positions[i] + g["shift_vectors"]
    d = vec.norm(dim=-1)
    attrs = _expand(vec, L)
    t = math.pi * d / R_MAX  # cosine-mapped Chebyshev polynomials of the distance
    radial = torch.stack([torch.cos(k * torch.acos(torch.cos(t).clamp(-1 + 1e-15, 1 - 1e-15))) if k > 1 else
                          (torch.cos(t) if k == 1 else torch.ones_like(t)) for k in range(8)], dim=-1)
    radial = radial * _cutoff(d).unsqueeze(-1)

    def maps(key, x, l_in, l_out, paths=None):
        return _map([sd[f"{key}.weight.{l}"] for l in range(min(l_in, l_out) + 1)], x, l_in, l_out, C, paths)

    def counts(l1, l2, lo):
        return [sum(p[2] == l for p in _paths(l1, l2, lo)) for l in range(lo + 1)]

    def norm(key, x, l_max):
        b = x.reshape(n, -1, C)
        sq = 0
        for l in range(l_max + 1):
            B = _tensor(_coupling(l, l, 0)[0], x)
            bl = b[:, l * l:(l + 1) ** 2]
            sq = sq + ((B @ bl) * bl).sum(1) / ((2 * l + 1) * (l_max + 1))
        gain = torch.cat([sd[f"{key}.weights.{l}"].repeat(2 * l + 1) for l in range(l_max + 1)])
        return x * (sq.mean(-1, keepdim=True) + 1e-6) ** -0.5 * gain

    def convolution(h, attrs, radial, i, j, lin, key):
        w = _mlp(sd, f"{key}.radial_mlp", radial).reshape(radial.shape[0], -1, C)
        return _product(h[j], attrs, w, lin, L, L, C, receivers=i, rows=n)

    x = sd["embedding.weight"][g["atom_types"]]
    scalars = []
    for k in range(2):
        key, lin, out = f"interactions.{k}", 0 if k == 0 else Lh, Lh if k == 0 else 0
        h = maps(f"{key}.linear_first", x, lin, lin)
        agg, step = 0, 40000  # edges in blocks that the backward forms again
        for a in range(0, i.shape[0], step):
            s = slice(a, a + step)
            agg = agg + torch.utils.checkpoint.checkpoint(convolution, h, attrs[s], radial[s], i[s], j[s], lin, key,
                                                          use_reentrant=False)
        agg = agg / sd[f"{key}.sqrt_avg_neighbors"]
        y = maps(f"{key}.linear_second", agg, L, L, counts(lin, L, L))
        if k == 0:
            y = torch.cat([y[:, :C] + _dense(sd, f"{key}.skip_projection", x), y[:, C:]], dim=1)
        else:
            y = y + maps(f"{key}.skip_projection", x, lin, L)
        y = norm(f"{key}.layer_norm", y, L)
        gate = _f32(1.8462285453386054) * torch.sigmoid(_dense(sd, f"nonlinearities.{k}.gate_linear", y[:, :C]))
        gate = gate.reshape(n, L + 1, C)
        values = maps(f"nonlinearities.{k}.value_linear", y, L, L).reshape(n, -1, C)
        gated = torch.cat([values[:, l * l:(l + 1) ** 2] * gate[:, l:l + 1] for l in range(L + 1)], dim=1)
        y = y + maps(f"nonlinearities.{k}.output_linear", gated.reshape(n, -1), L, L)
        key, feats, x = f"products.{k}", y, 0
        for s in range(3):
            p_out = out if s == 2 else L
            if s > 0:
                P = len(_paths(L, L, p_out))
                delta = sd.get(f"{key}.path_weights.{s}.delta")
                w = y.new_ones(P, C) if delta is None else 1 + delta.reshape(P, C)
                feats = _product(feats, y, w, L, L, p_out, C)
            feats = maps(f"{key}.product_linears.{s}", feats, p_out, p_out,
                         counts(L, L, p_out) if s else [1] * (L + 1))
            x = x + feats[:, :(out + 1) ** 2 * C]
        x = x + maps(f"{key}.skip_projection", y, L, out)
        x = norm(f"{key}.layer_norm", x, out)
        scalars.append(x[:, :C])
    e = _mlp(sd, "readout.readout_mlp", torch.cat(scalars, dim=1)).squeeze(-1)
    return sd["scale_shift.scales"][g["atom_types"]] * e


def _model64(case, seed):
    elements, graph = _system(case, seed)
    model = _model(case, seed, elements, graph)
    to64 = lambda t: t.detach().to(DEVICE, torch.float64 if t.is_floating_point() else t.dtype)
    sd = {k: to64(v) for k, v in model.state_dict().items()}
    train = case["path"] == "train"
    names = [k for k, _ in model.named_parameters()]
    for k in names:
        sd[k].requires_grad_(train)
    g = {k: to64(getattr(graph, k)) for k in ("edge_index", "atom_types", "batch", "shifts", "cell", "n_atoms")}
    cells = g["cell"][g["batch"][g["edge_index"][0]]]
    g["shift_vectors"] = (g["shifts"].double().unsqueeze(1) @ cells).squeeze(1)
    pos = to64(graph.positions).requires_grad_(True)
    site = _potential(sd, case, g, pos)
    energy = site.new_zeros(g["n_atoms"].shape[0]).index_add(0, g["batch"], site)
    (grad,) = torch.autograd.grad(energy.sum(), pos, create_graph=train)
    if not train:
        return dict(node_energies=site.detach(), energy=energy.detach(), forces=-grad)
    e_ref, f_ref = (t.to(DEVICE, torch.float64) for t in _targets(graph, seed))
    loss = ((energy - e_ref) / g["n_atoms"]).square().mean() + (-grad - f_ref).square().mean()
    grads = torch.autograd.grad(loss, [sd[k] for k in names], allow_unused=True)
    return dict(energy=energy.detach(), forces=-grad.detach(), **_buckets(names, grads))


def _neighbors64(case, seed):
    pos, cell, _ = _box(case, seed)
    x = torch.as_tensor(pos, device=DEVICE)
    side = torch.as_tensor(np.diag(cell).copy(), device=DEVICE)
    reach = [range(-r, r + 1) for r in (int(math.ceil(case["cutoff"] / float(s))) for s in side)]
    n, found = x.shape[0], []
    for a in range(0, n, 2048):
        for S in itertools.product(*reach):
            shift = torch.tensor(S, dtype=torch.float64, device=DEVICE)
            v = x.unsqueeze(0) - x[a:a + 2048].unsqueeze(1) + shift * side
            near = v.square().sum(-1) < case["cutoff"] ** 2
            i, j = near.nonzero(as_tuple=True)
            i = i + a
            if not any(S):
                keep = i != j
                i, j = i[keep], j[keep]
            found.append(torch.stack([i, j, *(torch.full_like(i, s) for s in S)], dim=1))
    pairs = torch.cat(found).cpu().numpy()
    pairs = pairs[np.lexsort(pairs.T[::-1])]
    return torch.as_tensor(pairs[:, :2].T.copy()), torch.as_tensor(pairs[:, 2:].astype(np.int32))


def exact(case, seed):
    path = case["path"]
    if path in ("model", "train"):
        return _model64(case, seed)
    if path in ("conv", "rows"):
        t = _tp_inputs(case, seed)
        C, ls = case["channels"], (case["l1"], case["l2"], case["lo"])
        in1, in2, w = (t[k].double().requires_grad_(True) for k in ("in1", "in2", "w"))
        wp = w.reshape(*w.shape[:-1], -1, C)
        go = t["go"].double()
        if path == "rows":
            out = _product(in1, in2, wp, *ls, C, reduced=case["reduced"])
        else:
            out, step = 0, 20000
            for a in range(0, case["edges"], step):
                s = slice(a, a + step)
                i, j = t["edges"][0, s], t["edges"][1, s]
                out = out + torch.utils.checkpoint.checkpoint(
                    lambda in1, y, wp, i, j: _product(in1[j], y, wp, *ls, C, receivers=i, rows=case["rows"]),
                    in1, in2[s], wp[s], i, j, use_reentrant=False)
        return (out.detach(),) + torch.autograd.grad(out, (in1, in2, w), go)
    if path == "linear":
        x, go, weights, paths = _linear_inputs(case, seed)
        x, go = x.double().requires_grad_(True), go.double()
        weights = [w.double().requires_grad_(True) for w in weights]
        out = _map(weights, x, case["l_in"], case["l_out"], case["fout"], paths)
        return (out.detach(),) + torch.autograd.grad(out, [x, *weights], go)
    if path == "basis":
        vec, g_attrs, g_feats = (t.double() for t in _basis_inputs(case, seed))
        vec.requires_grad_(True)
        d = vec.norm(dim=-1)
        k = torch.arange(1, case["n_radial"] + 1, dtype=torch.float64, device=DEVICE)
        bessel = math.sqrt(2.0 / R_MAX) * torch.sin(k * math.pi * d.unsqueeze(-1) / R_MAX) / d.unsqueeze(-1)
        attrs, feats = _expand(vec, case["l_max"]), bessel * _cutoff(d).unsqueeze(-1)
        return (attrs.detach(), feats.detach()) + torch.autograd.grad((attrs, feats), vec, (g_attrs, g_feats))
    return _neighbors64(case, seed)
