"""The work that users of this framework have it do, as measurable cases.

Whole calls: a molecular-dynamics step of one molecule and of a small crystal through the
calculator, energies and forces of molecule batches, and the replayed step of liquid boxes up to
100,000 atoms. Single layers: the two drop-in operators (factor density, node algebra), the CP
pooling, the moment mixing and projections, the readout, each forward and backward; and the pair
list build. Everything is float32, as the framework computes.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program has
in hand before the call, run() makes one call, exact() is the same result in plain 64-bit torch.
"""
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "face-mlip_amd"))
from face_amd import kernels, neighbors, node_kernel, ops  # noqa: E402
from face_amd.calculator import FACECalculator  # noqa: E402
from face_amd.model import FACE  # noqa: E402
from face_amd.runner import StepGraph  # noqa: E402

DEV = "cuda"
N_BASIS, HIDDEN, K_DIR = 8, 64, 16
RANK_K = (1, 3, 6, 10)
KINDS = ("md", "batch", "step", "pairs", "density", "algebra", "pooling", "moments", "readout")


# ----------------------------------------------------------------------------- the cases
def listed():
    return [
        # one MD step of a single 21-atom molecule: the smallest call a program makes, bound by launches
        _whole("md_molecule21_c96", "md", "molecules", 21, 1, C=96, K=32, rc=4.5),
        # one MD step of an 864-atom metal crystal (one element, 18 neighbours), tabulated radial functions
        _whole("md_fcc864_c96", "md", "fcc", 864, 1, C=96, K=32, rc=4.5),
        # a replayed step of a batch of 64 equal molecules: trajectories of replicas run side by side
        _whole("step_molecules64_c96", "step", "molecules", 1344, 64, C=96, K=32, rc=4.5),
        # energies and forces of 512 molecules of unequal sizes, call by call: scoring a data set
        _whole("batch_molecules512_cp160", "batch", "molecules", 10773, 512, C=160, K=32, rc=4.5, cp=True),
        # the replayed step of a 24,000-atom molecular liquid, CP pooling: production MD of a large box
        _whole("step_liquid24k_cp160", "step", "liquid", 24000, 1, C=160, K=32, rc=5.0, cp=True),
        # the replayed step of a 100,000-atom liquid with the widest model: the largest box
        _whole("step_liquid100k_c256", "step", "liquid", 100000, 1, C=256, K=64, rc=5.5),
        # the pair list of the 24,000-atom box: rebuilt every few tens of MD steps
        {"name": "pairs_liquid24k", "kind": "pairs", "system": "liquid", "atoms": 24000, "structures": 1, "rc": 5.5},
        # the factor density operator on padded rows, forward and backward: used inside another model
        {"name": "density_padded", "kind": "density", "atoms": 3000, "slots": 37, "B": 16, "K": 32},
        # the node-invariant algebra operator, forward and backward, with gated outputs
        {"name": "algebra_24k_c160", "kind": "algebra", "atoms": 24000, "C": 160, "eq": True},
        # the CP pooling layer fed by the radial network, forward and backward, on a liquid's pair list
        {"name": "pooling_cp160", "kind": "pooling", "system": "liquid", "atoms": 6000, "structures": 1, "rc": 5.0, "C": 160},
        # mixing of the pooled moments and the projections of two moment sets, forward and backward
        {"name": "moments_24k_c160", "kind": "moments", "atoms": 24000, "C": 160, "width": 160, "transport": 512,
         "elements": 3},
        # normalised invariants through the readout network, forward and backward
        {"name": "readout_10k_c160", "kind": "readout", "atoms": 10752, "C": 160, "last": False},
    ]


def _whole(name, kind, system, atoms, structures, C, K, rc, cp=False, passes=2, equivariant=True):
    c = {"kind": kind, "system": system, "atoms": atoms, "structures": structures, "C": C, "K": K, "rc": rc, "cp": cp,
         "passes": passes, "equivariant": equivariant}
    return dict(c, name=name) if name else c


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(KINDS)
    C = rng.choice((32, 64, 96, 128, 160))
    rc = rng.choice((4.5, 5.0))
    cp = rng.random() < 0.5
    if kind == "md":
        system = rng.choice(("molecules", "fcc"))
        atoms = size(9, 60) if system == "molecules" else 4 * rng.choice((4, 5, 6, 7, 8)) ** 3
        return _whole(None, kind, system, atoms, 1, C, rng.choice((16, 32, 64)), rc)
    if kind == "batch":
        structures = size(2, 500)
        return _whole(None, kind, "molecules", structures * 9 + size(structures, 12 * structures), structures, C,
                      rng.choice((16, 32)), rc, cp, rng.choice((1, 2, 3)), rng.random() < 0.75)
    if kind == "step":
        return _whole(None, kind, "liquid", size(1200, 24000), 1, C, rng.choice((16, 32, 64)), rc, cp)
    if kind == "pairs":
        system = rng.choice(("molecules", "liquid"))
        structures = size(2, 400) if system == "molecules" else 1
        atoms = structures * rng.randint(10, 30) if system == "molecules" else size(1500, 60000)
        return {"kind": kind, "system": system, "atoms": atoms, "structures": structures, "rc": rc}
    if kind == "density":
        return {"kind": kind, "atoms": size(20, 6000), "slots": rng.randint(8, 60), "B": 16,
                "K": rng.choice((16, 32, 48, 64))}
    if kind == "algebra":
        return {"kind": kind, "atoms": size(50, 24000), "C": rng.choice((24, 32, 64, 96, 128, 160)),
                "eq": rng.random() < 0.7}
    if kind == "pooling":
        return {"kind": kind, "system": "liquid", "atoms": size(1200, 9000), "structures": 1, "rc": rc, "C": C}
    if kind == "moments":
        return {"kind": kind, "atoms": size(60, 24000), "C": C, "width": rng.choice((C, 16 * rng.choice((16, 32)))),
                "transport": rng.choice((0, 512)), "elements": rng.randint(1, 5)}
    return {"kind": kind, "atoms": size(60, 24000), "C": C, "last": rng.random() < 0.4}


# ----------------------------------------------------------------------------- inputs
def _rng(seed, salt):
    return np.random.default_rng([int(seed), salt])


def _structures(case, seed):
    """Structures {'pos','Z','cell','pbc'} as a program hands them to the pair list build. Where the
    number of pairs shapes the outputs, every seed has the same geometry, moved, mirrored and with
    the atoms in another order."""
    if case["kind"] not in ("pairs", "pooling"):
        return _drawn_structures(case, _rng(seed, 1))
    out, rng = [], _rng(seed, 4)
    for s in _drawn_structures(case, _rng(0, 1)):
        order, L = rng.permutation(len(s["pos"])), s["cell"][0, 0]
        pos = s["pos"][order][:, rng.permutation(3)] * rng.choice((-1.0, 1.0), 3) + rng.uniform(0, 20, 3)
        out.append(dict(s, pos=np.mod(pos, L) if L else pos, Z=s["Z"][order]))
    return out


def _drawn_structures(case, rng):
    n, count = case["atoms"], case["structures"]
    if case["system"] == "fcc":
        cells = round((n / 4) ** (1 / 3))
        basis = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
        grid = np.stack(np.meshgrid(*[np.arange(cells)] * 3, indexing="ij"), -1).reshape(-1, 3)
        pos = ((grid[:, None] + basis[None]) * 4.09).reshape(-1, 3)
        L = 4.09 * cells
        return [{"pos": np.mod(pos + rng.normal(0, 0.1, pos.shape), L), "Z": np.full(len(pos), 47), "cell": np.eye(3) * L,
                 "pbc": np.ones(3, bool)}]
    if case["system"] == "liquid":
        L = (n / 0.10) ** (1 / 3)                       # 0.10 atoms per cubic Angstrom, H:C:O = 8:9:4
        m = math.ceil(n ** (1 / 3) - 1e-9)
        a = L / m
        site = rng.permutation(m ** 3)[:n]
        grid = np.stack(np.unravel_index(site, (m, m, m)), -1)
        pos = (grid + 0.5) * a + rng.uniform(-1, 1, (n, 3)) * 0.5 * (a - 0.9)
        Z = rng.permutation(np.resize(np.repeat([1, 6, 8], [8, 9, 4]), n))
        return [{"pos": np.mod(pos, L), "Z": Z, "cell": np.eye(3) * L, "pbc": np.ones(3, bool)}]
    # molecules: sites of a 1.55 A lattice near a centre, displaced; sizes even, or spread about the mean
    mean = n / count
    sizes = np.full(count, n // count)
    if n % count:
        sizes = np.maximum(4, np.round(mean * rng.uniform(0.55, 1.45, count)).astype(int))
        while sizes.sum() != n:
            k = rng.integers(count)
            sizes[k] = max(4, sizes[k] + np.sign(n - sizes.sum()))
    g = np.arange(-4, 5)
    grid = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) * 1.55
    far = np.linalg.norm(grid, axis=1)
    out = []
    for k in sizes:
        pos = grid[np.argsort(far + rng.uniform(0, 1.6, len(far)))[:k]] + rng.uniform(-0.25, 0.25, (k, 3))
        out.append({"pos": pos, "Z": rng.permutation(np.resize(np.repeat([6, 8, 1], [9, 4, 8]), k)),
                    "cell": np.zeros((3, 3)), "pbc": np.zeros(3, bool)})
    return out


def _elements(case):
    return [47] if case["system"] == "fcc" else [1, 6, 8]


def _neighbours(case):
    """Mean neighbours per atom, for the model's normalisation and for the counts of work()."""
    if case["system"] == "molecules":
        return 0.93 * (case["atoms"] / case["structures"] - 1)
    rho = 4 / 4.09 ** 3 if case["system"] == "fcc" else 0.10
    return 4 / 3 * math.pi * case["rc"] ** 3 * rho


def _weights(case, seed):
    """A model's parameters and buffers by their names, with the spread that trained ones have."""
    rng = _rng(seed, 2)
    C, n_el = case["C"], len(_elements(case))
    cp, eq, B = case["cp"], case["equivariant"], 16
    K = C if cp else case["K"]
    w = {}

    def linear(name, n_out, n_in, bias=True):
        b = 1 / math.sqrt(n_in)
        w[name + ".weight"] = rng.uniform(-b, b, (n_out, n_in)).astype(np.float32)
        if bias:
            w[name + ".bias"] = rng.uniform(-b, b, n_out).astype(np.float32)

    def near(name, centre, spread, *shape):
        w[name] = (centre + spread * rng.standard_normal(shape)).astype(np.float32)

    near("embed.weight", 0, 1, n_el, C)
    near("E0", 0, 1, n_el)
    w["scale"], w["avg_nb"] = np.float32(0.8), np.float32(max(1.0, _neighbours(case)))
    for t in range(case["passes"]):
        p = "blocks.%d." % t
        linear(p + "rad_in", HIDDEN, N_BASIS)
        near(p + "pair.weight", 0, 0.2, n_el * n_el, HIDDEN)
        linear(p + "radial.0", HIDDEN, HIDDEN)
        linear(p + "radial.2", B + (4 * C if cp else 0), HIDDEN)
        linear(p + "msg", K, C)
        near(p + "elem_scale.weight", 1, 0.1, n_el, 4 * C)
        near(p + "norm.weight", 1, 0.1, 9 * C)
        near(p + "norm.bias", 0, 0.1, 9 * C)
        linear(p + "out.0", 2 * C, 10 * C + 4)
        linear(p + "out.2", 2 * C, 2 * C)
        linear(p + "out.4", C + 1, 2 * C)
        for k in range(4):
            linear(p + "proj.%d" % k, 3 * C, C * (t + 1), False)
            linear(p + "mix.%d" % k, C, C if cp else B * K, False)
        if eq and t < case["passes"] - 1:
            near(p + "vpath", 1, 0.2, 4, C)
            near(p + "mpath", 1, 0.2, 4, C)
            linear(p + "gate", 2 * C, 9 * C)
            w[p + "gate.bias"] += np.float32(1)
        if t > 0:
            prev = C if eq else C * t
            linear(p + "dir_mix", K, 4 * K_DIR)
            for name in ("pvt", "pmt"):
                linear(p + name, (2 if eq else 1) * K_DIR, prev, False)
            if eq:
                for name in ("tmix1", "tmix2", "tmix3"):
                    linear(p + name, C, B * 2 * K_DIR, False)
    return {k: torch.as_tensor(v) for k, v in w.items()}


def _model(case, seed):
    m = FACE(_elements(case), C=case["C"], n_basis=N_BASIS, rc=case["rc"], n_passes=case["passes"], radial_hidden=HIDDEN,
             K_dir=K_DIR, transport=case["equivariant"], eqmsg=case["equivariant"], B=16, K=case["K"], cp=case["cp"])
    m.load_state_dict(_weights(case, seed), strict=False)
    return m.to(DEV).eval()


def _normal(seed, salt, *shape, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(int(seed) * 64 + salt)
    return torch.randn(*shape, device=DEV, generator=g) * scale


def _edge_inputs(case, seed, E, C):
    """Last hidden activations, envelope, messages and monomials of E edges."""
    h2 = F.silu(_normal(seed, 3, E, HIDDEN))
    env = torch.sigmoid(_normal(seed, 4, E))
    msg = _normal(seed, 5, E, C)
    u = F.normalize(_normal(seed, 6, E, 3), dim=1)
    w = _normal(seed, 7, 4 * C, HIDDEN, scale=1 / math.sqrt(HIDDEN))
    b = _normal(seed, 8, 4 * C, scale=0.1)
    return h2, w, b, env, msg, _monomials(u)


def _layer_inputs(case, seed):
    """(inputs with gradients, constants, upstream gradients) of a single layer."""
    kind, N = case["kind"], case["atoms"]
    if kind == "density":
        M, B, K = case["slots"], case["B"], case["K"]
        rows = torch.randint(max(1, M // 2), M + 1, (N, 1), generator=torch.Generator().manual_seed(int(seed))).to(DEV)
        mask = (torch.arange(M, device=DEV)[None] < rows).float()[..., None]
        u = F.normalize(_normal(seed, 6, N, M, 3), dim=-1)
        return [_normal(seed, 1, N, M, B) * mask, _normal(seed, 2, N, M, K), _monomials(u)], [], \
            [_normal(seed, 9, N, 20, B * K)]
    C = case["C"]
    if kind == "algebra":
        ins = [_normal(seed, 10 + i, N, C, k) for i, k in enumerate((3, 3, 3, 6, 6, 6, 10, 10))]
        ab = [1 + _normal(seed, 20 + i, 4, C, scale=0.2) for i in range(2)]
        return ins, ab, [_normal(seed, 30, N, C, 8), _normal(seed, 31, N, C, 3), _normal(seed, 32, N, C, 3, 3)]
    if kind == "moments":
        W, T = case["width"], case["transport"]
        ins = [_normal(seed, 10 + i, k, N, W) for i, k in enumerate(RANK_K)]
        ins += [_normal(seed, 20 + i, k, N, C) for i, k in enumerate(RANK_K)]
        ins += [_normal(seed, 24 + i, k, N, T) for i, k in enumerate((3, 6)[: 2 if T else 0])]
        z = torch.randint(0, case["elements"], (N,), generator=torch.Generator().manual_seed(int(seed))).to(DEV)
        s = 1 + _normal(seed, 30, case["elements"], 4 * C, scale=0.1)
        wm = [_normal(seed, 31 + i, C, W, scale=W ** -0.5) for i in range(4)]
        wt = [_normal(seed, 35 + i, C, T, scale=T ** -0.5) if T else None for i in range(2)]
        wp = [_normal(seed, 37 + i, (C, 3 * C, 3 * C, 2 * C)[i], 2 * C, scale=(2 * C) ** -0.5) for i in range(4)]
        up = [_normal(seed, 41 + i, k, N, w.shape[0]) for i, (k, w) in enumerate(zip(RANK_K, wp))]
        return ins, [z, s, wm, wt, wp], up
    # readout
    ins = [F.layer_norm(_normal(seed, 10, N, 9 * C) * torch.exp(_normal(seed, 11, N, 9 * C)), (9 * C,)), _normal(seed, 12, N, C)]
    shapes = [(2 * C, 10 * C), (2 * C,), (2 * C, 2 * C), (2 * C,), (C + 1, 2 * C), (C + 1,), (2 * C, 9 * C), (2 * C,)]
    ws = [_normal(seed, 13 + i, *s, scale=s[1] ** -0.5 if len(s) > 1 else 0.1) for i, s in enumerate(shapes)]
    up = [_normal(seed, 21, N, 1)] + ([] if case["last"] else [_normal(seed, 22, N, C), _normal(seed, 23, N, 2 * C)])
    return ins, ws, up


# ----------------------------------------------------------------------------- prepare and run
def prepare(case, seed):
    kind = case["kind"]
    if kind == "pairs":
        return {"kind": kind, "structures": _structures(case, seed), "rc": case["rc"]}
    if kind in ("md", "batch", "step"):
        model, st = _model(case, seed), _structures(case, seed)
        if kind == "md":
            calc = FACECalculator(model, DEV)
            s = st[0]
            moved = torch.as_tensor(s["pos"] + _rng(seed, 3).normal(0, 0.03, s["pos"].shape), dtype=torch.float32, device=DEV)
            calc.compute(s["pos"], s["Z"], s["cell"], s["pbc"])
            return {"kind": kind, "calc": calc, "pos": moved, "Z": s["Z"], "cell": s["cell"], "pbc": s["pbc"]}
        graph = neighbors.build_graph(st, case["rc"], DEV)
        if kind == "step":
            return {"kind": kind, "step": StepGraph(model, graph), "pos": graph.pos.clone()}
        return {"kind": kind, "model": model, "graph": graph, "pos": graph.pos.clone()}
    if kind == "pooling":
        graph = neighbors.build_graph(_structures(case, seed), case["rc"], DEV)
        h2, w, b, env, msg, Y = _edge_inputs(case, seed, graph.E, case["C"])
        up = [_normal(seed, 9 + i, k, graph.N, case["C"]) for i, k in enumerate(RANK_K)]
        ins = [t.requires_grad_(True) for t in (h2, env, msg, Y)]
        return {"kind": kind, "case": case, "graph": graph, "ins": ins, "consts": [w, b], "up": up}
    ins, consts, up = _layer_inputs(case, seed)
    if kind == "moments":
        consts[0] = consts[0].to(torch.int32)
    return {"kind": kind, "case": case, "ins": [t.requires_grad_(True) for t in ins], "consts": consts, "up": up}


def run(state):
    kind = state["kind"]
    if kind == "md":
        e, f = state["calc"].compute(state["pos"], state["Z"], state["cell"], state["pbc"])
        return {"energy": e, "forces": f}
    if kind == "step":
        e, f = state["step"](state["pos"])
        return {"energy": e, "forces": f}
    if kind == "batch":
        o = state["model"](state["graph"].with_pos(state["pos"].detach().requires_grad_(True)))
        return {"energy": o["energy"].detach(), "atom_energy": o["atom_energy"].detach(), "forces": o["forces"]}
    if kind == "pairs":
        g = neighbors.build_graph(state["structures"], state["rc"], DEV)
        return {"row_ptr": g.row_ptr, "col": g.col, "recv": g.recv, "S": g.S, "rev": g.rev, "shift": g.shift}
    outs = _layer(state)
    grads = torch.autograd.grad(outs, state["ins"], state["up"])
    return {"outputs": [o.detach() for o in outs], "gradients": list(grads)}


def _layer(state):
    kind, ins, consts = state["kind"], state["ins"], state["consts"]
    if kind == "density":
        return [kernels.factor_density(*ins)]
    if kind == "algebra":
        inv, V, M = node_kernel.node_algebra(*ins, *consts, state["case"]["eq"])
        if not state["case"]["eq"]:
            state["up"] = state["up"][:1]
            return [inv]
        return [inv, V, M]
    if kind == "pooling":
        h2, env, msg, Y = ins
        return list(ops.cp_radial_density(h2, *consts, env, msg, Y, state["graph"]))
    if kind == "moments":
        z, s, wm, wt, wp = consts
        D1, D2 = ins[8:] if len(ins) > 8 else (None, None)
        A = ops.scaled_mix(s, z, wm, wt, D1, D2, ins[:4])
        return list(ops.rank_proj(wp, [tuple(ins[4:8]), tuple(A)]))
    W0, b0, W1, b1, W2, b2, Wg, bg = consts
    last, nf = state["case"]["last"], 9 * state["case"]["C"]
    gate = (None, None) if last else (Wg, bg)
    e, h_new, gvm = ops.readout_mlp(ins[0], ins[1], W0[:, :nf], W0[:, nf:], b0, W1, b1, W2, b2, *gate, last)
    return [e] if last else [e, h_new, gvm]


# ----------------------------------------------------------------------------- work and tolerance
def work(case):
    kind, N, f4 = case["kind"], case["atoms"], 4
    if kind in ("md", "batch", "step"):
        C, E, H, B, Kd = case["C"], N * _neighbours(case), HIDDEN, 16, K_DIR
        cp, eq = case["cp"], case["equivariant"]
        K = C if cp else case["K"]
        linear = density = weights = 0
        for t in range(case["passes"]):
            out = 0 if t == case["passes"] - 1 else C
            radial = N_BASIS * H + H * H + H * (B + (4 * C if cp else 0))
            mix, proj = (C if cp else B * K) * C, (1 + 3 * 3 + 6 * 3 + 10 * 2) * C * C * (t + 1)
            read = 10 * C * 2 * C + 4 * C * C + 2 * C * (1 + out) + (9 * C * 2 * C if eq and out else 0)
            linear += 2 * (E * radial + 20 * N * mix + N * proj + N * read + N * C * K)
            density += 2 * 20 * E * (C if cp else B * K)
            weights += radial + 4 * mix + 9 * C * C * (t + 1) + read
            if t > 0:
                nt, prev = (2 if eq else 1), (C if eq else C * t)
                linear += 2 * (9 * N * prev * nt * Kd + E * 4 * Kd * K)
                density += 2 * 9 * E * 2 * Kd + (2 * 9 * E * B * 2 * Kd if eq else 0)
                linear += 2 * 9 * N * B * 2 * Kd * C if eq else 0
        return {"bytes": f4 * (weights + 7 * N + 4 * E), "flops": 2 * linear + 3 * density}
    if kind == "pairs":
        E = N * _neighbours(case)
        return {"bytes": 28 * N + f4 * 9 * E, "flops": 8 * E}
    if kind == "density":
        M, B, K = case["slots"], case["B"], case["K"]
        rows = N * M
        return {"bytes": f4 * (2 * rows * (B + K + 20) + 2 * N * 20 * B * K), "flops": 4 * 2 * 20 * rows * B * K}
    C = case["C"]
    if kind == "algebra":
        return {"bytes": f4 * N * C * (2 * 47 + 2 * (20 if case["eq"] else 8)), "flops": 3 * 300 * N * C}
    if kind == "pooling":
        E = N * _neighbours(case)
        return {"bytes": f4 * (2 * E * (HIDDEN + 1 + C + 20) + 2 * 20 * N * C),
                "flops": 2 * 2 * E * HIDDEN * 4 * C + 3 * 2 * 20 * E * C + 4 * 2 * E * 4 * C}
    if kind == "moments":
        W, T, P = case["width"], case["transport"], (1 + 9 + 18 + 20) * C
        return {"bytes": f4 * 2 * N * (20 * W + 20 * C + 9 * T + P),
                "flops": 2 * 2 * N * (20 * W * C + 9 * T * C + P * 2 * C)}
    out = 1 if case["last"] else 1 + C
    gate = 0 if case["last"] else 2 * C
    return {"bytes": f4 * N * 2 * (10 * C + out + gate),
            "flops": 2 * 2 * N * (10 * C * 2 * C + 4 * C * C + 2 * C * out + 9 * C * gate)}


def tolerance(case):
    """float32 sums in another order; about four times what the framework's results are off the 64-bit ones."""
    kind = case["kind"]
    if kind == "pairs":
        return "exact"
    if kind == "md":                          # slopes of tables stored in float32: 6e-5 to 3e-4 off
        return {"rel": 2e-4, "max": 4e-3}
    if kind in ("batch", "step"):             # 0.6e-6 to 2.1e-6 off
        return {"rel": 8e-6, "max": 4e-4}
    return {"rel": 4e-6, "max": 1e-4}         # single layers: 0.05e-6 to 1e-6 off


# ----------------------------------------------------------------------------- 64-bit results
SYM = ((), (0,), (1,), (2,), (0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2), (0, 0, 0), (1, 1, 1), (2, 2, 2), (0, 0, 1),
       (0, 0, 2), (0, 1, 1), (1, 1, 2), (0, 2, 2), (1, 2, 2), (0, 1, 2))
RANK_AT = (0, 1, 4, 10, 20)


def _monomials(u):
    cols = []
    for t in SYM:
        v = torch.ones_like(u[..., 0])
        for a in t:
            v = v * u[..., a]
        cols.append(v)
    return torch.stack(cols, -1)


def _full(x, rank):
    """(..., k) distinct components of a symmetric tensor -> (..., 3, ..., 3)."""
    at = {t: k for k, t in enumerate(SYM[RANK_AT[rank]:RANK_AT[rank + 1]])}
    idx = np.ndindex(*[3] * rank)
    return x[..., [at[tuple(sorted(t))] for t in idx]].reshape(*x.shape[:-1], *[3] * rank)


def _algebra(P1, Q1, S1, P2, Q2, S2, P3, Q3, a, b):
    """The eight invariants and the two gated products (rank 2 unsymmetrised)."""
    P2, Q2, S2, P3, Q3 = _full(P2, 2), _full(Q2, 2), _full(S2, 2), _full(P3, 3), _full(Q3, 3)
    v = lambda M, x: (M * x[..., None, :]).sum(-1)  # noqa: E731
    PQ = P2 @ Q2
    Q2S1, P3Q2 = v(Q2, S1), (P3 * Q2[..., None, :, :]).sum((-1, -2))
    P3S1 = (P3 * S1[..., None, None, :]).sum(-1)
    G = P3.flatten(-3, -2).transpose(-1, -2) @ Q3.flatten(-3, -2)
    inv = torch.stack([(P1 * Q1).sum(-1), (P2 * Q2).sum((-1, -2)), (P3 * Q3).sum((-1, -2, -3)), (P1 * Q2S1).sum(-1),
                       (PQ * S2.transpose(-1, -2)).sum((-1, -2)), (P3Q2 * S1).sum(-1), (G * S2).sum((-1, -2)),
                       (v(P3S1, Q1) * Q1).sum(-1)], -1)
    a, b = a.t(), b.t()
    V = a[:, 0:1] * P1 + a[:, 1:2] * Q2S1 + a[:, 2:3] * P3Q2 + a[:, 3:4] * v(P2, Q1)
    M = b[:, 0, None, None] * P2 + b[:, 1, None, None] * P1[..., :, None] * Q1[..., None, :]
    return inv, V, M + b[:, 2, None, None] * PQ + b[:, 3, None, None] * P3S1


def _pairs64(st, rc):
    """(i, j, shift) of all pairs within rc: cubic boxes wider than 2 rc, or free structures."""
    out, base = [], 0
    for s in st:
        pos = torch.as_tensor(np.asarray(s["pos"], np.float64), device=DEV)
        L = float(s["cell"][0, 0])
        for lo in range(0, len(pos), 2048):
            d = pos[None] - pos[lo:lo + 2048, None]
            k = -torch.round(d / L) if L else torch.zeros_like(d)
            d = d + k * L
            near = (d * d).sum(-1) < rc * rc
            near[torch.arange(near.shape[0], device=DEV), torch.arange(lo, lo + near.shape[0], device=DEV)] = False
            i, j = near.nonzero(as_tuple=True)
            out.append((i + lo + base, j + base, k[i, j] * float(np.float32(L))))
        base += len(pos)
    return [torch.cat(x) for x in zip(*out)]


def _pool(w, Y, i, N, X=None):
    """Per rank, the sums over each atom's edges of w (E, F) (or of X[rank]) times the monomials: 4 x (k, N, F)."""
    out = []
    for k in range(4):
        x = w if X is None else X[k]
        out.append(torch.stack([x.new_zeros(N, x.shape[1]).index_add(0, i, x * Y[:, c:c + 1])
                                for c in range(RANK_AT[k], RANK_AT[k + 1])]))
    return out


def _tables(W, p, rc, freq, B_cols, n=4096):
    """Values and slopes of a pass's radial functions on the grid, stored in float32."""
    r = torch.linspace(0, rc, n, device=DEV, dtype=torch.float64).clamp_min(1e-4)
    P = W[p + "pair.weight"].shape[0]

    def f(x):
        rb, _ = _basis(x, rc, freq)
        h = F.silu(F.linear(rb, W[p + "rad_in.weight"], W[p + "rad_in.bias"])[None] + W[p + "pair.weight"][:, None])
        h = F.silu(F.linear(h, W[p + "radial.0.weight"], W[p + "radial.0.bias"]))
        return F.linear(h, W[p + "radial.2.weight"], W[p + "radial.2.bias"])

    T, dT = torch.func.jvp(f, (r,), (torch.ones_like(r),))
    return T.float().double(), dT.float().double(), rc / (n - 1), P


def _basis(r, rc, freq):
    x = r / rc
    env = (1 - 28 * x ** 6 + 48 * x ** 7 - 21 * x ** 8) * (x < 1)
    return torch.sin(freq * r[..., None]) / r[..., None] * math.sqrt(2 / rc) * env[..., None], env


def _spline(tab, r, pair):
    T, dT, dr, _ = tab
    x = (r / dr).clamp(0, T.shape[1] - 1)
    k = x.detach().floor().long().clamp(max=T.shape[1] - 2)
    t = (x - k)[:, None]
    p0, p1, m0, m1 = T[pair, k], T[pair, k + 1], dT[pair, k] * dr, dT[pair, k + 1] * dr
    return p0 + t * t * (3 - 2 * t) * (p1 - p0) + t * (1 - t) ** 2 * m0 - t * t * (1 - t) * m1


def _whole64(case, seed):
    W = {k: v.to(DEV).double() for k, v in _weights(case, seed).items()}
    st, rc, C, B, Kd = _structures(case, seed), case["rc"], case["C"], 16, K_DIR
    start = torch.as_tensor(np.concatenate([s["pos"] for s in st]), device=DEV)
    pos = start.float().double()
    if case["kind"] == "md":                                      # the moved positions of the same list
        pos = torch.as_tensor(st[0]["pos"] + _rng(seed, 3).normal(0, 0.03, st[0]["pos"].shape), device=DEV).float().double()
    pos.requires_grad_(True)
    i, j, shift = _pairs64(st, rc + 0.4)
    N, n_el = len(pos), len(_elements(case))
    z = torch.as_tensor(np.searchsorted(_elements(case), np.concatenate([s["Z"] for s in st])), device=DEV)
    vec = pos[j] - pos[i] + shift
    keep = (vec.detach() ** 2).sum(-1) < rc * rc
    i, j, vec = i[keep], j[keep], vec[keep]
    pair = z[i] * n_el + z[j]
    r = vec.norm(dim=-1)
    u = vec / r[:, None]
    Y = _monomials(u)
    freq = torch.arange(1, N_BASIS + 1, device=DEV, dtype=torch.float32).mul(math.pi / rc).double()
    rb, env = _basis(r, rc, freq)
    h, sets, eq = W["embed.weight"][z], [], None
    e_at = W["E0"][z]
    lin = lambda x, name: F.linear(x, W[name + ".weight"], W.get(name + ".bias"))  # noqa: E731
    seg = lambda x: x.new_zeros(N, *x.shape[1:]).index_add(0, i, x)  # noqa: E731
    for t in range(case["passes"]):
        p = "blocks.%d." % t
        if case["kind"] == "md":
            rad = _spline(_tables(W, p, rc, freq, B), r, pair)
        else:
            rad = lin(F.silu(lin(F.silu(lin(rb, p + "rad_in") + W[p + "pair.weight"][pair]), p + "radial.0")), p + "radial.2")
        rad = rad * env[:, None]
        phi, mj = rad[:, :B], lin(h, p + "msg")[j]
        if t > 0:
            s1, s2 = eq if case["equivariant"] else (torch.cat([S[1] for S in sets], -1), torch.cat([S[2] for S in sets], -1))
            Vb, Mb = lin(s1, p + "pvt"), lin(s2, p + "pmt")                     # (3, N, nt Kd), (6, N, nt Kd)
            Y2 = Y[:, 4:10] * Y.new_tensor([1, 1, 1, 2, 2, 2])
            dot = lambda y, T: sum(y[:, q:q + 1] * T[q] for q in range(len(T)))  # noqa: E731
            d = torch.cat([dot(u, Vb[:, j, :Kd]), dot(Y2, Mb[:, j, :Kd]), dot(u, Vb[:, i, :Kd]), dot(Y2, Mb[:, i, :Kd])], 1)
            mj = mj + lin(d, p + "dir_mix")
        s = W[p + "elem_scale.weight"][z].view(N, 4, C) / W["avg_nb"]
        if case["cp"]:
            Af = _pool(None, Y, i, N, [rad[:, B + k * C:B + (k + 1) * C] * mj for k in range(4)])
        else:
            Af = _pool((phi[:, :, None] * mj[:, None, :]).flatten(1), Y, i, N)
        A = [lin(Af[k], p + "mix.%d" % k) for k in range(4)]
        if t > 0 and case["equivariant"]:
            V, M = Vb[:, j, Kd:], Mb[:, j, Kd:]
            full = ((0, 3, 4), (3, 1, 5), (4, 5, 2))
            Mu = torch.stack([sum(M[full[a][b]] * u[:, b:b + 1] for b in range(3)) for a in range(3)])
            uV = torch.stack([0.5 * (u[:, a:a + 1] * V[b] + u[:, b:b + 1] * V[a]) for a, b in SYM[4:10]])
            mom = lambda X: torch.stack([seg((phi[:, :, None] * x[:, None, :]).flatten(1)) for x in X])  # noqa: E731
            A[1] = A[1] + lin(mom(torch.cat([V, Mu], -1)), p + "tmix1")
            A[2] = A[2] + lin(mom(torch.cat([M, uV], -1)), p + "tmix2")
        A = [A[k] * s[None, :, k] for k in range(4)]
        sets.append(A)
        PQS = [lin(torch.cat([S[k] for S in sets], -1), p + "proj.%d" % k).permute(1, 2, 0).split(C, 1) for k in range(4)]
        (P0, _, _), (P1, Q1, S1), (P2, Q2, S2), (P3, Q3, _) = PQS
        gated = case["equivariant"] and t < case["passes"] - 1
        zero = P1.new_zeros(4, C)
        ab = (W[p + "vpath"], W[p + "mpath"]) if gated else (zero, zero)
        inv, V, M = _algebra(P1, Q1, S1, P2, Q2, S2, P3, Q3, *ab)
        inv = torch.cat([P0[..., 0]] + list(inv.unbind(-1)), 1)
        inv = F.layer_norm(inv, (9 * C,), W[p + "norm.weight"], W[p + "norm.bias"])
        o = lin(F.silu(lin(F.silu(lin(torch.cat([inv, h, inv.new_zeros(N, 4)], 1), p + "out.0")), p + "out.2")), p + "out.4")
        if gated:
            gv, gm = lin(inv, p + "gate").chunk(2, -1)
            M = torch.stack([0.5 * (M[..., a, b] + M[..., b, a]) for a, b in SYM[4:10]])
            eq = (V.permute(2, 0, 1) * gv, M * gm)
        e_at, h = e_at + W["scale"] * o[:, 0], h + o[:, 1:]
    owner = torch.repeat_interleave(torch.arange(len(st), device=DEV), torch.tensor([len(s["pos"]) for s in st], device=DEV))
    E = e_at.new_zeros(len(st)).index_add(0, owner, e_at)
    forces = -torch.autograd.grad(E.sum(), pos)[0]
    out = {"energy": (E[0] if case["kind"] == "md" else E).detach(), "forces": forces}
    return dict(out, atom_energy=e_at.detach()) if case["kind"] == "batch" else out


def exact(case, seed):
    kind = case["kind"]
    if kind == "pairs":
        return None
    if kind in ("md", "batch", "step"):
        wide = case["C"] if case["cp"] else 16 * case["K"]
        if case["atoms"] * _neighbours(case) * wide > 2.5e8:     # the unfused 64-bit edge tensors outgrow the card
            return None
        return _whole64(case, seed)
    f8 = lambda v: [f8(x) for x in v] if isinstance(v, (list, tuple)) else v.double() if v is not None and v.is_floating_point() else v  # noqa: E731
    if kind == "pooling":
        i = _graph_rows(case, seed)
        h2, w, b, env, msg, Y = f8(_edge_inputs(case, seed, len(i), case["C"]))
        N, C = case["atoms"], case["C"]
        up = f8([_normal(seed, 9 + k, n, N, C) for k, n in enumerate(RANK_K)])
        ins = [t.requires_grad_(True) for t in (h2, env, msg, Y)]
        R = F.linear(h2, w, b) * env[:, None]
        outs = _pool(None, Y, i, N, [R[:, k * C:(k + 1) * C] * msg for k in range(4)])
    else:
        ins, consts, up = (f8(v) for v in _layer_inputs(case, seed))
        ins = [t.requires_grad_(True) for t in ins]
        if kind == "density":
            phi, msg, Y = ins
            x = (phi[..., :, None] * msg[..., None, :]).flatten(2)
            outs = [torch.stack([(x * Y[..., c:c + 1]).sum(1) for c in range(20)], 1)]
        elif kind == "algebra":
            outs = list(_algebra(*ins, *consts))[: 3 if case["eq"] else 1]
            up = up[: len(outs)]
        elif kind == "moments":
            z, s, wm, wt, wp = consts
            C, D = case["C"], dict(zip((1, 2), ins[8:]))
            outs = []
            for k in range(4):
                A = F.linear(ins[k], wm[k])
                if k in D:
                    A = A + F.linear(D[k], wt[k - 1])
                A = A * s[z].view(-1, 4, C)[None, :, k]
                outs.append(F.linear(torch.cat([ins[4 + k], A], -1), wp[k]))
        else:
            W0, b0, W1, b1, W2, b2, Wg, bg = consts
            o = F.linear(F.silu(F.linear(F.silu(F.linear(torch.cat(ins, 1), W0, b0)), W1, b1)), W2, b2)
            outs = [o[:, :1]] if case["last"] else [o[:, :1], ins[1] + o[:, 1:], F.linear(ins[0], Wg, bg)]
    grads = torch.autograd.grad(outs, ins, up)
    return {"outputs": [o.detach() for o in outs], "gradients": list(grads)}


def _graph_rows(case, seed):
    """Receiver of every edge, grouped by receiver."""
    i, _, _ = _pairs64(_structures(case, seed), case["rc"])
    return torch.sort(i).values
