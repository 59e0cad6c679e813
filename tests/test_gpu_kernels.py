"""GPU parity of the HIP kernels against the CPU oracle (fp64 einsums + autograd).

Tolerances follow the reference's own kernel tests: max-abs error / max-abs reference
< 1e-4 for every output and gradient (tests/test_kernels.py:17-19, tests/test_node_kernel.py:84-89).
"""
import itertools
import sys

import numpy as np
import pytest
import torch

from oracle import cartesian
from oracle import ops as oops

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 1e-4


def rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return ((a - b).abs().max() / b.abs().max().clamp_min(1e-30)).item()


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


# ----------------------------------------------------------------------------- factor density
@pytest.mark.parametrize("B,K", [(16, 32), (32, 32), (8, 16), (16, 64)])
def test_factor_density_dropin_matches_reference_spec(B, K):
    """tests/test_kernels.py:7-20: N=300, M=37, seed 0, randn inputs and upstream G."""
    from face_amd.kernels import factor_density
    say("factor_density", B, K)
    N, M = 300, 37
    torch.manual_seed(0)
    phi = torch.randn(N, M, B, device=DEV, requires_grad=True)
    msg = torch.randn(N, M, K, device=DEV, requires_grad=True)
    Y = torch.randn(N, M, 20, device=DEV, requires_grad=True)
    G = torch.randn(N, 20, B * K, device=DEV)
    D1 = factor_density(phi, msg, Y)
    g1 = torch.autograd.grad((D1 * G).sum(), (phi, msg, Y))
    ins = [t.detach().double().cpu().requires_grad_(True) for t in (phi, msg, Y)]
    D2 = oops.factor_density(*ins)
    g2 = torch.autograd.grad((D2 * G.double().cpu()).sum(), ins)
    errs = [rel(D1, D2)] + [rel(a, b) for a, b in zip(g1, g2)]
    assert max(errs) < TOL, errs


class _G:
    """Random symmetric CSR graph for operator tests: unique undirected pairs, a hub row,
    isolated atoms; rows sorted by neighbour; reverse map computed on the host."""

    def __init__(self, N, n_pairs, seed, hub=70):
        from face_amd.ops import Graph
        rng = np.random.default_rng(seed)
        pairs = set()
        while len(pairs) < n_pairs:
            i, j = rng.integers(0, N - 3, 2)          # the last 3 atoms stay isolated
            if i != j:
                pairs.add((min(i, j), max(i, j)))
        for j in range(1, min(hub, N - 3)):
            pairs.add((0, j))
        directed = sorted([(i, j) for i, j in pairs] + [(j, i) for i, j in pairs])
        index = {e: k for k, e in enumerate(directed)}
        recv = np.array([e[0] for e in directed], np.int32)
        col = np.array([e[1] for e in directed], np.int32)
        rev = np.array([index[(j, i)] for i, j in directed], np.int32)
        counts = np.bincount(recv, minlength=N)
        row_ptr = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
        self.counts = counts.tolist()
        t = lambda a: torch.as_tensor(a, device=DEV)
        self.G = Graph(torch.zeros(N, 3, device=DEV), None, None, 1, None, t(row_ptr), t(col), t(recv), None, t(rev),
                       int(counts.max()))


def _pad(x_edge, counts, M):
    """(E, ...) edge tensor -> (N, M, ...) zero padded (for the padded oracle): one gather and a
    mask, so that autograd through it stays linear in the size."""
    N = len(counts)
    if x_edge.shape[0] == 0:
        return x_edge.new_zeros(N, M, *x_edge.shape[1:])
    cnt = torch.as_tensor(counts, dtype=torch.int64, device=x_edge.device)
    start = torch.cumsum(cnt, 0) - cnt
    slot = torch.arange(M, device=x_edge.device)
    valid = slot[None, :] < cnt[:, None]
    idx = (start[:, None] + slot[None, :]).clamp(max=x_edge.shape[0] - 1)
    out = x_edge[idx.reshape(-1)].reshape(N, M, *x_edge.shape[1:])
    return out * valid.reshape(N, M, *([1] * (x_edge.dim() - 1))).to(x_edge.dtype)


@pytest.mark.parametrize("nx,gathered,B,K", [(20, False, 16, 32), (20, True, 16, 32), (4, True, 16, 144), (20, False, 8, 16),
                                             (4, True, 8, 36), (20, False, 16, 64), (20, False, 16, 48),
                                             (20, True, 16, 80)])
def test_csr_density_ragged_rows(nx, gathered, B, K):
    """Factor density forward / backward on ragged CSR rows (a 53-edge hub row, isolated atoms)
    against the oracle: the split-product kernels (20 monomials, B = 16, K up to 64) and the general
    ones (other B, K and the 4-monomial set)."""
    from face_amd import ops
    say("csr density", nx, gathered, B, K)
    g = _G(57, 500, 2)
    counts = g.counts
    E = sum(counts)
    torch.manual_seed(3)
    phi = torch.randn(E, B + 5, device=DEV)[:, :B].requires_grad_(True)   # strided rows
    tab_rows = 57 if gathered else E
    msg = torch.randn(tab_rows, K, device=DEV, requires_grad=True)
    Y = torch.randn(E, 20, device=DEV, requires_grad=True)
    out = ops.density(phi, msg, Y, g.G, nx, gathered)
    D = torch.cat(out, 0) if nx == 20 else out              # monomial-major (nx, N, B*K)
    assert D.shape == (nx, 57, B * K)
    D = D.permute(1, 0, 2)
    G = torch.randn_like(D)
    gr = torch.autograd.grad((D * G).sum(), (phi, msg, Y))
    # oracle on the padded layout
    M = max(counts)
    col = g.G.col.long().cpu()
    pd = lambda t: _pad(t, counts, M)
    ph = phi.detach().double().cpu().requires_grad_(True)
    ms = msg.detach().double().cpu().requires_grad_(True)
    Yc = Y.detach().double().cpu().requires_grad_(True)
    msg_e = ms[col] if gathered else ms
    D2 = oops.factor_density(pd(ph), pd(msg_e), pd(Yc)[..., :nx])
    gr2 = torch.autograd.grad((D2 * G.double().cpu()).sum(), (ph, ms, Yc))
    errs = [rel(D, D2)] + [rel(a, b) for a, b in zip(gr, gr2)]
    assert max(errs) < TOL, errs
    # bitwise reproducible (no atomics)
    out3 = ops.density(phi, msg, Y, g.G, nx, gathered)
    D3 = (torch.cat(out3, 0) if nx == 20 else out3).permute(1, 0, 2)
    assert torch.equal(D, D3)


@pytest.mark.parametrize("gathered,C", [(False, 160), (True, 160), (False, 96), (True, 40)])
def test_cp_density_ragged_rows(gathered, C):
    from face_amd import ops
    say("cp density", gathered, C)
    g = _G(41, 600, 5)
    counts = g.counts
    E = sum(counts)
    torch.manual_seed(6)
    R = torch.randn(E, 16 + 4 * C, device=DEV)[:, 16:].requires_grad_(True)
    env = torch.rand(E, device=DEV, requires_grad=True)
    msg = torch.randn(41 if gathered else E, C, device=DEV, requires_grad=True)
    Y = torch.randn(E, 20, device=DEV, requires_grad=True)
    A = torch.cat(ops.cp_density(R, env, msg, Y, g.G, gathered), 0).permute(1, 0, 2)   # (N, 20, C)
    G = torch.randn_like(A)
    gr = torch.autograd.grad((A * G).sum(), (R, env, msg, Y))
    M = max(counts)
    col = g.G.col.long().cpu()
    pd = lambda t: _pad(t, counts, M)
    Rc = R.detach().double().cpu().requires_grad_(True)
    ec = env.detach().double().cpu().requires_grad_(True)
    ms = msg.detach().double().cpu().requires_grad_(True)
    Yc = Y.detach().double().cpu().requires_grad_(True)
    A2 = oops.cp_density(pd((Rc * ec[:, None]).view(E, 4, C)), pd(ms[col] if gathered else ms), pd(Yc))
    gr2 = torch.autograd.grad((A2 * G.double().cpu()).sum(), (Rc, ec, ms, Yc))
    errs = [rel(A, A2)] + [rel(a, b) for a, b in zip(gr, gr2)]
    assert max(errs) < TOL, errs


@pytest.mark.parametrize("gathered,C,H,N,pairs", [(False, 160, 64, 41, 600), (True, 160, 64, 41, 600),
                                                  (True, 96, 32, 41, 600), (False, 64, 16, 41, 600),
                                                  (True, 32, 48, 41, 600), (False, 160, 64, 3000, 20000),
                                                  (True, 192, 64, 300, 3000), (False, 320, 64, 41, 600)])
def test_cp_radial_density_fused_backward(gathered, C, H, N, pairs):
    """R = h2 W^T + b feeding the CP pooling, whose backward returns d h2 = dR W from inside the
    pooling kernel: with W^T resident in LDS (H x 4C fp32 up to 160 KB; the 3000-atom graph gives
    every wave of the grid a share of rows), with W^T staged in channel slabs (C = 192, H = 64), or,
    at C = 320 where neither fits, by the pooling backward writing dR and a separate product.
    Outputs and gradients (h2, env, msg, Y) vs the oracle in fp64."""
    from face_amd import ops
    say("cp radial density", gathered, C, H, N, pairs)
    g = _G(N, pairs, 5, hub=70 if N < 100 else 16)
    counts = g.counts
    E = sum(counts)
    torch.manual_seed(C + H)
    h2 = torch.randn(E, H, device=DEV, requires_grad=True)
    W = torch.randn(4 * C, H, device=DEV) / H ** 0.5
    b = torch.randn(4 * C, device=DEV) * 0.1
    env = torch.rand(E, device=DEV, requires_grad=True)
    msg = torch.randn(N if gathered else E, C, device=DEV, requires_grad=True)
    Y = torch.randn(E, 20, device=DEV, requires_grad=True)
    A = torch.cat(ops.cp_radial_density(h2, W, b, env, msg, Y, g.G, gathered), 0).permute(1, 0, 2)   # (N, 20, C)
    G = torch.randn_like(A)
    gr = torch.autograd.grad((A * G).sum(), (h2, env, msg, Y))
    M = max(counts)
    col = g.G.col.long().cpu()
    pd = lambda t: _pad(t, counts, M)
    hc = h2.detach().double().cpu().requires_grad_(True)
    ec = env.detach().double().cpu().requires_grad_(True)
    ms = msg.detach().double().cpu().requires_grad_(True)
    Yc = Y.detach().double().cpu().requires_grad_(True)
    Rc = hc @ W.double().cpu().T + b.double().cpu()
    A2 = oops.cp_density(pd((Rc * ec[:, None]).view(E, 4, C)), pd(ms[col] if gathered else ms), pd(Yc))
    gr2 = torch.autograd.grad((A2 * G.double().cpu()).sum(), (hc, ec, ms, Yc))
    errs = [rel(A, A2)] + [rel(a, b) for a, b in zip(gr, gr2)]
    say("   errs", errs)
    assert max(errs) < TOL, errs


def _ragged_counts(N, seed):
    """Row lengths with runs of empty rows at the start, inside and at the end, a run of one-edge
    rows (16-edge tiles holding up to 16 atom segments) and rows longer than a tile."""
    rng = np.random.default_rng(seed)
    body = rng.integers(0, 60, N - 3 - 40 - 6 - 5)
    body[rng.integers(0, body.size, body.size // 8)] = 0
    return [0, 0, 0] + [1] * 40 + [0] * 6 + body.tolist() + [70, 0, 0, 0, 0]


@pytest.mark.parametrize("C,H,N,gathered,with_b,with_env,with_R", [
    (160, 64, 700, False, True, True, True), (160, 64, 700, True, True, True, True),
    (96, 32, 700, True, False, True, True), (16, 16, 300, False, True, False, True),
    (320, 64, 300, False, True, True, False), (48, 48, 300, True, True, True, True),
    (192, 64, 3000, False, True, True, True), (160, 64, 60, True, True, True, True),
    (160, 64, 24000, False, True, True, True)])
def test_cp_radial_fused_forward_matches_two_launch_route(C, H, N, gathered, with_b, with_env, with_R):
    """The fused CP radial forward (R = h2 W^T + b computed, written and pooled in one launch)
    through the C ABI against the two-launch route on the same inputs (face_edge_linear_fwd then
    face_cp_density_fwd): R bitwise equal, A within fp32 rounding of the edge-serial pooling and
    within TOL of the fp64 oracle; every output row written (outputs start as NaN), empty rows
    exactly zero. Channel widths give 1 to 5 16-channel blocks per part and 1 to 4 parts. The
    24,000-atom case (rows of 30-74 edges, 1.25 M edges: the benchmark liquid's shape, every wave
    of the grid on its own share) is checked against the two-launch route only (the padded fp64
    oracle would need ~10 GB there)."""
    from face_amd import _lib, ops
    say("cp radial fused fwd", C, H, N, gathered, with_b, with_env, with_R)
    full = N >= 10000
    counts = (np.random.default_rng(N).integers(30, 75, N).tolist() if full else _ragged_counts(N, C + H))
    E = int(sum(counts))
    rng = np.random.default_rng(N + C)
    row_ptr = torch.as_tensor(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), device=DEV)
    col = torch.as_tensor(rng.integers(0, N, E).astype(np.int32), device=DEV)
    torch.manual_seed(C * H + N)
    h2 = torch.randn(E, H, device=DEV)
    W = torch.randn(4 * C, H, device=DEV) / H ** 0.5
    b = torch.randn(4 * C, device=DEV) * 0.1 if with_b else None
    env = torch.rand(E, device=DEV) if with_env else None
    msg = torch.randn(N if gathered else E, C, device=DEV)
    Y = torch.randn(E, 20, device=DEV)
    row = col if gathered else None
    st = _lib.stream_of(h2)
    outs = [torch.full((k, N, C), float("nan"), device=DEV) for k in ops.RANK_K]
    R = torch.full((E, 4 * C), float("nan"), device=DEV) if with_R else None
    P = _lib.ptr
    _lib.call("face_cp_radial_fwd", P(h2), H, H, P(W), P(b), P(env), P(msg), C, P(row), P(Y), 20, P(row_ptr), N, E,
              C, *_lib.ranks_of_blocks(outs), P(R), 4 * C, st)
    R2 = ops.edge_linear(h2, W, b)
    outs2 = [torch.empty(k, N, C, device=DEV) for k in ops.RANK_K]
    _lib.call("face_cp_density_fwd", P(R2), 4 * C, P(env), P(msg), C, P(row), P(Y), 20, P(row_ptr), N, 0, C,
              *_lib.ranks_of_blocks(outs2), st)
    torch.cuda.synchronize()
    if with_R:
        assert torch.equal(R, R2)
    A = torch.cat(outs, 0).permute(1, 0, 2)                               # (N, 20, C)
    A2 = torch.cat(outs2, 0).permute(1, 0, 2)
    assert torch.isfinite(A).all()
    empty = torch.as_tensor(counts, device=DEV) == 0
    assert (A[empty] == 0).all()
    scale = A2.abs().max().item()
    assert (A - A2).abs().max().item() <= 2e-6 * scale
    if full:
        return
    M = max(counts)
    pd = lambda t: _pad(t, counts, M)
    Rc = h2.double().cpu() @ W.double().cpu().T + (b.double().cpu() if with_b else 0)
    ec = env.double().cpu() if with_env else torch.ones(E, dtype=torch.float64)
    ms = msg.double().cpu()
    A3 = oops.cp_density(pd((Rc * ec[:, None]).view(E, 4, C)), pd(ms[col.long().cpu()] if gathered else ms),
                         pd(Y.double().cpu()))
    assert rel(A, A3) < TOL


def test_cp_radial_fused_forward_without_edges():
    """No edges at all: every row of A is zero, and h2 / W may be NULL."""
    from face_amd import _lib, ops
    N, C = 37, 32
    row_ptr = torch.zeros(N + 1, dtype=torch.int32, device=DEV)
    msg = torch.randn(N, C, device=DEV)
    Y = torch.randn(1, 20, device=DEV)
    outs = [torch.full((k, N, C), float("nan"), device=DEV) for k in ops.RANK_K]
    _lib.call("face_cp_radial_fwd", None, 64, 64, None, None, None, _lib.ptr(msg), C, None, _lib.ptr(Y), 20,
              _lib.ptr(row_ptr), N, 0, C, *_lib.ranks_of_blocks(outs), None, 4 * C, _lib.stream_of(msg))
    torch.cuda.synchronize()
    assert all((o == 0).all() for o in outs)


@pytest.mark.parametrize("what", ["Y", "Yinf", "env", "msg", "h2"])
@pytest.mark.parametrize("C,H,gathered", [(160, 64, True), (160, 64, False), (48, 16, True)])
def test_cp_radial_fused_forward_contains_non_finite_edges(C, H, gathered, what):
    """A NaN or an infinity on some edges (coincident atoms have NaN directions) stays with the receivers of
    those edges: every other atom keeps its bits, though tiles of 32 edges span atoms, and a NaN in the
    directions leaves the receiver's monomial of rank 0 alone."""
    from face_amd import _lib, ops
    say("cp radial fwd non-finite", C, H, gathered, what)
    N = 300
    counts = _ragged_counts(N, C + H)
    E = int(sum(counts))
    rec = np.repeat(np.arange(N), counts)
    row_ptr = torch.as_tensor(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), device=DEV)
    rng = np.random.default_rng(C)
    col = torch.as_tensor(rng.integers(1, N, E).astype(np.int32), device=DEV)
    torch.manual_seed(C + H)
    t = {"h2": torch.randn(E, H, device=DEV), "env": torch.rand(E, device=DEV), "Y": torch.randn(E, 20, device=DEV),
         "msg": torch.randn(N if gathered else E, C, device=DEV)}
    W, b = torch.randn(4 * C, H, device=DEV) / H ** 0.5, torch.randn(4 * C, device=DEV)
    bad = np.concatenate([[0, 7, 31, 32, E - 1], rng.integers(0, E, 12)])     # edges of tiles and of the list
    if what == "msg" and gathered:
        col[torch.as_tensor(bad, device=DEV)] = 0                             # the one bad table row

    def run():
        outs = [torch.full((k, N, C), 7.0, device=DEV) for k in ops.RANK_K]
        P = _lib.ptr
        _lib.call("face_cp_radial_fwd", P(t["h2"]), H, H, P(W), P(b), P(t["env"]), P(t["msg"]), C,
                  P(col) if gathered else None, P(t["Y"]), 20, P(row_ptr), N, E, C, *_lib.ranks_of_blocks(outs), None,
                  4 * C, _lib.stream_of(W))
        return torch.cat(outs, 0)                                             # (20, N, C)

    clean = run()
    assert torch.isfinite(clean).all()
    at = torch.as_tensor([0] if what == "msg" and gathered else bad, device=DEV)
    if what[0] == "Y":
        t["Y"][at, 1:] = float("nan") if what == "Y" else float("inf")
    else:
        t[what][at] = float("nan")
    out = run()
    hit = torch.zeros(N, dtype=torch.bool, device=DEV)
    hit[torch.as_tensor(rec[bad], device=DEV)] = True
    assert torch.equal(out[:, ~hit], clean[:, ~hit])
    assert not torch.isfinite(out[1:, hit]).any()
    assert torch.equal(out[0, hit], clean[0, hit]) if what[0] == "Y" else torch.isnan(out[0, hit]).all()


@pytest.mark.parametrize("where", ["x", "w"])
@pytest.mark.parametrize("C,H,gathered", [(160, 64, True), (48, 16, False), (16, 48, True)])
def test_edge_products_of_values_past_bf16(C, H, gathered, where):
    """Inputs or weights between the largest bf16 and the largest float32, and an infinity, take the plain float32
    products of the CP pooling forward and of the per-edge linear: last tiles of 21 edges, 16-channel tails, rows of
    several tiles. Bounds: one rounding (2^-24 of the sum of magnitudes) per term of the dot product and, for A, per
    edge of the row, plus four for the factors of a term."""
    from face_amd import _lib
    say("edge products past bf16", C, H, gathered, where)
    N = 300
    counts = _ragged_counts(N, C + H)
    counts[60] += (21 - sum(counts)) % 32
    E, rec = int(sum(counts)), np.repeat(np.arange(N), counts)
    assert E % 32 == 21
    row_ptr = torch.as_tensor(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), device=DEV)
    col = torch.as_tensor(np.random.default_rng(C).integers(0, N, E).astype(np.int32), device=DEV)
    torch.manual_seed(C + H)
    h2, W, b = torch.randn(E, H, device=DEV), torch.randn(4 * C, H, device=DEV) / H ** 0.5, torch.randn(4 * C, device=DEV)
    env, Y = torch.rand(E, device=DEV), 2 * torch.rand(E, 20, device=DEV) - 1
    msg = 2 * torch.rand(N if gathered else E, C, device=DEV) - 1
    tab = torch.randn(N, 4 * C, device=DEV)
    big, inf = 3.395e38, E // 2
    if where == "x":
        W[:, 1] = W[:, 1].clamp(-0.25, 0.25)
        W[:, 2] = W[:, 2].abs() + 0.1                                 # a definite sign against the infinity
        h2[[0, 33, E - 1], 1] = big
        h2[inf, 2] = float("inf")
    else:
        h2[:, 1] = 0.002 * h2[:, 1].clamp(-1, 1)                      # sums over a row of edges stay finite
        W[[0, 2 * C + 17 % C, 4 * C - 1], 1] = big
    P, st = _lib.ptr, _lib.stream_of(h2)
    outs = [torch.full((k, N, C), float("nan"), device=DEV) for k in (1, 3, 6, 10)]
    R, L = torch.full((E, 4 * C), 7.0, device=DEV), torch.full((E, 4 * C), 7.0, device=DEV)
    _lib.call("face_cp_radial_fwd", P(h2), H, H, P(W), P(b), P(env), P(msg), C, P(col) if gathered else None, P(Y), 20,
              P(row_ptr), N, E, C, *_lib.ranks_of_blocks(outs), P(R), 4 * C, st)
    _lib.call("face_edge_linear_fwd", P(h2), H, E, H, P(W), P(b), 4 * C, P(tab), 4 * C, P(col), P(L), 4 * C, st)
    torch.cuda.synchronize()
    edges = torch.ones(E, dtype=torch.bool, device=DEV)
    if where == "x":
        edges[inf] = False
        assert bool((R[inf] == float("inf")).all()) and bool((L[inf] == float("inf")).all())
    u = 2.0 ** -24
    ref = h2.double() @ W.double().t().contiguous() + b.double()
    mag = h2.double().abs() @ W.double().abs().t().contiguous() + b.double().abs()
    assert bool(((R.double() - ref).abs() <= (H + 1) * u * mag)[edges].all())
    t = tab.double()[col.long()]
    assert bool(((L.double() - ref - t).abs() <= (H + 2) * u * (mag + t.abs()))[edges].all())
    atoms = torch.ones(N, dtype=torch.bool, device=DEV)
    if where == "x":
        atoms[int(rec[inf])] = False
        assert not bool(torch.isfinite(outs[0][0, int(rec[inf])]).any())
        ref[inf], mag[inf] = 0.0, 0.0
    m = (msg[col.long()] if gathered else msg).double() * env.double()[:, None]
    at = torch.as_tensor(rec, device=DEV)
    x0 = 0
    for l, k in enumerate((1, 3, 6, 10)):
        for x in range(k):
            y = Y[:, x0 + x].double()[:, None]
            want = torch.zeros(N, C, dtype=torch.float64, device=DEV).index_add_(0, at, y * m * ref[:, l * C:(l + 1) * C])
            size = torch.zeros_like(want).index_add_(0, at, (y * m).abs() * mag[:, l * C:(l + 1) * C])
            assert bool(((outs[l][x].double() - want).abs() <= (H + max(counts) + 4) * u * size)[atoms].all()), (l, x)
        x0 += k


# ----------------------------------------------------------------------------- gated outputs
@pytest.mark.parametrize("N,C", [(1000, 160), (37, 96), (1, 4)])
def test_eq_gate_matches_torch(N, C):
    """V * gv, Ms * gm (face/model.py:286-287): outputs bit-exact against torch fp32, gradients of
    V, Ms and the gate row within fp32 rounding of torch's autograd."""
    from face_amd import ops
    say("eq_gate", N, C)
    torch.manual_seed(N + C)
    V = torch.randn(3, N, C, device=DEV, requires_grad=True)
    Ms = torch.randn(6, N, C, device=DEV, requires_grad=True)
    gvm = torch.randn(N, 2 * C, device=DEV, requires_grad=True)
    Vo, Mo = ops.eq_gate(V, Ms, gvm)
    gv, gm = gvm.chunk(2, dim=-1)
    Vr, Mr = V * gv[None], Ms * gm[None]
    assert torch.equal(Vo, Vr) and torch.equal(Mo, Mr)
    gV, gM = torch.randn_like(Vo), torch.randn_like(Mo)
    g1 = torch.autograd.grad((Vo * gV).sum() + (Mo * gM).sum(), (V, Ms, gvm))
    g2 = torch.autograd.grad((Vr * gV).sum() + (Mr * gM).sum(), (V, Ms, gvm))
    for a, b in zip(g1, g2):
        assert (a - b).abs().max().item() <= 1e-6 * (1 + b.abs().max().item())


@pytest.mark.parametrize("N,F", [(24000, 1440), (37, 864), (5, 4), (300, 2048)])
def test_layer_norm_matches_torch(N, F):
    """Readout LayerNorm (face/model.py:332) and its input gradient against torch's fp32
    LayerNorm on the same device, within fp32 rounding."""
    from face_amd import ops
    say("layer_norm", N, F)
    torch.manual_seed(N + F)
    x = (torch.randn(N, F, device=DEV) * 3 + 1).requires_grad_(True)
    w = torch.randn(F, device=DEV)
    b = torch.randn(F, device=DEV)
    y1 = ops.layer_norm(x, w, b, 1e-5)
    y2 = torch.nn.functional.layer_norm(x, (F,), w, b, 1e-5)
    assert (y1 - y2).abs().max().item() < 1e-5 * (1 + y2.abs().max().item())
    dy = torch.randn_like(y1)
    g1, = torch.autograd.grad((y1 * dy).sum(), x)
    g2, = torch.autograd.grad((y2 * dy).sum(), x)
    assert (g1 - g2).abs().max().item() < 1e-5 * (1 + g2.abs().max().item())


# ----------------------------------------------------------------------------- node algebra
@pytest.mark.parametrize("eq", [True, False])
def test_node_algebra_dropin_matches_reference_spec(eq):
    """tests/test_node_kernel.py:8-28: N=50, C=24, seed 1, outputs and every gradient incl. da, db."""
    from face_amd.node_kernel import node_algebra
    say("node_algebra eq", eq)
    torch.manual_seed(1)
    N, C = 50, 24
    shapes = [(3,), (3,), (3,), (6,), (6,), (6,), (10,), (10,)]
    xs = [torch.randn(N, C, *s, device=DEV, requires_grad=True) for s in shapes]
    a = torch.randn(4, C, device=DEV, requires_grad=True)
    b = torch.randn(4, C, device=DEV, requires_grad=True)
    gI, gV, gM = torch.randn(N, C, 8, device=DEV), torch.randn(N, C, 3, device=DEV), torch.randn(N, C, 3, 3, device=DEV)
    o1 = node_algebra(*xs, a, b, eq)
    L = lambda o, gi, gv, gm: (o[0] * gi).sum() + (((o[1] * gv).sum() + (o[2] * gm).sum()) if eq else 0)
    vars1 = xs + ([a, b] if eq else [])
    g1 = torch.autograd.grad(L(o1, gI, gV, gM), vars1, allow_unused=True)
    xc = [t.detach().double().cpu().requires_grad_(True) for t in xs]
    ac, bc = a.detach().double().cpu().requires_grad_(True), b.detach().double().cpu().requires_grad_(True)
    o2 = oops.node_algebra_sym(*xc, ac, bc)
    vars2 = xc + ([ac, bc] if eq else [])
    g2 = torch.autograd.grad(L(o2, gI.double().cpu(), gV.double().cpu(), gM.double().cpu()), vars2,
                             allow_unused=True)
    outs1 = list(o1[:3] if eq else o1[:1])
    outs2 = list(o2[:3] if eq else o2[:1])
    errs = [rel(u, v) for u, v in zip(outs1 + list(g1), outs2 + list(g2))]
    assert max(errs) < TOL, errs


@pytest.mark.parametrize("eq", [True, False])
@pytest.mark.parametrize("N,C", [(1, 1), (1, 255), (2, 128), (1, 257), (37, 48)])
def test_node_algebra_dense_rows_equal_strided(N, C, eq):
    """The kernels of dense (N, C, k) operands, 256 rows per workgroup (1, 255, 256, 257 and 1,776 rows),
    against the strided ones on the same values stored component-major: outputs and all gradients. Both
    form the same sums of at most 27 terms; contraction may differ (1e-6 of the largest value)."""
    from face_amd.node_kernel import node_algebra
    say("node dense", N, C, eq)
    torch.manual_seed(N * C)
    base = [torch.randn(N, C, k, device=DEV) for k in (3, 3, 3, 6, 6, 6, 10, 10)]
    ab = [torch.randn(4, C, device=DEV) for _ in range(2)]
    ups = [torch.randn(N, C, 8, device=DEV), torch.randn(N, C, 3, device=DEV), torch.randn(N, C, 3, 3, device=DEV)]
    res = []
    for dense in (True, False):
        if dense:
            ins = [x.clone().requires_grad_(True) for x in base]
        else:                                        # strides (C, 1, N C)
            ins = [x.permute(2, 0, 1).contiguous().permute(1, 2, 0).requires_grad_(True) for x in base]
        a, b = [x.clone().requires_grad_(True) for x in ab]
        outs = node_algebra(*ins, a, b, eq)[:3 if eq else 1]
        grads = torch.autograd.grad(outs, ins + ([a, b] if eq else []), ups[:len(outs)])
        res.append(list(outs) + list(grads))
    for x, y in zip(*res):
        assert x.shape == y.shape and rel(x, y) < 1e-6


def test_node_features_product_layout():
    """Strided P/Q/S read from projection outputs, families written into the readout row,
    symmetrised gated products (face/model.py:244-249,274-276)."""
    from face_amd import ops
    say("node features")
    torch.manual_seed(2)
    N, C = 37, 20
    y0 = torch.randn(1, N, C, device=DEV, requires_grad=True)
    y1 = torch.randn(3, N, 3 * C, device=DEV, requires_grad=True)
    y2 = torch.randn(6, N, 3 * C, device=DEV, requires_grad=True)
    y3 = torch.randn(10, N, 2 * C, device=DEV, requires_grad=True)
    a = torch.randn(4, C, device=DEV, requires_grad=True)
    b = torch.randn(4, C, device=DEV, requires_grad=True)
    feats, V, Ms = ops.node_features(y0, y1, y2, y3, a, b, True, C)
    gf, gv, gm = torch.randn_like(feats), torch.randn_like(V), torch.randn_like(Ms)
    vars1 = [y0, y1, y2, y3, a, b]
    g1 = torch.autograd.grad((feats * gf).sum() + (V * gv).sum() + (Ms * gm).sum(), vars1)
    yc = [t.detach().double().cpu().requires_grad_(True) for t in vars1]
    c0, c1, c2, c3, ac, bc = yc
    split = lambda y, k: [y[..., j * C:(j + 1) * C].permute(1, 2, 0) for j in range(k)]
    P1, Q1, S1 = split(c1, 3)
    P2, Q2, S2 = split(c2, 3)
    P3, Q3 = split(c3, 2)
    inv, Vr, Mf = oops.node_algebra_sym(P1, Q1, S1, P2, Q2, S2, P3, Q3, ac, bc)
    feats2 = torch.cat([c0[0]] + list(inv.unbind(-1)), 1)
    Ms2 = cartesian.to_sym2(0.5 * (Mf + Mf.transpose(-1, -2))).permute(2, 0, 1)
    V2 = Vr.permute(2, 0, 1)
    L2 = (feats2 * gf.double().cpu()).sum() + (V2 * gv.double().cpu()).sum() + (Ms2 * gm.double().cpu()).sum()
    g2 = torch.autograd.grad(L2, yc)
    errs = [rel(feats, feats2), rel(V, V2), rel(Ms, Ms2)] + [rel(u, v) for u, v in zip(g1, g2)]
    assert max(errs) < TOL, errs


@pytest.mark.parametrize("N,C,eq,wide", [(37, 20, True, False), (50, 96, True, True), (23, 160, False, False),
                                         (9, 256, True, False), (5, 40, False, True)])
def test_node_layer_norm_fused_matches_oracle(N, C, eq, wide):
    """Node algebra with the readout LayerNorm in one kernel each way (face/model.py:244-264, :332)
    against the oracle's node algebra + torch layer_norm in fp64: the normalised row, V, Ms and
    every input gradient; C not a multiple of the wave width, y0 rows wider than C."""
    from face_amd import ops
    say("node + layer norm", N, C, eq, wide)
    torch.manual_seed(N + C)
    y0 = torch.randn(1, N, 2 * C if wide else C, device=DEV, requires_grad=True)
    y1 = torch.randn(3, N, 3 * C, device=DEV, requires_grad=True)
    y2 = torch.randn(6, N, 3 * C, device=DEV, requires_grad=True)
    y3 = torch.randn(10, N, 2 * C, device=DEV, requires_grad=True)
    a = torch.randn(4, C, device=DEV) if eq else None
    b = torch.randn(4, C, device=DEV) if eq else None
    lw = torch.rand(9 * C, device=DEV) + 0.5
    lb = torch.randn(9 * C, device=DEV) * 0.1
    inv, V, Ms = ops.node_ln(y0, y1, y2, y3, a, b, eq, C, lw, lb, 1e-5)
    gi = torch.randn_like(inv)
    L = (inv * gi).sum()
    if eq:
        gv, gm = torch.randn_like(V), torch.randn_like(Ms)
        L = L + (V * gv).sum() + (Ms * gm).sum()
    vars1 = [y0, y1, y2, y3]
    g1 = torch.autograd.grad(L, vars1)
    yc = [t.detach().double().cpu().requires_grad_(True) for t in vars1]
    c0, c1, c2, c3 = yc
    ac = a.double().cpu() if eq else torch.zeros(4, C, dtype=torch.float64)
    bc = b.double().cpu() if eq else torch.zeros(4, C, dtype=torch.float64)
    split = lambda y, k: [y[..., j * C:(j + 1) * C].permute(1, 2, 0) for j in range(k)]
    P1, Q1, S1 = split(c1, 3)
    P2, Q2, S2 = split(c2, 3)
    P3, Q3 = split(c3, 2)
    invr, Vr, Mf = oops.node_algebra_sym(P1, Q1, S1, P2, Q2, S2, P3, Q3, ac, bc)
    feats = torch.cat([c0[0, :, :C]] + list(invr.unbind(-1)), 1)
    inv2 = torch.nn.functional.layer_norm(feats, (9 * C,), lw.double().cpu(), lb.double().cpu(), 1e-5)
    L2 = (inv2 * gi.double().cpu()).sum()
    outs, refs = [inv], [inv2]
    if eq:
        Ms2 = cartesian.to_sym2(0.5 * (Mf + Mf.transpose(-1, -2))).permute(2, 0, 1)
        V2 = Vr.permute(2, 0, 1)
        L2 = L2 + (V2 * gv.double().cpu()).sum() + (Ms2 * gm.double().cpu()).sum()
        outs += [V, Ms]
        refs += [V2, Ms2]
    g2 = torch.autograd.grad(L2, yc)
    errs = [rel(u, v) for u, v in zip(outs, refs)] + [rel(u, v) for u, v in zip(g1, g2)]
    say("   errs", errs)
    assert max(errs) < TOL, errs
    if wide:
        assert float(g1[0][0, :, C:].abs().max()) == 0.0


# ----------------------------------------------------------------------------- gathers / scatter
def test_gathers_and_force_scatter_match_index_add():
    from face_amd import ops
    from face_amd.neighbors import build_graph
    from face_amd import systems
    say("gathers / scatter")
    (liq,) = [systems.liquid(500, np.random.default_rng(9), rho=0.1, dmin=0.9)]
    g = build_graph([liq], 4.0)
    torch.manual_seed(0)
    X = torch.randn(g.N, 7, device=DEV, requires_grad=True)
    Xj = ops.gather_neighbour(X, g)
    Xi = ops.gather_receiver(X, g)
    col, recv = g.col.long(), g.recv.long()
    assert torch.equal(Xj, X[col]) and torch.equal(Xi, X[recv])
    w1, w2 = torch.randn_like(Xj), torch.randn_like(Xi)
    (gx,) = torch.autograd.grad((Xj * w1).sum() + (Xi * w2).sum(), X)
    ref = torch.zeros_like(X).index_add(0, col, w1).index_add(0, recv, w2)
    assert rel(gx, ref) < 1e-5
    gvec = torch.randn(g.E, 3, device=DEV)
    grad = torch.empty(g.N, 3, device=DEV)
    from face_amd._lib import call, ptr, stream_of
    call("face_force_scatter", ptr(gvec), ptr(g.row_ptr), ptr(g.rev), g.N, 1.0, ptr(grad), stream_of(gvec))
    ref = torch.zeros(g.N, 3, device=DEV).index_add(0, col, gvec).index_add(0, recv, -gvec)
    assert rel(grad, ref) < 1e-5
    # the contiguous row form: reverse slots and per-window own-row sums laid out as the edge backward
    # (face_edge_geom_bwd_seg) writes them, wsum filled only at the last edge of each row in each
    # 64-edge window (NaN elsewhere: never read), then the row pass (both lane widths)
    # (16-byte rows: x, y, z and an unused fourth float, NaN here)
    gvec_rev = torch.full((g.E, 4), float("nan"), device=DEV)
    gvec_rev[:, :3] = gvec[g.rev.long()]
    e_idx = torch.arange(g.E, device=DEV)
    seg = recv * ((g.E + 63) // 64) + e_idx // 64
    _, inv, cnt = torch.unique_consecutive(seg, return_inverse=True, return_counts=True)
    sums = torch.zeros(cnt.numel(), 3, device=DEV).index_add(0, inv, gvec)
    wsum = torch.full((g.E, 4), float("nan"), device=DEV)
    wsum[torch.cumsum(cnt, 0) - 1, :3] = sums
    for mean_row in (16, 40):
        grad2 = torch.full((g.N, 3), float("nan"), device=DEV)
        call("face_force_scatter_rows", ptr(gvec_rev), ptr(wsum), ptr(g.row_ptr), g.N, mean_row, -1.0, ptr(grad2),
             stream_of(gvec))
        assert rel(-grad2, ref) < 1e-5


# ----------------------------------------------------------------------------- edge geometry
@pytest.mark.parametrize("system", ["molecules", "liquid"])
def test_edge_geometry_forward_and_backward(system):
    """Edge geometry, basis and envelope and their backward into dE/dpos (the row-organised edge
    backward and the contiguous force scatter; short molecule rows and ~40-pair periodic rows)."""
    from face_amd import ops
    from face_amd.neighbors import build_graph
    from face_amd import systems
    say("edge geometry", system)
    rc = 4.5
    if system == "molecules":
        st = systems.molecules(6, np.random.default_rng(2))
    else:
        st = [systems.liquid(400, np.random.default_rng(4), rho=0.1, dmin=0.9)]
    g = build_graph(st, rc)
    pos = g.pos.clone().requires_grad_(True)
    freq = (torch.arange(1, 9) * np.pi / rc).float().to(DEV)
    Y, rb, env, rr = ops.edge_geometry(pos, g, freq, rc, with_r=True)
    wY, wr, we, wd = torch.randn_like(Y), torch.randn_like(rb), torch.randn_like(env), torch.randn_like(rr)
    (gp,) = torch.autograd.grad((Y * wY).sum() + (rb * wr).sum() + (env * we).sum() + (rr * wd).sum(), pos)
    # each input handed to several readers as views of one tensor: their gradients, summed in the
    # edge backward, give the same forces as one reader with the summed upstream gradient
    outs = ops.edge_geometry(pos, g, freq, rc, with_r=True, counts=(3, 2, 4, 2))
    assert len(outs) == 11 and all(torch.equal(t, Y) for t in outs[:3]) and torch.equal(outs[3], rb)
    parts = [(outs[0], 0.5 * wY), (outs[1], 0.25 * wY), (outs[2], 0.25 * wY), (outs[3], 0.5 * wr), (outs[4], 0.5 * wr),
             (outs[5], we), (outs[6], 0 * we), (outs[9], 0.5 * wd), (outs[10], 0.5 * wd)]   # one env view unread
    (gp_v,) = torch.autograd.grad(sum((t * w).sum() for t, w in parts), pos)
    assert (gp_v - gp).abs().max() <= 1e-5 * gp.abs().max()
    # without the Bessel rows (compiled radial): rb is empty and the rest unchanged
    Y3, rb3, env3, r3 = ops.edge_geometry(pos.detach(), g, freq, rc, with_rb=False, with_r=True)
    assert rb3.numel() == 0 and torch.equal(Y3, Y.detach()) and torch.equal(r3, rr.detach())
    # oracle: the reference formulas in fp64 on the CPU (face/model.py:670-677, :28-40)
    pc = g.pos.detach().double().cpu().requires_grad_(True)
    col, recv = g.col.long().cpu(), g.recv.long().cpu()
    vec = pc[col] - pc[recv] + g.shift.double().cpu()
    r = torch.sqrt((vec * vec).sum(-1))
    u = vec / r[:, None]
    x = r / rc
    e_ref = (1 - 28 * x ** 6 + 48 * x ** 7 - 21 * x ** 8) * (x < 1)
    bes = torch.sin(torch.arange(1, 9, dtype=torch.float64) * np.pi / rc * r[:, None]) / r[:, None] * np.sqrt(2 / rc)
    Y2, rb2 = cartesian.monomials(u), bes * e_ref[:, None]
    (gp2,) = torch.autograd.grad((Y2 * wY.double().cpu()).sum() + (rb2 * wr.double().cpu()).sum()
                                 + (e_ref * we.double().cpu()).sum() + (r * wd.double().cpu()).sum(), pc)
    errs = [rel(Y, Y2), rel(rb, rb2), rel(env, e_ref), rel(rr, r), rel(gp, gp2)]
    assert max(errs) < TOL, errs


@pytest.mark.parametrize("P,G,F,nb", [(9, 4096, 16, 16), (9, 4096, 16 + 4 * 160, 16), (1, 300, 16, 16),
                                       (4, 64, 37, 5), (2, 33, 6, 0)])
def test_radial_spline_matches_oracle(P, G, F, nb):
    """Compiled radial (face/model.py:407-418, :466-467): phi = S[:, :nb] * env and R = S[:, nb:]
    with their r / env gradients, against the oracle's RadialSpline in fp64 (autograd), for radii
    inside the grid, on grid points, and beyond its end (clamped, zero r-derivative). The tables
    sample smooth functions, as compiled radial functions are: with random, non-smooth tables the
    fp32 rounding of r / dr alone (2e-4 of a cell at 4096 points) moves the value by ~1e-4."""
    from face_amd import ops
    from oracle.model import RadialSpline
    say("spline", P, G, F, nb)
    gen = torch.Generator().manual_seed(G + F)
    rc = 5.0
    dr = rc / (G - 1)
    rg = (torch.arange(G, dtype=torch.float64) * dr)[None, :, None]
    amp, k, ph = (torch.randn(P, 1, F, generator=gen, dtype=torch.float64) for _ in range(3))
    k = 0.3 + 2.5 * k.abs()
    T = (amp * torch.sin(k * rg + ph) + 0.1 * amp * rg ** 2).float()
    dT = (amp * k * torch.cos(k * rg + ph) + 0.2 * amp * rg).float()
    E = 3000
    rng = np.random.default_rng(F)
    r = rng.uniform(1e-4, rc + 0.7, E)
    r[:50] = np.arange(50) % G * dr                              # on grid points
    r = torch.tensor(r, dtype=torch.float32)
    pair = torch.tensor(rng.integers(0, P, E), dtype=torch.int32)
    env = torch.rand(E, generator=gen)
    rd, envd = r.to(DEV).requires_grad_(True), env.to(DEV).requires_grad_(True)
    phi, R = ops.radial_spline(rd, envd, pair.to(DEV), T.to(DEV), dT.to(DEV), dr, nb)
    assert phi.shape == (E, nb) and R.shape == (E, F - nb)
    wp, wq = torch.randn(E, nb, generator=gen), torch.randn(E, F - nb, generator=gen)
    gr, ge = torch.autograd.grad((phi * wp.to(DEV)).sum() + (R * wq.to(DEV)).sum(), (rd, envd))
    sp = RadialSpline(T.double(), dT.double(), dr)
    rc_, ec = r.double().requires_grad_(True), env.double().requires_grad_(True)
    S = sp(rc_, pair.long())
    phi2, R2 = S[:, :nb] * ec[:, None], S[:, nb:]
    gr2, ge2 = torch.autograd.grad((phi2 * wp.double()).sum() + (R2 * wq.double()).sum(), (rc_, ec))
    errs = [rel(phi, phi2) if nb else 0.0, rel(R, R2) if F > nb else 0.0, rel(gr, gr2), rel(ge, ge2) if nb else 0.0]
    assert max(errs) < TOL, errs
    assert float(gr[r.to(DEV) > rc + 1e-3].abs().max()) == 0.0   # clamped: no r-derivative


def test_radial_spline_without_envelope_as_a_reference_binding():
    """The call pattern of a binding inside the reference's RadialSpline.forward (padded (N, M)
    radii and pair indices flattened, no envelope pointer, nb = F): values and r-gradient equal
    the oracle's RadialSpline in fp64."""
    from face_amd._lib import call, ptr, stream_of
    from oracle.model import RadialSpline
    say("spline binding")
    P, G, F, N, M = 9, 4096, 16, 40, 23
    dr = 4.5 / (G - 1)
    gen = torch.Generator().manual_seed(4)
    rg = (torch.arange(G, dtype=torch.float64) * dr)[None, :, None]
    amp, k = torch.randn(P, 1, F, generator=gen, dtype=torch.float64), 0.5 + torch.rand(P, 1, F, generator=gen)
    T, dT = (amp * torch.cos(k * rg)).float(), (-amp * k * torch.sin(k * rg)).float()
    r = torch.rand(N, M, generator=gen) * 4.4 + 0.05
    pair = torch.randint(0, P, (N, M), generator=gen)
    rd, pd = r.reshape(-1).to(DEV), pair.reshape(-1).to(torch.int32).to(DEV)
    E = N * M
    S = torch.empty(E, F, device=DEV)
    Td, dTd = T.to(DEV), dT.to(DEV)
    st = stream_of(rd)
    call("face_radial_spline_fwd", ptr(rd), ptr(pd), E, ptr(Td), ptr(dTd), P, G, F, dr, None, F, None, ptr(S), F,
         None, 0, st)
    w = torch.randn(E, F, generator=gen)
    gr = torch.empty(E, device=DEV)
    call("face_radial_spline_bwd", ptr(rd), ptr(pd), E, ptr(Td), ptr(dTd), P, G, F, dr, None, F, None,
         ptr(w.to(DEV)), F, None, 0, ptr(gr), None, st)
    sp = RadialSpline(T.double(), dT.double(), dr)
    rc = r.double().requires_grad_(True)
    S2 = sp(rc, pair)
    (gr2,) = torch.autograd.grad((S2 * w.double().view(N, M, F)).sum(), rc)
    assert max(rel(S, S2.reshape(E, F)), rel(gr, gr2.reshape(-1))) < TOL


@pytest.mark.parametrize("P,G,F,nb,E", [(5, 700, 24, 8, 20000), (9, 4096, 16 + 4 * 160, 16, 150000),
                                         (4, 4096, 16 + 4 * 256, 16, 40000), (2, 40, 8 + 4 * 32, 8, 3001)])
def test_radial_spline_order_is_a_cell_sorted_permutation(P, G, F, nb, E):
    """face_radial_spline_order: a permutation of the edges with non-decreasing table cell
    (pair * G + grid interval, the same cell the spline kernels use), including radii past the
    grid's end (last interval); the spline outputs in that order (the cell-run kernels, which
    keep each cell's table rows in registers over its run of edges) equal the unordered per-edge
    kernels' bitwise, at the CP widths (16 + 4C columns, C = 160 and 256) too."""
    from face_amd._lib import call, ptr, stream_of
    say("spline order", P, G, F, nb, E)
    rc = 4.0
    dr = rc / (G - 1)
    rng = np.random.default_rng(9)
    r = torch.tensor(rng.uniform(1e-4, rc + 0.5, E), dtype=torch.float32, device=DEV)
    pair = torch.tensor(rng.integers(0, P, E), dtype=torch.int32, device=DEV)
    work = torch.empty(P * G, dtype=torch.int32, device=DEV)
    order = torch.empty(E, dtype=torch.int32, device=DEV)
    st = stream_of(r)
    call("face_radial_spline_order", ptr(r), ptr(pair), E, P, G, dr, ptr(work), ptr(order), st)
    o = order.long().cpu()
    assert torch.equal(torch.sort(o).values, torch.arange(E))
    x = (r.cpu() / dr).clamp(0, G - 1)
    cell = pair.long().cpu() * G + torch.floor(x).long().clamp(max=G - 2)
    assert bool((cell[o][1:] >= cell[o][:-1]).all())
    T = torch.randn(P, G, F, device=DEV)
    dT = torch.randn(P, G, F, device=DEV)
    env = torch.rand(E, device=DEV)
    outs = []
    for od in (None, order):
        phi = torch.empty(E, nb, device=DEV)
        R = torch.empty(E, F - nb, device=DEV)
        call("face_radial_spline_fwd", ptr(r), ptr(pair), E, ptr(T), ptr(dT), P, G, F, dr, ptr(env), nb, ptr(od),
             ptr(phi), nb, ptr(R), F - nb, st)
        gp, gq = torch.ones(E, nb, device=DEV), torch.ones(E, F - nb, device=DEV)
        gr, ge = torch.empty(E, device=DEV), torch.empty(E, device=DEV)
        call("face_radial_spline_bwd", ptr(r), ptr(pair), E, ptr(T), ptr(dT), P, G, F, dr, ptr(env), nb, ptr(od),
             ptr(gp), nb, ptr(gq), F - nb, ptr(gr), ptr(ge), st)
        outs.append((phi, R, gr, ge))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("Kd,B,transport", [(16, 16, True), (4, 8, True), (5, 4, False), (16, 16, False)])
def test_dir_transport_and_gradients(Kd, B, transport, packed, monkeypatch):
    """Directional features d = [u.V_j, u^T M_j u, u.V_i, u^T M_i u] (face/model.py:474-493) and the
    transport sums D1 = [sum phi V, sum phi M u], D2 = [sum phi M, sum phi sym(u V)] (face/model.py:
    514-528) vs gathered einsums and the oracle's explicit per-edge transport tensors, with the
    tables read in place and packed node-major."""
    from face_amd import ops
    monkeypatch.setattr(ops, "DIR_PACK_MIN_BYTES", 0 if packed else 1 << 40)
    say("dir/transport", Kd, B, transport, "packed" if packed else "in place")
    g = _G(37, 300, Kd + 10)
    counts = g.counts
    E = sum(counts)
    nt = 2 if transport else 1
    torch.manual_seed(Kd)
    Vb = torch.randn(3, 37, nt * Kd, device=DEV, requires_grad=True)
    Mb = torch.randn(6, 37, nt * Kd, device=DEV, requires_grad=True)
    phi = torch.randn(E, B, device=DEV, requires_grad=True)
    Y = torch.randn(E, 20, device=DEV, requires_grad=True)
    d, D1, D2 = ops.dir_transport(Vb, Mb, phi, Y, g.G, Kd, transport)
    wd = torch.randn_like(d)
    L = (d * wd).sum()
    if transport:
        w1, w2 = torch.randn_like(D1), torch.randn_like(D2)
        L = L + (D1 * w1).sum() + (D2 * w2).sum()
    ins = [Vb, Mb, Y] + ([phi] if transport else [])
    grads = torch.autograd.grad(L, ins)
    # oracle (fp64, CPU)
    c = [t.detach().double().cpu().requires_grad_(True) for t in ins]
    Vc, Mc, Yc = c[:3]
    col, recv = g.G.col.long().cpu(), g.G.recv.long().cpu()
    u = Yc[:, 1:4]
    Y2 = Yc[:, 4:10] * torch.tensor([1.0, 1, 1, 2, 2, 2], dtype=torch.float64)
    Vj, Mj = Vc[:, col, :Kd], Mc[:, col, :Kd]            # (3|6, E, Kd)
    Vi, Mi = Vc[:, recv, :Kd], Mc[:, recv, :Kd]
    d2 = torch.cat([torch.einsum("ea,aek->ek", u, Vj), torch.einsum("ea,aek->ek", Y2, Mj),
                    torch.einsum("ea,aek->ek", u, Vi), torch.einsum("ea,aek->ek", Y2, Mi)], -1)
    L2 = (d2 * wd.double().cpu()).sum()
    outs, refs = [d], [d2]
    if transport:
        pc = c[3]
        M = max(counts)
        pd = lambda t: _pad(t, counts, M)
        Vt = Vc[:, col, Kd:].permute(1, 2, 0)            # (E, Kd, 3)
        Mt = Mc[:, col, Kd:].permute(1, 2, 0)            # (E, Kd, 6)
        R1, R2 = oops.transport_sums(pd(pc), pd(u), pd(Vt), pd(Mt), 1.0)   # (N, B*2Kd, 3|6)
        R1, R2 = R1.permute(2, 0, 1), R2.permute(2, 0, 1)
        L2 = L2 + (R1 * w1.double().cpu()).sum() + (R2 * w2.double().cpu()).sum()
        outs += [D1, D2]
        refs += [R1, R2]
    grads2 = torch.autograd.grad(L2, c)
    errs = [rel(a, b) for a, b in zip(outs, refs)] + [rel(a, b) for a, b in zip(grads, grads2)]
    assert max(errs) < TOL, errs


# ----------------------------------------------------------------------------- radial MLP
@pytest.mark.parametrize("E,H,F,offset", [(100000, 64, 640, 0), (1001, 16, 128, 0), (37, 48, 640, 0),
                                          (5, 32, 1024, 0), (300, 64, 1280, 0), (4099, 64, 640, 4), (0, 64, 640, 0)])
def test_radial_head_matches_torch(E, H, F, offset):
    """R = h2 w^T + b for the CP columns of the last radial layer vs torch fp64: whole-LDS weight
    images with the rotated (H = 64, F = 640) and padded row layouts, the feature-chunked grid
    (H = 64, F = 1280), ragged edge tiles and a row stride / base offset that is not the width."""
    from face_amd import ops
    say("radial head", E, H, F, offset)
    torch.manual_seed(E + F)
    base = torch.randn(E * (H + offset) + offset, device=DEV)
    h2 = base[offset:offset + E * (H + offset)].view(E, H + offset)[:, :H] if E else torch.empty(0, H, device=DEV)
    w = torch.randn(F, H, device=DEV) / H ** 0.5
    b = torch.randn(F, device=DEV)
    R = ops.radial_head(h2, w, b)
    assert R.shape == (E, F)
    if E == 0:
        return
    ref = h2.double() @ w.double().T + b.double()
    err = rel(R, ref)
    say("   err", err)
    assert err < 1e-5, err


@pytest.mark.parametrize("F,K", [(160, 64), (32, 64), (16, 16), (256, 48), (48, 32)])
def test_edge_message_matches_torch(F, K):
    """gather(msg(h)) + dir_mix(d) (face/model.py:488-493) as one launch, m[e] = T[col e] + d[e] W^T
    + b, and its backward (d T by the reverse-edge reduction, d d = dm W) vs torch fp64 on a
    random symmetric graph with a 70-neighbour hub row (5 edge tiles) and isolated atoms."""
    from face_amd import ops
    say("edge message", F, K)
    gr = _G(700, 9000, F + K)
    g = gr.G
    torch.manual_seed(F * K)
    T = torch.randn(g.N, F, device=DEV, requires_grad=True)
    d = torch.randn(g.E, K, device=DEV, requires_grad=True)
    w = torch.randn(F, K, device=DEV) / K ** 0.5
    b = torch.randn(F, device=DEV)
    m = ops.edge_message(T, d, w, b, g)
    gm = torch.randn_like(m)
    gT, gd = torch.autograd.grad((m * gm).sum(), (T, d))
    Tc = T.detach().double().cpu().requires_grad_(True)
    dc = d.detach().double().cpu().requires_grad_(True)
    mr = Tc[g.col.long().cpu()] + dc @ w.double().cpu().T + b.double().cpu()
    gT2, gd2 = torch.autograd.grad((mr * gm.double().cpu()).sum(), (Tc, dc))
    errs = [rel(m, mr), rel(gT, gT2), rel(gd, gd2)]
    say("   errs", errs)
    assert max(errs) < 1e-5, errs
    assert float(gT[-3:].abs().max()) == 0.0                   # isolated atoms: exact zero rows


@pytest.mark.parametrize("E,nb,H,B,n_pair,want_h2",[(20000, 8, 64, 16, 9, True), (20000, 8, 64, 16, 1, False),
                                                      (1001, 8, 16, 8, 9, False), (37, 8, 32, 20, 4, True),
                                                      (5, 12, 48, 32, 9, True), (0, 8, 64, 16, 9, True)])
def test_radial_mlp_matches_torch(E, nb, H, B, n_pair, want_h2):
    """phi = (silu(silu(rb W_in^T + b_in + pair_tab[pair]) W1^T + b1) W_phi^T + b_phi) * env and h2
    (face/model.py:465-469) vs the same layers in torch fp64, with the gradients of rb and env."""
    from face_amd import ops
    say("radial", E, nb, H, B, n_pair, want_h2)
    torch.manual_seed(E + H)
    rb = torch.randn(E, nb, device=DEV, requires_grad=True)
    env = torch.rand(E, device=DEV, requires_grad=True)
    pair = torch.randint(0, n_pair, (E,), device=DEV, dtype=torch.int32)
    ws = [torch.randn(H, nb) / nb ** 0.5, torch.randn(H) * 0.1, torch.randn(n_pair, H) * 0.3,
          torch.randn(H, H) / H ** 0.5, torch.randn(H) * 0.1, torch.randn(B, H) / H ** 0.5, torch.randn(B) * 0.1]
    ws = [w.to(DEV) for w in ws]
    phi, phi_b, h2 = ops.radial_mlp(rb, env, pair, *ws, want_h2)
    assert phi.shape == (E, B) and h2.shape == ((E, H) if want_h2 else (0, H))
    assert torch.equal(phi, phi_b)
    if E == 0:
        return
    gp = torch.randn_like(phi)
    # the upstream gradient split over the two readers' views (summed in the backward kernel)
    L = (phi * (0.25 * gp)).sum() + (phi_b * (0.75 * gp)).sum()
    gh = torch.randn(E, H, device=DEV)
    if want_h2:
        L = L + (h2 * gh).sum()
    grads = torch.autograd.grad(L, [rb, env])
    # torch fp64 reference
    rc = rb.detach().double().requires_grad_(True)
    ec = env.detach().double().requires_grad_(True)
    w = [t.double() for t in ws]
    hid = torch.nn.functional.silu(rc @ w[0].T + w[1] + w[2][pair.long()])
    h2r = torch.nn.functional.silu(hid @ w[3].T + w[4])
    phir = (h2r @ w[5].T + w[6]) * ec[:, None]
    L2 = (phir * gp.double()).sum() + ((h2r * gh.double()).sum() if want_h2 else 0)
    grads2 = torch.autograd.grad(L2, [rc, ec])
    outs, refs = [phi] + ([h2] if want_h2 else []), [phir] + ([h2r] if want_h2 else [])
    errs = [rel(a, b) for a, b in zip(outs, refs)] + [rel(a, b) for a, b in zip(grads, grads2)]
    say("   errs", errs)
    assert max(errs) < TOL, errs


@pytest.mark.parametrize("E,n_sets,want_h2", [(15552, 2, False), (20000, 2, True), (1001, 3, True), (37, 4, False)])
def test_radial_mlp_sets_equal_single_launches(E, n_sets, want_h2):
    """The radial MLPs of several passes in one launch each way give bitwise the outputs and
    input gradients of one launch per pass (the same instructions per set): rb / envelope read
    through per-pass views, a second phi reader on some passes, no gradient on others."""
    from face_amd import ops
    say("radial sets", E, n_sets, want_h2)
    torch.manual_seed(E + n_sets)
    nb, H, B, n_pair = 8, 64, 16, 9
    base_rb = torch.randn(E, nb, device=DEV, requires_grad=True)
    base_env = torch.rand(E, device=DEV, requires_grad=True)
    pair = torch.randint(0, n_pair, (E,), device=DEV, dtype=torch.int32)
    wsets = []
    for _ in range(n_sets):
        ws = [torch.randn(H, nb) / nb ** 0.5, torch.randn(H) * 0.1, torch.randn(n_pair, H) * 0.3,
              torch.randn(H, H) / H ** 0.5, torch.randn(H) * 0.1, torch.randn(B, H) / H ** 0.5, torch.randn(B) * 0.1]
        wsets.append([w.to(DEV) for w in ws])
    gps = [torch.randn(E, B, device=DEV) for _ in range(n_sets)]
    ghs = [torch.randn(E, H, device=DEV) for _ in range(n_sets)]

    def loss(outs):
        L = 0
        for k, (phi, phi_b, h2) in enumerate(outs):
            L = L + (phi * gps[k]).sum()
            if k % 2 == 1:
                L = L + (phi_b * (0.5 * gps[k])).sum()
            if want_h2 and k != 1:
                L = L + (h2 * ghs[k]).sum()
        return L
    rbs = [base_rb.view(base_rb.shape) for _ in range(n_sets)]
    envs = [base_env.view(base_env.shape) for _ in range(n_sets)]
    outs = ops.radial_mlp_sets(pair, wsets, want_h2, rbs, envs)
    got = torch.autograd.grad(loss(outs), rbs + envs)
    rbs2 = [base_rb.view(base_rb.shape) for _ in range(n_sets)]
    envs2 = [base_env.view(base_env.shape) for _ in range(n_sets)]
    outs2 = [ops.radial_mlp(rbs2[k], envs2[k], pair, *wsets[k], want_h2) for k in range(n_sets)]
    want = torch.autograd.grad(loss(outs2), rbs2 + envs2)
    for a, b in zip(outs, outs2):
        for x, y in zip(a, b):
            assert torch.equal(x, y)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


# ----------------------------------------------------------------------------- row-block linear layers
def _lin_ref(x, w, w_kn, y0, beta, bias, xs, ys, grp, period, s_off):
    x, w = x.double().cpu(), w.double().cpu()
    g = grp.long().cpu()[torch.arange(x.shape[0]) % period] if grp is not None else None
    if xs is not None:
        x = x * xs.double().cpu()[g][:, s_off:s_off + x.shape[1]]
    y = x @ (w if w_kn else w.T)
    if beta:
        y = y + beta * y0.double().cpu()
    if bias is not None:
        y = y + bias.double().cpu()
    if ys is not None:
        y = y * ys.double().cpu()[g][:, s_off:s_off + y.shape[1]]
    return y


@pytest.mark.parametrize("case,shape", [("single", None), ("ranks_proj", None), ("ranks_scaled", None),
                                        ("kn_xscale", None), ("k512", None), ("empty", None), ("k1024", None),
                                        ("single", "-4"), ("ranks_proj", "-4"), ("ranks_scaled", "-4"), ("kn_xscale", "-4"),
                                        ("k512", "8"), ("empty", "8")])
def test_rows_linear_matches_torch(case, shape, monkeypatch):
    """y = (beta y + (x * xs) w^T + bias) * ys over up to four problems per launch (mix / tmix /
    proj with the elem_scale factor and their input gradients) vs torch fp64: ragged row counts,
    weight column slices (ld_w > k), (k, n) weights, K = 512 and 1024, sliced outputs (n = 480), an
    empty problem beside full ones. shape forces the kernel the size would not choose: "-4" the direct
    one, "8" the staged one in workgroups of eight waves."""
    from face_amd import ops
    say("rows_linear", case, shape)
    torch.manual_seed(len(case))
    N, C = 1000, 160
    grp = torch.randint(0, 3, (N,), device=DEV, dtype=torch.int32)
    tab = torch.rand(3, 4 * C, device=DEV) + 0.5
    bias = xs = ys = None
    w_kn = False
    probs, refs = [], []
    if case == "single":
        x = torch.randn(10007, C, device=DEV)
        w = torch.randn(C, C, device=DEV) / C ** 0.5
        probs = [(x, w, torch.empty(10007, C, device=DEV), 0, 0.0)]
    elif case == "ranks_proj":
        wide = torch.randn(3 * C, 2 * C, device=DEV) / C ** 0.5           # proj weight over two sets
        for l, (k, n) in enumerate(((1, C), (3, 3 * C), (6, 3 * C), (10, 2 * C))):
            x = torch.randn(k * N, C, device=DEV)
            probs.append((x, wide[:n, C:], torch.randn(k * N, n, device=DEV), 0, 1.0 if l % 2 else 0.0))
    elif case == "ranks_scaled":                                             # mix (+ tmix) * elem_scale
        ys, bias = tab, torch.randn(C, device=DEV)
        for l, k in enumerate((1, 3, 6, 10)):
            x = torch.randn(k * N, C, device=DEV)
            w = torch.randn(C, C, device=DEV) / C ** 0.5
            probs.append((x, w, torch.randn(k * N, C, device=DEV), l * C, 1.0 if l in (1, 2) else 0.0))
    elif case == "kn_xscale":
        w_kn, xs = True, tab
        for l, k in enumerate((1, 3, 6, 10)):
            x = torch.randn(k * N, C, device=DEV)
            w = torch.randn(C, 2 * C + 32, device=DEV)[:, 16:16 + 2 * C] / C ** 0.5   # (k, n), ld_w > n
            probs.append((x, w, torch.empty(k * N, 2 * C, device=DEV), l * C, 0.0))
    elif case == "k512":
        x = torch.randn(6 * N, 512, device=DEV)
        w = torch.randn(C, 512, device=DEV) / 512 ** 0.5
        probs = [(x, w, torch.randn(6 * N, C, device=DEV), 0, 1.0)]
    elif case == "k1024":                                                    # the mix of a K = 64 model
        ys = tab
        x = torch.randn(40 * N, 1024, device=DEV)
        w = torch.randn(C, 1024, device=DEV) / 32
        probs = [(x, w, torch.randn(40 * N, C, device=DEV), C, 1.0)]
    else:
        x = torch.randn(0, C, device=DEV)
        probs = [(x, torch.randn(C, C, device=DEV), torch.empty(0, C, device=DEV), 0, 0.0),
                 (torch.randn(77, C, device=DEV), torch.randn(C, C, device=DEV), torch.empty(77, C, device=DEV), 0, 0.0)]
    for (x, w, y, s, b) in probs:
        refs.append(_lin_ref(x, w, w_kn, y, b, bias, xs, ys, grp if (xs is not None or ys is not None) else None, N, s))
    if shape is not None:
        monkeypatch.setenv("FACE_GEMM_SHAPE", f"{shape},{-(-max(p[2].shape[1] for p in probs) // 32)},0")
    ops.rows_linear(probs, w_kn=w_kn, bias=bias, xs=xs, ys=ys, group=grp, period=N)
    errs = [rel(p[2], r) if r.numel() else 0.0 for p, r in zip(probs, refs)]
    say("   errs", errs)
    assert max(errs) < 1e-5, errs


def test_rows_linear_rows_do_not_depend_on_their_number():
    """Launches past one workgroup per CU take the staged kernel, whose sums are the same sequence for any
    number of rows, whatever launch shape the size chooses: the 864-atom factor mix backward (17,280
    rows of 96 -> 512 columns, (k, n) weight, input scale) against its first 2,000 rows and against 17,279 of
    them, plus torch fp64."""
    from face_amd import ops
    say("rows_linear number of rows")
    torch.manual_seed(11)
    N, C, BK = 864, 96, 512
    tab = torch.rand(1, 4 * C, device=DEV) + 0.5
    grp = torch.zeros(N, device=DEV, dtype=torch.int32)
    xs = [torch.randn(k * N, C, device=DEV) for k in (1, 3, 6, 10)]
    ws = [torch.randn(C, BK, device=DEV) / C ** 0.5 for _ in range(4)]

    def run(rows):
        ys = [torch.empty(min(rows, x.shape[0]), BK, device=DEV) for x in xs]
        ops.rows_linear([(x[:y.shape[0]], w, y, l * C, 0.0) for l, (x, w, y) in enumerate(zip(xs, ws, ys))],
                        w_kn=True, xs=tab, group=grp, period=N)
        torch.cuda.synchronize()
        return ys

    full, part, most = run(10 * N), run(2000), run(10 * N - 1)
    for l, (x, w) in enumerate(zip(xs, ws)):
        ref = (x.double() * tab.double()[0, l * C:(l + 1) * C]) @ w.double()
        assert (full[l].double() - ref).abs().max() <= 1e-5 * ref.abs().max()
        assert torch.equal(part[l], full[l][:part[l].shape[0]])
        assert torch.equal(most[l], full[l][:most[l].shape[0]])


def _gemm_shapes(n_widest):
    """Every (waves per workgroup, column slices) pair that gives another launch of the staged kernel: slices
    of 1 to 8 blocks of 32 columns."""
    return [(nw, ns) for nw in (8, 4) for ns in sorted({-(-n_widest // (32 * nb)) for nb in range(1, 9)})]


@pytest.mark.parametrize("case", ["fcc864_mix_bwd", "liquid24k_mix_fwd"])
def test_rows_linear_every_launch_shape_gives_bitwise_equal_rows(case, monkeypatch):
    """Every launch shape of the staged kernel (4 or 8 waves per workgroup, every slice width, plain and
    XCD-aware item order, forced through FACE_GEMM_SHAPE) gives the same bits as the rules' shape: the
    864-atom factor mix backward ((k, n) weight 96 -> 512, input scale, split in the kernel) and the
    24,000-atom CP mix forward (480,000 rows of 160 -> 160 over four ranks, (n, k) weights split ahead where
    the shape has such a kernel, output scale)."""
    from face_amd import ops
    say("rows_linear every shape", case)
    torch.manual_seed(13)
    if case == "fcc864_mix_bwd":
        N, C, n = 864, 96, 512
        w_kn, scale = True, "xs"
        ws = [torch.randn(C, n, device=DEV) / C ** 0.5 for _ in range(4)]
    else:
        N, C, n = 24000, 160, 160
        w_kn, scale = False, "ys"
        ws = [torch.randn(n, C, device=DEV) / C ** 0.5 for _ in range(4)]
    tab = torch.rand(3, 4 * max(C, n), device=DEV) + 0.5
    grp = torch.randint(0, 3, (N,), device=DEV, dtype=torch.int32)
    xs = [torch.randn(k * N, C, device=DEV) for k in (1, 3, 6, 10)]

    def run():
        ys = [torch.empty(x.shape[0], n, device=DEV) for x in xs]
        ops.rows_linear([(x, w, y, l * (C if scale == "xs" else n), 0.0)
                         for l, (x, w, y) in enumerate(zip(xs, ws, ys))], w_kn=w_kn,
                        xs=tab if scale == "xs" else None, ys=tab if scale == "ys" else None, group=grp, period=N)
        torch.cuda.synchronize()
        return ys

    rule = run()
    for l, (x, w) in enumerate(zip(xs, ws)):
        g = grp.long().repeat(x.shape[0] // N)
        if scale == "xs":
            ref = (x.double() * tab.double()[g, l * C:(l + 1) * C]) @ w.double()
        else:
            ref = (x.double() @ w.double().T) * tab.double()[g, l * n:(l + 1) * n]
        assert (rule[l].double() - ref).abs().max() <= 1e-5 * ref.abs().max()
    ran = refused = 0
    for nw, n_sl in _gemm_shapes(n):
        for xcd in (0, 1):
            monkeypatch.setenv("FACE_GEMM_SHAPE", f"{nw},{n_sl},{xcd}")
            try:
                out = run()
            except RuntimeError as err:                  # a slice width without a kernel
                assert "(code -2)" in str(err), err
                refused += 1
                continue
            for a, b in zip(out, rule):
                assert torch.equal(a, b), (nw, n_sl, xcd)
            ran += 1
    say(f"   {ran} shapes bitwise equal to the rules' shape, {refused} refused")
    assert ran == 16, (ran, refused)


def _rows_launch(x, w, y, w_kn, ahead, beta=0.0, xs=None, ys=None, grp=None, s_off=0):
    """face_rows_linear_ws with the weights split in the kernel (ahead False) or ahead into a
    workspace sized here from the header's rule, whatever face_rows_linear_work suggests."""
    from face_amd import _lib
    arr = (_lib.LinProblem * 1)(_lib.LinProblem(x.data_ptr(), x.stride(0), x.shape[0], w.data_ptr(), w.stride(0),
                                                y.data_ptr(), y.stride(0), y.shape[1], x.shape[1], s_off, beta, None, 0,
                                                x.shape[1], 0, None, 0, None, None, 0, 0, 0, None, 0, None, None))
    need = -(-x.shape[1] // 32) * 2 * -(-y.shape[1] // 32) * 3072 if ahead else 0
    work = torch.empty(need, dtype=torch.uint8, device=DEV) if ahead else None
    tab = xs if xs is not None else ys
    _lib.call("face_rows_linear_ws", arr, 1, 1 if w_kn else 0, _lib.ptr(xs), _lib.ptr(ys),
              0 if tab is None else tab.stride(0), 0 if tab is None else tab.shape[0], _lib.ptr(grp),
              0 if grp is None else grp.shape[0], _lib.ptr(work), need, _lib.stream_of(y))
    torch.cuda.synchronize()


@pytest.mark.parametrize("w_kn", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 16, 16), (31, 48, 16), (33, 32, 48), (127, 176, 32), (129, 144, 80), (300, 304, 160),
                                   (64, 528, 112)])
def test_rows_linear_edges_and_weights_split_ahead(m, n, k, w_kn, monkeypatch):
    """Edges of the 32-row, 32-column and 32-k blocks (odd 16-column blocks of n and k, one row to one
    past a tile), accumulating onto y: the direct kernel (K in four parts, the rules' choice at these
    sizes) and the staged kernel with the weights split in it and ahead, the latter two with the same
    bits, all within float32 of torch fp64 (2^-22 |x| |w| per product covers the three-way split and the
    float32 sums)."""
    say("rows_linear edges", m, n, k, w_kn)
    torch.manual_seed(m + n + k)
    x = torch.randn(m, k + 4, device=DEV)[:, :k]
    w = torch.randn(k, n + 4, device=DEV)[:, :n] if w_kn else torch.randn(n, k + 4, device=DEV)[:, :k]
    y0 = torch.randn(m, n + 8, device=DEV)
    wd = w.double() if w_kn else w.double().t().contiguous()
    ref = 0.5 * y0[:, :n].double() + x.double().contiguous() @ wd.contiguous()
    bound = 2.0 ** -22 * (x.double().abs().contiguous() @ wd.abs().contiguous() + y0[:, :n].double().abs())
    outs = []
    for shape, ahead in ((None, False), (f"-4,{-(-n // 64)},0", False), (f"4,{-(-n // 96)},1", False),
                         (f"8,{-(-n // 160)},0", False), (None, True)):
        if shape is None:
            monkeypatch.delenv("FACE_GEMM_SHAPE", raising=False)
        else:
            monkeypatch.setenv("FACE_GEMM_SHAPE", shape)
        y = y0.clone()
        _rows_launch(x, w, y[:, :n], w_kn, ahead, beta=0.5)
        assert torch.equal(y[:, n:], y0[:, n:])                      # nothing past the last column
        assert bool(((y[:, :n].double() - ref).abs() <= bound).all()), (shape, ahead)
        outs.append(y[:, :n])
    assert torch.equal(outs[2], outs[3]) and torch.equal(outs[2], outs[4])


@pytest.mark.parametrize("w_kn", [False, True])
def test_rows_linear_rows_far_apart(w_kn):
    """Seven rows 2^28 elements apart (just below the 2^31 elements an operand may span), where 32 bits do
    not hold a row's byte offset: every operand that has a row stride, plain and with transforms, with and
    without a workspace for the split weights."""
    from face_amd import ops
    say("rows_linear far rows", w_kn)
    torch.manual_seed(6)
    m, ld, k1, k2, n = 7, 1 << 28, 48, 16, 80
    buf = torch.empty(6 * ld + 4096, device=DEV)
    far = lambda at, w: buf.as_strided((m, w), (ld, 1), at)
    x, x2, xz, y0, y = far(0, k1), far(512, k2), far(1024, k1), far(1536, n), far(2048, n)
    for t in (x, x2, xz, y0):
        t.copy_(torch.randn(t.shape, device=DEV))
    w = torch.randn(k1 + k2, n, device=DEV) if w_kn else torch.randn(n, k1 + k2, device=DEV)
    d = lambda t: t.double().cpu()
    wd = d(w) if w_kn else d(w).T
    w1 = w[:k1] if w_kn else w[:, :k1]
    for ahead in (False, True):
        y.fill_(7.0)
        _rows_launch(x, w1, y, w_kn, ahead)
        assert rel(y, d(x) @ wd[:k1]) < 1e-5
    for op in (0, 2):
        y.fill_(7.0)
        ops.rows_linear([ops.lin(x, w, y, x2=x2, x_op=op, xz=xz if op else None, y0=y0, beta=0.5)], w_kn=w_kn)
        z, xi = d(xz), d(x)
        s = torch.sigmoid(z)
        xi = xi * s * (1 + z * (1 - s)) if op else xi
        assert rel(y, 0.5 * d(y0) + torch.cat([xi, d(x2)], 1) @ wd) < 1e-5


@pytest.mark.parametrize("m", [0, 40])
def test_rows_linear_split_ahead_beside_a_problem_of_no_rows(m):
    """Weights split ahead where one problem has no rows and NULL operands, which are then never read
    (and no rows at all: nothing is launched)."""
    from face_amd import _lib
    say("rows_linear split ahead, no rows", m)
    torch.manual_seed(5)
    k, n = 48, 64
    x, w, y = torch.randn(40, k, device=DEV), torch.randn(n, k, device=DEV), torch.full((40, n), 7.0, device=DEV)
    P = lambda rows, *p: _lib.LinProblem(p[0], k, rows, p[1], k, p[2], n, n, k, 0, 0.0, None, 0, k, 0, None, 0, None,
                                         None, 0, 0, 0, None, 0, None, None)
    arr = (_lib.LinProblem * 3)(P(0, None, None, None), P(m, x.data_ptr(), w.data_ptr(), y.data_ptr()),
                                P(0, None, None, None))
    need = 3 * 4 * 2 * 3072
    work = torch.empty(need, dtype=torch.uint8, device=DEV)
    _lib.call("face_rows_linear_ws", arr, 3, 0, None, None, 0, 0, None, 0, _lib.ptr(work), need, _lib.stream_of(y))
    torch.cuda.synchronize()
    ref = x.double() @ w.double().t().contiguous()
    assert rel(y, ref) < 1e-5 if m else bool((y == 7.0).all())


@pytest.mark.parametrize("route", ["direct", "staged", "ahead"])
@pytest.mark.parametrize("where", ["x", "w"])
def test_rows_linear_values_past_bf16(where, route, monkeypatch):
    """Operands that round to a bf16 infinity (3.4e38), infinities and NaN: the results are those of
    plain float32 products, and all other rows, of the same 32-row tile too, keep their bits."""
    say("rows_linear past bf16", where, route)
    ahead = route == "ahead"
    monkeypatch.setenv("FACE_GEMM_SHAPE", "-4,3,0" if route == "direct" else "4,1,0")
    torch.manual_seed(3)
    m, n, k = 200, 96, 64
    x, w = torch.randn(m, k, device=DEV), torch.randn(n, k, device=DEV)
    w[:, 1] = w[:, 1].abs() + 0.5                                    # a definite sign against the infinity
    plain = torch.empty(m, n, device=DEV)
    _rows_launch(x, w, plain, False, ahead)
    big = x.clone() if where == "x" else w.clone()
    big[5, 0], big[70, 1], big[70, 2], big[80, 3] = 3.4e38, float("inf"), 1e30, float("nan")
    small = w if where == "x" else x
    small[:, 0] = small[:, 0].clamp(-0.5, 0.5)                       # 3.4e38 * 0.5 stays finite
    if where == "w":
        small[:, 1] = small[:, 1].abs() + 0.5
    _rows_launch(x, w, plain, False, ahead)
    out = torch.empty(m, n, device=DEV)
    _rows_launch(big if where == "x" else x, big if where == "w" else w, out, False, ahead)
    if where == "w":
        plain, out = plain.t(), out.t()
    ref = (big.double() @ small.double().t().contiguous())
    touched = torch.zeros(out.shape[0], dtype=torch.bool, device=DEV)
    touched[[5, 70, 80]] = True
    if where == "x":
        assert torch.equal(out[~touched], plain[~touched])
    rest = ref[~touched]
    assert (out[~touched].double() - rest).abs().max() <= 1e-5 * rest.abs().max()
    assert bool((out[70] == float("inf")).all()) and bool(torch.isnan(out[80]).all())
    assert (out[5].double() - ref[5]).abs().max() <= 1e-6 * ref[5].abs().max()


@pytest.mark.parametrize("route", ["direct", "staged"])
@pytest.mark.parametrize("e", [-100, -109, -112, -120])
def test_rows_linear_smallest_values(e, route, monkeypatch):
    """Values near the end of the float32 range (identity weights: the sum of the three limbs): exact down to
    2^-110, held to 2^-134 below."""
    monkeypatch.setenv("FACE_GEMM_SHAPE", "-4,1,0" if route == "direct" else "4,1,0")
    torch.manual_seed(2)
    x = (1 + torch.rand(64, 32, device=DEV)) * 2.0 ** e
    y = torch.empty(64, 32, device=DEV)
    _rows_launch(x, torch.eye(32, device=DEV), y, False, False)
    err = (y.double() - x.double()).abs().max().item()
    say("rows_linear smallest values", e, route, err * 2.0 ** 134)
    assert err <= (0 if e >= -110 else 2.0 ** -134)


@pytest.mark.parametrize("last,gate,const_h", [(False, True, False), (False, False, True), (True, False, False),
                                               (True, True, False)])
@pytest.mark.parametrize("N,C", [(1, 16), (33, 48), (700, 160), (40, 24)])
def test_readout_mlp_matches_torch(N, C, last, gate, const_h):
    """ops.readout_mlp on the row-block kernels (C a multiple of 16) and on the library products (24)
    against torch in fp64: outputs and the gradients of the invariant row and h, with h given or folded
    into a constant (hb), the gate row, and the last pass's energy row alone. 5e-6 of the largest value:
    four float32 layers of at most 10 C = 1,600 terms."""
    from face_amd import ops
    say("readout_mlp", N, C, last, gate, const_h)
    torch.manual_seed(N + C)
    r = lambda *s: torch.randn(*s, device=DEV) / s[-1] ** 0.5
    inv, h = torch.randn(N, 9 * C, device=DEV, requires_grad=True), torch.randn(N, C, device=DEV, requires_grad=True)
    W0, b0, W1, b1, W2, b2 = r(2 * C, 10 * C + 4), r(2 * C), r(2 * C, 2 * C), r(2 * C), r(C + 1, 2 * C), r(C + 1)
    Wg, bg = (r(2 * C, 9 * C), r(2 * C)) if gate else (None, None)
    W0a, W0b = W0[:, :9 * C], W0[:, 9 * C:10 * C]
    hb = (h.detach().double() @ W0b.double().t().contiguous() + b0.double()).float() if const_h else None
    outs = ops.readout_mlp(inv, h, W0a, W0b, b0, W1, b1, W2, b2, Wg, bg, last, hb)
    ups = [None if o is None else torch.randn_like(o) for o in outs]
    F = torch.nn.functional
    d = lambda t: t.detach().cpu().double()
    inv_, h_ = d(inv).requires_grad_(True), d(h).requires_grad_(True)
    z0 = F.linear(inv_, d(W0a)) + (d(hb) if const_h else F.linear(h_, d(W0b), d(b0)))
    o = F.linear(F.silu(F.linear(F.silu(z0), d(W1), d(b1))), d(W2), d(b2))
    refs = [o[:, :1], None if last else h_ + o[:, 1:], F.linear(inv_, d(Wg), d(bg)) if gate else None]
    loss = lambda os, us: sum((x * u).sum() for x, u in zip(os, us) if x is not None)
    got = torch.autograd.grad(loss(outs, ups), [inv, h], allow_unused=True)
    want = torch.autograd.grad(loss(refs, [None if u is None else d(u) for u in ups]), [inv_, h_], allow_unused=True)
    for a, b in zip(outs, refs):
        assert (a is None) == (b is None) and (a is None or rel(a, b) < 5e-6)
    assert rel(got[0], want[0]) < 5e-6
    if not const_h:
        assert rel(got[1], want[1]) < 5e-6


@pytest.mark.parametrize("w_kn", [False, True])
@pytest.mark.parametrize("route", ["direct", "staged", "ahead"])
@pytest.mark.parametrize("k", [32, 48, 64, 96, 160, 320, 512, 1440])
def test_rows_linear_sums_do_not_drift(k, route, w_kn):
    """The mean error of many random sums, whose instructions all cut towards minus infinity: -0.7e-8
    (k = 64) to -2.7e-8 (512) and -7.7e-8 (1440) of the results' rms when nothing turns their sign. With the
    turns the drifts of single 16-k steps (1 to 6e-9 each) cancel but for about one step's, 2e-9; below k = 80
    for what the first chunk of 32 has over the others, 5e-9, and a chunk alone keeps its 7e-9."""
    torch.manual_seed(k)
    m, n, reps = (40, 160, 200) if route == "direct" else (8192, 160, 1)
    w = (torch.randn(k, n, device=DEV) if w_kn else torch.randn(n, k, device=DEV)) / k ** 0.5
    wd = w.double() if w_kn else w.double().t().contiguous()
    err, ref = [], []
    for _ in range(reps):
        x, y = torch.randn(m, k, device=DEV), torch.empty(m, n, device=DEV)
        _rows_launch(x, w, y, w_kn, route == "ahead")
        ref.append(x.double() @ wd)
        err.append(y.double() - ref[-1])
    err, rms = torch.cat(err), torch.cat(ref).pow(2).mean().sqrt()
    mean, se = (err.mean() / rms).item(), (err.std() / rms / err.numel() ** 0.5).item()
    say(f"rows_linear drift k {k} {route} kn {w_kn} mean {mean:+.2e} se {se:.1e} rms {(err.pow(2).mean().sqrt() / rms).item():.2e}")
    assert abs(mean) < (2e-9 if k >= 80 else 5.5e-9 if k > 32 else 8e-9)


@pytest.mark.parametrize("op", [0, 1])
@pytest.mark.parametrize("m", [40, 20000, 170000])
def test_rows_linear_adds_a_residual_once(m, op):
    """An initial sum of its own (y0, a thousand times the products) is added to the finished products: one
    rounding of the result and the products' own error (below 2^-21 |x| |w|), in the direct kernel, the staged one
    and the one with the weights split ahead; not a rounding at the residual's size per instruction."""
    from face_amd import ops
    say("rows_linear residual", m, op)
    torch.manual_seed(m)
    k, n = 320, 160
    x, w = torch.randn(m, k, device=DEV), torch.randn(n, k, device=DEV) / k ** 0.5
    y0, y = 1000 * torch.randn(m, n, device=DEV), torch.empty(m, n, device=DEV)
    ops.rows_linear([ops.lin(x, w, y, x_op=op, y0=y0, beta=0.5)])
    xd = torch.nn.functional.silu(x.double()) if op else x.double()
    wd = w.double().t().contiguous()
    ref = 0.5 * y0.double() + xd @ wd
    bound = 2.0 ** -24 * ref.abs() + 2.0 ** -21 * (xd.abs() @ wd.abs())
    assert bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("lo,hi", [(-20.0, -6.0), (-6.0, -1.0), (-1.0, 0.0), (0.0, 1.0), (1.0, 20.0)])
def test_silu_on_load_is_rounded_without_bias(lo, hi):
    """silu and the silu derivative as the row kernels form them (identity weights: the products are exact)
    and as the energy row does, in ulps of the fp64 values: the hardware exponential's ulp and at most six
    roundings to nearest (0.29 rms each), so an rms below 1 and a mean within 0.1 (raw exp2 and reciprocal:
    rms 1 to 5 and mean 0.3 to 0.8 for x < 0; 1 - sigmoid for the slope: rms 2.8 for x > 1)."""
    from face_amd import _lib, ops
    say("silu on load", lo, hi)
    torch.manual_seed(9)
    m, k = 4096, 64
    z = torch.rand(m, k, device=DEV) * (hi - lo) + lo
    one, eye = torch.ones(m, k, device=DEV), torch.eye(k, device=DEV)
    y1, y2, e = torch.empty(m, k, device=DEV), torch.empty(m, k, device=DEV), torch.empty(m, device=DEV)
    ops.rows_linear([ops.lin(z, eye, y1, x_op=1)])
    ops.rows_linear([ops.lin(one, eye, y2, x_op=2, xz=z)])
    _lib.call("face_silu_dot", _lib.ptr(z), k, m, k, _lib.ptr(eye[3].contiguous()), None, _lib.ptr(e), _lib.stream_of(e))
    zd = z.double()
    s = torch.sigmoid(zd)
    for what, got, ref in (("silu", y1, zd * s), ("energy row", e, (zd * s)[:, 3]), ("slope", y2, s * (1 + zd * (1 - s)))):
        ok = ref.abs() > (0.2 if what == "slope" else 0)             # away from the slope's zero at -1.278
        if not ok.any():
            continue
        err = ((got.double() - ref) / 2.0 ** (torch.floor(torch.log2(ref.abs())) - 23))[ok]
        say(f"   {what} mean {err.mean():+.3f} rms {err.pow(2).mean().sqrt():.3f}")
        assert err.pow(2).mean().sqrt() < 1.0
        assert err.mean().abs() < 0.1


def _readout_case(N, C, seed=0):
    """Random operands of ops.readout_mlp with the gate: (inv, h, weights)."""
    torch.manual_seed(seed)
    r = lambda *s: torch.randn(*s, device=DEV) / s[-1] ** 0.5
    ws = [r(2 * C, 9 * C), r(2 * C, C), r(2 * C), r(2 * C, 2 * C), r(2 * C), r(C + 1, 2 * C), r(C + 1), r(2 * C, 9 * C),
          r(2 * C)]
    return torch.randn(N, 9 * C, device=DEV), torch.randn(N, C, device=DEV), ws


@pytest.mark.parametrize("N", [1, 70])
def test_readout_mlp_takes_broadcast_rows(N):
    """Expanded operands and upstream gradients (row stride 0, as a sum over atoms gives; strides of
    one-row tensors; transposed ones) give the results of their dense copies."""
    from face_amd import ops
    say("readout_mlp broadcast", N)
    C = 32
    inv, h, ws = _readout_case(N, C)
    row = lambda w: torch.randn(1, w, device=DEV).expand(N, w)
    odd = lambda w: torch.randn(w, N, device=DEV).t()
    hb = row(2 * C)

    def run(inv, h, hb, ups):
        i, x = inv.detach().requires_grad_(True), h.detach().requires_grad_(True)
        outs = ops.readout_mlp(i, x, *ws, False, hb)
        return list(outs) + list(torch.autograd.grad(outs, [i, x], ups))

    for give_hb in (False, True):
        for ins in ((row(9 * C), row(C)), (odd(9 * C), odd(C)), (inv, h)):
            for ups in ([row(1), row(C), row(2 * C)], [odd(1), odd(C), odd(2 * C)]):
                got = run(*ins, hb if give_hb else None, ups)
                want = run(*(t.clone(memory_format=torch.contiguous_format) for t in ins), hb.clone(
                    memory_format=torch.contiguous_format) if give_hb else None,
                    [u.clone(memory_format=torch.contiguous_format) for u in ups])
                assert all(torch.equal(a, b) for a, b in zip(got, want))
    # a loss over sums of the outputs, as a user writes it
    i, x = inv.requires_grad_(True), h.requires_grad_(True)
    v = torch.randn(C, device=DEV)
    outs = ops.readout_mlp(i, x, *ws, False)
    got = torch.autograd.grad(outs[0].sum() + (outs[1].sum(0) * v).sum() + outs[2].sum(), [i, x])
    outs = ops.readout_mlp(i, x, *ws, False)
    want = torch.autograd.grad(outs, [i, x], [torch.ones(N, 1, device=DEV), v.repeat(N, 1), torch.ones(N, 2 * C, device=DEV)])
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_readout_mlp_refuses_or_broadcasts_other_shapes():
    """Operands whose shape, type or place is not the row-block kernels': refused where the library products
    refuse them (a row of other width, a weight of other shape, another type, host memory), and broadcast where
    these broadcast (a bias of one value, one row for all atoms)."""
    from face_amd import ops
    say("readout_mlp shapes")
    C, N = 32, 70
    inv, h, ws = _readout_case(N, C)
    hb = torch.randn(1, 2 * C, device=DEV)
    swap = lambda k, t: ws[:k] + [t] + ws[k + 1:]
    refused = [(inv[:, :8 * C], h, ws, None), (torch.randn(N, 10 * C, device=DEV), h, ws, None), (inv, h[:, :16], ws, None),
               (inv, h[:64], ws, None), (inv, h.cpu(), ws, None), (inv, h.double(), ws, None),
               (inv, h, ws, hb.expand(N, -1).double()), (inv, h, ws, hb.expand(N, -1).cpu())]
    refused += [(inv, h, swap(k, ws[k][..., :16]), None) for k in (1, 2, 3, 4, 5, 6, 7, 8)]        # of the weights and biases
    refused += [(inv, h, swap(k, ws[k].cpu()), None) for k in range(9)]
    for i, (x, y, w, b) in enumerate(refused):
        assert not ops.ReadoutMLP.takes_rows(x, y, *w, b), i
        with pytest.raises(RuntimeError):
            ops.readout_mlp(x, y, *w, False, b)
    assert ops.ReadoutMLP.takes_rows(inv, h, *ws, None)
    for k in (2, 4, 8):                                                # b0, b1, bg of one value
        one = torch.full((1,), 0.3, device=DEV)
        got, want = ops.readout_mlp(inv, h, *swap(k, one), False), ops.readout_mlp(inv, h, *swap(k, one.repeat(2 * C)), False)
        assert all(rel(a, b) < 5e-6 for a, b in zip(got, want))
    got, want = ops.readout_mlp(inv, h, *ws, False, hb), ops.readout_mlp(inv, h, *ws, False, hb.repeat(N, 1))
    assert all(rel(a, b) < 5e-6 for a, b in zip(got, want))


@pytest.mark.parametrize("side", ["xs", "ys"])
def test_rows_linear_scale_tables_larger_than_lds(side):
    """64 groups whose scale rows do not fit in LDS beside the weights: read from memory instead, the
    results of a launch whose tables fit."""
    say("rows_linear wide scale tables", side)
    torch.manual_seed(4)
    N, k, n = 500, 768, 512
    x, w = torch.randn(N, k, device=DEV), torch.randn(n, k, device=DEV) / k ** 0.5
    tab = torch.rand(64, 1024, device=DEV) + 0.5
    grp = torch.randint(0, 64, (N,), device=DEV, dtype=torch.int32)
    kw = {side: tab}
    y = torch.empty(N, n, device=DEV)
    _rows_launch(x, w, y, False, False, grp=grp, **kw)
    ref = _lin_ref(x, w, False, None, 0.0, None, kw.get("xs"), kw.get("ys"), grp, N, 0)
    assert rel(y, ref) < 1e-5


@pytest.mark.parametrize("shape", [None, "-4,2,0", "8,1,1"])
@pytest.mark.parametrize("w_kn", [False, True])
def test_rows_linear_split_input_transforms_and_initial_sum(w_kn, shape, monkeypatch):
    """The readout forms of face_rows_linear vs torch fp64: input columns from two tensors
    ([x | x2], the split at k1), silu(x) and x * silu'(xz) applied to the x columns as they load,
    a bias per problem, and the sum started at beta * y0 over the first n_y0 columns of another
    tensor (a residual); four problems of different K in one launch, ragged rows, strided views.
    shape forces the direct kernel and the staged one in workgroups of eight waves."""
    from face_amd import ops
    if shape is not None:
        monkeypatch.setenv("FACE_GEMM_SHAPE", shape)
    say("rows_linear split/ops", w_kn, shape)
    torch.manual_seed(7)
    m = 1203
    silu = lambda t: t * torch.sigmoid(t)
    dsilu = lambda g, z: g * torch.sigmoid(z) * (1 + z * (1 - torch.sigmoid(z)))
    base = torch.randn(m, 400, device=DEV)
    cases = []
    # (x cols k1, x2 cols, n, x_op, bias, y0 cols)
    for k1, k2, n, op, has_b, ny0 in ((144, 16, 64, 0, True, 0), (96, 0, 48, 1, True, 32), (64, 32, 80, 2, False, 80),
                                      (32, 0, 16, 1, True, 16)):
        x = base[:, :k1] if op != 2 else torch.randn(m, k1, device=DEV)          # a strided view
        x2 = torch.randn(m, k2 + 8, device=DEV)[:, :k2] if k2 else None
        xz = torch.randn(m, k1, device=DEV) if op == 2 else None
        k = k1 + k2
        w = torch.randn(k, n, device=DEV) / k ** 0.5 if w_kn else torch.randn(n, k + 4, device=DEV)[:, :k] / k ** 0.5
        bias = torch.randn(n, device=DEV) if has_b else None
        y0 = torch.randn(m, ny0 + 4, device=DEV)[:, :ny0] if ny0 else None
        y = torch.empty(m, n, device=DEV)
        cases.append((ops.lin(x, w, y, x2=x2, x_op=op, xz=xz, bias=bias, y0=y0, beta=1.0 if ny0 else 0.0,
                              n_y0=ny0 if ny0 else None), (x, x2, xz, w, bias, y0, op, ny0)))
    ops.rows_linear([c[0] for c in cases], w_kn=w_kn)
    errs = []
    for pr, (x, x2, xz, w, bias, y0, op, ny0) in cases:
        d = lambda t: None if t is None else t.double().cpu()
        xi = d(x)
        xi = silu(xi) if op == 1 else (dsilu(xi, d(xz)) if op == 2 else xi)
        if x2 is not None:
            xi = torch.cat([xi, d(x2)], 1)
        ref = xi @ (d(w) if w_kn else d(w).T)
        if bias is not None:
            ref = ref + d(bias)
        if ny0:
            ref[:, :ny0] += d(y0)
        errs.append(rel(pr["y"], ref))
    say("   errs", errs)
    assert max(errs) < 1e-5, errs


@pytest.mark.parametrize("C,gate", [(160, True), (160, False), (96, True), (32, False)])
def test_readout_matches_torch(C, gate):
    """The pass readout on the row GEMM (face/model.py:331-339, the gate row of :286-287):
    LayerNorm -> [inv | h] W0^T + b0 -> SiLU -> W1 -> SiLU -> W2 with the energy column and the
    residual h + o[:, 1:], and gvm = inv Wg^T + bg; values and the gradients of feats and h (with
    the gate row's gradient entering the backward) vs torch fp64 autograd."""
    from face_amd import ops
    say("readout", C, gate)
    torch.manual_seed(C + gate)
    N, nf = 777, 9 * C
    feats = torch.randn(N, nf, device=DEV) * 2 + 0.3
    h = torch.randn(N, C + 16, device=DEV)[:, :C]                  # a strided residual, like a previous h_new
    lnw, lnb = torch.rand(nf, device=DEV) + 0.5, torch.randn(nf, device=DEV) * 0.1
    W0 = torch.randn(2 * C, 10 * C + 4, device=DEV) / (10 * C) ** 0.5
    b0 = torch.randn(2 * C, device=DEV) * 0.1
    W1, b1 = torch.randn(2 * C, 2 * C, device=DEV) / (2 * C) ** 0.5, torch.randn(2 * C, device=DEV) * 0.1
    W2, b2 = torch.randn(C + 1, 2 * C, device=DEV) / (2 * C) ** 0.5, torch.randn(C + 1, device=DEV) * 0.1
    Wg, bg = torch.randn(2 * C, nf, device=DEV) / nf ** 0.5, torch.randn(2 * C, device=DEV)
    n_pad = C + 16
    W2p = W2.new_zeros(n_pad, 2 * C)
    W2p[:C], W2p[C] = W2[1:], W2[0]
    b2p = b2.new_zeros(n_pad)
    b2p[:C], b2p[C] = b2[1:], b2[0]
    Wst = torch.cat([W0[:, :nf], Wg], 0).contiguous()
    fd, hd = feats.clone().requires_grad_(True), h.clone().requires_grad_(True)
    e, hn, gvm = ops.readout(fd, hd, lnw, lnb, 1e-5, W0, b0, W1, b1, W2p, b2p, *((Wg, bg, Wst) if gate else (None, None, None)))
    ge, gh = torch.randn(N, 1, device=DEV), torch.randn(N, C, device=DEV)
    gg = torch.randn(N, 2 * C, device=DEV)
    loss = (e * ge).sum() + (hn * gh).sum() + ((gvm * gg).sum() if gate else 0.0)
    gf, ghh = torch.autograd.grad(loss, (fd, hd))
    c = lambda t: t.detach().double().cpu()
    f2, h2 = c(feats).requires_grad_(True), c(h).requires_grad_(True)
    inv = torch.nn.functional.layer_norm(f2, (nf,), c(lnw), c(lnb), 1e-5)
    z = torch.cat([inv, h2, torch.zeros(N, 4, dtype=torch.float64)], 1) @ c(W0).T + c(b0)
    z = torch.nn.functional.silu(z) @ c(W1).T + c(b1)
    o = torch.nn.functional.silu(z) @ c(W2).T + c(b2)
    e2, hn2 = o[:, :1], h2 + o[:, 1:]
    loss2 = (e2 * c(ge)).sum() + (hn2 * c(gh)).sum()
    if gate:
        gvm2 = inv @ c(Wg).T + c(bg)
        loss2 = loss2 + (gvm2 * c(gg)).sum()
    gf2, gh2 = torch.autograd.grad(loss2, (f2, h2))
    errs = [rel(e, e2), rel(hn, hn2), rel(gf, gf2), rel(ghh, gh2)] + ([rel(gvm, gvm2)] if gate else [])
    say("   errs", errs)
    assert max(errs) < 1e-5, errs


@pytest.mark.parametrize("transport,Cin,merge", [(True, 160, True), (True, 160, False), (False, 160, True),
                                                  (False, 512, True), (True, 32, True)])
def test_scaled_mix_forward_backward(transport, Cin, merge, monkeypatch):
    """A_l = (Af_l W_l^T [+ D_l T_l^T]) * s[z] for the four ranks (face/model.py:498-501, :530-533)
    and the gradients of Af_l and D_l vs torch fp64 autograd (the transport-mix backward in the
    mix backward's launch and on its own)."""
    from face_amd import ops
    monkeypatch.setattr(ops, "MIX_MERGE_MAX_ATOMS", 1 << 30 if merge else 0)
    say("scaled mix", transport, Cin, merge)
    torch.manual_seed(Cin + transport)
    N, C, Dw = 517, 96 if Cin != 32 else 32, 64
    grp = torch.randint(0, 3, (N,), device=DEV, dtype=torch.int32)
    s_tab = torch.rand(3, 4 * C, device=DEV) + 0.5
    Af = [torch.randn(k, N, Cin, device=DEV, requires_grad=True) for k in (1, 3, 6, 10)]
    wm = [torch.randn(C, Cin, device=DEV) / Cin ** 0.5 for _ in range(4)]
    D1 = torch.randn(3, N, Dw, device=DEV, requires_grad=True) if transport else None
    D2 = torch.randn(6, N, Dw, device=DEV, requires_grad=True) if transport else None
    wt = [torch.randn(C, Dw, device=DEV) / 8, torch.randn(C, Dw, device=DEV) / 8] if transport else [None, None]
    A = ops.scaled_mix(s_tab, grp, wm, wt, D1, D2, Af)
    G = [torch.randn_like(a) for a in A]
    ins = Af + ([D1, D2] if transport else [])
    gr = torch.autograd.grad(sum((a * g).sum() for a, g in zip(A, G)), ins)
    c = lambda t: t.detach().double().cpu()
    insc = [c(t).requires_grad_(True) for t in ins]
    s = c(s_tab)[grp.long().cpu()].view(N, 4, C)
    A2 = []
    for l in range(4):
        y = insc[l] @ c(wm[l]).T
        if transport and l in (1, 2):
            y = y + insc[3 + l] @ c(wt[l - 1]).T
        A2.append(y * s[None, :, l, :])
    gr2 = torch.autograd.grad(sum((a * c(g)).sum() for a, g in zip(A2, G)), insc)
    errs = [rel(a, b) for a, b in zip(A, A2)] + [rel(a, b) for a, b in zip(gr, gr2)]
    say("   errs", errs)
    assert max(errs) < 1e-5, errs


@pytest.mark.parametrize("wrong", ["width", "weight", "weight_rows", "host", "host_weight", "type"])
def test_scaled_mix_refuses_other_transport_operands(wrong):
    """Transport sums or weights that do not fit the mix (width, shape, host memory, type) are refused."""
    from face_amd import ops
    say("scaled mix wrong transport operands", wrong)
    N, C, Dw = 40, 32, 64
    grp = torch.zeros(N, device=DEV, dtype=torch.int32)
    s_tab = torch.rand(1, 4 * C, device=DEV)
    Af = [torch.randn(k, N, C, device=DEV) for k in (1, 3, 6, 10)]
    wm = [torch.randn(C, C, device=DEV) for _ in range(4)]
    D, w = torch.randn(3, N, Dw, device=DEV), torch.randn(C, Dw, device=DEV)
    D = {"width": D[..., :48], "host": D.cpu(), "type": D.double()}.get(wrong, D)
    w = {"weight": w[:, :32], "weight_rows": w[:16], "host_weight": w.cpu()}.get(wrong, w)
    with pytest.raises(RuntimeError):
        ops.scaled_mix(s_tab, grp, wm, [w, None], D, None, Af)


@pytest.mark.parametrize("last", [False, True])
def test_readout_mlp_refuses_a_second_derivative(last):
    """The input gradients have no derivative of their own: asked for with create_graph they are refused when
    differentiated, alone or in a sum with something that has one, never dropped from it."""
    from face_amd import ops
    say("readout_mlp double backward", last)
    inv, h, ws = _readout_case(50, 32)
    inv.requires_grad_(True)
    outs = [o for o in ops.readout_mlp(inv, h, *ws, last) if o is not None]
    ups = [torch.randn_like(o).requires_grad_(True) for o in outs]
    want = torch.autograd.grad(outs, inv, [u.detach() for u in ups], retain_graph=True)[0]
    d_inv = torch.autograd.grad(outs, inv, ups, create_graph=True)[0]
    assert rel(d_inv, want) < 1e-5
    with pytest.raises(RuntimeError, match="not implemented"):
        torch.autograd.grad(d_inv.sum() + sum((u * u).sum() for u in ups), ups)


def test_readout_and_mix_past_the_span_of_a_row_block(monkeypatch):
    """Operands of 2^31 elements and more (eight rows 2^28 apart), which the row-block kernels refuse, and,
    with the limit lowered, as many rows: the results of small dense operands, bit for bit where the
    operands are copied, to the rounding of two float32 routes where the library products take over."""
    from face_amd import ops
    say("readout and mix past the span")
    N, C, Dw, ld = 8, 32, 64, 1 << 28
    inv, h, ws = _readout_case(N, C)
    buf = torch.empty(7 * ld + 8192, device=DEV)

    def far(t, at):
        v = buf.as_strided(t.shape, (ld, 1), at)
        return v.copy_(t)

    def readout(inv, h, ups):
        i, x = inv.detach().requires_grad_(True), h.detach().requires_grad_(True)
        outs = ops.readout_mlp(i, x, *ws, False)
        return [o.detach() for o in outs] + list(torch.autograd.grad(outs, [i, x], ups))

    ups = [torch.randn(N, w, device=DEV) for w in (1, C, 2 * C)]
    want = readout(inv, h, ups)
    got = readout(far(inv, 0), far(h, 1024), [ups[0], far(ups[1], 2048), far(ups[2], 3072)])
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    grp = torch.zeros(N, device=DEV, dtype=torch.int32)
    s_tab = torch.rand(1, 4 * C, device=DEV) + 0.5
    Af = [torch.randn(k, N, C, device=DEV) for k in (1, 3, 6, 10)]
    wm = [torch.randn(C, C, device=DEV) / C ** 0.5 for _ in range(4)]
    D1, D2 = torch.randn(3, N, Dw, device=DEV), torch.randn(6, N, Dw, device=DEV)
    wt = [torch.randn(C, Dw, device=DEV) / 8 for _ in range(2)]
    want_mix = ops.scaled_mix(s_tab, grp, wm, wt, D1, D2, Af)
    spread = torch.empty(23 * (1 << 27) + Dw, device=DEV)
    Df = spread.as_strided(D1.shape, (8 << 27, 1 << 27, 1), 0).copy_(D1)      # 24 rows 2^27 elements apart
    got_mix = ops.scaled_mix(s_tab, grp, wm, wt, Df, D2, Af)
    monkeypatch.setattr(ops, "GEMM_SPAN", N * 9 * C)                          # the readout's widest rows reach it
    got = readout(inv, h, ups)
    assert all(rel(a, b) < 1e-5 for a, b in zip(got + list(got_mix), want + list(want_mix)))


def test_scaled_mix_takes_broadcast_transport_sums():
    """Transport sums and weights whose rows are one row repeated (stride 0) give the results of their dense
    copies (to the rounding of two float32 routes)."""
    from face_amd import ops
    say("scaled mix broadcast")
    torch.manual_seed(8)
    N, C, Dw = 45, 32, 64
    grp = torch.zeros(N, device=DEV, dtype=torch.int32)
    s_tab = torch.rand(1, 4 * C, device=DEV) + 0.5
    Af = [torch.randn(k, N, C, device=DEV) for k in (1, 3, 6, 10)]
    wm = [torch.randn(C, C, device=DEV) / C ** 0.5 for _ in range(4)]
    D = [torch.randn(1, 1, Dw, device=DEV).expand(k, N, Dw) for k in (3, 6)]
    wt = [torch.randn(C, Dw, device=DEV) / 8, torch.randn(1, Dw, device=DEV).expand(C, Dw)]
    dense = lambda ts: [t.clone(memory_format=torch.contiguous_format) for t in ts]
    got = ops.scaled_mix(s_tab, grp, wm, wt, *D, Af)
    want = ops.scaled_mix(s_tab, grp, wm, dense(wt), *dense(D), Af)
    assert all(rel(a, b) < 1e-5 for a, b in zip(got, want))


@pytest.mark.parametrize("n_sets,C,in_row", [(1, 160, False), (2, 160, False), (2, 96, False), (3, 32, False),
                                             (2, 96, True)])
def test_rank_proj_forward_backward(n_sets, C, in_row):
    """proj of the concatenated moment sets for the four ranks (face/model.py:537-544) as one launch
    per set, with the row-sliced weights the node algebra uses (P0 | PQS | PQS | PQ), and the
    sets' gradients, vs torch fp64 autograd; in_row: rank 0 written into the first C columns of a
    wider row buffer (as for the readout row), the other columns left as they were."""
    from face_amd import ops
    say("rank proj", n_sets, C, in_row)
    torch.manual_seed(n_sets * C)
    N = 613
    full = [torch.randn(3 * C, n_sets * C, device=DEV) / C ** 0.5 for _ in range(4)]
    ws = [w[:n] for w, n in zip(full, (C, 3 * C, 3 * C, 2 * C))]
    sets = [[torch.randn(k, N, C, device=DEV, requires_grad=True) for k in (1, 3, 6, 10)] for _ in range(n_sets)]
    buf = torch.full((N, 9 * C), 7.0, device=DEV) if in_row else None
    ys = ops.rank_proj(ws, sets, out0=buf[:, :C] if in_row else None)
    if in_row:
        assert ys[0].data_ptr() == buf.data_ptr() and ys[0].stride(1) == 9 * C
        assert (buf[:, C:] == 7.0).all()
    G = [torch.randn_like(y) for y in ys]
    flat = [t for S in sets for t in S]
    gr = torch.autograd.grad(sum((y * g).sum() for y, g in zip(ys, G)), flat)
    c = lambda t: t.detach().double().cpu()
    flatc = [c(t).requires_grad_(True) for t in flat]
    ys2 = [sum(flatc[4 * s + l] @ c(ws[l][:, s * C:(s + 1) * C]).T for s in range(n_sets)) for l in range(4)]
    gr2 = torch.autograd.grad(sum((y * c(g)).sum() for y, g in zip(ys2, G)), flatc)
    errs = [rel(a, b) for a, b in zip(ys, ys2)] + [rel(a, b) for a, b in zip(gr, gr2)]
    say("   errs", max(errs))
    assert max(errs) < 1e-5, errs


@pytest.mark.parametrize("gathered,K,C,transport", [(False, 32, 96, True), (True, 32, 96, False),
                                                    (False, 64, 256, True), (True, 16, 160, True),
                                                    (False, 48, 32, False)])
def test_density_mix_fused_matches_reference(gathered, K, C, transport):
    """Factor density fused with the per-rank mix and element scale (face/kernels.py:170-178 then
    face/model.py:503-506, :530-533), forward and the gradients of phi, msg, Y and the transport
    sums, against the oracle's factor density + F.linear + scale in fp64 autograd. Ragged rows:
    a hub row, isolated atoms, N not a multiple of the 4-atom tile."""
    from face_amd import ops
    say("density+mix fused", gathered, K, C, transport)
    B, N, Dw = 16, 57, 64
    g = _G(N, 500, 5)
    counts = g.counts
    E = sum(counts)
    torch.manual_seed(K + C)
    phi = torch.randn(E, B, device=DEV, requires_grad=True)
    msg = torch.randn(N if gathered else E, K, device=DEV, requires_grad=True)
    Y = torch.randn(E, 20, device=DEV, requires_grad=True)
    grp = torch.randint(0, 3, (N,), device=DEV, dtype=torch.int32)
    s_tab = torch.rand(3, 4 * C, device=DEV) + 0.5
    wm = [torch.randn(C, B * K, device=DEV) / (B * K) ** 0.5 for _ in range(4)]
    wmt = [w.t().contiguous() for w in wm]
    D1 = torch.randn(3, N, Dw, device=DEV, requires_grad=True) if transport else None
    D2 = torch.randn(6, N, Dw, device=DEV, requires_grad=True) if transport else None
    wt = [torch.randn(C, Dw, device=DEV) / 8, torch.randn(C, Dw, device=DEV) / 8] if transport else [None, None]
    A = ops.density_mix(s_tab, grp, wm, wmt, wt, D1, D2, phi, msg, Y, g.G, gathered)
    assert [tuple(a.shape) for a in A] == [(k, N, C) for k in (1, 3, 6, 10)]
    Gs = [torch.randn_like(a) for a in A]
    ins = [phi, msg, Y] + ([D1, D2] if transport else [])
    gr = torch.autograd.grad(sum((a * gg).sum() for a, gg in zip(A, Gs)), ins)
    # oracle: padded factor density, then the four mixes with the scale
    c = lambda t: t.detach().double().cpu()
    insc = [c(t).requires_grad_(True) for t in ins]
    M = max(counts)
    col = g.G.col.long().cpu()
    pd = lambda t: _pad(t, counts, M)
    msg_e = insc[1][col] if gathered else insc[1]
    Dd = oops.factor_density(pd(insc[0]), pd(msg_e), pd(insc[2]))             # (N, 20, B K)
    s = c(s_tab)[grp.long().cpu()].view(N, 4, C)
    A2 = []
    for l, (x0, x1) in enumerate(((0, 1), (1, 4), (4, 10), (10, 20))):
        y = Dd[:, x0:x1, :].permute(1, 0, 2) @ c(wm[l]).T                      # (k_l, N, C)
        if transport and l in (1, 2):
            y = y + insc[2 + l] @ c(wt[l - 1]).T
        A2.append(y * s[None, :, l, :])
    gr2 = torch.autograd.grad(sum((a * c(gg)).sum() for a, gg in zip(A2, Gs)), insc)
    errs = [rel(a, b) for a, b in zip(A, A2)] + [rel(a, b) for a, b in zip(gr, gr2)]
    say("   errs", [f"{e:.1e}" for e in errs])
    assert max(errs) < TOL, errs
    # bitwise reproducible (fixed summation order)
    A3 = ops.density_mix(s_tab, grp, wm, wmt, wt, D1, D2, phi, msg, Y, g.G, gathered)
    assert all(torch.equal(a, b) for a, b in zip(A, A3))


@pytest.mark.parametrize("with_at,sizes", [(False, [5, 300, 1, 700, 33, 260]), (True, [5, 300, 1, 700, 33, 260]),
                                           (True, [300000]), (False, [140000, 7, 160000])])
def test_atom_energy_matches_index_add(with_at, sizes):
    """Atom energies e0 + scale * e_p added pass by pass and their per-structure sums (face/model.py:
    680-690) against index_add, ragged structures (one of a single atom; structures larger than one
    pass of the per-atom grid) and strided (N, 1) column views; the backward against autograd
    through the torch expression; a second call bitwise equal."""
    from face_amd import ops
    say("atom energy", with_at, len(sizes), sum(sizes))
    torch.manual_seed(3)
    N, nstr = sum(sizes), len(sizes)
    batch = torch.repeat_interleave(torch.arange(nstr), torch.tensor(sizes)).to(DEV)
    sp = torch.tensor([0] + list(np.cumsum(sizes)), dtype=torch.int32, device=DEV)
    e0 = torch.randn(N, device=DEV)
    scale = torch.tensor(0.7, device=DEV)
    rows = [torch.randn(N, w, device=DEV, requires_grad=True) for w in (1, 17, 9)]
    es = [r[:, :1] for r in rows]
    E, e_at = ops.atom_energy(e0, scale, sp, nstr, es)
    ref_at = e0.clone()
    for e in es:
        ref_at = ref_at + scale * e.squeeze(-1)
    ref_E = torch.zeros(nstr, device=DEV).index_add(0, batch, ref_at)
    assert torch.allclose(e_at, ref_at, rtol=1e-6, atol=1e-6)
    assert torch.allclose(E, ref_E, rtol=1e-5, atol=1e-4 * max(1.0, N ** 0.5 / 30))
    E2, e_at2 = ops.atom_energy(e0, scale, sp, nstr, es)
    assert torch.equal(E, E2) and torch.equal(e_at, e_at2)
    gE = torch.randn(nstr, device=DEV)
    g_at = torch.randn(N, device=DEV) if with_at else None
    outs, gouts = ([E, e_at], [gE, g_at]) if with_at else ([E], [gE])
    got = torch.autograd.grad(outs, rows, gouts)
    routs = [ref_E, ref_at] if with_at else [ref_E]
    want = torch.autograd.grad(routs, rows, gouts)
    for a, b in zip(got, want):
        assert torch.allclose(a, b, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("N,C,n", [(864, 96, 32), (37, 160, 48)])
def test_table_linears_match_torch(N, C, n):
    """The pass's directional table linears V pvt^T, Ms pmt^T (face/model.py:474-479) in one
    launch each way, forward and input gradients against torch fp64."""
    from face_amd import ops
    say("table linears", N, C, n)
    torch.manual_seed(N + C)
    V = torch.randn(3, N, C, device=DEV, requires_grad=True)
    Ms = torch.randn(6, N, C, device=DEV, requires_grad=True)
    wv = torch.randn(n, C, device=DEV) / C ** 0.5
    wm = torch.randn(n, C, device=DEV) / C ** 0.5
    Vb, Mb = ops.table_linears(V, Ms, wv, wm)
    gv, gm = torch.randn_like(Vb), torch.randn_like(Mb)
    got = torch.autograd.grad((Vb * gv).sum() + (Mb * gm).sum(), (V, Ms))
    Vc, Mc = V.detach().double().cpu().requires_grad_(True), Ms.detach().double().cpu().requires_grad_(True)
    Vr, Mr = Vc @ wv.double().cpu().T, Mc @ wm.double().cpu().T
    want = torch.autograd.grad((Vr * gv.double().cpu()).sum() + (Mr * gm.double().cpu()).sum(), (Vc, Mc))
    errs = [rel(Vb, Vr), rel(Mb, Mr)] + [rel(a, b) for a, b in zip(got, want)]
    assert max(errs) < 1e-5, errs


@pytest.mark.parametrize("counts,K,huge", [
    ([1, 0, 31, 32, 33, 5], 16, None), ([64, 65, 0, 2, 40], 32, None), ([96, 97, 130, 1, 64], 48, None),
    ([70, 96, 33, 200, 0], 64, None), ([7, 30], 64, None), ([40, 3, 70], 32, "msg"), ([40, 3, 70], 32, "G"),
    ([40, 3, 70], 32, "Y")])
def test_factor_density_row_lengths(counts, K, huge):
    """Row lengths around the 16- and 32-edge tiles and the chunks of 32, 64 and 96 edges, gathered messages,
    both directions against fp64; one value past the largest bf16 (no finite limbs) leaves every other atom's results finite and
    its own as plain fp32 gives them."""
    from face_amd import _lib, ops
    N, E, M = len(counts), sum(counts), max(counts)
    say("factor density bwd", counts, K, huge)
    torch.manual_seed(K + E)
    row_ptr = torch.as_tensor(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), device=DEV)
    col = torch.randint(0, N, (E,), dtype=torch.int32, device=DEV)
    phi, Y = torch.randn(E, 21, device=DEV)[:, :16], torch.randn(E, 20, device=DEV)
    msg = torch.randn(N, K, device=DEV)
    G = [torch.randn(k, N, 16 * K, device=DEV) for k in ops.RANK_K]
    if huge in ("msg", "Y"):                 # the other factors small: fp32 sums of the products stay in range
        G = [g * 1e-3 for g in G]
        phi *= 1e-3
        if huge == "msg":
            msg[1, 3] = 3.39e38
            Y *= 1e-3
        else:
            Y[1, 4] = 3.4e38
            msg *= 1e-3
    if huge == "G":
        G[2][1, 2, 5] = float("inf")
    dphi, dmsg, dY = (torch.full((E, w), float("nan"), device=DEV) for w in (16, K, 20))
    D = [torch.full((k, N, 16 * K), float("nan"), device=DEV) for k in ops.RANK_K]
    P = _lib.ptr
    _lib.call("face_density_bwd", P(phi), 21, P(msg), K, P(col), P(Y), 20, 20, P(row_ptr), N, 0, M, 16, K,
              *_lib.ranks_of_blocks(G), P(dphi), 16, P(dmsg), K, P(dY), 20, _lib.stream_of(phi))
    _lib.call("face_density_fwd", P(phi), 21, P(msg), K, P(col), P(Y), 20, 20, P(row_ptr), N, 0, 16, K,
              *_lib.ranks_of_blocks(D), _lib.stream_of(phi))
    rec = torch.repeat_interleave(torch.arange(N, device=DEV), torch.as_tensor(counts, device=DEV))
    Gd = torch.cat(G, 0).permute(1, 0, 2).reshape(N, 20, 16, K).double()[rec]            # (E, 20, 16, K)
    md, pd, Yd = msg.double()[col.long()], phi.double(), Y.double()
    W = torch.einsum("exbk,ek->exb", Gd, md)
    want = (torch.einsum("exb,ex->eb", W, Yd), torch.einsum("exbk,ex,eb->ek", Gd, Yd, pd),
            torch.einsum("exb,eb->ex", W, pd))
    Dw = torch.zeros(N, 20, 16, K, dtype=torch.float64, device=DEV)
    Dw.index_add_(0, rec, torch.einsum("ex,eb,ek->exbk", Yd, pd, md))
    want += (Dw.reshape(N, -1),)
    D = torch.cat(D, 0).permute(1, 0, 2).reshape(N, -1)
    for got, w in zip((dphi, dmsg, dY, D), want):
        w32 = w.float()
        assert torch.equal(torch.isnan(got), torch.isnan(w32))
        inf = torch.isinf(w32)
        assert torch.equal(got[inf], w32[inf])
        ok = torch.isfinite(w32)
        assert torch.isfinite(got[ok]).all()
        # sums of at most 320 fp32 products: relative to each row's scale
        scale = torch.where(ok, w32.abs(), torch.zeros_like(w32)).amax(1, keepdim=True).expand_as(w32)
        assert ((got - w32).abs()[ok] <= 4e-6 * scale[ok]).all()
