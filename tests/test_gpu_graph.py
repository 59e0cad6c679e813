"""GPU pair-list build vs the fp64 brute-force oracle: bit-exact pair sets, canonical order,
bit-exact shifts, reverse map and padded view (face/neighbors.py:7-37)."""
import sys

import numpy as np
import pytest
import torch

from oracle.neighbors import pair_list, pair_list_cells, padded_graph as oracle_padded

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def oracle_csr(structures, rc, pairs=pair_list):
    I, J, S, off = [], [], [], 0
    for st in structures:
        i, j, s = pairs(st["pos"], st["cell"], st["pbc"], rc)
        I.append(i + off); J.append(j + off); S.append(s)
        off += len(st["pos"])
    return np.concatenate(I), np.concatenate(J), np.concatenate(S)


def check_graph(structures, rc, method="auto", pairs=pair_list):
    from face_amd.neighbors import build_graph
    g = build_graph(structures, rc, method=method)
    i, j, S = oracle_csr(structures, rc, pairs)
    recv, col, Sg = g.recv.cpu().numpy(), g.col.cpu().numpy(), g.S.cpu().numpy()
    assert len(col) == len(j), (len(col), len(j))
    assert np.array_equal(recv, i) and np.array_equal(col, j) and np.array_equal(Sg, S)
    cells = np.concatenate([np.repeat(np.asarray(st["cell"], np.float64)[None], len(st["pos"]), 0)
                            for st in structures])
    sv = np.einsum("ea,eab->eb", S.astype(np.float64), cells[i])
    assert np.array_equal(g.shift.cpu().numpy(), sv.astype(np.float32))
    rev = g.rev.cpu().numpy()
    assert np.array_equal(col[rev], recv) and np.array_equal(recv[rev], col) and np.array_equal(Sg[rev], -Sg)
    assert np.array_equal(rev[rev], np.arange(len(rev)))
    return g


def test_molecule_batch_exact():
    from face_amd import systems
    say("molecule batch")
    check_graph(systems.molecules(64, systems.stream(0)), 4.5)


def test_fcc_864_exact():
    from face_amd import systems
    say("fcc 864")
    st = systems.fcc(4.09, 6, 0.1, systems.stream(2))
    g = check_graph([st], 4.5)
    assert g.max_row == 18


@pytest.mark.parametrize("method", ["cell", "small"])
def test_liquid_3000_exact(method):
    from face_amd import systems
    say("liquid 3000", method)
    st = systems.liquid(3000, np.random.default_rng(5))
    check_graph([st], 5.0, method=method)


@pytest.mark.parametrize("method", ["cell", "small"])
@pytest.mark.parametrize("n,rc", [(130, 4.0), (150, 6.4), (63, 7.5)])
def test_dense_rows_of_many_images_exact(n, rc, method):
    """Rows past 256 pairs (the cell list's keys in LDS; 130 atoms stay below, the others reach ~ 330 and
    more), several images per neighbour and bins that wrap more than once, in a skewed cell."""
    say("dense rows", n, rc, method)
    rng = np.random.default_rng(n)
    cell = np.array([[8.0, 0, 0], [1.5, 7.5, 0], [-0.7, 0.9, 8.3]])
    st = {"pos": rng.random((n, 3)) @ cell + rng.integers(-1, 2, (n, 3)) @ cell, "Z": np.full(n, 6), "cell": cell,
          "pbc": np.ones(3, bool)}
    check_graph([st], rc, method=method)


@pytest.mark.parametrize("k", [3, 4])
def test_liquid_full_size_exact(k):
    """The 24,000-atom (1.25 M pairs) and 100,000-atom (6.9 M pairs) liquids at full size against
    the bin-candidate fp64 oracle (equal to the brute-force one, pinned on the CPU)."""
    from face_amd import systems
    sts, kw, el, desc = systems.workload(k)
    say("full-size pair list", desc)
    g = check_graph(sts, kw["rc"], pairs=pair_list_cells)
    say(f"  N {g.N} E {g.E} max_row {g.max_row}")
    assert g.N == len(sts[0]["pos"]) and g.E > (1_000_000 if k == 3 else 6_000_000)


@pytest.mark.parametrize("method", ["cell", "small"])
def test_triclinic_and_thin_cells(method):
    say("triclinic", method)
    rng = np.random.default_rng(8)
    cell = np.array([[6.1, 0.0, 0.0], [2.3, 5.7, 0.0], [-1.1, 1.7, 4.2]])   # thinner than 2 rc along c
    pos = rng.random((70, 3)) @ cell + rng.normal(0, 3.0, (70, 3))       # unwrapped positions
    st = {"pos": pos, "Z": np.full(70, 6), "cell": cell, "pbc": np.ones(3, bool)}
    check_graph([st], 4.5, method=method)


def test_mixed_pbc_and_empty_rows():
    say("mixed pbc")
    rng = np.random.default_rng(3)
    cell = np.diag([7.0, 30.0, 7.5])
    st1 = {"pos": rng.random((25, 3)) @ cell, "Z": np.full(25, 8), "cell": cell, "pbc": np.array([1, 0, 1], bool)}
    st2 = {"pos": np.array([[0.0, 0, 0], [20.0, 0, 0]]), "Z": np.array([1, 1]), "cell": np.zeros((3, 3)),
           "pbc": np.zeros(3, bool)}                                      # two isolated atoms
    check_graph([st1, st2], 4.0)


def test_boundary_decisions_match_fp64_oracle():
    """Pairs within a few ulp of rc: the accept test (fp64, fixed order, correctly rounded
    sqrt) must agree with the oracle bit for bit."""
    say("boundary ulps")
    rng = np.random.default_rng(11)
    rc = 4.5
    n = 400
    dirs = rng.normal(size=(n, 3))
    dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
    scale = rc * (1 + rng.integers(-6, 7, n) * np.finfo(np.float64).eps)
    pos = []
    for k in range(n):
        a = rng.uniform(-50, 50, 3)
        pos += [a, a + dirs[k] * scale[k]]
    pos = np.asarray(pos)
    structures = [{"pos": pos[2 * k:2 * k + 2], "Z": np.array([1, 1]), "cell": np.zeros((3, 3)),
                   "pbc": np.zeros(3, bool)} for k in range(n)]
    g = check_graph(structures, rc)
    say("accepted pairs", g.E, "of", 2 * n)


def test_padded_view_matches_reference_layout():
    from face_amd import systems
    from face_amd.neighbors import padded_graph
    say("padded view")
    mols = systems.molecules(5, np.random.default_rng(4))
    box = [systems.fcc(4.09, 2, 0.1, np.random.default_rng(1))]
    for sts in (mols, box):
        got = padded_graph(sts, 4.5)
        want = oracle_padded(sts, 4.5)
        assert np.array_equal(got["nbr"].cpu().numpy(), want["nbr"].numpy())
        assert np.array_equal(got["mask"].cpu().numpy(), want["mask"].numpy())
        assert np.array_equal(got["shift"].cpu().numpy(), want["shift"].numpy())
        assert np.array_equal(got["batch"].cpu().numpy(), want["batch"].numpy())
        assert np.array_equal(got["pos"].cpu().numpy(), want["pos"].numpy())


@pytest.mark.parametrize("n", [0, 1, 63, 64, 511, 513, 8191, 8192, 8193, 20003])
def test_scan_of_row_counts(n):
    from face_amd.neighbors import _scan
    from face_amd import _lib
    counts = torch.randint(0, 150, (n,), dtype=torch.int32, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    row_ptr, total, longest = _scan(counts, counts.device, _lib.stream_of(counts))
    want = np.concatenate([[0], np.cumsum(counts.cpu().numpy())])
    assert np.array_equal(row_ptr.cpu().numpy(), want)
    assert total == want[-1] and longest == (int(counts.max()) if n else 0)


@pytest.mark.parametrize("method", ["cell", "small"])
def test_positions_of_any_strides(method):
    rng = np.random.default_rng(8)
    pos = rng.uniform(0, 9.0, (3, 150)).T                # column-major, as a transposed file read gives
    st = dict(pos=pos, Z=np.ones(150, int), cell=np.eye(3) * 9.0, pbc=True)
    check_graph([dict(st, pbc=np.ones(3, bool))], 4.0, method)
    check_graph([dict(st, pbc=np.ones(3, bool), pos=np.repeat(pos, 2, 0)[::2])], 4.0, method)
    if method == "small":                                # several of them: their concatenation is column-major too
        check_graph([dict(pos=rng.uniform(0, 6, (3, n)).T, Z=np.ones(n, int), cell=np.zeros((3, 3)),
                          pbc=np.zeros(3, bool)) for n in (20, 1, 31)], 4.0, method)


def test_overflowing_rows_hold_valid_pairs():
    """A row whose space is too small, and images past the sort key's range, count as overflows; every row
    of the cell list then still holds pairs of existing atoms (a short row its first ones), and the reverse
    map answers for a list with indexes that are no atoms, without following them."""
    from face_amd import _lib, neighbors
    say("overflowing rows")
    rng = np.random.default_rng(2)
    N, L, rc = 400, 16.0, 4.5
    st = {"pos": rng.uniform(0, L, (N, 3)), "Z": np.ones(N, int), "cell": np.eye(3) * L, "pbc": np.ones(3, bool)}
    g = neighbors.build_graph([st], rc, method="cell")
    counts = (g.row_ptr[1:] - g.row_ptr[:-1]).cpu().numpy()
    i32 = dict(dtype=torch.int32, device="cuda")
    P, strm = _lib.ptr, _lib.stream_of(g.col)

    def fill(pos, row_ptr):
        nbh = neighbors._grid(st["cell"], rc)
        nb = (_lib.I32 * 6)(*nbh)
        pos = torch.as_tensor(pos, dtype=torch.float64, device="cuda")
        cell = torch.as_tensor(st["cell"].reshape(9), dtype=torch.float64, device="cuda")
        inv = torch.as_tensor(np.linalg.inv(st["cell"]).reshape(9), dtype=torch.float64, device="cuda")
        nbins = nbh[0] * nbh[1] * nbh[2]
        bin_of, wrap, cnt, start, slots, atoms = (torch.empty(s, **i32) for s in (N, (N, 3), nbins, nbins + 1, nbins, N))
        _lib.call("face_nbr_bin", P(pos), N, P(inv), nb, P(bin_of), P(wrap), P(cnt), P(start), P(slots), P(atoms), strm)
        E = int(row_ptr[-1])
        key = torch.empty(E, dtype=torch.int64, device="cuda")
        col, S = torch.full((E,), 1 << 30, **i32), torch.empty(E, 3, **i32)
        shift, over = torch.empty(E, 3, device="cuda"), torch.zeros(1, **i32)
        rp = torch.as_tensor(row_ptr.astype(np.int32), device="cuda")
        _lib.call("face_nbr_fill", P(pos), N, None, None, P(cell), None, None, rc, nb, P(bin_of), P(wrap), P(start),
                  P(atoms), P(rp), P(key), P(col), P(S), P(shift), P(over), strm)
        return rp, col, S, int(over)

    # one row five pairs short
    short = counts.copy()
    short[7] -= 5
    rp, col, S, over = fill(st["pos"], np.concatenate([[0], np.cumsum(short)]))
    assert over == 5
    full = [set(zip(c.tolist(), map(tuple, s.tolist()))) for c, s in
            ((g.col[g.row_ptr[i]:g.row_ptr[i + 1]].cpu(), g.S[g.row_ptr[i]:g.row_ptr[i + 1]].cpu()) for i in range(N))]
    rph = rp.cpu().numpy()
    for i in range(N):
        got = list(zip(col[rph[i]:rph[i + 1]].tolist(), map(tuple, S[rph[i]:rph[i + 1]].tolist())))
        assert set(got) <= full[i] and len(set(got)) == short[i], i
    # atom 3 lies 600 cells away: its images do not fit the key
    far = st["pos"].copy()
    far[3, 0] += 600 * L
    rp, col, S, over = fill(far, np.concatenate([[0], np.cumsum(counts)]))
    assert over > 0 and int(col.min()) >= 0 and int(col.max()) < N
    # indexes that are no atoms
    col = g.col.clone()
    bad = torch.tensor([0, 100, g.E - 1], device="cuda")
    col[bad] = torch.tensor([-5, N, 1 << 30], **i32)
    rev, missing = torch.empty(g.E, **i32), torch.zeros(1, **i32)
    _lib.call("face_nbr_rev", P(g.row_ptr), P(col), P(g.S), N, P(rev), P(missing), strm)
    assert int(missing) >= 3 and torch.equal(rev[bad].long(), bad)
