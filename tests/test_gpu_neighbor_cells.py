"""The cell search against the brute-force one, bit for bit, over the forms its dispatch tells apart: cells with
enough atoms for a block each (up to 2,048 candidates, up to 4,096, three cells in one direction or more), few
atoms, sparse cells, fewer than three cells in a direction or more candidates than LDS holds in the average cell
(atom by atom), single cells with more than that, one block or several per cell, triclinic boxes, cutoffs per
type, coordinates outside [0, 1). _form restates the dispatch, so that each case is known to reach what it is
for. The reverse map against its definition."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return "cuda"


CUBE = np.eye(3)
TRI = np.array([[1.0, 0.1, 0.0], [-0.2, 1.1, 0.15], [0.05, -0.1, 0.95]])

def _cells(lat, frac, rc):
    """(cells per direction, candidates of every occupied cell): the atoms of the 27 cells around it."""
    vol = abs(np.linalg.det(lat))
    nc = [max(1, int(np.floor(vol / np.linalg.norm(np.cross(lat[(d + 1) % 3], lat[(d + 2) % 3])) / rc))) for d in range(3)]
    own = np.zeros(nc)
    np.add.at(own, tuple(np.minimum((np.mod(frac, 1.0) * nc).astype(int), np.array(nc) - 1).T), 1)
    tot = sum(np.roll(own, s, (0, 1, 2)) for s in np.ndindex(3, 3, 3)) if min(nc) >= 3 else None
    return nc, None if tot is None else tot[own > 0]


def _form(lat, frac, rc):
    """The search that a call takes: atom by atom, or cells' blocks of a capacity and which cells exceed it."""
    nc, tot = _cells(lat, frac, rc)
    n, ncells = len(frac), int(np.prod(nc))
    avg = n / ncells * 27.0
    if min(nc) < 3 or n < 5000 or n < 6 * ncells or 1.08 * avg > 4096:
        return "by_atom"
    cap = 4096 if 1.5 * avg > 2048 else 2048
    return f"blocks_{cap}" + ("" if tot.max() <= cap else "_overfull")


# name, lattice (A), atoms, types, cutoff, slots per type, cutoffs per type, spread (1: fills the box), offset
CASES = [
    ("blocks", 39.5 * CUBE, 5200, 2, 6.5, 160, None, 1.0, 0.0),
    ("blocks_tri", 42.0 * TRI, 5100, 3, 6.0, 128, (6.0, 5.0, 5.5), 1.0, 0.0),
    ("by_atom", 33.0 * CUBE, 3000, 2, 6.5, 160, None, 1.0, 0.0),
    ("three_cells", 20.0 * CUBE, 5001, 1, 6.5, 900, None, 1.0, 0.0),
    ("two_cells", np.diag([14.0, 35.0, 49.0]), 5123, 4, 6.9, 400, None, 1.0, 0.0),
    ("one_cell", 30.0 * np.array([[1.0, 0, 0], [0.9, 0.5, 0], [0, 0, 1.0]]), 5000, 2, 8.0, 600, None, 1.0, 0.0),
    ("sparse", 80.0 * CUBE, 5500, 2, 6.5, 64, (6.5, 4.0), 1.0, 0.0),
    ("overfull", 60.0 * CUBE, 6000, 2, 6.0, 1400, None, 0.28, 0.0),
    ("fuller_lds", 30.0 * CUBE, 5000, 5, 9.0, 300, None, 0.96, 0.0),
    ("outside", 39.5 * CUBE, 5200, 2, 6.5, 160, None, 1.0, -13.0),
    ("edge_cells", 39.2 * CUBE, 65 * 216, 16, 6.5, 100, None, 1.0, 0.0),
    ("three_along_x", np.diag([20.0, 41.0, 41.0]), 5400, 2, 6.5, 250, None, 1.0, 0.0),
    ("three_along_y_z", np.diag([81.0, 20.0, 20.5]), 5100, 3, 6.5, 190, (6.5, 6.0, 5.0), 1.0, 0.0),
    ("three_tri", np.diag([24.0, 44.0, 24.0]) @ TRI, 6100, 2, 6.5, 260, None, 1.0, -13.0),
    ("upper_half", 39.5 * CUBE, 27200, 2, 6.5, 340, None, 1.0, 0.0),
]
FORMS = dict(blocks="blocks_2048", blocks_tri="blocks_2048", by_atom="by_atom", three_cells="by_atom",
             two_cells="by_atom", one_cell="by_atom", sparse="by_atom", overfull="blocks_2048_overfull",
             fuller_lds="by_atom", outside="blocks_2048", edge_cells="blocks_4096", three_along_x="blocks_2048",
             three_along_y_z="blocks_2048", three_tri="blocks_4096", upper_half="blocks_4096")


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("want_dR", [False, True])
def test_cell_search_is_the_brute_force_one(dev, case, want_dR):
    from matpl_amd.neighbor import find_neighbore_gpu
    name, lat, n, T, rc, m, rct, spread, offset = case
    rng = np.random.Generator(np.random.PCG64([len(name), n]))
    frac = rng.random((n, 3)) * spread
    if offset:
        frac[::3] += offset
        frac[1::3] += 7.0
    types = rng.integers(0, T, n)
    assert _form(lat, frac, rc) == FORMS[name]
    if name.startswith("three_a") or name == "three_tri":
        assert min(_cells(lat, frac, rc)[0]) == 3
    if name == "upper_half":
        assert (_cells(lat, frac, rc)[1] > 2048).all()
    kw = dict(rc_type=rct, want_dR=want_dR, want_shift=True, device=dev)
    print(f"{name} n={n} T={T}", flush=True)
    a = find_neighbore_gpu(lat, frac, types, T, m, rc, **kw)
    b = find_neighbore_gpu(lat, frac, types, T, m, rc, force_brute=True, **kw)
    assert int(b.counts.sum()) > 0
    for k in ("counts", "list", "shift", "frac_wrapped") + (("dR",) if want_dR else ()):
        assert torch.equal(getattr(a, k), getattr(b, k)), k


def test_cell_search_overflow_zeroes_the_row(dev):
    from matpl_amd.neighbor import find_neighbore_gpu
    rng = np.random.Generator(np.random.PCG64(5))
    frac, types = rng.random((5200, 3)), rng.integers(0, 2, 5200)
    frac[:80] = 0.5 + 0.02 * rng.random((80, 3))
    kw = dict(want_dR=False, want_shift=True, device=dev, check=False)
    a = find_neighbore_gpu(39.5 * CUBE, frac, types, 2, 60, 6.0, **kw)
    b = find_neighbore_gpu(39.5 * CUBE, frac, types, 2, 60, 6.0, force_brute=True, **kw)
    over = (b.counts.sum(1) == 0)
    assert int(over.sum()) >= 80 and not bool(over.all())
    assert int(a.status) > 0 and bool(over[int(a.status) - 1])
    assert torch.equal(a.counts, b.counts)
    assert torch.equal(a.list[~over], b.list[~over])
    assert int(a.list[over].abs().sum()) == 0


@pytest.mark.parametrize("lat,n,m", [(39.5 * CUBE, 1601, 27), (13.2 * CUBE, 130, 130), (8.0 * CUBE, 37, 150)])
def test_reverse_map_names_the_partner(dev, lat, n, m):
    """Odd slot counts (unaligned four-wide loads), buckets shorter than four, several images of one atom."""
    from matpl_amd.neighbor import find_neighbore_gpu, reverse_map
    rng = np.random.Generator(np.random.PCG64(n))
    frac, types = rng.random((n, 3)), rng.integers(0, 3, n)
    types[:2] = (3, 4)
    tm = torch.as_tensor(types, dtype=torch.int32, device=dev)
    nl = find_neighbore_gpu(lat, frac, tm, 5, m, 6.0, want_dR=False, want_shift=True, device=dev)
    rev, status = reverse_map(nl, tm, m)
    assert int(status) == 0
    lst, rv, sh = (x.cpu().numpy().reshape(-1) for x in (nl.list, rev, nl.shift))
    used = lst > 0
    assert used.any() and np.array_equal(rv[~used], np.full((~used).sum(), -1))
    slots = np.nonzero(used)[0]
    partner = rv[slots]
    centre = slots // (5 * m)
    assert np.array_equal(partner // (5 * m), lst[slots] - 1)
    assert np.array_equal(lst[partner], centre + 1)
    assert np.array_equal(partner % (5 * m) // m, types[centre])
    image = lambda p: np.stack([(p >> k & 255) - 128 for k in (0, 8, 16)])
    assert np.array_equal(image(sh[partner]), -image(sh[slots]))
    # a list that lacks one partner is refused, its other entries are mapped as before
    k = slots[len(slots) // 2]
    i = k // (5 * m)
    c = nl.counts.clone()
    c[i, k % (5 * m) // m] = 0
    nl2 = type(nl)(nl.list, None, c, nl.shift, nl.frac_wrapped, nl.status)
    rev2, status2 = reverse_map(nl2, tm, m)
    assert int(status2) > 0


@pytest.mark.parametrize("order,scattered", [("space", False), ("type_space", False), ("random", True),
                                             ("type_random", True)])
def test_reverse_map_in_any_order(dev, order, scattered):
    """The search starts at the bucket's middle, or where atoms in no spatial order put the partner."""
    from matpl_amd.neighbor import find_neighbore_gpu, reverse_map
    rng = np.random.Generator(np.random.PCG64(17))
    n, T, m, L = 9001, 2, 121, 62.0
    frac, types = rng.random((n, 3)), rng.integers(0, T, n)
    if "space" in order:
        o = np.argsort(frac[:, 0])
        frac, types = frac[o], types[o]
    if "type" in order:
        o = np.argsort(types, kind="stable")
        frac, types = frac[o], types[o]
    tm = torch.as_tensor(types, dtype=torch.int32, device=dev)
    nl = find_neighbore_gpu(L * CUBE, frac, tm, T, m, 6.0, want_dR=False, want_shift=True, device=dev)
    lst, cnt = nl.list.cpu().numpy().reshape(n, T, m), nl.counts.cpu().numpy()
    span = []
    for a in (n // 8, 3 * n // 8, 5 * n // 8, 7 * n // 8):
        f, l = lst[a, :, 0], lst[a, np.arange(T), cnt[a] - 1]
        assert (cnt[a] > 4).all()
        span.append(min((l - f).sum(), l.max() - f.min()))
    assert (sum(4 * x > 3 * n for x in span) >= 3) == scattered
    rev, status = reverse_map(nl, tm, m)
    assert int(status) == 0
    rv, sh = rev.cpu().numpy().reshape(-1), nl.shift.cpu().numpy().reshape(-1)
    lst = lst.reshape(-1)
    slots = np.nonzero(lst > 0)[0]
    partner = rv[slots]
    assert (rv[lst == 0] == -1).all() and (partner >= 0).all()
    assert np.array_equal(rv[partner], slots)
    assert np.array_equal(partner // (T * m), lst[slots] - 1)
    assert np.array_equal(lst[partner], slots // (T * m) + 1)
    image = lambda p: np.stack([(p >> k & 255) - 128 for k in (0, 8, 16)])
    assert np.array_equal(image(sh[partner]), -image(sh[slots]))
