"""The reverse map against its definition."""
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
