"""The launch shape that the fused DP kernels take by size, types and precision gives the plain launch's results:
energies bit for bit, forces and the virial within the rounding of the 8-wavefront
instantiation (1e-6 of the largest component, the bound of the launch-shape tests). A shape that is set also holds
where the default takes groups of atoms."""
import numpy as np
import pytest
import torch

from matpl_amd import _lib, autotune
from matpl_amd import structures as st
from matpl_amd.dp_fused import FusedDP, short_buckets
from matpl_amd.dpnet import DPConfig, DPWeights
from matpl_amd.neighbor import find_neighbore_gpu, reverse_map

pytestmark = pytest.mark.gpu

PLAIN = {"max_blocks": 4095, "lds_weights": -1, "xcd": 0, "waves": 4}      # any shape but the default is taken as set


@pytest.mark.parametrize("precision", ["bf16", "fp32"])
@pytest.mark.parametrize("system,reps", [("hfo2", (9, 9, 8)), ("hfo2", (9, 9, 9)), ("cu", (13, 13, 13))])
def test_default_launch_matches_the_plain_one(dev, system, reps, precision):
    f = (st.fluorite_hfo2 if system == "hfo2" else st.fcc_cu)(reps, seed=3)
    T = 2 if system == "hfo2" else 1
    cfg = DPConfig(ntypes=T, m=130)
    w = DPWeights.random(cfg, seed=5, davg=np.tile([0.1, 0, 0, 0], (T, 1)), dstd=np.tile([0.2, 0.1, 0.1, 0.1], (T, 1)))
    nl = find_neighbore_gpu(f.lattice, f.frac(), f.types, T, cfg.m, cfg.rcut, device=dev, want_dR=False,
                            want_shift=True)
    L = torch.as_tensor(f.lattice, device=dev)
    pos = (nl.frac_wrapped @ L).contiguous()
    tm = torch.as_tensor(f.types, device=dev)
    rev, rst = reverse_map(nl, tm, cfg.m)
    assert int(rst.item()) == 0
    model = FusedDP(w, precision, dev)
    ranges = [(int(np.searchsorted(f.types, t, "left")), int(np.searchsorted(f.types, t, "right"))) for t in range(T)]
    run = lambda: [x.clone() for x in model(pos, L.reshape(1, 9).contiguous(), tm, nl.list, nl.shift, nl.counts,
                                            cfg.m, type_ranges=ranges, rev=rev)]
    print(f"{system} {f.natoms} {precision}", flush=True)
    try:
        for k in (0, 1):
            autotune.set_launch(k, **PLAIN)
        Ei0, F0, V0, s0 = run()
        autotune.reset()
        Ei, F, V, s = run()
    finally:
        autotune.reset()
    assert int(s0.item()) == 0 and int(s.item()) == 0
    assert torch.equal(Ei, Ei0)
    assert float((F - F0).abs().max()) <= 1e-6 * float(F0.abs().max())
    assert float((V - V0).abs().max()) <= 1e-6 * float(V0.abs().max())


def test_a_set_launch_replaces_the_groups(dev):
    """Four types in equal parts, 4,200 atoms: groups by default, FP32 sums in another order (the FP32 bound against the
    oracle, 1e-5 eV/A, for the difference of the two), and a shape that does not fit is refused as for two types."""
    rng = np.random.default_rng(12)
    n, T, m, side = 4200, 4, 150, 17
    L = (n / 0.05) ** (1 / 3)
    site = rng.permutation(side ** 3)[:n]
    frac = (np.stack([site // side ** 2, site // side % side, site % side], -1) + 0.5 + rng.uniform(-0.1, 0.1, (n, 3))) / side
    types = np.sort(rng.integers(0, T, n)).astype(np.int32)
    cfg = DPConfig(ntypes=T, m=m)
    w = DPWeights.random(cfg, seed=5, davg=np.tile([0.1, 0, 0, 0], (T, 1)), dstd=np.tile([0.2, 0.1, 0.1, 0.1], (T, 1)))
    nl = find_neighbore_gpu(L * np.eye(3), frac, types, T, m, cfg.rcut, device=dev, want_dR=False, want_shift=True)
    pos = (nl.frac_wrapped * L).contiguous()
    tm, lat = torch.as_tensor(types, device=dev), torch.as_tensor(L * np.eye(3), device=dev).reshape(1, 9)
    rev, rst = reverse_map(nl, tm, m)
    assert int(rst.item()) == 0
    model = FusedDP(w, "fp32", dev)
    run = lambda: [x.clone() for x in model(pos, lat, tm, nl.list, nl.shift, nl.counts, m, rev=rev)]
    print(f"set launch against groups {n}", flush=True)
    try:
        autotune.reset()
        Ei0, F0, V0, s0 = run()
        assert short_buckets(np.bincount(types))
        for k in (0, 1):
            autotune.set_launch(k, **PLAIN)
        Ei, F, V, s = run()
        assert int(s0.item()) == 0 and int(s.item()) == 0
        assert float((F - F0).abs().max()) <= 1e-5 * max(1.0, float(F0.abs().max()))
        assert float((Ei - Ei0).abs().max()) <= 1e-6 * max(1.0, float(Ei0.abs().max()))
        for k in (0, 1):
            autotune.reset()
            autotune.set_launch(k, 4096, 1, 0)          # weights of 16 pairs in LDS
            with pytest.raises(_lib.MatplError):
                run()
    finally:
        autotune.reset()
