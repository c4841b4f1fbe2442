"""The launch shape that the fused DP kernels take by size, types and precision gives the plain launch's results:
energies bit for bit, forces and the virial within the rounding of the 8-wavefront
instantiation (1e-6 of the largest component, the bound of the launch-shape tests)."""
import numpy as np
import pytest
import torch

from matpl_amd import autotune
from matpl_amd import structures as st
from matpl_amd.dp_fused import FusedDP
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
