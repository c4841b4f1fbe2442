"""The NEP model's fused descriptor, force and virial path (matpl_nep_descriptor, matpl_nep_model_forces and their
backward) against the operators' sequence it stands for (calculateNepFeat / calculateNepMbFeat, autograd for dE/dRi,
nep_force_virial) in double, at the edges of its windows: frames of 1 atom, several frames in a window, frames above
the LDS copy of F (device atomics), sizes other than the default, no angular part.

Tolerances: outputs and gradients are sums of at most ~1e5 terms; 1e-11 (double, about 5e4 eps) and 2e-4 (float) of
the largest entry bound any order of summation and are far above what is measured."""
import numpy as np
import pytest
import torch

from matpl_amd import nep as mn
from matpl_amd import nep_ops
from matpl_amd.nepnet import NEPConfig, NEPWeights
from matpl_amd.structures import Frame

pytestmark = pytest.mark.gpu


def _frames(sizes, T, seed):
    rng = np.random.default_rng(seed)
    out = []
    for n in sizes:
        side = int(np.ceil(n ** (1 / 3)))
        L = side * 2.6
        site = rng.permutation(side ** 3)[:n]
        pos = np.stack([site // (side * side), site // side % side, site % side], -1) * 2.6
        out.append(Frame(np.diag([L] * 3), pos + rng.uniform(0, 0.3, (n, 3)), rng.integers(0, T, n).astype(np.int32)))
    return out


def _by_ops(model, nb, p):
    """(E, F, V) through the operators, differentiable in the parameters."""
    cfg = model.cfg
    ins = [nb["Ri_r"].detach().requires_grad_(), nb["Ri_a"].detach().requires_grad_()]
    q = model.features(ins[0], nb["NL_r"], ins[1], nb["NL_a"], p["atom_type_map"])
    Ei, gq = model.energies_and_grad(q, p["atom_type_map"])      # gq = dEi/dq, differentiable
    E = model._frame_sum(Ei, p["num_atoms"])
    ins = ins[:1] if cfg.l_max[0] == 0 else ins
    F = V = 0
    for Ri, NL, dE in zip(ins, (nb["NL_r"], nb["NL_a"]), torch.autograd.grad([q], ins, [gq], create_graph=True)):
        f, v = nep_ops.nep_force_virial(NL, dE, Ri, p["num_atoms"])
        F, V = F - f, V - v
    return E, F, V


CASES = [([1, 2, 3, 70, 64, 5, 1, 130], 3, 4, 12, [4, 2, 0]),       # many frames in a window
         ([2500], 2, 4, 12, [4, 2, 0]),                              # above the LDS copy in double
         ([40, 9, 300], 2, 3, 7, [4, 2, 1]),                         # other sizes, 5-body
         ([50, 20], 5, 4, 12, [0, 0, 0]),                            # radial only
         ([3] * 40 + [1900] + [2] * 30, 2, 4, 12, [4, 2, 0])]        # one large frame among many tiny ones


@pytest.mark.parametrize("sizes,T,n_max,basis,l_max", CASES)
def test_model_path_equals_operator_sequence(dev, sizes, T, n_max, basis, l_max):
    print(f"case nep model path sizes={sizes} T={T} n_max={n_max} basis={basis} l_max={l_max}", flush=True)
    cfg = NEPConfig(ntypes=T, n_max_radial=n_max, n_max_angular=n_max, basis_radial=basis, basis_angular=basis,
                    l_max=l_max)
    w = NEPWeights.random(cfg, seed=31, q_scaler=np.full(cfg.nfeat, 0.3))
    p = mn.pack_frames(_frames(sizes, T, 5), cfg.rcut_radial, dev)
    nb = mn.neighbors(p, cfg.rcut_radial, cfg.rcut_angular, T)
    g = torch.Generator(device=dev).manual_seed(3)
    n, nf = sum(sizes), len(sizes)
    wE, wF, wV = (torch.randn(*s, dtype=torch.float64, device=dev, generator=g) for s in ((nf, 1), (n, 3), (nf, 9)))
    ref = mn.NEPTorch(w, torch.float64, dev)
    want = _by_ops(ref, nb, p)
    names = [k for k, q in ref.named_parameters() if l_max[0] > 0 or q is not ref.c3]
    params = [q for q in ref.parameters() if l_max[0] > 0 or q is not ref.c3]
    partial = {k: [torch.zeros_like(q) if g is None else g for q, g in zip(params, torch.autograd.grad(
        (x * wx).sum(), params, retain_graph=True, allow_unused=True))] for k, x, wx in ((2, want[1], wF), (3, want[2], wV))}
    want += torch.autograd.grad((want[0] * wE).sum() + (want[1] * wF).sum() + 0.1 * (want[2] * wV).sum(), params)
    for dtype, tol in ((torch.float64, 1e-11), (torch.float32, 2e-4)):
        model = mn.NEPTorch(w, dtype, dev)
        args = (nb["NN_r"], nb["NL_r"], nb["Ri_r"], nb["NN_a"], nb["NL_a"], nb["Ri_a"], p["num_atoms"],
                p["atom_type_map"])
        E, _, F, V = model(*args, create_graph=True)
        loss = (E * wE).sum() + (F * wF).sum() + 0.1 * (V * wV).sum()
        params = [q for q in model.parameters() if l_max[0] > 0 or q is not model.c3]
        got = (E, F, V) + torch.autograd.grad(loss, params)
        for k, (a, b) in enumerate(zip(got, want)):
            a, b = a.detach().double(), b.detach()
            err = float((a - b).abs().max())
            assert err <= tol * max(float(b.abs().max()), 1e-2), (dtype, k, err, float(b.abs().max()))
        # without a graph: the same values, detached forces
        E1, _, F1, V1 = model(*args, create_graph=False)
        assert not F1.requires_grad and not V1.requires_grad
        assert float((F1 - F.detach()).abs().max()) <= tol * float(F.detach().abs().max().clamp_min(1e-2))
        # only the forces, or only the virials, in the loss: a bias b1 of the nets (the last tensor of each) reaches
        # neither
        for k, wx in ((2, wF), (3, wV)):
            x = model(*args, create_graph=True)[k]
            gs = torch.autograd.grad((x * wx).sum(), params, allow_unused=True)
            for q, a, b in zip(names, gs, partial[k]):
                a = torch.zeros_like(b) if a is None else a.double()
                assert a.abs().max() > 0 or q.endswith("b.1"), q
                err = float((a - b).abs().max())
                assert err <= tol * max(float(b.abs().max()), 1e-2), (dtype, k, q, err, float(b.abs().max()))


def test_work_buffer_grows_with_the_atoms():
    """100,000 frames of 10 atoms and one of 2,000: rows of 2,000 for each frame would be gigabytes."""
    from matpl_amd import _lib
    small = _lib.query("matpl_nep_model_forces_work", 0, 1_000_000, 100_000, 10, 4, 5, 13)
    mixed = _lib.query("matpl_nep_model_forces_work", 0, 1_002_000, 100_001, 2000, 4, 5, 13)
    # three floats an atom and window of its frame, 72 bytes for each window and frame
    assert small <= 1_000_000 * 12 * 2 + 72 * (1_000_000 // 64 + 100_001)
    assert mixed <= 1_002_000 * 12 * (2000 // 64 + 2) + 72 * (1_002_000 // 64 + 100_002)


def test_energies_ask_nothing_of_the_frames(dev):
    """One frame whose num_atom is not the list's atom count: energies as for the whole list, forces refused."""
    cfg = NEPConfig(ntypes=2)
    w = NEPWeights.random(cfg, seed=3, q_scaler=np.full(cfg.nfeat, 0.3))
    p = mn.pack_frames(_frames([40], 2, 6), cfg.rcut_radial, dev)
    nb = mn.neighbors(p, cfg.rcut_radial, cfg.rcut_angular, 2)
    model = mn.NEPTorch(w, torch.float64, dev)
    args = (nb["NN_r"], nb["NL_r"], nb["Ri_r"], nb["NN_a"], nb["NL_a"], nb["Ri_a"])
    E0, Ei0, _, _ = model(*args, p["num_atoms"], p["atom_type_map"])
    E, Ei, F, V = model(*args, torch.ones_like(p["num_atoms"]), p["atom_type_map"], is_calc_f=False)
    assert torch.equal(E, E0) and torch.equal(Ei, Ei0) and F is None and V is None
    (g,) = torch.autograd.grad(E.sum(), [model.c2])
    assert torch.isfinite(g).all()
    with pytest.raises(ValueError):
        model(*args, torch.ones_like(p["num_atoms"]), p["atom_type_map"])
