"""The fused DP kernels' group passes (three types and more, several atoms per wavefront from 4,096 atoms on) at
their edges: frames of 1 and 2 atoms, types in no order, atoms without neighbors, buckets of more than a tile and
atoms whose lists exceed a wavefront's buffer (256 entries), against the FP64 oracle frame by frame; and a training
step on a batch large enough for whole groups against the sum of its parts, which are small enough to run atom by
atom. The embedding gradients' two forms (no more wavefronts than SIMDs, and more) against each other. Tolerances: as tests/test_gpu_dp_fused.py (FP32 1e-5 eV/A per force component, 1e-6 relative energy; BF16
force RMSE 1e-3 eV/A); gradients in FP32 are sums of ~1e6 products added in another order, 2e-5 of their norm."""
import numpy as np
import pytest
import torch

import oracle
from matpl_amd.dp_fused import FusedDP
from matpl_amd.dp_train_fused import DPTrainFused, pack_fused_batch
from matpl_amd.dpnet import DPConfig, DPWeights
from matpl_amd.neighbor import find_neighbore_batch, reverse_map
from matpl_amd.structures import Frame

pytestmark = pytest.mark.gpu


def _frame(n, density, T, rng, sort):
    side = int(np.ceil(n ** (1 / 3)))
    L = (n / density) ** (1 / 3)
    site = rng.permutation(side ** 3)[:n]
    pos = np.stack([site // (side * side), site // side % side, site % side], -1) + 0.5
    pos = (pos + rng.uniform(-0.12, 0.12, (n, 3))) * (L / side)
    t = rng.integers(0, T, n).astype(np.int32)
    return Frame(np.diag([L] * 3), pos, np.sort(t) if sort else t, ["A"] * T)


def _frames(T, sort, dense, seed):
    rng = np.random.default_rng(seed)
    sizes = [1, 2, 3, 230, 150] + [int(x) for x in rng.integers(180, 300, 36)]
    out = [_frame(n, 0.0005 if n <= 3 else 0.05, T, rng, sort) for n in sizes]
    if dense:
        out.insert(4, _frame(700, 0.36, T, rng, sort))          # ~330 neighbors an atom
    return out


def _weights(T, m, seed, E=25):
    cfg = DPConfig(ntypes=T, m=m, emb_sizes=[E] * 3)
    davg = np.tile([0.05, 0, 0, 0], (T, 1))
    dstd = np.tile([0.1, 0.07, 0.07, 0.07], (T, 1))
    return DPWeights.random(cfg, seed=seed, davg=davg, dstd=dstd)


@pytest.mark.parametrize("T,m,sort,dense", [(4, 60, True, False), (3, 150, True, True), (5, 40, False, False)])
def test_group_evaluation_vs_oracle(dev, T, m, sort, dense):
    frames = _frames(T, sort, dense, 11 + T)
    sizes = [f.natoms for f in frames]
    n = sum(sizes)
    print(f"case dp group T={T} m={m} sorted={sort} dense={dense} atoms={n}", flush=True)
    assert n > 8192
    w = _weights(T, m, 3)
    nl = find_neighbore_batch([f.lattice for f in frames], [f.frac() for f in frames], [f.types for f in frames], T, m,
                              w.cfg.rcut, want_dR=False, want_shift=True, device=dev)
    start = np.concatenate([[0], np.cumsum(sizes)])
    fs = torch.as_tensor(start.astype(np.int64), device=dev)
    af = torch.as_tensor(np.repeat(np.arange(len(sizes), dtype=np.int32), sizes), device=dev)
    tm = torch.as_tensor(np.concatenate([f.types for f in frames]), device=dev)
    lat = torch.as_tensor(np.stack([f.lattice.reshape(9) for f in frames]), device=dev)
    pos = torch.cat([nl.frac_wrapped[start[k]:start[k + 1]] @ lat[k].view(3, 3) for k in range(len(sizes))]).contiguous()
    rev, st = reverse_map(nl, tm, m, frame_start=fs, atom_frame=af)
    assert int(st.item()) == 0
    ref = [oracle.dp_evaluate(f, w) for f in frames]
    E = np.concatenate([np.asarray(r["Ei"]).reshape(-1) for r in ref])
    F = np.concatenate([np.asarray(r["F"]).reshape(-1, 3) for r in ref])
    V = np.stack([np.asarray(r["V"]).reshape(9) for r in ref])
    for precision in ("fp32", "bf16"):
        for gather in (True, False):
            model = FusedDP(w, precision, dev)
            Ei, Fg, Vg, status = model(pos, lat, tm, nl.list, nl.shift, nl.counts, m, atom_frame=af, frame_start=fs,
                                       nframes=len(sizes), rev=rev if gather else None)
            assert int(status.item()) == 0
            dF = Fg.cpu().numpy() - F
            dE, dV = np.abs(Ei.cpu().numpy() - E).max(), np.abs(Vg.cpu().numpy() - V).max()
            print(precision, gather, np.abs(dF).max(), np.sqrt((dF ** 2).mean()), dE, dV, flush=True)
            if precision == "fp32":
                assert np.abs(dF).max() < 1e-5 * max(1.0, np.abs(F).max())
                assert dE < 2e-6 * max(1.0, np.abs(E).max()) and dV < 1e-5 * max(1.0, np.abs(V).max())
            else:
                assert np.sqrt((dF ** 2).mean()) < 1e-3 * max(1.0, np.sqrt((F ** 2).mean()))


def test_group_training_step_equals_its_parts(dev):
    """All 41 frames (whole groups) against pieces of at most 2,047 atoms (one atom per wavefront)."""
    frames = _frames(4, True, False, 5)
    w = _weights(4, 60, 9)
    model = DPTrainFused(w, "fp32", dev)
    n, nf = sum(f.natoms for f in frames), len(frames)
    print(f"case dp group training atoms={n}", flush=True)
    batch = pack_fused_batch(frames, w.cfg, dev, seed=4)
    loss, grads = model.loss_and_grads(batch)
    cuts, k = [0], 0
    while k < nf:
        tot = 0
        while k < nf and tot + frames[k].natoms < 2048:
            tot += frames[k].natoms
            k += 1
        cuts.append(k)
    total, parts = 0.0, None
    first = np.concatenate([[0], np.cumsum([f.natoms for f in frames])])
    for a, b in zip(cuts[:-1], cuts[1:]):
        piece = pack_fused_batch(frames[a:b], w.cfg, dev, seed=4)
        piece.E_label = batch.E_label[a:b].contiguous()
        piece.F_label = batch.F_label[first[a]:first[b]].contiguous()
        model.pe, model.pf = (b - a) / nf, piece.natoms / n
        l, g = model.loss_and_grads(piece)
        total = total + l.double()
        g = [None if x is None else x.double() for x in g]
        parts = g if parts is None else [x if y is None else (y if x is None else x + y) for x, y in zip(parts, g)]
    assert abs(float(loss) - float(total)) < 1e-5 * abs(float(total))
    for x, y in zip(grads, parts):
        assert (x is None) == (y is None)
        if x is not None:
            assert float((x.double() - y).norm()) <= 2e-5 * float(y.norm()) + 1e-12


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("E", [25, 16])
def test_gradient_kernel_forms_agree(dev, E, precision):
    """One batch by atoms per wavefront: 1 (some 3,500 wavefronts) and 40 (fewer than SIMDs). Both round the same operands,
    so that in BF16 too only the order of the sums differs."""
    frames = _frames(4, True, False, 3)[:7]
    n = sum(f.natoms for f in frames)
    print(f"case embedding gradient forms E={E} {precision} atoms={n}", flush=True)
    model = DPTrainFused(_weights(4, 60, 9, E), precision, dev)
    batch = pack_fused_batch(frames, model.cfg, dev, seed=4)
    got = []
    for chunk in (1, 40):
        assert (-(-n // chunk) * 4 > 1024) == (chunk == 1)
        model.chunk = chunk
        got.append(model.loss_and_grads(batch)[1])
    assert sum(x is not None for x in got[0]) > 0
    for x, y in zip(*got):
        assert (x is None) == (y is None)
        if x is not None:
            assert float((x - y).norm()) <= 2e-5 * float(y.norm()) + 1e-12
