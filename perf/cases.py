"""The workloads this framework's speed is judged on, each through its public entry points.

Seven kinds of call, which are what a user has the framework do:

  dp_eval     energy, forces and virial of a DP se_e2_a model from a neighbor list with a skin: what every MD
              step asks for (matpl_amd.dp_fused.FusedDP). Small systems run as a captured HIP graph, as
              matpl_amd.md.DPMD.capture does; large ones run eagerly.
  dp_rebuild  the neighbor list of an MD run and its reverse slot map, rebuilt every few steps.
  dp_train    one DP training step's loss and gradients on a packed batch (matpl_amd.dp_train_fused).
  nep_eval    energy, forces and virial of a NEP model, neighbor search included, either replayed as one HIP
              graph (matpl_amd.nep.NEPGraph) or called eagerly (several frames, validation).
  nep_train   one NEP training step: neighbor search, forward, forces and virials, loss, gradients of every
              parameter (matpl_amd.nep.NEPTorch).
  dp_ops      the reference's operator sequence on a padded list: environment matrix, calculateForce,
              calculateVirial and their backward (torch.ops.CalcOps_cuda), which a DP model that keeps its own
              torch nets calls.

The systems are those of this repository's benchmark and tests: fcc Cu (one type), fluorite HfO2 (two), a
Li10GeP2S12 composition (four), zincblende SiC (two) and a random Ag-Au-Si-C alloy (four).
"""
import math

import numpy as np
import torch

DEV = "cuda"

# ------------------------------------------------------------------------------------------------ cases


def listed():
    return [
        # the smallest DP evaluation a user runs: 108 Cu atoms, one MD step's graph; launches and latency count
        dict(name="dp_eval_cu_108_bf16", kind="dp_eval", system="cu", nx=3, ny=3, nz=3, precision="bf16",
             embedding="net", graph=True),
        # a small two-type cell with the compressed embedding (the reference's DP compress), odd cell counts
        dict(name="dp_eval_hfo2_1500_table", kind="dp_eval", system="hfo2", nx=5, ny=5, nz=5, precision="bf16",
             embedding="table", graph=True),
        # an ordinary MD cell in FP32
        dict(name="dp_eval_hfo2_11880_fp32", kind="dp_eval", system="hfo2", nx=9, ny=10, nz=11, precision="fp32",
             embedding="net", graph=False),
        # the benchmark's MD cell
        dict(name="dp_eval_hfo2_99636_bf16", kind="dp_eval", system="hfo2", nx=19, ny=19, nz=23, precision="bf16",
             embedding="net", graph=False),
        # its neighbor list and reverse map, the other part of an MD run
        dict(name="dp_rebuild_hfo2_99636", kind="dp_rebuild", system="hfo2", nx=19, ny=19, nz=23),
        # the benchmark's training batch: 256 frames of 64 to 512 atoms, four types
        dict(name="dp_train_lgps_256_bf16", kind="dp_train", frames=256, nmin=64, nmax=512, precision="bf16"),
        # a small batch in FP32
        dict(name="dp_train_lgps_24_fp32", kind="dp_train", frames=24, nmin=64, nmax=512, precision="fp32"),
        # the benchmark's NEP cell as one replayed graph (MD), float model
        dict(name="nep_eval_sic_1728_f32", kind="nep_eval", system="sic", frames=1, nmin=1728, nmax=1728,
             dtype="f32", graph=True),
        # validation of a batch of alloy frames in double, eager
        dict(name="nep_eval_alloy_32_f64", kind="nep_eval", system="alloy", frames=32, nmin=32, nmax=1024,
             dtype="f64", graph=False),
        # the benchmark's NEP training batch
        dict(name="nep_train_alloy_128_f32", kind="nep_train", frames=128, nmin=32, nmax=1024, dtype="f32"),
        # a small batch in double, the precision the reference trains in
        dict(name="nep_train_alloy_16_f64", kind="nep_train", frames=16, nmin=32, nmax=1024, dtype="f64"),
        # the drop-in operators of a DP model with torch nets, in the reference's precision
        dict(name="dp_ops_hfo2_6144_f64", kind="dp_ops", system="hfo2", nx=8, ny=8, nz=8, dtype="f64"),
    ]


def _cells(rng, lo, hi, per_cell):
    """Three cell counts, odd ones among them, whose atom count is log-uniform in [lo, hi]."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    side = (n / per_cell) ** (1.0 / 3.0)
    out = [max(2, int(round(side * rng.uniform(0.8, 1.25)))) for _ in range(3)]
    while out[0] * out[1] * out[2] * per_cell > hi:
        out[out.index(max(out))] -= 1
    return out


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dp_eval", "dp_eval", "dp_rebuild", "dp_train", "nep_eval", "nep_train", "dp_ops"])
    if kind in ("dp_eval", "dp_rebuild"):
        system = rng.choice(["cu", "hfo2", "hfo2"])
        hi = 90000 if system == "hfo2" else 30000
        nx, ny, nz = _cells(rng, 100, hi, 12 if system == "hfo2" else 4)
        if kind == "dp_rebuild":
            return dict(kind=kind, system=system, nx=nx, ny=ny, nz=nz)
        n = nx * ny * nz * (12 if system == "hfo2" else 4)
        precision = rng.choice(["bf16", "bf16", "fp32"]) if n <= 30000 else "bf16"
        return dict(kind=kind, system=system, nx=nx, ny=ny, nz=nz, precision=precision,
                    embedding=rng.choice(["net", "net", "table"]), graph=n <= 4000)
    if kind == "dp_train":
        precision = rng.choice(["bf16", "fp32"])
        nmin = rng.randint(40, 120)
        return dict(kind=kind, frames=_log_int(rng, 4, 220 if precision == "bf16" else 100), nmin=nmin,
                    nmax=nmin + rng.randint(1, 400), precision=precision)
    if kind == "nep_eval":
        if rng.random() < 0.5:
            n = rng.randint(3, 7) * rng.randint(3, 7) * rng.randint(3, 7) * 8
            return dict(kind=kind, system="sic", frames=1, nmin=n, nmax=n, dtype=rng.choice(["f32", "f64"]),
                        graph=True)
        nmin = rng.randint(20, 300)
        return dict(kind=kind, system="alloy", frames=_log_int(rng, 1, 100), nmin=nmin,
                    nmax=nmin + rng.randint(1, 700), dtype=rng.choice(["f32", "f64"]), graph=False)
    if kind == "nep_train":
        dtype = rng.choice(["f32", "f64"])
        nmin = rng.randint(20, 200)
        return dict(kind=kind, frames=_log_int(rng, 4, 100 if dtype == "f32" else 48), nmin=nmin,
                    nmax=nmin + rng.randint(1, 800), dtype=dtype)
    nx, ny, nz = _cells(rng, 100, 8000, 12)
    return dict(kind=kind, system="hfo2", nx=nx, ny=ny, nz=nz, dtype=rng.choice(["f32", "f64"]))


# -------------------------------------------------------------------------------------------- structures

RC, RS = 6.0, 5.5                  # DP cutoff and smoothing start (A)
SKIN = 0.5                         # of the MD neighbor list
MNL = 160                          # slots per type in the MD neighbor list
DP_M = {"cu": 100, "hfo2": 120, "lgps": 150}
DP_T = {"cu": 1, "hfo2": 2, "lgps": 4}
# mean and deviation of the environment matrix per centre type, of these systems' own statistics
# (the first of the four columns has a mean; the deviations of the other three are one number)
DP_STAT = {"cu": ([0.1656], [[0.1257, 0.1200]]),
           "hfo2": ([0.0740, 0.0755], [[0.1213, 0.0820], [0.1188, 0.0813]]),
           "lgps": ([0.0154] * 4, [[0.0616, 0.0367]] * 4)}
DENSITY = {"lgps": 0.0499, "alloy": 0.06}
TYPES = {"lgps": (0.40, 0.04, 0.08, 0.48), "alloy": (0.25, 0.25, 0.25, 0.25)}
NEP_RC, NEP_RCA = 6.0, 4.0


def _rng(case, seed):
    return np.random.Generator(np.random.PCG64([int(seed) & 0x7FFFFFFF, 77]))


def _crystal(system, nx, ny, nz, rng):
    """(lattice, positions, types) of a supercell with thermal displacements, atoms grouped by type."""
    fcc = np.array([[0, 0, 0], [0, .5, .5], [.5, 0, .5], [.5, .5, 0]])
    if system == "cu":
        a, sigma, basis, types = 3.615, 0.1, fcc, [0] * 4
    elif system == "hfo2":
        oxy = np.array([[x, y, z] for x in (.25, .75) for y in (.25, .75) for z in (.25, .75)])
        a, sigma, basis, types = 5.08, 0.1, np.concatenate([fcc, oxy]), [0] * 4 + [1] * 8
    else:
        a, sigma, basis, types = 4.36, 0.08, np.concatenate([fcc, fcc + 0.25]), [0] * 4 + [1] * 4
    cells = np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"), -1).reshape(-1, 1, 3)
    pos = ((cells + basis[None]) * a).reshape(-1, 3)
    t = np.tile(np.asarray(types, np.int32), nx * ny * nz)
    pos = pos + rng.normal(0.0, sigma, size=pos.shape)
    order = np.argsort(t, kind="stable")
    return np.diag([a * nx, a * ny, a * nz]).astype(np.float64), pos[order], t[order]


def _amorphous(system, n, rng):
    """(lattice, positions, types): n atoms on randomly chosen, jittered sites of a cubic grid."""
    side = math.ceil(n ** (1.0 / 3.0))
    length = (n / DENSITY[system]) ** (1.0 / 3.0)
    site = rng.permutation(side ** 3)[:n]
    g = np.stack([site // (side * side), site // side % side, site % side], -1)
    pos = (g + 0.5 + rng.uniform(-0.14, 0.14, size=(n, 3))) * (length / side)
    frac = TYPES[system]
    counts = [max(1, int(round(n * f))) for f in frac[:-1]]
    t = np.repeat(np.arange(len(frac), dtype=np.int32), counts + [n - sum(counts)])
    return np.diag([length] * 3), pos, t


def _frames(case, seed):
    rng = _rng(case, seed)
    if case["kind"] in ("dp_eval", "dp_rebuild", "dp_ops"):
        return [_crystal(case["system"], case["nx"], case["ny"], case["nz"], rng)]
    system = case.get("system", "lgps" if case["kind"] == "dp_train" else "alloy")
    if system == "sic":
        n8 = case["nmin"] // 8
        nx = max(d for d in range(1, int(round(n8 ** (1 / 3))) + 1) if n8 % d == 0)
        rest = n8 // nx
        ny = max(d for d in range(1, int(math.isqrt(rest)) + 1) if rest % d == 0)
        return [_crystal("sic", nx, ny, rest // ny, rng)]
    # the sizes belong to the case, not to the seed, so that other inputs are the same work
    sizes = np.random.Generator(np.random.PCG64([case["frames"], case["nmin"], case["nmax"]])).integers(
        case["nmin"], case["nmax"] + 1, size=case["frames"])
    return [_amorphous(system, int(n), rng) for n in sizes]


def _natoms(case):
    if case["kind"] in ("dp_eval", "dp_rebuild", "dp_ops"):
        return case["nx"] * case["ny"] * case["nz"] * (4 if case["system"] == "cu" else 12)
    if case.get("system") == "sic":
        return case["nmin"]
    return int(np.random.Generator(np.random.PCG64([case["frames"], case["nmin"], case["nmax"]])).integers(
        case["nmin"], case["nmax"] + 1, size=case["frames"]).sum())


# ----------------------------------------------------------------------------------------------- weights


def _net(rng, sizes, rdt):
    out = []
    for k in range(len(sizes) - 1):
        W = rng.normal(0.0, 1.0 / math.sqrt(sizes[k]), size=(sizes[k], sizes[k + 1]))
        r = rng.normal(0.1, 0.001, size=sizes[k + 1]) if rdt and 0 < k < len(sizes) - 2 else None
        out.append((W, rng.normal(0.0, 1.0, size=sizes[k + 1]), r))
    return out


def _dp_model(system, seed):
    """(embedding nets [T*T], fitting nets [T], davg [T, 4], dstd [T, 4]): 1-25-25-25 and 400-50-50-50-1."""
    rng = np.random.Generator(np.random.PCG64([int(seed) & 0x7FFFFFFF, 78]))
    T = DP_T[system]
    emb = [_net(rng, [1, 25, 25, 25], False) for _ in range(T * T)]
    fit = [_net(rng, [400, 50, 50, 50, 1], True) for _ in range(T)]
    mean, dev = DP_STAT[system]
    davg = np.array([[a, 0.0, 0.0, 0.0] for a in mean])
    dstd = np.array([[d[0], d[1], d[1], d[1]] for d in dev])
    return emb, fit, davg, dstd


def _dp_weights(system, seed):
    from matpl_amd.dpnet import DPConfig, DPWeights
    cfg = DPConfig(ntypes=DP_T[system], rcut=RC, rcut_smooth=RS, m=DP_M[system])
    return DPWeights(cfg, *_dp_model(system, seed))


def _nep_model(T, seed):
    """(c2, c3, q_scaler, fitting nets): n_max 4/4, basis 12, l_max [4, 2, 0], 30 hidden units."""
    rng = np.random.Generator(np.random.PCG64([int(seed) & 0x7FFFFFFF, 79]))
    c2 = rng.uniform(-0.5, 0.5, size=(T, T, 5, 13)) + 0.1 * rng.normal(size=(T, T, 5, 13))
    c3 = rng.uniform(-0.5, 0.5, size=(T, T, 5, 13)) + 0.1 * rng.normal(size=(T, T, 5, 13))
    qs = np.concatenate([np.full(5, 0.1), np.full(20, 1.0), np.full(5, 2.0)])
    return c2, c3, qs, [_net(rng, [30, 30, 1], False) for _ in range(T)]


def _nep_weights(T, seed):
    from matpl_amd.nepnet import NEPConfig, NEPWeights
    return NEPWeights(NEPConfig(ntypes=T, l_max=[4, 2, 0]), *_nep_model(T, seed))


def _labels(case, seed, sizes):
    rng = np.random.Generator(np.random.PCG64([int(seed) & 0x7FFFFFFF, 80]))
    n = np.asarray(sizes, np.float64)
    return (rng.normal(0.0, 0.1, len(n)) * n, rng.normal(0.0, 0.5, (int(n.sum()), 3)),
            rng.normal(0.0, 0.2, (len(n), 9)) * n[:, None])


def _dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=DEV)


# ----------------------------------------------------------------------------------------------- prepare


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_list(case, seed):
    from matpl_amd.neighbor import find_neighbore_gpu, reverse_map
    (lat, pos, types), = _frames(case, seed)
    T = DP_T[case["system"]]
    tm = _dev(types, torch.int32)
    frac = _dev(pos @ np.linalg.inv(lat))
    nl = find_neighbore_gpu(lat, frac, tm, T, MNL, RC + SKIN, device=DEV, want_dR=False, want_shift=True)
    rev, status = reverse_map(nl, tm, MNL)
    return dict(case=case, lat=lat, frac=frac, types=tm, T=T, nl=nl, rev=rev, rev_status=status)


def _table(w):
    """The reference's DP compress defaults: spacing 0.01, cubic, tabulated up to a 1 A bond."""
    from matpl_amd.compress import build_table
    from matpl_amd.dp import DPTorch
    return build_table(list(DPTorch(w, torch.float64, DEV).emb), w.davg, w.dstd, 1.0, dx=0.01, order=3, device=DEV)


def _prepare_dp_eval(case, seed):
    from matpl_amd.dp_fused import FusedDP
    s = _prepare_list(case, seed)
    w = _dp_weights(case["system"], seed)
    s["lattice"] = _dev(s["lat"].reshape(1, 9))
    s["pos"] = (s["nl"].frac_wrapped @ s["lattice"].view(3, 3)).contiguous()
    tm = s["types"].cpu().numpy()
    s["ranges"] = [(int(np.searchsorted(tm, t, "left")), int(np.searchsorted(tm, t, "right"))) for t in range(s["T"])]
    s["model"] = FusedDP(w, case["precision"], DEV, compress=_table(w) if case["embedding"] == "table" else None)
    if case["graph"]:
        for _ in range(2):
            _dp_call(s)
        torch.cuda.synchronize()
        s["replay"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["replay"]):
            s["out"] = _dp_call(s)
    return s


def _dp_call(s):
    nl = s["nl"]
    Ei, F, V, status = s["model"](s["pos"], s["lattice"], s["types"], nl.list, nl.shift, nl.counts, MNL,
                                  type_ranges=s["ranges"], rev=s["rev"])
    return dict(Ei=Ei, F=F, V=V, status=status)


def _prepare_dp_train(case, seed):
    from matpl_amd.dp_train_fused import DPTrainFused, pack_fused_batch
    from matpl_amd.structures import Frame
    frames = [Frame(*f, ["Li", "Ge", "P", "S"]) for f in _frames(case, seed)]
    w = _dp_weights("lgps", seed)
    batch = pack_fused_batch(frames, w.cfg, DEV)
    E, F, _ = _labels(case, seed, [f.natoms for f in frames])
    batch.E_label, batch.F_label = _dev(E), _dev(F)
    return dict(case=case, batch=batch, model=DPTrainFused(w, case["precision"], DEV))


def _prepare_nep(case, seed):
    from matpl_amd import nep, nep_ops
    from matpl_amd.structures import Frame
    raw = _frames(case, seed)
    T = 2 if case.get("system") == "sic" else 4
    dtype = torch.float32 if case["dtype"] == "f32" else torch.float64
    w = _nep_weights(T, seed)
    p = nep.pack_frames([Frame(*f) for f in raw], w.cfg.rcut_radial, DEV)
    s = dict(case=case, packed=p, T=T, dtype=dtype, cfg=w.cfg, model=nep.NEPTorch(w, dtype, DEV))
    if case["kind"] == "nep_train":
        s["labels"] = [_dev(x, dtype) for x in _labels(case, seed, [len(f[1]) for f in raw])]
        s["natoms"] = p["num_atoms"].to(dtype)
        s["params"] = list(s["model"].parameters())
    elif case["graph"]:
        nr, na = nep_ops.calculate_maxneigh(p["num_atoms"], p["box"], p["box_orig"], p["num_cell"], p["position"],
                                            w.cfg.rcut_radial, w.cfg.rcut_angular, T, p["atom_type_map"], False)
        s["replay"] = nep.NEPGraph(s["model"], p, T, int(nr.max()), int(na.max()))
    return s


def _prepare_dp_ops(case, seed):
    from matpl_amd import calcops
    from matpl_amd.neighbor import find_neighbore_gpu, image_dr
    calcops.register()
    (lat, pos, types), = _frames(case, seed)
    T, m = DP_T[case["system"]], DP_M[case["system"]]
    dtype = torch.float32 if case["dtype"] == "f32" else torch.float64
    tm = _dev(types, torch.int32)
    nl = find_neighbore_gpu(lat, _dev(pos @ np.linalg.inv(lat)), tm, T, m, RC, device=DEV)
    _, _, davg, dstd = _dp_model(case["system"], seed)
    N, S = nl.list.shape
    rng = np.random.Generator(np.random.PCG64([int(seed) & 0x7FFFFFFF, 81]))
    g = torch.Generator(device=DEV).manual_seed(int(rng.integers(1 << 31)))

    def normal(*shape):
        return torch.randn(*shape, dtype=dtype, device=DEV, generator=g)
    return dict(case=case, types=tm, list0=(nl.list - 1).view(1, N, 1, S).contiguous(),
                image_dr=image_dr(nl.list, nl.dR).to(dtype).unsqueeze(0).contiguous(),
                rij=nl.dR.to(dtype).unsqueeze(0).contiguous(),
                davg=_dev(np.tile(davg, (1, S)), dtype), dstd=_dev(np.tile(dstd, (1, S)), dtype),
                dE=normal(1, N, 1, S * 4).requires_grad_(), F0=normal(1, N, 3), gF=normal(1, N, 3), gV=normal(1, 9))


_PREPARE = dict(dp_eval=_prepare_dp_eval, dp_rebuild=_prepare_list, dp_train=_prepare_dp_train, nep_eval=_prepare_nep,
                nep_train=_prepare_nep, dp_ops=_prepare_dp_ops)

# --------------------------------------------------------------------------------------------------- run


def run(s):
    return _RUN[s["case"]["kind"]](s)


def _run_dp_eval(s):
    if "replay" in s:
        s["replay"].replay()
        return s["out"]
    return _dp_call(s)


def _run_dp_rebuild(s):
    from matpl_amd.neighbor import find_neighbore_gpu, reverse_map
    nl = find_neighbore_gpu(s["lat"], s["frac"], s["types"], s["T"], MNL, RC + SKIN, device=DEV, want_dR=False,
                            want_shift=True, check=False, out=s["nl"])
    rev, status = reverse_map(nl, s["types"], MNL, out=(s["rev"], s["rev_status"]))
    return dict(list=nl.list, shift=nl.shift, counts=nl.counts, frac=nl.frac_wrapped, status=nl.status, rev=rev,
                rev_status=status)


def _run_dp_train(s):
    loss, grads = s["model"].loss_and_grads(s["batch"])
    # the flat gradient vectors of the embedding and the fitting nets (what a data-parallel trainer reduces)
    n = len(list(s["model"].emb.parameters()))
    return dict(loss=loss, emb=torch.cat([g.reshape(-1) for g in grads[:n] if g is not None]),
                fit=torch.cat([g.reshape(-1) for g in grads[n:] if g is not None]))


def _nep_call(s, **kw):
    from matpl_amd import nep
    p, cfg = s["packed"], s["cfg"]
    nb = nep.neighbors(p, cfg.rcut_radial, cfg.rcut_angular, s["T"], ri_dtype=s["dtype"])
    return s["model"](nb["NN_r"], nb["NL_r"], nb["Ri_r"], nb["NN_a"], nb["NL_a"], nb["Ri_a"], p["num_atoms"],
                      p["atom_type_map"], **kw)


def _run_nep_eval(s):
    E, Ei, F, V = s["replay"].replay() if "replay" in s else _nep_call(s, create_graph=False)
    return dict(E=E.detach(), Ei=Ei.detach(), F=F.detach(), V=V.detach())


def _run_nep_train(s):
    E, Ei, F, V = _nep_call(s, create_graph=True)
    El, Fl, Vl = s["labels"]
    n = s["natoms"]
    loss = (((E[:, 0] - El) / n) ** 2).mean() + ((F - Fl) ** 2).mean() + (((V - Vl) / n[:, None]) ** 2).mean()
    return dict(loss=loss.detach(), grads=list(torch.autograd.grad(loss, s["params"])))


def _run_dp_ops(s):
    from matpl_amd.neighbor import env_mat
    ops = torch.ops.CalcOps_cuda
    Ri, Ri_d = env_mat(s["image_dr"], s["types"], s["davg"], s["dstd"], RS, RC)
    N, S = Ri.shape[1:3]
    Ri_d = Ri_d.view(1, N, S * 4, 3)
    nghost = torch.zeros((), dtype=torch.int64)
    F = ops.calculateForce(s["list0"], s["dE"], Ri_d, s["F0"], nghost)[0]
    V, AV = ops.calculateVirial(s["list0"], s["dE"], s["rij"], Ri_d, nghost)
    g, = torch.autograd.grad([F, V], [s["dE"]], [s["gF"], s["gV"]])
    return dict(Ri=Ri, Ri_d=Ri_d, F=F.detach(), V=V.detach(), AV=AV, dE=g)


_RUN = dict(dp_eval=_run_dp_eval, dp_rebuild=_run_dp_rebuild, dp_train=_run_dp_train, nep_eval=_run_nep_eval,
            nep_train=_run_nep_train, dp_ops=_run_dp_ops)

# -------------------------------------------------------------------------------------- work, tolerance


def _neighbors(case, rc):
    if "system" in case and case["system"] in ("cu", "hfo2", "sic"):
        density = {"cu": 4 / 3.615 ** 3, "hfo2": 12 / 5.08 ** 3, "sic": 8 / 4.36 ** 3}[case["system"]]
    else:
        density = DENSITY["lgps" if case["kind"] == "dp_train" else "alloy"]
    return density * 4.0 / 3.0 * math.pi * rc ** 3


def work(case):
    """Every input read once and every output written once, and the model's arithmetic (a multiply-add is two)."""
    N, kind = _natoms(case), case["kind"]
    fb = 4 if case.get("dtype") == "f32" else 8
    if kind == "dp_rebuild":
        T = DP_T[case["system"]]
        return dict(bytes=N * (24 + 4 + 24 + 4 * T + 3 * 4 * T * MNL), flops=N * _neighbors(case, RC + SKIN) * 20)
    if kind == "dp_ops":
        S = DP_T[case["system"]] * DP_M[case["system"]]
        # image_dr and dE read, Ri and Ri_d written, Rij and the list read, dE's gradient written
        return dict(bytes=N * S * (4 + fb * (4 + 4 + 4 + 12 + 3 + 4)) + N * fb * (3 * 3 + 9),
                    flops=N * _neighbors(case, RC) * 150)
    if kind in ("dp_eval", "dp_train"):
        n_in = N * _neighbors(case, RC)
        n_list = N * _neighbors(case, RC + SKIN) if kind == "dp_eval" else n_in
        # per neighbor: the embedding net or the table forward, and its derivative; per atom the fitting net
        # (400-50-50-50-1, forward and input gradient) and the descriptor products
        net = 2 * (25 + 2 * 625) if case.get("embedding") != "table" else 2 * 25 * 3
        per_pair, per_atom = net + 200, 2 * (20000 + 5000 + 50) + 2 * 6400
        flops = 2.0 * (n_in * per_pair + N * per_atom)
        if kind == "dp_train":
            flops *= 2.0
        # list and shift entries and the reverse map, positions and types read; energies and forces written
        return dict(bytes=n_list * 12 + N * (24 + 4 + 4 + 12), flops=flops)
    nr, na = N * _neighbors(case, NEP_RC), N * _neighbors(case, NEP_RCA)
    flops = nr * (13 * 5 * 2 + 40) + na * (13 * 5 * 2 + 5 * 24 * 2 + 60) + N * 30 * 30 * 4
    # positions and types read, energies and forces written; the lists are the path's own affair
    return dict(bytes=N * (24 + 8 + 4 * fb), flops=flops * (2.0 if kind == "nep_eval" else 6.0))


def tolerance(case):
    # about four times the largest error against 64 bits that was measured over these ranges
    kind = case["kind"]
    if kind == "dp_rebuild":
        return "exact"
    if kind in ("dp_eval", "dp_train"):
        if case["precision"] == "bf16":
            return {"rel": 2.5e-2, "max": 0.6}        # measured 6.4e-3
        return {"rel": 8e-6}                          # measured 1.8e-6
    if case["dtype"] == "f32":
        return {"rel": 8e-6}                          # measured 1.5e-6
    return {"rel": 1e-13}                             # measured 7.4e-15 (cancellation varies with the sizes)


# --------------------------------------------------------------------- the same results in 64 bits, plain torch


def _pairs(lat, pos, rc):
    """Every ordered pair within rc under periodic images: (i, j, image shift in A), chunk by chunk over i."""
    L = _dev(lat)
    height = 1.0 / np.linalg.norm(np.linalg.inv(lat), axis=0)
    frac = _dev(pos) @ torch.linalg.inv(L)
    N = frac.shape[0]
    x = frac @ L
    minimum = bool((height >= 2 * rc).all())
    if minimum:
        images = torch.zeros((1, 3), dtype=torch.float64, device=DEV)
    else:
        frac_range = float((frac.max(0)[0] - frac.min(0)[0]).max())
        k = [int(math.ceil(rc / h + frac_range)) for h in height]
        images = torch.cartesian_prod(*[torch.arange(-c, c + 1, dtype=torch.float64, device=DEV) for c in k])
    step = max(1, 40_000_000 // (N * len(images)))
    out = []
    for a in range(0, N, step):
        d = frac[None, :, :] - frac[a:a + step, None, :]
        if minimum:
            n = -torch.round(d).unsqueeze(2)
        else:
            n = images.expand(d.shape[0], N, -1, 3)
        r2 = ((d.unsqueeze(2) + n) @ L).square().sum(-1)
        i, j, q = torch.nonzero((r2 < rc * rc) & (r2 > 1e-10), as_tuple=True)
        out.append((i + a, j, n[i, j, q] @ L))
    return x, torch.cat([o[0] for o in out]), torch.cat([o[1] for o in out]), torch.cat([o[2] for o in out])


def _all_pairs(frames, rc):
    """The frames' pairs packed along the atom axis: dR of each pair, its atoms, and each atom's frame."""
    dR, ii, jj, base, frame = [], [], [], 0, []
    for k, (lat, pos, _) in enumerate(frames):
        x, i, j, s = _pairs(lat, pos, rc)
        dR.append(x[j] - x[i] + s)
        ii.append(i + base)
        jj.append(j + base)
        base += len(pos)
        frame.append(torch.full((len(pos),), k, dtype=torch.int64, device=DEV))
    return torch.cat(dR), torch.cat(ii), torch.cat(jj), torch.cat(frame)


def _dp_energy(dR, i, j, frame, types, params, davg, dstd, m, listed_types):
    """Per-atom DP energies as a function of the pairs' displacements and the nets' parameters."""
    emb, fit = params
    T, N = len(fit), types.shape[0]
    r = dR.square().sum(-1).sqrt()
    u = (r - RS) / (RC - RS)
    sw = torch.where(r < RS, torch.ones_like(r), u ** 3 * (-6 * u * u + 15 * u - 10) + 1)
    s = sw / r
    raw = torch.cat([s[:, None], s[:, None] * dR / r[:, None]], -1)
    ti = types[i]
    Ri = (raw - davg[ti]) / dstd[ti]
    pad = -davg / dstd

    def net(layers, x):
        for k, (W, b, _) in enumerate(layers):
            h = torch.tanh(x @ W + b)
            x = h + x if k else h
        return x
    A = torch.zeros((N, 4, 25), dtype=torch.float64, device=DEV)
    for a in range(T):
        for t in range(T):
            at = types == a
            sel = torch.nonzero((ti == a) & (types[j] == t)).reshape(-1)
            G = net(emb[a * T + t], Ri[sel, 0:1])
            Rs = Ri[sel]
            A = A + torch.stack([torch.zeros((N, 25), dtype=torch.float64, device=DEV).index_add(
                0, i[sel], Rs[:, c:c + 1] * G) for c in range(4)], 1)
            n = torch.bincount(i[sel], minlength=N)
            empty = (at & listed_types[:, t]) * (m - n).to(torch.float64)
            A = A + empty[:, None, None] * (pad[a][:, None] * net(emb[a * T + t], pad[a, 0].view(1, 1)))
    A = A / (m * listed_types.sum(1).to(torch.float64))[:, None, None]
    D = (A.transpose(1, 2) @ A[:, :, :16]).reshape(N, 400)
    Ei = torch.zeros(N, dtype=torch.float64, device=DEV)
    for a in range(T):
        at = torch.nonzero(types == a).reshape(-1)
        x = D[at]
        for k, (W, b, rdt) in enumerate(fit[a]):
            z = x @ W + b
            if k == len(fit[a]) - 1:
                x = z
            else:
                h = torch.tanh(z)
                x = h if k == 0 else h * rdt + x
        Ei = Ei.index_copy(0, at, x.reshape(-1))
    return Ei


def _leaves(nets, grad):
    return [[tuple(None if x is None else _dev(x).requires_grad_(grad) for x in layer) for layer in net]
            for net in nets]


def _force_virial(g, dR, i, j, frame, natoms, nframes):
    F = torch.zeros((natoms, 3), dtype=torch.float64, device=DEV).index_add(0, i, g).index_add(0, j, -g)
    W = -(g[:, :, None] * dR.detach()[:, None, :]).reshape(-1, 9)
    return F, torch.zeros((nframes, 9), dtype=torch.float64, device=DEV).index_add(0, frame[i], W)


def _exact_dp_eval(case, seed):
    frames = _frames(case, seed)
    emb, fit, davg, dstd = _dp_model(case["system"], seed)
    dR, i, j, frame = _all_pairs(frames, RC)
    dR.requires_grad_()
    types = _dev(frames[0][2], torch.int64)
    every = torch.ones((len(types), len(fit)), dtype=torch.bool, device=DEV)
    Ei = _dp_energy(dR, i, j, frame, types, (_leaves(emb, False), _leaves(fit, False)), _dev(davg), _dev(dstd),
                    DP_M[case["system"]], every)
    g, = torch.autograd.grad(Ei.sum(), dR)
    F, V = _force_virial(g, dR, i, j, frame, len(types), 1)
    return dict(Ei=Ei.detach(), F=F, V=V, status=None)


def _exact_dp_rebuild(case, seed):
    (lat, pos, _), = _frames(case, seed)
    f = _dev(pos @ np.linalg.inv(lat))
    return dict(list=None, shift=None, counts=None, frac=f - torch.floor(f), status=None, rev=None, rev_status=None)


def _exact_dp_train(case, seed):
    frames = _frames(case, seed)
    emb, fit, davg, dstd = _dp_model("lgps", seed)
    params = (_leaves(emb, True), _leaves(fit, True))
    dR, i, j, frame = _all_pairs(frames, RC)
    dR.requires_grad_()
    types = _dev(np.concatenate([f[2] for f in frames]), torch.int64)
    present = torch.zeros((len(frames), 4), dtype=torch.bool, device=DEV)
    present[frame, types] = True
    Ei = _dp_energy(dR, i, j, frame, types, params, _dev(davg), _dev(dstd), DP_M["lgps"], present[frame])
    g, = torch.autograd.grad(Ei.sum(), dR, create_graph=True)
    F, _ = _force_virial(g, dR, i, j, frame, len(types), len(frames))
    n = torch.bincount(frame).to(torch.float64)
    E = torch.zeros(len(frames), dtype=torch.float64, device=DEV).index_add(0, frame, Ei)
    El, Fl, _ = (_dev(x) for x in _labels(case, seed, [len(f[1]) for f in frames]))
    loss = (((E - El) / n) ** 2).mean() + ((F - Fl) ** 2).mean()
    # per net its weights, then its biases, then its residual scales
    flat = [[layer[c] for net in nets for c in range(3) for layer in net if layer[c] is not None]
            for nets in params]
    grads = torch.autograd.grad(loss, flat[0] + flat[1])
    k = len(flat[0])
    return dict(loss=loss.detach(), emb=torch.cat([x.reshape(-1) for x in grads[:k]]),
                fit=torch.cat([x.reshape(-1) for x in grads[k:]]))


_C3B = [0.238732414637843, 0.119366207318922, 0.119366207318922, 0.099471839432435, 0.596831036594608,
        0.596831036594608, 0.149207759148652, 0.149207759148652, 0.139260575205408, 0.104445431404056,
        0.104445431404056, 1.044454314040563, 1.044454314040563, 0.174075719006761, 0.174075719006761,
        0.011190581936149, 0.223811638722978, 0.223811638722978, 0.111905819361489, 0.111905819361489,
        1.566681471060845, 1.566681471060845, 0.195835183882606, 0.195835183882606]
_C4B = [-0.007499480826664, -0.134990654879954, 0.067495327439977, 0.404971964639861, -0.809943929279723]


def _radial(r, c, rc):
    """g_n(r) of each pair from its coefficients c [P, n, k] on the Chebyshev basis."""
    fc = 0.5 * torch.cos(math.pi * r / rc) + 0.5
    x = 2.0 * (r / rc - 1.0) ** 2 - 1.0
    t = [torch.ones_like(r), x]
    while len(t) < c.shape[-1]:
        t.append(2.0 * x * t[-1] - t[-2])
    f = (torch.stack(t, -1) + 1.0) * 0.5 * fc[:, None]
    return (c @ f[:, :, None])[:, :, 0]


def _harmonics(u):
    x, y, z = u.unbind(-1)
    x2, y2, z2 = x * x, y * y, z * z
    d = x2 - y2
    return torch.stack([
        z, x, y, 3 * z2 - 1, x * z, y * z, d, 2 * x * y,
        (5 * z2 - 3) * z, (5 * z2 - 1) * x, (5 * z2 - 1) * y, d * z, 2 * x * y * z, (x2 - 3 * y2) * x,
        (3 * x2 - y2) * y,
        (35 * z2 - 30) * z2 + 3, (7 * z2 - 3) * x * z, (7 * z2 - 3) * y * z, (7 * z2 - 1) * d,
        (7 * z2 - 1) * x * y * 2, (x2 - 3 * y2) * x * z, (3 * x2 - y2) * y * z, d * d - 4 * x2 * y2,
        4 * x * y * d], -1)


def _nep_energy(dR, i, j, types, c2, c3, qs, fit):
    N = types.shape[0]
    r = dR.square().sum(-1).sqrt()
    zero = torch.zeros((N, 5), dtype=torch.float64, device=DEV)
    q = [zero.index_add(0, i, _radial(r, c2[types[i], types[j]], NEP_RC))]
    near = torch.nonzero(r < NEP_RCA).reshape(-1)
    ra, ia, ja = r[near], i[near], j[near]
    g = _radial(ra, c3[types[ia], types[ja]], NEP_RCA)
    b = _harmonics(dR[near] / ra[:, None])
    s = torch.zeros((N, 5, 24), dtype=torch.float64, device=DEV).index_add(0, ia, g[:, :, None] * b[:, None, :])
    w = _dev([c if k in (0, 3, 8, 15) else 2 * c for k, c in enumerate(_C3B)])
    sq = w * s * s
    q += [sq[..., a:e].sum(-1) for a, e in ((0, 3), (3, 8), (8, 15), (15, 24))]
    q.append(_C4B[0] * s[..., 3] ** 3 + _C4B[1] * s[..., 3] * (s[..., 4] ** 2 + s[..., 5] ** 2) +
             _C4B[2] * s[..., 3] * (s[..., 6] ** 2 + s[..., 7] ** 2) +
             _C4B[3] * s[..., 6] * (s[..., 5] ** 2 - s[..., 4] ** 2) + _C4B[4] * s[..., 4] * s[..., 5] * s[..., 7])
    x = torch.cat(q, -1) * qs
    Ei = torch.zeros(N, dtype=torch.float64, device=DEV)
    for t, ((W0, b0, _), (W1, b1, _)) in enumerate(fit):
        at = torch.nonzero(types == t).reshape(-1)
        Ei = Ei.index_copy(0, at, (torch.tanh(x[at] @ W0 + b0) @ W1 + b1).reshape(-1))
    return Ei


def _exact_nep(case, seed):
    train = case["kind"] == "nep_train"
    frames = _frames(case, seed)
    c2, c3, qs, fit = _nep_model(2 if case.get("system") == "sic" else 4, seed)
    c2, c3 = _dev(c2).requires_grad_(train), _dev(c3).requires_grad_(train)
    fit = _leaves(fit, train)
    dR, i, j, frame = _all_pairs(frames, NEP_RC)
    dR.requires_grad_()
    types = _dev(np.concatenate([f[2] for f in frames]), torch.int64)
    Ei = _nep_energy(dR, i, j, types, c2, c3, _dev(qs), fit)
    g, = torch.autograd.grad(Ei.sum(), dR, create_graph=train)
    F, V = _force_virial(g, dR, i, j, frame, len(types), len(frames))
    E = torch.zeros(len(frames), dtype=torch.float64, device=DEV).index_add(0, frame, Ei)
    if not train:
        return dict(E=E.detach()[:, None], Ei=Ei.detach(), F=F, V=V)
    n = torch.bincount(frame).to(torch.float64)
    El, Fl, Vl = (_dev(x) for x in _labels(case, seed, [len(f[1]) for f in frames]))
    loss = (((E - El) / n) ** 2).mean() + ((F - Fl) ** 2).mean() + (((V - Vl) / n[:, None]) ** 2).mean()
    params = [c2, c3] + [layer[c] for net in fit for c in range(2) for layer in net]
    return dict(loss=loss.detach(), grads=list(torch.autograd.grad(loss, params)))


def _exact_dp_ops(case, seed):
    s = _prepare_dp_ops(case, seed)          # for the inputs; what follows is plain torch
    f8 = torch.float64
    idr = s["image_dr"][0].to(f8)
    N, S = idr.shape[:2]
    x = idr[..., 1:].clone().requires_grad_()
    inside = idr[..., 0] > 0
    r = torch.where(inside[..., None], x, torch.ones_like(x)).square().sum(-1).sqrt()
    u = (r - RS) / (RC - RS)
    sw = torch.where(r < RS, torch.ones_like(r), torch.where(r < RC, u ** 3 * (-6 * u * u + 15 * u - 10) + 1,
                                                              torch.zeros_like(r)))
    sr = torch.where(inside, sw / r, torch.zeros_like(r))
    raw = torch.cat([sr[..., None], sr[..., None] * x / r[..., None]], -1)
    ti = s["types"].long()
    av, sd = (s[k].to(f8).view(-1, S, 4)[ti] for k in ("davg", "dstd"))
    Ri = (raw - av) / sd
    Rd = torch.stack([-torch.autograd.grad(raw[..., w].sum(), x, retain_graph=True)[0] / sd[..., w:w + 1]
                      for w in range(4)], -2).detach()
    dE = s["dE"].detach().to(f8).view(N, S, 4)
    lst = s["list0"].view(N, S).long()
    at = torch.nonzero(lst.reshape(-1) >= 0).reshape(-1)
    j = lst.reshape(-1)[at]
    f = (dE[..., None] * Rd).sum(-2)
    rij = s["rij"][0].to(f8)
    outer = (f[..., :, None] * rij[..., None, :]).reshape(-1, 9)
    F = s["F0"][0].to(f8).index_add(0, j, f.reshape(-1, 3)[at])
    AV = torch.zeros((N, 9), dtype=f8, device=DEV).index_add(0, j, outer[at])
    gF, gV = s["gF"][0].to(f8), s["gV"].to(f8).view(3, 3)
    back = -gF[:, None, :].expand(N, S, 3).clone()
    back.view(-1, 3)[at] += gF[j] + rij.reshape(-1, 3)[at] @ gV.T
    return dict(Ri=Ri.detach()[None], Ri_d=Rd.view(1, N, S * 4, 3), F=F[None], V=AV.sum(0)[None], AV=AV[None],
                dE=(Rd * back[..., None, :]).sum(-1).view(1, N, 1, S * 4))


_EXACT = dict(dp_eval=_exact_dp_eval, dp_rebuild=_exact_dp_rebuild, dp_train=_exact_dp_train, nep_eval=_exact_nep,
              nep_train=_exact_nep, dp_ops=_exact_dp_ops)


def exact(case, seed):
    out = _EXACT[case["kind"]](case, seed)
    torch.cuda.empty_cache()
    return out
