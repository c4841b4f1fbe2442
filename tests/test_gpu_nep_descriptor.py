"""The NEP descriptor kernels (matpl_nep_feat, matpl_nep_descriptor) at the edges of their passes, against
the FP64 oracle's features and their torch autograd: lists of 0, 1, 63, 64, 65 and more entries, types in no
order, one type and many, the reference's default sizes and others up to the largest, 3-body alone and with
the 4- and 5-body terms.

Tolerances: the sums run over at most ~130 slots, 16 types x 20 basis functions and 24 harmonics of values of
order one; n terms added in any order are within n eps of the exact sum, n below 2,000 in every output, hence
2,000 eps of the largest entry (float 1.2e-4 (eps 6e-8), double 2.2e-13), measured far below."""
import numpy as np
import pytest
import torch

import oracle.nep as on
from matpl_amd import _lib
from matpl_amd.calcops import _ptr, _stream

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1.2e-4, torch.float64: 2.2e-13}
RC = 5.0


def _inputs(T, S, counts, seed):
    """Ri [N, S, 4] with |(x, y, z)| = r, some slots beyond the cutoff, NL with the given prefix lengths."""
    rng = np.random.default_rng(seed)
    N = len(counts)
    am = rng.integers(0, T, N)
    NL = np.full((N, S), -1, np.int64)
    Ri = np.zeros((N, S, 4))
    for i, c in enumerate(counts):
        NL[i, :c] = rng.integers(0, N, c)
        u = rng.normal(size=(c, 3))
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        r = rng.uniform(1.0, RC * 1.03, c)
        Ri[i, :c, 0] = r
        Ri[i, :c, 1:] = u * r[:, None]
    return am, NL, Ri, rng


def _close(got, want, dtype, what):
    want = want.detach()
    got = got.detach().cpu().double().reshape(want.shape)
    err = float((got - want).abs().max()) if want.numel() else 0.0
    assert err <= TOL[dtype] * max(float(want.abs().max()) if want.numel() else 0.0, 1e-3), (what, err)


CASES = [(1, 5, 13, (4, 2, 0), 70, [0, 1, 63, 64, 65, 70, 2, 0, 5]),
         (4, 5, 13, (4, 2, 1), 64, [64, 0, 17, 16, 15, 16, 1, 30, 33, 64]),
         (3, 3, 8, (4, 0, 0), 130, [130, 129, 7, 64, 65, 0]),
         (2, 8, 20, (4, 2, 1), 9, [9, 0, 4, 5, 3, 9, 9, 1]),
         (8, 5, 13, (2, 0, 0), 21, [21, 20, 3, 0, 21]),
         (2, 1, 16, (1, 0, 0), 40, [40, 8, 33]),
         (4, 4, 17, (4, 2, 0), 12, [12] * 23)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("angular", [0, 1])
@pytest.mark.parametrize("T,nm,nb,l,S,counts", CASES)
def test_descriptor_modes(dev, dtype, angular, T, nm, nb, l, S, counts):
    print(f"case descriptor {dtype} angular={angular} T={T} nm={nm} nb={nb} l={l} S={S} N={len(counts)}", flush=True)
    am, NL, Ri, rng = _inputs(T, S, counts, 100 * T + nb)
    N = len(counts)
    nf = nm * (l[0] + (l[1] > 0) + (l[2] > 0)) if angular else nm
    ld, col0 = nf + 3, 2
    c = rng.normal(size=(T, T, nm, nb)) * 0.3
    gq = rng.normal(size=(N, nf))
    gg = rng.normal(size=(N, S, 4)) * (NL >= 0)[..., None]
    if not angular:
        gg[..., 1:] = 0
    f32 = lambda a: torch.as_tensor(a).to(dtype).double()        # the values the kernels see, in FP64
    c_, Ri_, gq_ = f32(c).requires_grad_(), f32(Ri).requires_grad_(), f32(gq).requires_grad_()
    gg_ = f32(gg)
    if angular:
        q = on.angular_feats(c_, Ri_, NL, am, RC, *l)
    else:
        q = on.radial_feats(c_, Ri_, NL, am, RC)
    gc1, gRi = torch.autograd.grad(q, [c_, Ri_], gq_, create_graph=True)
    valid = torch.as_tensor(NL >= 0).unsqueeze(-1)
    gRi = torch.where(valid, gRi, torch.zeros_like(gRi))
    ggq, gc2 = torch.autograd.grad((gRi * gg_).sum(), [gq_, c_], retain_graph=True)
    # the same for gradients of model forces and of two frames' virials: q = gF[i] - gF[j] - gV x, gg = [q . u, q]
    gF, gV = f32(rng.normal(size=(N, 3))), f32(rng.normal(size=(2, 9)))
    frame = (torch.arange(N) >= N // 2).to(torch.int32)
    x, r = Ri_.detach()[..., 1:], Ri_.detach()[..., :1]
    qf = gF[:, None] - gF[torch.as_tensor(NL).clamp(min=0)] - (gV.view(2, 1, 3, 3)[frame.long()] @ x[..., None])[..., 0]
    ggf_ = torch.where(valid, torch.cat([(qf * x).sum(-1, keepdim=True) / torch.where(valid, r, 1.0), qf], -1), 0.0)
    ggq_f, gc2_f = torch.autograd.grad((gRi * ggf_).sum(), [gq_, c_])

    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev).to(dtype).contiguous()
    cd, Rd, gqd, ggd = d(c), d(Ri), torch.zeros((N, ld), dtype=dtype, device=dev), d(gg)
    gqd[:, col0:col0 + nf] = d(gq)
    NLd, amd = torch.as_tensor(NL, device=dev), torch.as_tensor(am, device=dev)
    gFd, gVd, frame = gF.to(dtype).to(dev), gV.to(dtype).to(dev), frame.to(dev)
    f64 = int(dtype == torch.float64)
    new = lambda *s: torch.full(s, float("nan"), dtype=dtype, device=dev)
    save = new(N, nm * 24 if angular else T * nb)

    def call(name, mode, *rest):
        _lib.call(name, f64, angular, mode, _ptr(cd), _ptr(Rd), _ptr(NLd), _ptr(amd), N, S, T, nm, nb, ld, col0, *l, RC,
                  *[_ptr(x) for x in rest], _stream())

    cut = lambda t: t[:, col0:col0 + nf]
    for name in ("matpl_nep_feat", "matpl_nep_descriptor"):
        feats = new(N, ld)
        if name == "matpl_nep_feat":
            call(name, 0, feats, save if angular else None, None, None, None, None, None)
            _close(cut(feats), q, dtype, "feats")
            g, gc = new(N, S, 4), torch.zeros_like(cd)
            call(name, 1, None, save, gqd, None, g, gc, None)
            _close(g, gRi, dtype, "gRi")
            _close(gc, gc1, dtype, "gc")
            gc, ggf = torch.zeros_like(cd), new(N, ld)
            call(name, 2, None, save, gqd, ggd, None, gc, ggf)
            _close(cut(ggf), ggq, dtype, "ggfeat")
            _close(gc, gc2, dtype, "gc second order")
        else:
            call(name, 0, feats, save, *[None] * 8)
            _close(cut(feats), q, dtype, "feats")
            assert torch.isnan(feats[:, :col0]).all() and torch.isnan(feats[:, col0 + nf:]).all()
            gc, ggf, gs = torch.zeros_like(cd), new(N, ld), new(N, nm * 24)
            call(name, 1, None, save, gqd, None, gFd, gVd, frame, gc, ggf, gs if angular else None)
            _close(cut(ggf), ggq_f, dtype, "ggfeat")
            # the second order's rest and the first order in one coefficient pass
            call(name, 2, None, save, gqd, gs if angular else None, *[None] * 3, gc, None, None)
            _close(gc, gc1 + gc2_f, dtype, "gc of both orders")
            if angular:
                gc = torch.zeros_like(cd)
                call(name, 2, None, save, None, gs, *[None] * 3, gc, None, None)
                gc3 = torch.zeros_like(cd)
                call(name, 2, None, save, gqd, gs, *[None] * 3, gc3, None, None)
                _close(gc3 - gc, gc1, dtype, "gc without gs")
