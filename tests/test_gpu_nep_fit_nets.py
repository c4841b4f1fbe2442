"""The NEP fitting kernels with one weight pointer per type (matpl_nep_fit_forward_nets / _backward_nets), forward
and first and second derivative, against float64 torch autograd: atoms counts around the block's 8 and the tile's 64,
weights above the forward's LDS budget (D = 35, H = 100 in double: 28 KB), an empty type. Tolerances as
tests/test_gpu_nep_fit.py: float64 1e-12, float32 2e-5 of the largest entry."""
import numpy as np
import pytest
import torch

from matpl_amd import nep as mn

pytestmark = pytest.mark.gpu

CASES = [(1, 1, 30, 30), (8, 1, 5, 3), (9, 2, 30, 30), (64, 1, 33, 31), (65, 3, 30, 32), (1000, 4, 35, 100),
         (20000, 2, 30, 30)]


@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 2e-5)])
@pytest.mark.parametrize("N,T,D,H", CASES)
def test_nets_entry(dev, dtype, tol, N, T, D, H):
    print(f"case nep fit nets {dtype} N={N} T={T} D={D} H={H}", flush=True)
    rng = np.random.default_rng(N + D)
    types = rng.integers(0, max(T - 1, 1), N)                    # the last of several types has no atom
    mk = lambda *s, sc=1.0: torch.tensor(rng.normal(size=s) * sc, dtype=dtype, device=dev).double()
    q, qs = mk(N, D, sc=0.7).requires_grad_(), mk(D)
    params = [x.requires_grad_() for _ in range(T)
              for x in (mk(D, H, sc=D ** -0.5), mk(H), mk(H, 1, sc=H ** -0.5), mk(1))]
    gE, gg = mk(N), mk(N, D)
    tm = torch.as_tensor(types, device=dev)
    E = torch.zeros(N, dtype=torch.float64, device=dev)
    for t in range(T):
        W0, b0, w1, b1 = params[4 * t:4 * t + 4]
        ix = torch.nonzero(tm == t).reshape(-1)
        E = E.index_put((ix,), (torch.tanh((q * qs)[ix] @ W0 + b0) @ w1 + b1).reshape(-1))
    (g,) = torch.autograd.grad(E.sum(), q, create_graph=True)
    want = [E, g] + list(torch.autograd.grad((E * gE).sum() + (g * gg).sum(), [q] + params, allow_unused=True))
    plan = mn.FitPlan([torch.nonzero(tm == t).reshape(-1) for t in range(T)], dtype == torch.float64, D, H, dev)
    qd = q.detach().to(dtype).requires_grad_()
    pd = [x.detach().to(dtype).requires_grad_() for x in params]
    Ed, gd = mn._NepFitNetsFn.apply(qd, qs.to(dtype), plan, *pd)
    got = [Ed, gd] + list(torch.autograd.grad((Ed * gE.to(dtype)).sum() + (gd * gg.to(dtype)).sum(), [qd] + pd))
    for k, (a, b) in enumerate(zip(got, want)):
        a = a.detach().double()
        b = torch.zeros_like(a) if b is None else b.detach()
        err = float((a - b).abs().max())
        assert err <= tol * max(float(b.abs().max()), 1.0), (k, err)
