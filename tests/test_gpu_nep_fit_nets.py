"""The NEP fitting kernels with one weight pointer per type (matpl_nep_fit_forward_nets / _backward_nets), forward
and first and second derivative, against float64 torch autograd: atoms counts around the block's 8 and the tile's 64,
enough atoms for two and four at a time (20,000 and 40,000) with remainders, weights that the forward stages in parts
(D = 56, H = 120 in double: 54 KB; D = 480, H = 8, whose rows leave less room), an empty type. Tolerances as
tests/test_gpu_nep_fit.py: float64 1e-12, float32 2e-5 of the largest entry. A parameter gradient is a sum of N terms
of order one, whose partial sums reach sqrt(N) whatever the total is; it takes at most 64 additions in a tile, N / 512
over tiles and 8 over groups, about 150 roundings of half an ulp of sqrt(N)."""
import numpy as np
import pytest
import torch

from matpl_amd import nep as mn

pytestmark = pytest.mark.gpu

CASES = [(1, 1, 30, 30), (8, 1, 5, 3), (9, 2, 30, 30), (64, 1, 33, 31), (65, 3, 30, 32), (1000, 4, 35, 100),
         (20000, 2, 30, 30), (40003, 3, 5, 10), (36001, 2, 56, 120), (700, 2, 480, 8), (9001, 1, 56, 64)]


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
        summed = 75 * torch.finfo(dtype).eps * N ** 0.5 if k >= 3 else 0.0
        assert err <= tol * max(float(b.abs().max()), 1.0) + summed, (k, err)
