"""Force and virial scatter where the block's row table fills up, wraps and is left unused, against float64 sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("B,N,S,ng,rows", [
    (1, 1, 1, 0, 1), (2, 7, 9, 0, 7), (1, 8, 33, 5, 13), (3, 9, 64, 0, 2),      # one block, its edges
    (1, 700, 130, 40, 740),         # about 1040 slots a block over 740 rows: the table overflows
    (1, 4000, 70, 0, 4000),         # hardly any row twice in a block
    (1, 20, 300, 0, 1),             # every slot the same row
    (300, 2, 8, 1, 3), (77, 1, 17, 0, 1),       # frames of few slots: directly up to 16 a block, by the table from 17 on
])
def test_scatter_row_sums(B, N, S, ng, rows, dtype):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from matpl_amd import _lib
    from matpl_amd.calcops import _ptr, _stream
    g = torch.Generator().manual_seed(N * S)
    r = lambda *shape: torch.randn(*shape, generator=g, dtype=torch.float64).to(dtype).cuda()
    NA = N + ng
    nl = torch.randint(-1, rows, (B, N, S), generator=g, dtype=torch.int32).cuda()
    dE, Rid, Rij, Fc = r(B, N, S, 4), r(B, N, S, 4, 3), r(B, N, S, 3), r(B, N, 3)
    sfx = "f64" if dtype == torch.float64 else "f32"
    F = torch.empty(B, NA, 3, dtype=dtype, device="cuda")
    AV = torch.empty(B, NA, 9, dtype=dtype, device="cuda")
    V = torch.empty(B, 9, dtype=dtype, device="cuda")
    ws = torch.empty(B * 256 * 9, dtype=dtype, device="cuda")
    print(f"B={B} N={N} S={S} {sfx}", flush=True)
    _lib.call(f"matpl_dp_force_{sfx}", _ptr(nl), _ptr(dE), _ptr(Rid), _ptr(Fc), B, N, S, ng, _ptr(F), _stream())
    _lib.call(f"matpl_dp_virial_{sfx}", _ptr(nl), _ptr(dE), _ptr(Rij), _ptr(Rid), B, N, S, ng, _ptr(V), _ptr(AV),
              _ptr(ws), ws.numel(), _stream())
    f = (dE.double().unsqueeze(-1) * Rid.double()).sum(3)
    w = (f.unsqueeze(-1) * Rij.double().unsqueeze(3)).reshape(B, N * S, 9)
    used = (nl >= 0).reshape(B, N * S)
    row = nl.clamp(min=0).long().reshape(B, N * S)
    # a term is a sum of 4 products (and one more product), a row at most N S of them added one by one
    # (plus the centre's force): errors below (terms + 8) eps times the sum of the magnitudes
    eps = torch.finfo(dtype).eps / 2
    for b in range(B):
        k, j = used[b], row[b][used[b]]
        n = torch.zeros(NA, 1, dtype=torch.float64, device="cuda").index_add(0, j, torch.ones_like(j).double()[:, None])
        mag = (dE.double().unsqueeze(-1) * Rid.double()).abs().sum(3)
        want = torch.zeros(NA, 3, dtype=torch.float64, device="cuda").index_add(0, j, f[b].reshape(-1, 3)[k])
        size = torch.zeros_like(want).index_add(0, j, mag[b].reshape(-1, 3)[k])
        want[:N] += Fc[b].double()
        size[:N] += Fc[b].double().abs()
        assert bool(((F[b].double() - want).abs() <= (n + 8) * eps * size).all())
        magw = (mag.unsqueeze(-1) * Rij.double().abs().unsqueeze(3)).reshape(B, N * S, 9)
        want = torch.zeros(NA, 9, dtype=torch.float64, device="cuda").index_add(0, j, w[b][k])
        size = torch.zeros_like(want).index_add(0, j, magw[b][k])
        assert bool(((AV[b].double() - want).abs() <= (n + 8) * eps * size).all())
