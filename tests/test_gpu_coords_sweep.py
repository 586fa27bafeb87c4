"""Sweeps over a never-stored cost at the edges of their tiles and of the split of
their work, against the same iterations in plain FP64 torch."""
import math

import pytest

pytestmark = pytest.mark.gpu


def _reference(torch, x, y, G, lam1, lam2, eps, n_iter):
    C = torch.zeros((len(x), len(y)), dtype=torch.float64, device='cuda')
    for k in range(x.shape[1]):
        t = x[:, k, None] - y[None, :, k]
        C.addcmul_(t, t)
    s = C.flatten().sort().values
    C /= 0.5 * (s[(s.numel() - 1) // 2] + s[s.numel() // 2])
    del s
    f = torch.zeros(C.shape[0], dtype=torch.float64, device='cuda')
    g = torch.zeros(C.shape[1], dtype=torch.float64, device='cuda')
    logq = torch.log(G.mean())
    for _ in range(n_iter):
        lse = torch.logsumexp((g[None, :] - C) / eps, 1)
        f = lam1 / (lam1 + eps) * eps * (torch.log(G) + math.log(len(g)) - lse)
        lse = torch.logsumexp((f[:, None] - C) / eps, 0)
        g = lam2 / (lam2 + eps) * eps * (logq + math.log(len(f)) - lse)
    R = torch.exp((f[:, None] + g[None, :] - C) / eps)
    return f, g, R.sum(1) / len(g)


# one unit; a last unit of rows and a last tile of columns that are nearly empty; fewer units than
# CUs; more units than places, so that units are cut and their sums handed over, with the last
# split shorter (8300 x 8450, 8 splits of 34 tiles) and with another split per direction (16500 x 900)
@pytest.mark.parametrize('n_i,n_j,d,terms', [(1, 1, 3, 6), (33, 130, 5, 3), (129, 257, 50, 6), (1500, 3001, 33, 6),
                                             (8300, 8450, 20, 6), (8300, 8450, 17, 3), (16500, 900, 70, 6),
                                             (9000, 8200, 100, 3)])
def test_sweeps_match_fp64(n_i, n_j, d, terms):
    import torch
    from wot_amd.ot import large
    gen = torch.Generator(device='cuda').manual_seed(n_i + d)
    x = torch.randn(n_i, d, dtype=torch.float64, device='cuda', generator=gen)
    y = torch.randn(n_j, d, dtype=torch.float64, device='cuda', generator=gen) + 0.2
    G = torch.exp(0.3 * torch.randn(n_i, dtype=torch.float64, device='cuda', generator=gen))
    eps, lam1, lam2, n_iter = 0.5, 1.0, 50.0, 4
    args = dict(lambda1=lam1, lambda2=lam2, epsilon=eps, epsilon0=eps, scaling_iter=n_iter, extra_iter=0,
                inner_iter_max=50, tau=1e4, terms=terms, want_row_sums=True)
    r = large.transport_stablev2_coords(x, y, G, **args)
    f, g, rows = _reference(torch, x, y, G, lam1, lam2, eps, n_iter)
    # Per sweep: exponents of at most 40 rounded at 2^-24, exp2 to 1 ulp and at most 128 FP32 additions
    # per lane: ln S is off by at most 40 ln 2 2^-24 + 130 * 2^-24 = 1e-5.  With 3 terms the cross
    # term (at most 5 here) also lacks 2^-16 of itself, twice over eps: 3.1e-4.  The errors of the
    # 2 n_iter sweeps add up at most (an iteration is non-expansive), each times eps.
    ln_s = 1e-5 + (3.1e-4 if terms == 3 else 0.0)
    tol = 2 * n_iter * ln_s * eps
    assert float((r.f - f).abs().max()) < tol
    assert float((r.g - g).abs().max()) < tol
    # a row sum is exp of the potentials' errors over eps and of its own sweep's
    assert float((r.row_sums / rows - 1).abs().max()) < 2 * tol / eps + ln_s
    again = large.transport_stablev2_coords(x, y, G, **args)
    assert torch.equal(r.f, again.f) and torch.equal(r.g, again.g) and torch.equal(r.row_sums, again.row_sums)


# tau so low that absorptions follow each other, and the default that hardly ever fires; rows of a
# workgroup's 32 and of several, one column more than a tile
@pytest.mark.parametrize('n_i,n_j,tau', [(31, 33, 3.0), (129, 65, 20.0), (257, 300, 1e4)])
def test_gap_schedule_absorptions_match_oracle(n_i, n_j, tau):
    import numpy as np
    import wot_amd.ot as ot
    from oracle import ot_oracle as O
    from wot_amd.synthetic import day_pair
    dp = day_pair(n_i, n_j, dim=9, n_components=4, seed=n_i)
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, batch_size=5, tolerance=1e-8, tau=tau, epsilon0=1.0,
               max_iter=1e7)
    st, so = {}, {}
    res = ot.optimal_transport_duality_gap(None, dp.growth, coords=(dp.x, dp.y), stats=st, **prm)
    Ro = O.optimal_transport_duality_gap(O.default_cost_matrix(dp.x, dp.y), dp.growth, stats=so, **prm)
    # absorptions change nothing but the evolution check; exponents rounded at 2^-24 leave the plan
    # within 1e-5 and the checks at the same iteration or its neighbour
    assert abs(st['iterations'] - so['iterations']) <= 5
    assert abs(st['stabilisations'] - so['stabilisations']) <= abs(st['iterations'] - so['iterations'])
    R = res.dense().cpu().numpy()
    assert np.linalg.norm(R - Ro) / np.linalg.norm(Ro) <= 1e-5


# cut units whose sums do not come in time: rows with one and with several splits, both term counts
@pytest.mark.parametrize('n_i,n_j,d,terms', [(8300, 8450, 20, 6), (8300, 8450, 17, 3), (16500, 900, 70, 6)])
def test_sums_that_do_not_come_are_computed_again(n_i, n_j, d, terms):
    import ctypes
    import torch
    from wot_amd import _native
    from wot_amd.ot import device as dev
    gen = torch.Generator(device='cuda').manual_seed(n_i + d)
    x = torch.randn(n_i, d, dtype=torch.float64, device='cuda', generator=gen)
    y = torch.randn(n_j, d, dtype=torch.float64, device='cuda', generator=gen) + 0.2
    G = torch.exp(0.3 * torch.randn(n_i, dtype=torch.float64, device='cuda', generator=gen))
    L, p = _native.lib(), dev._ptr
    ws = dev.workspace(torch, L.wotk_fused_workspace_size(n_i, n_j, d), 'cuda')

    def solve(fn, *extra):
        out = [torch.empty(n, dtype=torch.float64, device='cuda') for n in (n_i, n_j, n_i, 1)]
        st = _native.Stats()
        _native.check(fn(p(x), p(y), n_i, n_j, d, p(G), 1.0, 50.0, 0.5, 3, 1e4, 0.5, 0, 50, terms,
                         *(p(t) for t in out), p(ws), ws.numel(), ctypes.byref(st),
                         ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), *extra))
        return out

    for a, b in zip(solve(L.wotk_transport_stablev2_coords), solve(L.wotk_probe_stablev2_coords_limits, 0)):
        assert torch.equal(a, b)
