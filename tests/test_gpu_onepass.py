"""The one-read iteration (pairs from 2^23 entries) against the two sweeps the
no-allocation entry point keeps, at the edges of its column chunks and row
steps, and where rows and columns leave its FP32 range."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# columns at and around the 3840-column chunks (1 to 5 chunks, 4 / 2 / 1 rows per step), the largest
# width, rows that do not divide by the 256 workgroups or by the rows of a step, one row less than a round
SHAPES = [(2049, 4095), (2500, 4096), (2051, 4097), (1100, 8192), (1023, 8193), (701, 12289), (513, 16384),
          (515, 16389), (415, 20288), (9000, 1001)]
# lanes sum in another order (FP32 partial sums of at most 60 terms each, then FP64): the plan moves by a few
# 1e-9 per sum, as between the sweep's own tile variants (1e-6 is what those are held to)
TOL = 1e-6


def _run(fn, cost, G, prm, ws=None):
    import torch
    from wot_amd import _native
    from wot_amd.ot import device as dev
    n_i, n_j = cost.shape
    f = torch.empty(n_i, dtype=torch.float64, device='cuda')
    g = torch.empty(n_j, dtype=torch.float64, device='cuda')
    p = dev._ptr
    st = _native.Stats()
    args = [p(cost.C), cost.ldc, p(cost.CT), cost.ldct, n_i, n_j, p(G), prm['lambda1'], prm['lambda2'], prm['epsilon'],
            prm['scaling_iter'], 1e4, prm['epsilon0'], prm['extra_iter'], prm['inner_iter_max'], None, n_j, None, p(f),
            p(g)]
    if ws is not None:
        args += [p(ws), ws.numel()]
    args += [ctypes.byref(st), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)]
    _native.check(fn(*args))
    return f, g, st.epsilon_final


def _both(x, y, G, **kw):
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    from wot_amd.ot import device as dev
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, epsilon0=1.0, scaling_iter=150, extra_iter=20,
               inner_iter_max=50)
    prm.update(kw)
    cost = ot.DeviceCost.from_coordinates(x, y)
    Gd = torch.from_numpy(np.ascontiguousarray(G)).cuda()
    L = _native.lib()
    ws = dev.workspace(torch, L.wotk_solver_workspace_size(*cost.shape), 'cuda')
    one = _run(L.wotk_transport_stablev2, cost, Gd, prm, ws)
    two = _run(L.wotk_transport_stablev2_noalloc, cost, Gd, prm)
    return cost, one, two


def _plan(cost, r):
    import torch
    return torch.exp((r[0][:, None] + r[1][None, :] - cost.dense().double()) / r[2])


@pytest.mark.parametrize('n_i,n_j', SHAPES)
def test_one_read_iteration_matches_two_sweeps(n_i, n_j):
    import torch
    from wot_amd.synthetic import day_pair
    dp = day_pair(n_i, n_j, dim=30, n_components=5, seed=n_i)
    cost, one, two = _both(dp.x, dp.y, dp.growth)
    a, b = _plan(cost, one), _plan(cost, two)
    assert float((a - b).norm() / b.norm()) < TOL
    for d in (0, 1):
        assert float(((a.sum(d) - b.sum(d)).abs() / b.sum(d)).max()) < TOL


@pytest.mark.parametrize('eps', [0.05, 0.003])
def test_rows_and_columns_out_of_range(eps):
    """Outlier cells on both sides and a first eps far below the cost's scale: first sums under 2^-40."""
    import torch
    rng = np.random.default_rng(7)
    x, y = rng.standard_normal((2100, 30)), rng.standard_normal((4100, 30))
    x[::97] *= 12.0
    y[5::113] *= 15.0
    G = np.exp(0.3 * rng.standard_normal(2100))
    cost, one, two = _both(x, y, G, epsilon=eps, epsilon0=eps, scaling_iter=0, extra_iter=30)
    for a, b in zip(one[:2], two[:2]):
        assert torch.isfinite(a).all()
        # potentials of the scale of the cost; both paths round exponents of up to |C| / eps at 2^-24
        assert float((a - b).abs().max()) < 1e-6 * float(b.abs().max())


def test_zero_and_nan_growth_travel_as_in_the_sweeps():
    import torch
    rng = np.random.default_rng(8)
    x, y = rng.standard_normal((2100, 30)), rng.standard_normal((4100, 30))
    G = np.ones(2100)
    G[17] = 0.0
    _, one, two = _both(x, y, G, scaling_iter=0, extra_iter=3)
    assert torch.equal(torch.isinf(one[0]), torch.isinf(two[0])) and bool(torch.isinf(one[0])[17])
    assert float((one[1] - two[1]).abs().max()) < 1e-7 * float(two[1].abs().max())
    G[17] = np.nan
    _, one, two = _both(x, y, G, scaling_iter=0, extra_iter=2)
    for a, b in zip(one[:2], two[:2]):
        assert torch.equal(torch.isnan(a), torch.isnan(b))


@pytest.mark.parametrize('n_i,n_j,kw', [(2100, 4100, {}), (4300, 2049, dict(batch_size=3, epsilon=0.1)),
                                        (2100, 4100, dict(tau=2.0)), (2100, 4100, dict(tau=2.0, max_iter=23)),
                                        (2100, 4100, dict(max_iter=35)), (2100, 4100, dict(max_iter=452))])
def test_duality_gap_schedule_matches_fp64(n_i, n_j, kw):
    """Counts and plan of the schedule with the tau check inside the iteration, batches queued ahead of the
    evolution checks and the one-read gap pass, against the FP64 restatement on the device."""
    import torch
    import wot_amd.ot as ot
    from wot_amd import plain_gpu
    from wot_amd.synthetic import day_pair
    dp = day_pair(n_i, n_j, dim=30, n_components=5, seed=n_j)
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, batch_size=5, tolerance=1e-8, tau=1e4, epsilon0=1.0,
               max_iter=1e7)
    prm.update(kw)
    cost = ot.DeviceCost.from_coordinates(dp.x, dp.y)
    st, so = {}, {}
    R = ot.optimal_transport_duality_gap(cost, dp.growth, stats=st, device_out=True, **prm)
    ref = plain_gpu.optimal_transport_duality_gap(cost.dense().double(), torch.from_numpy(dp.growth).cuda(), stats=so,
                                                  **prm)
    assert st['iterations'] == so['iterations']
    assert bool(st['max_iter_reached']) == (st['iterations'] >= prm['max_iter'])
    if 'stabilisations' in so:
        assert st['stabilisations'] == so['stabilisations']
    assert float((R - ref).norm() / ref.norm()) < 1e-6


def _both_of_matrix(C, G, **kw):
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    from wot_amd.ot import device as dev
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, epsilon0=1.0, scaling_iter=150, extra_iter=20,
               inner_iter_max=50)
    prm.update(kw)
    cost = ot.DeviceCost.from_matrix(C)
    Gd = torch.from_numpy(np.ascontiguousarray(G)).cuda()
    L = _native.lib()
    ws = dev.workspace(torch, L.wotk_solver_workspace_size(*cost.shape), 'cuda')
    return (_run(L.wotk_transport_stablev2, cost, Gd, prm, ws),
            _run(L.wotk_transport_stablev2_noalloc, cost, Gd, prm))


# forbidden pairs (infinite) and costs beyond 2^31 / k, in the first, a middle and the last row and column and
# strewn; every width of the columns' chunks; some in the first eps already
@pytest.mark.parametrize('n_i,n_j', [(2201, 3839), (2100, 4101), (1021, 8221), (701, 12289), (517, 16389)])
@pytest.mark.parametrize('big', [np.inf, 1e9, 3e38])
def test_forbidden_pairs_are_terms_of_zero(n_i, n_j, big):
    import torch
    rng = np.random.default_rng(n_j)
    C = rng.gamma(6.0, 1 / 6.0, (n_i, n_j))
    C[rng.random((n_i, n_j)) < 0.01] = big
    for r in (0, n_i // 2, n_i - 1):
        C[r, :: 2] = big
    for c in (0, n_j // 2, n_j - 1):
        C[1:: 2, c] = big
    one, two = _both_of_matrix(C, np.exp(0.3 * rng.standard_normal(n_i)))
    for a, b in zip(one[:2], two[:2]):
        assert torch.isfinite(b).all()
        # exponents of a few times max C / eps = 100 rounded at 2^-24 by the sweeps, averaged over the terms,
        # times eps, over 340 half-iterations that do not expand: 340 * 0.05 * 100 * 2^-24 * ln 2
        assert float((a - b).abs().max()) < 7e-5


def test_nan_costs_stay_nan():
    import torch
    rng = np.random.default_rng(3)
    C = rng.gamma(6.0, 1 / 6.0, (2100, 4100))
    C[77, 1234] = np.nan
    one, two = _both_of_matrix(C, np.ones(2100), scaling_iter=0, extra_iter=1)
    for a, b in zip(one[:2], two[:2]):
        assert torch.equal(torch.isnan(a), torch.isnan(b))


@pytest.mark.parametrize('eps,lam1', [(0.05, 1.0), (0.003, 5.0), (0.003, 50.0)])
def test_rows_whose_terms_overflow(eps, lam1):
    """Zero growth: such a row has no shift, and its terms pass 2^128 where it lies on a target that only far
    cells serve."""
    import torch
    from wot_amd.synthetic import day_pair
    dp = day_pair(2100, 4100, dim=30, n_components=5, seed=2100)
    x, y, G = dp.x.copy(), dp.y.copy(), dp.growth.copy()
    zero = [0, 17, 900, 2099]
    y[[3, 1024, 2047, 4099]] *= 4.0
    x[zero] = y[[3, 1024, 2047, 4099]]
    G[zero] = 0.0
    cost, one, two = _both(x, y, G, epsilon=eps, epsilon0=1.0, lambda1=lam1, scaling_iter=300, extra_iter=20,
                           inner_iter_max=50)
    # the terms of such rows leave FP32: the case is the one that it is meant to be
    top = (two[1][None, :] - cost.dense()[zero].double()).max() / eps / np.log(2.0)
    assert float(top) > 128
    for a, b in zip(one[:2], two[:2]):
        assert torch.equal(torch.isinf(a), torch.isinf(b)) and not torch.isnan(a).any()
        fin = torch.isfinite(b)
        # exponents up to max |C| / eps rounded at 2^-24, times eps, over 640 half-iterations
        assert float((a - b)[fin].abs().max()) < 640 * 2.0 ** -24 * float(cost.dense().max())


@pytest.mark.parametrize('lam1,lam2', [(0.1, 50.0), (0.01, 0.1), (0.002, 0.002)])
def test_small_penalties(lam1, lam2):
    """Rows and columns that the plan hardly serves: their sums are far from 1 at every iteration."""
    import torch
    from wot_amd.synthetic import day_pair
    dp = day_pair(2100, 4100, dim=30, n_components=5, seed=4)
    cost, one, two = _both(dp.x, dp.y, dp.growth, lambda1=lam1, lambda2=lam2)
    for a, b in zip(one[:2], two[:2]):
        assert torch.isfinite(a).all()
        # exponents up to max |C| / eps rounded at 2^-24, times eps, over 340 half-iterations
        assert float((a - b).abs().max()) < 340 * 2.0 ** -24 * float(cost.dense().max())


# the one-read gap pass: pairs with a short side, and from 2^24 entries on, in whole and ragged tiles
@pytest.mark.parametrize('n_i,n_j,kw', [(1500, 6001, {}), (6017, 1500, dict(tau=2.0)), (4200, 4100, {}),
                                        (5003, 3401, dict(batch_size=3))])
def test_one_read_gap_pass_matches_fp64(n_i, n_j, kw):
    test_duality_gap_schedule_matches_fp64(n_i, n_j, kw)


def test_objectives_on_either_side_of_the_gap_pass_rule():
    """2900 x 2900 takes two passes, 4200 x 4100 and 1500 x 6001 one: both against FP64."""
    import torch
    import wot_amd.ot as ot
    from wot_amd.ot import device as dev
    from wot_amd.synthetic import day_pair
    for n_i, n_j in ((2900, 2900), (4200, 4100), (1500, 6001)):
        dp = day_pair(n_i, n_j, dim=30, n_components=5, seed=n_j)
        cost = ot.DeviceCost.from_coordinates(dp.x, dp.y)
        G = torch.from_numpy(dp.growth).cuda()
        r = dev.solve(cost, G, 'fixed_iters', dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, scaling_iter=60, tau=1e4,
                                                   epsilon0=1.0, extra_iter=0, inner_iter_max=20),
                      want_potentials=True)
        pri, dua = dev.primal_dual(cost, G, r['f'], r['g'], 1.0, 50.0, 0.05)
        C, f, g = cost.dense().double(), r['f'], r['g']
        y = (f[:, None] + g[None, :] - C) / 0.05
        R, K = torch.exp(y), torch.exp(-C / 0.05)
        q, n, m = G.mean(), n_i, n_j
        x1, x2 = R.sum(1) / m, R.sum(0) / n
        want_p = float((x1 * torch.log(x1 / G) - x1 + G).sum() / n + 50.0 * (x2 * torch.log(x2 / q) - x2 + q).sum() / m
                       + (0.05 * ((R * y).sum() - R.sum() + K.sum()) + (R * C).sum()) / (n * m))
        want_d = float(-(G * (torch.exp(-f) - 1)).sum() / n - 50.0 * (q * (torch.exp(-g / 50.0) - 1)).sum() / m
                       - 0.05 * (R.sum() - K.sum()) / (n * m))
        assert pri == pytest.approx(want_p, rel=1e-10) and dua == pytest.approx(want_d, rel=1e-10)
