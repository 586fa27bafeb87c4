"""The resident solver (pairs up to 2^23 entries, one persistent launch) against
the launched sweeps, which the no-allocation entry point keeps: the same bits,
at the edges of its teams, chunks and register pieces."""
import numpy as np
import pytest

from test_gpu_onepass import _run

pytestmark = pytest.mark.gpu

# one row or column; fewer rows than teams; chunk edges at 1024 columns; several rows per team; the most
# pieces per thread (9); long sides
SHAPES = [(1, 1), (1, 2), (2, 1), (3, 5), (64, 3), (300, 400), (1023, 1025), (1024, 1024), (1025, 1023), (1025, 2049),
          (2049, 2047), (2896, 2896), (2749, 3001), (200, 8704), (8704, 9), (900, 8000), (8191, 1024)]


def _pair(n_i, n_j, seed=0):
    rng = np.random.default_rng(n_i + 7 * n_j + seed)
    return rng.standard_normal((n_i, 20)), 0.3 + rng.standard_normal((n_j, 20)), np.exp(0.3 * rng.standard_normal(n_i))


def _both(n_i, n_j, G=None, **kw):
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    from wot_amd.ot import device as dev
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, epsilon0=1.0, scaling_iter=23, extra_iter=4, inner_iter_max=5)
    prm.update(kw)
    x, y, g = _pair(n_i, n_j)
    cost = (ot.DeviceCost.from_coordinates(x, y) if n_i * n_j > 1
            else ot.DeviceCost.from_matrix(np.array([[0.7]])))
    Gd = torch.from_numpy(np.ascontiguousarray(g if G is None else G)).cuda()
    L = _native.lib()
    ws = dev.workspace(torch, L.wotk_solver_workspace_size(n_i, n_j), 'cuda')
    ws.fill_(255)
    a = _run(L.wotk_transport_stablev2, cost, Gd, prm, ws)
    b = _run(L.wotk_transport_stablev2_noalloc, cost, Gd, prm)
    return a, b


@pytest.mark.parametrize('n_i,n_j', SHAPES)
def test_same_bits_as_the_launched_sweeps(n_i, n_j):
    import torch
    a, b = _both(n_i, n_j)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and a[2] == b[2]


def test_many_eps_segments_and_launches():
    """More eps values than one launch takes (96) and an iteration count over several launches."""
    import torch
    a, b = _both(70, 90, scaling_iter=205, inner_iter_max=1, extra_iter=3)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    a, b = _both(40, 50, scaling_iter=16390, inner_iter_max=20000, extra_iter=0)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_growth_zero_and_nan():
    import torch
    G = np.ones(300)
    G[17] = 0.0
    a, b = _both(300, 200, G=G)
    for x, y in zip(a[:2], b[:2]):
        assert torch.equal(torch.nan_to_num(x), torch.nan_to_num(y))
        assert torch.equal(torch.isnan(x), torch.isnan(y)) and torch.equal(torch.isinf(x), torch.isinf(y))
    G[17] = np.nan
    a, b = _both(300, 200, G=G, scaling_iter=3)
    for x, y in zip(a[:2], b[:2]):
        assert torch.equal(torch.isnan(x), torch.isnan(y))


@pytest.mark.parametrize('n_i,n_j,kw', [(120, 150, {}), (700, 1100, dict(batch_size=7)), (300, 360, dict(tau=3.0)),
                                        (60, 50, dict(max_iter=12)), (60, 50, dict(max_iter=303))])
def test_duality_gap_counts_and_plan(n_i, n_j, kw):
    from oracle import ot_oracle as O
    import wot_amd.ot as ot
    x, y, g = _pair(n_i, n_j, 1)
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, batch_size=5, tolerance=1e-8, tau=1e4, epsilon0=1.0,
               max_iter=1e7)
    prm.update(kw)
    cost = ot.DeviceCost.from_coordinates(x, y)
    st, so = {}, {}
    R = ot.optimal_transport_duality_gap(cost, g, stats=st, **prm)
    ref = O.optimal_transport_duality_gap(O.default_cost_matrix(x, y), G=g, stats=so, **prm)
    assert st['iterations'] == so['iterations'] and st['stabilisations'] == so['stabilisations']
    assert bool(st['max_iter_reached']) == so['max_iter_reached']
    assert np.linalg.norm(R - ref) / np.linalg.norm(ref) < 1e-5


def test_two_streams_and_threads_at_once():
    """Two resident solves from two threads on two streams: neither waits for the other for good."""
    import threading
    import torch
    import wot_amd.ot as ot
    x, y, g = _pair(800, 900, 2)
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, batch_size=5, tolerance=1e-8, tau=1e4, epsilon0=1.0,
               max_iter=1e7, device_out=True)
    ref = ot.optimal_transport_duality_gap(ot.DeviceCost.from_coordinates(x, y), g, **prm)
    out = [None, None]

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            cost = ot.DeviceCost.from_coordinates(x, y)
            for _ in range(3):
                out[k] = ot.optimal_transport_duality_gap(cost, g, **prm)
            torch.cuda.current_stream().synchronize()

    ts = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert torch.equal(out[0], ref) and torch.equal(out[1], ref)


@pytest.mark.parametrize('kw', [dict(tolerance=1e-2), dict(batch_size=1000)])
def test_first_duality_check_converges(kw):
    """The check behind the sum of K-tilde decides: its sums are complete in every workgroup or the solve stalls."""
    from oracle import ot_oracle as O
    import wot_amd.ot as ot
    x, y, g = _pair(300, 360, 1)
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, batch_size=5, tolerance=1e-8, tau=1e4, epsilon0=1.0,
               max_iter=1e7)
    prm.update(kw)
    st, so = {}, {}
    R = ot.optimal_transport_duality_gap(ot.DeviceCost.from_coordinates(x, y), g, stats=st, **prm)
    ref = O.optimal_transport_duality_gap(O.default_cost_matrix(x, y), G=g, stats=so, **prm)
    assert st['iterations'] == so['iterations']
    assert np.linalg.norm(R - ref) / np.linalg.norm(ref) < 1e-5


def test_threads_with_different_shapes():
    """Pairs that need different amounts of LDS in the same instance of the kernel, from several threads."""
    import threading
    import torch
    import wot_amd.ot as ot
    shapes = [(60, 50), (1000, 900), (40, 2000), (2000, 30)]
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, epsilon0=1.0, scaling_iter=40, extra_iter=0, inner_iter_max=50,
               tau=1e4, device_out=True)
    pairs = [_pair(i, j, 3) for i, j in shapes]
    costs = [ot.DeviceCost.from_coordinates(x, y) for x, y, _ in pairs]
    refs = [ot.transport_stablev2(c, G=p[2], **prm) for c, p in zip(costs, pairs)]
    torch.cuda.synchronize()
    same = [True] * len(shapes)

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(5):
                out = ot.transport_stablev2(costs[k], G=pairs[k][2], **prm)
                torch.cuda.current_stream().synchronize()
                same[k] = same[k] and torch.equal(out, refs[k])

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(shapes))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(same)


def test_duality_gap_over_several_launches():
    """An unattainable tolerance: more iterations than one launch takes, with absorptions on both sides of the cut."""
    from oracle import ot_oracle as O
    import wot_amd.ot as ot
    x, y, g = _pair(60, 50, 1)
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, batch_size=7, tolerance=-1.0, tau=1.0, epsilon0=1.0,
               max_iter=4100)
    st, so = {}, {}
    R = ot.optimal_transport_duality_gap(ot.DeviceCost.from_coordinates(x, y), g, stats=st, **prm)
    ref = O.optimal_transport_duality_gap(O.default_cost_matrix(x, y), G=g, stats=so, **prm)
    assert st['iterations'] == so['iterations'] == 4100 and st['max_iter_reached'] and so['max_iter_reached']
    assert np.linalg.norm(R - ref) / np.linalg.norm(ref) < 1e-5


# ---- the route: a solve that was refused or given up has the same bits, so the tests above cannot see it ----
def _route(ws, n_i, n_j):
    import ctypes
    import torch
    from wot_amd import _native
    route, launches = ctypes.c_int32(-1), ctypes.c_int64(-1)
    _native.check(_native.lib().wotk_solver_route(n_i, n_j, ctypes.c_void_p(ws.data_ptr()), ws.numel(),
                                                  ctypes.byref(route), ctypes.byref(launches),
                                                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return route.value, launches.value


def _workspace(n_i, n_j):
    import torch
    from wot_amd import _native
    from wot_amd.ot import device as dev
    ws = dev.workspace(torch, _native.lib().wotk_solver_workspace_size(n_i, n_j), 'cuda')
    ws.fill_(255)
    return ws


def _gap(cost, g, ws, fn='wotk_transport_duality_gap', extra=(), **kw):
    """One duality-gap solve through the C ABI: potentials and statistics."""
    import ctypes
    import torch
    from wot_amd import _native
    from wot_amd.ot import device as dev
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, batch_size=5, tolerance=1e-8, tau=1e4, epsilon0=1.0,
               max_iter=10 ** 7)
    prm.update(kw)
    n_i, n_j = cost.shape
    G = torch.from_numpy(np.ascontiguousarray(g)).cuda()
    f = torch.empty(n_i, dtype=torch.float64, device='cuda')
    h = torch.empty(n_j, dtype=torch.float64, device='cuda')
    st = _native.Stats()
    p = dev._ptr
    _native.check(getattr(_native.lib(), fn)(
        p(cost.C), cost.ldc, p(cost.CT), cost.ldct, n_i, n_j, p(G), prm['lambda1'], prm['lambda2'], prm['epsilon'],
        prm['batch_size'], prm['tolerance'], prm['tau'], prm['epsilon0'], prm['max_iter'], None, n_j, None, p(f), p(h),
        p(ws), ws.numel(), ctypes.byref(st), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), *extra))
    return f, h, st.as_dict()


@pytest.mark.parametrize('n_i,n_j', SHAPES)
def test_route_of_the_fixed_schedule(n_i, n_j):
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    x, y, g = _pair(n_i, n_j)
    cost = (ot.DeviceCost.from_coordinates(x, y) if n_i * n_j > 1
            else ot.DeviceCost.from_matrix(np.array([[0.7]])))
    ws = _workspace(n_i, n_j)
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, epsilon0=1.0, scaling_iter=23, extra_iter=4, inner_iter_max=5)
    _run(_native.lib().wotk_transport_stablev2, cost, torch.from_numpy(g).cuda(), prm, ws)
    assert _route(ws, n_i, n_j) == (_native.ROUTE_RESIDENT, 1)


# rows on one side for some workgroups only (wide and tall), several rows per workgroup; the first duality
# check decides; several launches
@pytest.mark.parametrize('n_i,n_j,kw,launches', [
    (120, 150, {}, 1), (300, 400, {}, 1), (400, 300, {}, 1), (300, 360, dict(tolerance=1e-2), 1),
    (300, 360, dict(batch_size=1000), 1), (900, 8000, dict(tau=3.0), 1), (8000, 900, dict(tau=3.0), 1),
    (2749, 3001, {}, 1), (60, 50, dict(tolerance=-1.0, max_iter=2048), 1),
    (60, 50, dict(tolerance=-1.0, max_iter=4097), 3)])
def test_route_of_the_duality_gap_schedule(n_i, n_j, kw, launches):
    import wot_amd.ot as ot
    from wot_amd import _native
    x, y, g = _pair(n_i, n_j, 1)
    ws = _workspace(n_i, n_j)
    _gap(ot.DeviceCost.from_coordinates(x, y), g, ws, **kw)
    assert _route(ws, n_i, n_j) == (_native.ROUTE_RESIDENT, launches)


def test_routes_beyond_the_resident_solver():
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    for n_i, n_j, want in [(2900, 2900, _native.ROUTE_ONE_READ), (40, 9000, _native.ROUTE_SWEEPS)]:
        x, y, g = _pair(n_i, n_j)
        ws = _workspace(n_i, n_j)
        prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, epsilon0=1.0, scaling_iter=2, extra_iter=0,
                   inner_iter_max=5)
        _run(_native.lib().wotk_transport_stablev2, ot.DeviceCost.from_coordinates(x, y), torch.from_numpy(g).cuda(),
             prm, ws)
        assert _route(ws, n_i, n_j) == (want, 0)


def test_route_beside_another_solve():
    """A solve that starts while another is under way takes the sweeps, and neither gives up."""
    import threading
    import time
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    shapes = [(300, 400), (1000, 260), (2000, 2500)]
    pairs = [_pair(i, j, 2) for i, j in shapes]
    costs = [ot.DeviceCost.from_coordinates(x, y) for x, y, _ in pairs]
    refs = [_fixed('wotk_transport_stablev2', c, p[2], _workspace(*s)) for c, p, s in zip(costs, pairs, shapes)]
    long_ws = _workspace(60, 50)
    x, y, g = _pair(60, 50, 1)
    long_cost = ot.DeviceCost.from_coordinates(x, y)
    torch.cuda.synchronize()
    seen = []

    def long_solve():
        with torch.cuda.stream(torch.cuda.Stream()):
            _gap(long_cost, g, long_ws, tolerance=-1.0, max_iter=300000)  # more than 1 s

    t = threading.Thread(target=long_solve)
    t.start()
    time.sleep(0.2)
    for c, p, s, ref in zip(costs, pairs, shapes, refs):
        ws = _workspace(*s)
        out = _fixed('wotk_transport_stablev2', c, p[2], ws)
        seen.append(_route(ws, *s)[0])
        assert torch.equal(out[0], ref[0]) and torch.equal(out[1], ref[1])
    assert t.is_alive()
    t.join()
    assert seen == [_native.ROUTE_SWEEPS] * 3
    assert _route(long_ws, 60, 50) == (_native.ROUTE_RESIDENT, 147)


def test_routes_of_several_threads():
    """Wide and tall pairs from four threads, by whichever route: the same bits, and resident attempts are
    not given up as a rule (one may be, where others' sweeps keep its CUs for 0.1 s)."""
    import threading
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    shapes = [(300, 400), (1000, 260), (2000, 2500), (30, 20)]
    costs = [ot.DeviceCost.from_coordinates(*_pair(i, j, 2)[:2]) for i, j in shapes]
    refs = [_gap(c, _pair(*s, 2)[2], _workspace(*s))[:2] for c, s in zip(costs, shapes)]
    torch.cuda.synchronize()
    routes, same = [[] for _ in shapes], [True] * len(shapes)

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            ws = _workspace(*shapes[k])
            for _ in range(4):
                f, h, _ = _gap(costs[k], _pair(*shapes[k], 2)[2], ws)
                same[k] = same[k] and torch.equal(f, refs[k][0]) and torch.equal(h, refs[k][1])
                routes[k].append(_route(ws, *shapes[k])[0])

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(shapes))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(same)
    assert sum(r == _native.ROUTE_GAVE_UP for rs in routes for r in rs) <= 2


@pytest.mark.parametrize('n_i,n_j', [(30, 20), (300, 400), (2049, 2047)])
def test_few_iterations_take_the_sweeps(n_i, n_j):
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    x, y, g = _pair(n_i, n_j)
    cost = ot.DeviceCost.from_coordinates(x, y)
    ws = _workspace(n_i, n_j)
    prm = dict(lambda1=1.0, lambda2=50.0, epsilon=0.05, epsilon0=1.0, inner_iter_max=5)
    for its, extra, route in ((1, 0, _native.ROUTE_SWEEPS), (10, 5, _native.ROUTE_SWEEPS),
                              (10, 6, _native.ROUTE_RESIDENT)):
        a = _run(_native.lib().wotk_transport_stablev2, cost, torch.from_numpy(g).cuda(),
                 dict(prm, scaling_iter=its, extra_iter=extra), ws)
        assert _route(ws, n_i, n_j) == (route, int(route == _native.ROUTE_RESIDENT))
        b = _run(_native.lib().wotk_transport_stablev2_noalloc, cost, torch.from_numpy(g).cuda(),
                 dict(prm, scaling_iter=its, extra_iter=extra))
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


# ---- what follows when a bound is met: the same bits by another route ----
def _fixed(fn, cost, g, ws, extra=()):
    import ctypes
    import torch
    from wot_amd import _native
    from wot_amd.ot import device as dev
    n_i, n_j = cost.shape
    G = torch.from_numpy(np.ascontiguousarray(g)).cuda()
    f = torch.empty(n_i, dtype=torch.float64, device='cuda')
    h = torch.empty(n_j, dtype=torch.float64, device='cuda')
    st = _native.Stats()
    p = dev._ptr
    _native.check(getattr(_native.lib(), fn)(
        p(cost.C), cost.ldc, p(cost.CT), cost.ldct, n_i, n_j, p(G), 1.0, 50.0, 0.05, 43, 1e4, 1.0, 4, 11, None, n_j,
        None, p(f), p(h), p(ws), ws.numel(), ctypes.byref(st),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), *extra))
    return f, h, st.as_dict()


# pairs of several workgroups, with rows on one side only for some of them
@pytest.mark.parametrize('n_i,n_j', [(30, 20), (300, 400), (1000, 260), (2049, 2047)])
def test_a_wait_that_is_given_up(n_i, n_j):
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    x, y, g = _pair(n_i, n_j, 4)
    cost = ot.DeviceCost.from_coordinates(x, y)
    ws = _workspace(n_i, n_j)
    a = _fixed('wotk_transport_stablev2', cost, g, ws)
    assert _route(ws, n_i, n_j)[0] == _native.ROUTE_RESIDENT
    b = _fixed('wotk_probe_stablev2_limits', cost, g, ws, (1, 0))
    assert _route(ws, n_i, n_j)[0] == _native.ROUTE_GAVE_UP
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    a = _gap(cost, g, ws, tau=3.0)
    assert _route(ws, n_i, n_j)[0] == _native.ROUTE_RESIDENT
    b = _gap(cost, g, ws, 'wotk_probe_duality_gap_limits', (1, 0), tau=3.0)
    assert _route(ws, n_i, n_j)[0] == _native.ROUTE_GAVE_UP
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    for key in ('iterations', 'stabilisations', 'gap_checks', 'epsilon_final'):
        assert a[2][key] == b[2][key]


# one iteration per launch, cuts inside and at the ends of batches
@pytest.mark.parametrize('n_i,n_j', [(30, 20), (300, 400), (1000, 260)])
@pytest.mark.parametrize('launch_iters', [1, 5, 7])
def test_launches_that_stop(n_i, n_j, launch_iters):
    import torch
    import wot_amd.ot as ot
    from wot_amd import _native
    x, y, g = _pair(n_i, n_j, 4)
    cost = ot.DeviceCost.from_coordinates(x, y)
    ws = _workspace(n_i, n_j)
    a = _fixed('wotk_transport_stablev2', cost, g, ws)
    b = _fixed('wotk_probe_stablev2_limits', cost, g, ws, (0, launch_iters))
    assert _route(ws, n_i, n_j) == (_native.ROUTE_RESIDENT, -(-47 // launch_iters))
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    for kw in (dict(tau=3.0), dict(tau=3.0, batch_size=3, max_iter=311)):
        a = _gap(cost, g, ws, **kw)
        b = _gap(cost, g, ws, 'wotk_probe_duality_gap_limits', (0, launch_iters), **kw)
        assert _route(ws, n_i, n_j) == (_native.ROUTE_RESIDENT, -(-a[2]['iterations'] // launch_iters))
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and a[2] == b[2]
