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
               max_iter=16390)
    st, so = {}, {}
    R = ot.optimal_transport_duality_gap(ot.DeviceCost.from_coordinates(x, y), g, stats=st, **prm)
    ref = O.optimal_transport_duality_gap(O.default_cost_matrix(x, y), G=g, stats=so, **prm)
    assert st['iterations'] == so['iterations'] == 16390 and st['max_iter_reached'] and so['max_iter_reached']
    assert np.linalg.norm(R - ref) / np.linalg.norm(ref) < 1e-5
