"""Cost and median from regenerated distances: tile edges, every selection
route (all entries kept, sampled bracket, ties that need the radix fallback),
against numpy on the device's own FP64 distances.  The median and its indices
are order statistics, so they are equal; C is FP32(D / median) with one FP64
division, so it is equal up to one FP32 rounding of a value that two correctly
rounded quotients cannot differ by more than one FP64 unit in."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _points(kind, n_i, n_j, d, seed):
    rng = np.random.default_rng(seed)
    if kind == 'normal':
        return rng.standard_normal((n_i, d)), 0.5 + rng.standard_normal((n_j, d))
    if kind == 'sorted_clusters':  # runs of similar tiles
        a = np.sort(rng.integers(0, 5, n_i))[:, None] * 4.0 + rng.standard_normal((n_i, d)) * 0.01
        b = np.sort(rng.integers(0, 5, n_j))[:, None] * 4.0 + rng.standard_normal((n_j, d)) * 0.01
        return a, b
    if kind == 'integers':  # a handful of distinct distances: the middle bins hold too many ties
        return rng.integers(0, 3, (n_i, d)).astype(float), rng.integers(0, 3, (n_j, d)).astype(float)
    if kind == 'outlier':
        a, b = rng.standard_normal((n_i, d)), rng.standard_normal((n_j, d))
        a[0] *= 1e6
        b[:min(n_j, n_i)] = a[:min(n_j, n_i)]  # exact zeros beside 1e12
        return a, b
    return np.ones((n_i, d)), np.ones((n_j, d))  # identical: the median is 0


CASES = [('normal', 1, 1, 1), ('normal', 1, 2, 3), ('normal', 5, 3, 33), ('normal', 127, 63, 30),
         ('normal', 128, 64, 32), ('normal', 129, 65, 31), ('normal', 512, 512, 30), ('normal', 513, 512, 30),
         ('normal', 900, 701, 50), ('normal', 2100, 2003, 30), ('sorted_clusters', 1500, 1300, 10),
         ('integers', 800, 701, 2), ('outlier', 700, 900, 30), ('identical', 640, 513, 4)]


@pytest.mark.parametrize('mode', ['f64', 'bf16x6', 'bf16x3'])
@pytest.mark.parametrize('kind,n_i,n_j,d', CASES)
def test_cost_and_median(kind, n_i, n_j, d, mode):
    import torch
    import wot_amd.ot as ot
    from wot_amd.ot import device as dev
    x, y = _points(kind, n_i, n_j, d, n_i + n_j)
    cost = ot.DeviceCost.from_coordinates(x, y, mode=mode)
    C = cost.dense().cpu().numpy()
    CT = cost.CT[:, :n_i].cpu().numpy()
    med = float(cost.median.cpu()[0])
    idx = cost.median_index.cpu().numpy()
    assert np.array_equal(C, CT.T, equal_nan=True)
    pad = cost.C[:, n_j:(n_j + 3) // 4 * 4]
    padt = cost.CT[:, n_i:(n_i + 3) // 4 * 4]
    assert not pad.any() and not padt.any()
    D = dev.sqeuclid_f64(x, y).cpu().numpy()
    from scipy.spatial.distance import cdist
    assert np.allclose(D, cdist(x, y, 'sqeuclidean'), rtol=1e-12, atol=0)
    if mode == 'f64':
        flat = np.sort(D.ravel())
        lo, hi = flat[(flat.size - 1) // 2], flat[flat.size // 2]
        assert med == (lo + hi) / 2 if flat.size % 2 == 0 else med == lo
        assert idx[0] == np.flatnonzero(D.ravel() == lo)[0] and idx[1] == np.flatnonzero(D.ravel() == hi)[0]
        with np.errstate(invalid='ignore', divide='ignore'):
            ref = (D / med).astype(np.float32)
        assert np.array_equal(np.isnan(C), np.isnan(ref))
        ok = ~np.isnan(ref)
        assert np.all(np.abs(C[ok] - ref[ok]) <= np.spacing(np.abs(ref[ok])))
        assert np.mean(C[ok] != ref[ok]) < 1e-6 if ok.any() else True
    elif kind in ('normal', 'sorted_clusters'):
        # an order statistic of the split distances: as many on either side as the rank says.
        # C keeps their order up to FP32 rounding, and the median entry is 1 (even counts: around 1)
        n = C.size
        one = np.float32(1.0)
        assert np.sum(C < one - 2 * np.spacing(one)) <= (n - 1) // 2 + 1
        assert np.sum(C > one + 2 * np.spacing(one)) <= n // 2 + 1
        mids = C.ravel()[idx]
        assert abs(float(mids.astype(np.float64).mean()) - 1.0) <= 2.0 ** -23
    if kind != 'identical' and mode == 'f64':
        stored = float(dev.median_f64(torch.from_numpy(D).cuda()).cpu()[0])
        assert stored == med


def test_median_of_the_never_stored_pair():
    """The counting and gathering passes (no candidate lists), with and without ties."""
    import wot_amd.ot as ot
    from wot_amd.ot import large
    for kind, n_i, n_j, d in (('normal', 700, 901, 30), ('integers', 800, 701, 2), ('normal', 40, 50, 7)):
        x, y = _points(kind, n_i, n_j, d, 3)
        r = large.transport_stablev2_coords(x, y, np.ones(n_i), scaling_iter=1, extra_iter=0)
        cost = ot.DeviceCost.from_coordinates(x, y)
        assert float(r.median.cpu()[0]) == float(cost.median.cpu()[0])


# more equal distances than the middle bins' list holds: one value, the two middle ranks in two values, a few
# values, one value among unequal ones; with the candidate lists and without (never stored)
@pytest.mark.parametrize('kind', ['one', 'halves', 'few', 'spike'])
@pytest.mark.parametrize('n_i,n_j', [(520, 514), (2100, 2003)])
def test_heavy_ties(kind, n_i, n_j):
    import wot_amd.ot as ot
    from wot_amd.ot import large
    rng = np.random.default_rng(n_i)
    x, y = np.zeros((n_i, 3)), np.ones((n_j, 3))
    if kind == 'halves':
        x[n_i // 2:] = 3.0
    elif kind == 'few':
        x, y = rng.integers(0, 3, (n_i, 3)).astype(float), rng.integers(0, 3, (n_j, 3)).astype(float)
    elif kind == 'spike':
        x[: 2 * n_i // 5] = rng.random((2 * n_i // 5, 3))
        y[: n_j // 5] = 4.0 + rng.random((n_j // 5, 3))
    cost = ot.DeviceCost.from_coordinates(x, y)
    D = np.zeros((n_i, n_j))
    for k in range(3):
        D += (x[:, k, None] - y[None, :, k]) ** 2
    # sums of three squares in another order of rounding than the device's: only the exact kinds compare by bits
    flat = np.sort(D.ravel())
    lo, hi = flat[(flat.size - 1) // 2], flat[flat.size // 2]
    med, idx = float(cost.median.cpu()[0]), cost.median_index.cpu().numpy()
    assert med == pytest.approx((lo + hi) / 2, rel=1e-15 if kind != 'spike' else 1e-14)
    if kind != 'spike':
        assert idx[0] == np.flatnonzero(D.ravel() == lo)[0] and idx[1] == np.flatnonzero(D.ravel() == hi)[0]
    r = large.transport_stablev2_coords(x, y, np.ones(n_i), scaling_iter=1, extra_iter=0)
    assert float(r.median.cpu()[0]) == med


# either side of the bounds of one list (24576 entries) and of 16 lists (2^22)
@pytest.mark.parametrize('n_i,n_j', [(128, 192), (157, 157), (2047, 2048), (2048, 2048)])
@pytest.mark.parametrize('kind', ['normal', 'sorted_clusters'])
def test_number_of_candidate_lists(kind, n_i, n_j):
    for mode in ('f64', 'bf16x6'):
        test_cost_and_median(kind, n_i, n_j, 30, mode)
