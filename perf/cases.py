"""The work users of wot_amd have it do, as cases that can be timed and checked.

Every case is one call chain through the public entry points on seeded
synthetic data of the shapes the package is configured, tested and benchmarked
with: cells in PCA coordinates (Gaussian mixtures, 20-50 dimensions), 200 to
20,000 cells per day, OTModel's default parameters.

kinds
    cost      the median-normalised squared-Euclidean cost of one day pair
    pair      one transport map from coordinates (cost, solve, growth loop)
    course    a time course over an (epsilon, lambda1) grid, batched
    coords    a pair whose cost is never stored
    chain     long-range coupling: product of consecutive FP32 maps
    walk      populations pulled back and pushed forward through stored maps
    gradient  the differentiable objective, forward and backward
    pca       local PCA of two days' expression matrices
"""
import math

import torch

import wot_amd.ot as ot
import wot_amd.tmap as tmap
from wot_amd.ot import batch, large

# OTModel's defaults
EPS0, TAU, LAMBDA2 = 1.0, 1e4, 50.0
SCALING_ITER, INNER_ITER, EXTRA_ITER = 3000, 50, 1000
BATCH, TOLERANCE, MAX_ITER = 5, 1e-8, 1e7

# a map of more entries than this is kept as an FP32 device map (half the
# memory, TransportMapModel's dtype='float32'); a smaller one as FP64
FP32_MAP_ENTRIES = 1 << 23


def listed():
    return [
        # the cost of the largest single pair: what every map of that size starts with
        dict(name='cost_15000x15000', kind='cost', n_i=15000, n_j=15000, d=30, mode='f64'),
        # a small pair with the fixed schedule: 8000 dependent sweeps of a cost that fits in cache
        dict(name='fixed_300x400', kind='pair', solver='fixed_iters', n_i=300, n_j=400, d=30, mode='f64',
             eps=0.05, lambda1=1.0, growth_iters=1),
        # the ordinary pair of the tests and the small benchmark, learning the growth once
        dict(name='fixed_2000x2500_growth2', kind='pair', solver='fixed_iters', n_i=2000, n_j=2500, d=30, mode='f64',
             eps=0.05, lambda1=1.0, growth_iters=2),
        # two large days, fixed schedule, the cost from the matrix cores
        dict(name='fixed_10000x8001', kind='pair', solver='fixed_iters', n_i=10000, n_j=8001, d=30, mode='bf16x6',
             eps=0.05, lambda1=1.0, growth_iters=1),
        # OTModel's default solver on an ordinary, odd-sized pair
        dict(name='gap_2749x3001', kind='pair', solver='duality_gap', n_i=2749, n_j=3001, d=30, mode='f64',
             eps=0.05, lambda1=1.0, growth_iters=1),
        # OTModel's default solver on the largest stored pair
        dict(name='gap_15000x15000', kind='pair', solver='duality_gap', n_i=15000, n_j=15000, d=30, mode='f64',
             eps=0.05, lambda1=1.0, growth_iters=1),
        # a short time course over the parameter grid of the benchmark
        dict(name='course_6days_9combos', kind='course', days=6, lo=1500, hi=3500, d=30, n_eps=3, n_lambda=3),
        # a pair kept as coordinates only
        dict(name='coords_20000x20000_d50', kind='coords', solver='duality_gap', n_i=20000, n_j=20000, d=50, terms=6,
             eps=0.05, lambda1=1.0),
        # day 0 to day 3 through FP32 maps
        dict(name='chain_5003_4000_6001_4500', kind='chain', dims='5003,4000,6001,4500'),
        # ten populations back to the first day and on to the last
        dict(name='walk_8days_10pops', kind='walk', days=8, lo=3000, hi=12000, pops=10, dtype='float64'),
        # one step of a training loop over FP32 embeddings
        dict(name='gradient_4000x3500', kind='gradient', n_i=4000, n_j=3500, d=30, eps=0.05, lambda1=1.0),
        # the PCA in front of one map
        dict(name='pca_7000_5000cells_2000genes', kind='pca', n_i=7000, n_j=5000, genes=2000, k=30),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['cost', 'pair', 'pair', 'course', 'coords', 'chain', 'walk', 'gradient', 'pca'])
    if kind == 'cost':
        return dict(kind=kind, n_i=_log_int(rng, 200, 15000), n_j=_log_int(rng, 200, 15000), d=rng.randint(10, 30),
                    mode=rng.choice(['f64', 'f64', 'bf16x6', 'bf16x3']))
    if kind == 'pair':
        solver = rng.choice(['fixed_iters', 'duality_gap'])
        top = 8900 if solver == 'fixed_iters' else 15000
        n_i, n_j = _log_int(rng, 200, top), _log_int(rng, 200, top)
        return dict(kind=kind, solver=solver, n_i=n_i, n_j=n_j, d=rng.randint(10, 50),
                    mode=rng.choice(['f64', 'f64', 'bf16x6']), eps=rng.choice([0.02, 0.05, 0.1]),
                    lambda1=rng.choice([0.5, 1.0, 5.0]), growth_iters=rng.choice([1, 2]) if n_i * n_j <= 1 << 22 else 1)
    if kind == 'course':
        lo = _log_int(rng, 300, 1500)
        return dict(kind=kind, days=rng.randint(3, 6), lo=lo, hi=lo + rng.randint(200, 2000), d=rng.randint(20, 50),
                    n_eps=rng.choice([1, 2, 3]), n_lambda=rng.choice([1, 2, 3]))
    if kind == 'coords':
        solver = rng.choice(['fixed_iters', 'duality_gap', 'duality_gap'])
        top = 6000 if solver == 'fixed_iters' else 20000
        return dict(kind=kind, solver=solver, n_i=_log_int(rng, 1500, top), n_j=_log_int(rng, 1500, top),
                    d=rng.randint(20, 50), terms=rng.choice([3, 6]), eps=0.05, lambda1=rng.choice([0.5, 1.0, 5.0]))
    if kind == 'chain':
        return dict(kind=kind, dims=','.join(str(_log_int(rng, 300, 5500)) for _ in range(rng.randint(3, 5))))
    if kind == 'walk':
        lo = _log_int(rng, 500, 5000)
        return dict(kind=kind, days=rng.randint(3, 8), lo=lo, hi=lo + rng.randint(500, 7000),
                    pops=rng.choice([1, 3, 10, 16, 24, 40]), dtype=rng.choice(['float64', 'float64', 'float32']))
    if kind == 'gradient':
        return dict(kind=kind, n_i=_log_int(rng, 300, 4000), n_j=_log_int(rng, 300, 3500), d=rng.randint(10, 50),
                    eps=rng.choice([0.05, 0.1]), lambda1=rng.choice([1.0, 5.0]))
    return dict(kind=kind, n_i=_log_int(rng, 600, 7000), n_j=_log_int(rng, 600, 5000), genes=_log_int(rng, 400, 2000),
                k=rng.choice([10, 20, 30]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device='cuda').manual_seed(int(seed))


def _randn(gen, *shape):
    return torch.randn(shape, dtype=torch.float64, device='cuda', generator=gen)


def _cells(gen, n, means):
    comp = torch.randint(0, means.shape[0], (n,), device='cuda', generator=gen)
    return means[comp] + _randn(gen, n, means.shape[1])


def _pair(gen, n_i, n_j, d):
    mu = 3.0 * _randn(gen, 10, d)
    return (_cells(gen, n_i, mu), _cells(gen, n_j, mu + 0.5 * _randn(gen, 10, d)),
            torch.exp(0.3 * _randn(gen, n_i)))


def _day_sizes(case, seed):
    """Cells per day: fixed by the case, so that every seed does the same work."""
    span = case['hi'] - case['lo']
    return [case['lo'] + (span * ((7 * t + 3) % 11)) // 10 + t % 2 for t in range(case['days'])]


def _grid(case):
    eps = {1: (0.05,), 2: (0.05, 0.1), 3: (0.01, 0.05, 0.1)}[case['n_eps']]
    lam = {1: (1.0,), 2: (0.5, 5.0), 3: (0.5, 1.0, 5.0)}[case['n_lambda']]
    return eps, lam


def _solver_args(case):
    a = dict(epsilon=case['eps'], lambda1=case['lambda1'], lambda2=LAMBDA2, epsilon0=EPS0, tau=TAU)
    if case['solver'] == 'fixed_iters':
        a.update(scaling_iter=SCALING_ITER, inner_iter_max=INNER_ITER, extra_iter=EXTRA_ITER)
    else:
        a.update(batch_size=BATCH, tolerance=TOLERANCE, max_iter=MAX_ITER)
    return a


def _maps(gen, dims, dtype):
    """Maps of log-normal entries over a few orders of magnitude, rows of mass about one."""
    out = []
    for a, b in zip(dims, dims[1:]):
        m = torch.empty((a, b), dtype=dtype, device='cuda')
        m.log_normal_(mean=-math.log(b) - 2.0, std=2.0, generator=gen)
        out.append(m)
    return out


def prepare(case, seed):
    gen = _gen(seed)
    kind = case['kind']
    st = dict(case=case)
    if kind in ('cost', 'pair', 'coords', 'gradient'):
        st['x'], st['y'], st['growth'] = _pair(gen, case['n_i'], case['n_j'], case['d'])
        if kind == 'gradient':
            st['x'] = st['x'].float().requires_grad_(True)
            st['y'] = st['y'].float()
            st['log_g'] = torch.log(st.pop('growth')).float().requires_grad_(True)
    elif kind == 'course':
        mu, w = 3.0 * _randn(gen, 20, case['d']), _randn(gen, 20, case['d'])
        sizes = _day_sizes(case, seed)
        st['coords'] = [_cells(gen, n, mu + 0.25 * t * w) for t, n in enumerate(sizes)]
        st['growth'] = [torch.exp(0.3 * _randn(gen, n)) for n in sizes]
    elif kind == 'chain':
        st['maps'] = _maps(gen, [int(v) for v in case['dims'].split(',')], torch.float32)
    elif kind == 'walk':
        sizes = _day_sizes(case, seed)
        st['mid'] = mid = len(sizes) // 2
        st['maps'] = [tmap.DeviceMap.upload(m, case['dtype'])
                      for m in _maps(gen, sizes, getattr(torch, case['dtype']))]
        for m in st['maps'][:mid]:
            m.make_transposed()  # TransportMapModel's default for the maps that pull backs take
        p = (torch.rand((sizes[mid], case['pops']), dtype=torch.float64, device='cuda', generator=gen) > 0.8).double()
        p[0] = 1.0
        st['pops'] = p / p.sum(0, keepdim=True)
        st['offs'] = [sum(sizes[:t]) for t in range(len(sizes) + 1)]
        st['out'] = torch.empty((st['offs'][-1], case['pops']), dtype=torch.float64, device='cuda')
    else:  # expression: 40 programs of falling weight plus noise
        n, g = case['n_i'] + case['n_j'], case['genes']
        load = 8.0 * 0.93 ** torch.arange(40, dtype=torch.float64, device='cuda')
        x = (_randn(gen, n, 40) * load) @ _randn(gen, 40, g) / math.sqrt(40.0) + 0.3 * _randn(gen, n, g) + 1.0
        st['m1'], st['m2'] = x[:case['n_i']].float().contiguous(), x[case['n_i']:].float().contiguous()
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    return globals()['_run_' + st['case']['kind']](st)


def _run_cost(st):
    c = ot.DeviceCost.from_coordinates(st['x'], st['y'], mode=st['case']['mode'])
    return dict(C=c.dense(), CT=c.CT[:, :c.n_i], median=c.median, median_index=c.median_index)


def _run_pair(st):
    case = st['case']
    cost = ot.DeviceCost.from_coordinates(st['x'], st['y'], mode=case['mode'])
    solver = ot.transport_stablev2 if case['solver'] == 'fixed_iters' else ot.optimal_transport_duality_gap
    plan, growth = ot.compute_transport_matrix(solver=solver, C=cost, G=st['growth'],
                                               growth_iters=case['growth_iters'], device_out=True,
                                               **_solver_args(case))
    if plan.numel() > FP32_MAP_ENTRIES:
        plan = tmap.DeviceMap.upload(plan, 'float32').X
    return dict(map=plan, growth=growth[1:])


def _run_course(st):
    eps, lam = _grid(st['case'])
    r = batch.solve_time_course(st['coords'], st['growth'], epsilons=eps, lambda1s=lam, lambda2=LAMBDA2,
                                scaling_iter=SCALING_ITER, tau=TAU, epsilon0=EPS0, extra_iter=EXTRA_ITER,
                                inner_iter_max=INNER_ITER)
    return dict(f=r.f, g=r.g)


def _run_coords(st):
    case = st['case']
    solve = (large.transport_stablev2_coords if case['solver'] == 'fixed_iters'
             else large.optimal_transport_duality_gap_coords)
    r = solve(st['x'], st['y'], st['growth'], terms=case['terms'], want_row_sums=True, **_solver_args(case))
    return dict(f=r.f, g=r.g, median=r.median, row_sums=r.row_sums)


def _run_chain(st):
    return tmap.chain_product(st['maps'])


def _run_walk(st):
    maps, p, mid, offs, out = st['maps'], st['pops'], st['mid'], st['offs'], st['out']
    last = len(maps)
    out[offs[mid]:offs[mid + 1]].copy_(p)
    if mid > 0:
        tmap.propagate([maps[t - 1] for t in range(mid, 0, -1)], p, tmap.PULL_BACK, normalize=True,
                       outs=[out[offs[t - 1]:offs[t]] for t in range(mid, 0, -1)])
    if mid < last:
        tmap.propagate([maps[t] for t in range(mid, last)], p, tmap.PUSH_FORWARD, normalize=True,
                       outs=[out[offs[t + 1]:offs[t + 2]] for t in range(mid, last)])
    return out


def _run_gradient(st):
    case = st['case']
    val = ot.ot_objective(st['x'], st['log_g'], st['y'], epsilon=case['eps'], lambda1=case['lambda1'],
                          lambda2=LAMBDA2)
    gx, gl = torch.autograd.grad(val, (st['x'], st['log_g']))
    return dict(value=val.detach(), grad_x=gx, grad_log_g=gl)


def _run_pca(st):
    v1, v2, pca, mean = ot.compute_pca(st['m1'], st['m2'], st['case']['k'])
    return dict(v1=v1, v2=v2, singular_values=pca.singular_values_, mean=mean)


# ---------------------------------------------------------------------------
# what one pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case['kind']
    if kind in ('chain', 'walk', 'course'):
        dims = [int(v) for v in case['dims'].split(',')] if kind == 'chain' else _day_sizes(case, 0)
        area = sum(float(a) * b for a, b in zip(dims, dims[1:]))
        if kind == 'chain':
            return dict(bytes=4.0 * (area + dims[0] * dims[-1]),
                        flops=2.0 * sum(float(dims[0]) * a * b for a, b in zip(dims[1:], dims[2:])))
        if kind == 'walk':
            size = 8 if case['dtype'] == 'float64' else 4
            return dict(bytes=size * area + 8.0 * case['pops'] * (sum(dims) + dims[len(dims) // 2]),
                        flops=2.0 * case['pops'] * area)
        combos = case['n_eps'] * case['n_lambda']
        return dict(bytes=8.0 * sum(dims) * (case['d'] + 1) + 16.0 * combos * sum(dims),
                    flops=2.0 * (SCALING_ITER + EXTRA_ITER) * area * (2.0 * combos + 3.0 * case['n_eps']))
    if kind == 'pca':
        n, g = case['n_i'] + case['n_j'], case['genes']
        return dict(bytes=4.0 * n * g + 8.0 * (n * case['k'] + g), flops=float(n) * g * min(n, g))
    n_i, n_j, d = case['n_i'], case['n_j'], case['d']
    area = float(n_i) * n_j
    read = 8.0 * (n_i + n_j) * d
    if kind == 'cost':
        return dict(bytes=read + 8.0 * area, flops=3.0 * area * d)
    # an iteration is two sweeps of a subtraction, a scaling, an exponential and a sum per entry
    iters = SCALING_ITER + EXTRA_ITER if case.get('solver') == 'fixed_iters' else 300
    sweeps = 8.0 * area * iters * case.get('growth_iters', 1)
    if kind == 'pair':
        return dict(bytes=read + 8.0 * n_i + (4.0 if area > FP32_MAP_ENTRIES else 8.0) * area,
                    flops=3.0 * area * d + sweeps)
    if kind == 'coords':
        return dict(bytes=read + 16.0 * n_i + 8.0 * n_j, flops=3.0 * area * d + sweeps)
    return dict(bytes=0.5 * read * 2 + 8.0 * n_i, flops=7.0 * area * d + sweeps)  # gradient


# ---------------------------------------------------------------------------
# the same results from plain torch in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    return globals()['_exact_' + case['kind']](case, prepare(case, seed))


def _distances(x, y):
    x, y = x.detach().double(), y.detach().double()
    D = torch.zeros((x.shape[0], y.shape[0]), dtype=torch.float64, device=x.device)
    for k in range(x.shape[1]):
        t = x[:, k, None] - y[None, :, k]
        D.addcmul_(t, t)
        del t
    return D


def _median(D):
    s = D.reshape(-1).sort().values
    n = s.numel()
    return 0.5 * (s[(n - 1) // 2] + s[n // 2])


def _kernel(f, g, C, eps):
    """exp((f + g - C) / eps) for stacked potentials f (E, I), g (E, J) and eps (E,)."""
    K = f[:, :, None] + g[:, None, :]
    K -= C
    K /= eps[:, None, None]
    return K.exp_()


def _exact_fixed(C, G, eps, lambda1):
    """Potentials after the fixed schedule for stacked eps, lambda1 (E,)."""
    E, (n_i, n_j) = eps.numel(), C.shape
    f = torch.zeros((E, n_i), dtype=torch.float64, device=C.device)
    g = torch.zeros((E, n_j), dtype=torch.float64, device=C.device)
    a = b = None
    for n in range(SCALING_ITER + EXTRA_ITER):
        if n % INNER_ITER == 0 and n <= SCALING_ITER:
            if a is not None:
                f, g = f + e * a.log(), g + e * b.log()
                del K
            e = ((EPS0 - eps) * math.exp(-(n // INNER_ITER)) + eps)[:, None]
            K = _kernel(f, g, C, e[:, 0])
            KT = K.transpose(1, 2)
            b = torch.ones_like(g)
            al1, al2 = lambda1[:, None] / (lambda1[:, None] + e), LAMBDA2 / (LAMBDA2 + e)
            fa = (G * n_j) ** al1 * torch.exp(-f / (lambda1[:, None] + e))
            fb = (G.mean() * n_i) ** al2 * torch.exp(-g / (LAMBDA2 + e))
        a = fa * torch.matmul(K, b[:, :, None])[:, :, 0] ** -al1
        b = fb * torch.matmul(KT, a[:, :, None])[:, :, 0] ** -al2
    return f + e * a.log(), g + e * b.log(), e[:, 0]


def _exact_gap(C, G, eps, lambda1):
    """Potentials at the end of the duality-gap schedule."""
    n_i, n_j = C.shape
    q = G.mean()
    f = torch.zeros(n_i, dtype=torch.float64, device=C.device)
    g = torch.zeros(n_j, dtype=torch.float64, device=C.device)
    for s in range(6):
        e = EPS0 * eps ** (s / 5.0)
        al1, al2 = lambda1 / (lambda1 + e), LAMBDA2 / (LAMBDA2 + e)
        sum_kt = float(torch.exp(-C / e).sum()) if s == 5 else 0.0
        u, v = f, g
        a, b = torch.ones_like(f), torch.ones_like(g)
        K = torch.exp((u[:, None] + v[None, :] - C) / e)
        gap = math.inf
        while gap > (TOLERANCE if s == 5 else 1e-6):
            for _ in range(BATCH):
                a0, b0 = a, b
                a = (G * n_j / torch.mv(K, b)) ** al1 * torch.exp(-u / (lambda1 + e))
                b = (q * n_i / torch.mv(K.t(), a)) ** al2 * torch.exp(-v / (LAMBDA2 + e))
                if float(torch.maximum(a.max(), b.max())) > TAU:
                    u, v = u + e * a.log(), v + e * b.log()
                    K = torch.exp((u[:, None] + v[None, :] - C) / e)
                    a, b = torch.ones_like(a), torch.ones_like(b)
            A, B = a * torch.exp(u / e), b * torch.exp(v / e)
            if s < 5:
                A0, B0 = a0 * torch.exp(u / e), b0 * torch.exp(v / e)
                gap = float(torch.maximum((A - A0).norm() / (1 + A.norm()), (B - B0).norm() / (1 + B.norm())))
                continue
            f, g = e * A.log(), e * B.log()
            pri, R = _primal(C, f, g, G, e, lambda1, sum_kt)
            dua = (-lambda1 * (G * (torch.exp(-f / lambda1) - 1)).mean()
                   - LAMBDA2 * (q * (torch.exp(-g / LAMBDA2) - 1)).mean() - e * (R.sum() - sum_kt) / (n_i * n_j))
            gap = float((pri - dua) / pri.abs())
            del R
        f, g = u + e * a.log(), v + e * b.log()
    return f, g, e


def _primal(C, f, g, G, e, lambda1, sum_kt):
    n_i, n_j = C.shape
    q = G.mean()
    R = torch.exp((f[:, None] + g[None, :] - C) / e)
    r, c = R.sum(1), R.sum(0)
    x, y = r / n_j, c / n_i
    # sum R (e log R + C) = sum f r + sum g c
    body = (f * r).sum() + (g * c).sum() + e * (sum_kt - r.sum())
    return (lambda1 * (x * torch.log(x / G) - x + G).mean() + LAMBDA2 * (y * torch.log(y / q) - y + q).mean()
            + body / (n_i * n_j)), R


def _exact_cost(case, st):
    D = _distances(st['x'], st['y'])
    m = _median(D)
    C = D.div_(m)
    return dict(C=C, CT=C.t(), median=m.reshape(1), median_index=None)


def _potentials(case, C, G):
    if case['solver'] == 'fixed_iters':
        one = torch.ones(1, dtype=torch.float64, device=C.device)
        f, g, e = _exact_fixed(C, G, case['eps'] * one, case['lambda1'] * one)
        return f[0], g[0], float(e[0])
    return _exact_gap(C, G, case['eps'], case['lambda1'])


def _exact_pair(case, st):
    C = _distances(st['x'], st['y'])
    C /= _median(C)
    G, growth = st['growth'], []
    for it in range(case['growth_iters']):
        f, g, e = _potentials(case, C, G)
        plan = f[:, None] + g[None, :]
        plan -= C
        plan = plan.div_(e).exp_().div_(C.shape[1])
        if it + 1 < case['growth_iters']:
            G = plan.sum(1)
            growth.append(G)
    return dict(map=plan, growth=growth)


def _exact_course(case, st):
    eps, lam = _grid(case)
    combos = [(e, v) for e in eps for v in lam]
    e = torch.tensor([c[0] for c in combos], dtype=torch.float64, device='cuda')
    v = torch.tensor([c[1] for c in combos], dtype=torch.float64, device='cuda')
    fs, gs = [], []
    for x, y, G in zip(st['coords'], st['coords'][1:], st['growth']):
        C = _distances(x, y)
        C /= _median(C)
        f, g, _ = _exact_fixed(C, G, e, v)
        fs.append(f)
        gs.append(g)
    return dict(f=fs, g=gs)


def _exact_coords(case, st):
    C = _distances(st['x'], st['y'])
    m = _median(C)
    C /= m
    f, g, e = _potentials(case, C, st['growth'])
    C.neg_().add_(f[:, None]).add_(g[None, :])
    return dict(f=f, g=g, median=m.reshape(1), row_sums=C.div_(e).exp_().sum(1) / C.shape[1])


def _exact_chain(case, st):
    out = st['maps'][0].double()
    for m in st['maps'][1:]:
        out = out @ m.double()
    return out


def _exact_walk(case, st):
    maps, mid, offs, out = [m.X.double() for m in st['maps']], st['mid'], st['offs'], st['out']
    out[offs[mid]:offs[mid + 1]] = st['pops']
    p = st['pops']
    for t in range(mid, 0, -1):
        p = maps[t - 1] @ p
        p = p / p.sum(0, keepdim=True)
        out[offs[t - 1]:offs[t]] = p
    p = st['pops']
    for t in range(mid, len(maps)):
        p = maps[t].t() @ p
        p = p / p.sum(0, keepdim=True)
        out[offs[t + 1]:offs[t + 2]] = p
    return out


def _exact_gradient(case, st):
    x = st['x'].detach().double().requires_grad_(True)
    log_g = st['log_g'].detach().double().requires_grad_(True)
    y = st['y'].double()
    with torch.no_grad():
        D = _distances(x, y)
        m = _median(D)
        f, g, e = _exact_gap(D / m, torch.exp(log_g), case['eps'], case['lambda1'])
        R = torch.exp((f[:, None] + g[None, :] - D / m) / e)
        s = D.reshape(-1).sort()
        mids = [int(s.indices[(D.numel() - 1) // 2]), int(s.indices[D.numel() // 2])]
        del D, s
    # the objective's partial derivative at the fixed optimal plan
    G = torch.exp(log_g)
    n_i, n_j = R.shape
    D = (x * x).sum(1)[:, None] + (y * y).sum(1)[None, :] - 2.0 * (x @ y.t())
    med = sum(0.5 * ((x[k // n_j] - y[k % n_j]) ** 2).sum() for k in mids)
    C = D / med
    xs, ys, q = R.sum(1) / n_j, R.sum(0) / n_i, G.mean()
    with torch.no_grad():
        logr = torch.nan_to_num(R.log())
        ent = (R * logr).sum() - R.sum()
    val = (case['lambda1'] * (xs * torch.log(xs / G) - xs + G).mean()
           + LAMBDA2 * (ys * torch.log(ys / q) - ys + q).mean()
           + (e * (ent + torch.exp(-C / e).sum()) + (R * C).sum()) / (n_i * n_j))
    gx, gl = torch.autograd.grad(val, (x, log_g))
    return dict(value=val.detach(), grad_x=gx, grad_log_g=gl)


def _exact_pca(case, st):
    x = torch.cat([st['m1'], st['m2']]).double()
    n, g = x.shape
    mean = x.mean(0)
    A = x - mean
    A -= A.mean(1, keepdim=True)
    k = case['k']
    if n <= g:
        w, V = torch.linalg.eigh(A @ A.t())
        S, V = w.flip(0)[:k].clamp(min=0).sqrt(), V.flip(1)[:, :k]
    else:
        w, U = torch.linalg.eigh(A.t() @ A)
        S = w.flip(0)[:k].clamp(min=0).sqrt()
        V = (A @ U.flip(1)[:, :k]) / S
    top = V.abs().argmax(0)
    V = V * V[top, torch.arange(k, device=V.device)].sign()
    return dict(v1=V[:case['n_i']], v2=V[case['n_i']:], singular_values=S, mean=mean)
