"""Workloads of the framework, each through its public entry points.

A case is one call that a variational-Monte-Carlo program makes over and over: a step of an optimiser
(parameters in, gradient and energy out), a stochastic-reconfiguration update, a distance gradient of a
time evolution, a batch of configurations to evaluate, a training call of the proposal network.  ``run``
gives the model its parameters first wherever an optimiser would, so that what a new parameter set costs
(upload, normalisation) is part of the pass.

Models of precision 32 and 16 compute in single precision and return their values in complex128 arrays;
``run`` narrows those to complex64, the type that they were computed in.  Values of precision=64 models
stay as they come.
"""
import math

import numpy as np
import torch

import rbmongpu_amd as R
from rbmongpu_amd import hamiltonians as H
from rbmongpu_amd.new_neural_network import deep_connections


def listed():
    return [
        # the smallest step: a chain that fits in exact summation, where launches and latency count
        dict(name="exact_n10_m20", kind="exact_gradient", N=10, M=20, precision=32),
        # the same step in double precision at the size where exact summation starts to take time
        dict(name="exact_n16_m64_fp64", kind="exact_gradient", N=16, M=64, precision=64),
        # Metropolis on a chain of 20 spins: few chains, long runs (one wavefront per SIMD)
        dict(name="mc_chain20_m80", kind="mc_gradient", lx=20, ly=1, M=80, chains=4096, therm=200, samples=1000),
        # Metropolis on the 10x10 lattice, the model whose weights exceed LDS
        dict(name="mc_10x10_m200", kind="mc_gradient", lx=10, ly=10, M=200, chains=8192, therm=40, samples=100),
        # the same model sampled through the proposal network
        dict(name="learned_10x10_m200", kind="learned_gradient", lx=10, ly=10, M=200, hidden=256, chains=8192,
             therm=20, samples=150),
        # the deep network on bfloat16 layers
        dict(name="deep_n40_bf16", kind="deep_mc_gradient", N=40, m1=160, m2=80, chains=32768, therm=50, samples=10),
        # a sparsely connected deep network, exact summation in single precision
        dict(name="deep_sparse_n14", kind="deep_exact_gradient", N=14, m1=28, m2=14, c1=7, c2=14, precision=32,
             invariant=False),
        # stochastic reconfiguration of a 6x6 Heisenberg model in its S_z = 0 sector
        dict(name="sr_6x6_m144", kind="sr_step", lx=6, ly=6, M=144, chains=16384, therm=20, samples=4),
        # one step of a time evolution: distance to (1 + i dt H) psi and its gradient
        dict(name="distance_n14_m56", kind="distance_gradient", N=14, M=56, precision=32),
        # configurations from elsewhere, an odd lattice size: log psi and E_loc
        dict(name="batch_n61_m122", kind="evaluate", N=61, M=122, n=20001, precision=32),
        # training the proposal network on recorded configurations, some steps of the schedule's last phase
        dict(name="made_train_n100_h256", kind="made_train", N=100, hidden=256, n=100000, batch=16384, steps=10),
        # the geometric tensor of a small model, as the reference computes it
        dict(name="s_matrix_n10_m20", kind="s_matrix", N=10, M=20, precision=32),
    ]


def _between(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["exact_gradient", "mc_gradient", "learned_gradient", "deep_mc_gradient", "deep_exact_gradient",
                       "sr_step", "distance_gradient", "evaluate", "made_train", "s_matrix"])
    if kind == "exact_gradient":
        N = rng.randint(6, 17)
        return dict(kind=kind, N=N, M=_between(rng, N, 4 * N), precision=rng.choice([32, 64]))
    if kind == "mc_gradient":
        if rng.random() < 0.5:
            lx, ly = rng.randint(9, 60), 1
        else:
            lx, ly = rng.randint(3, 11), rng.randint(3, 10)
        N = lx * ly
        return dict(kind=kind, lx=lx, ly=ly, M=_between(rng, max(N // 2, 8), min(2 * N, 220)),
                    chains=_between(rng, 500, 8192), therm=rng.randint(10, 40), samples=_between(rng, 10, 80))
    if kind == "learned_gradient":
        lx, ly = rng.randint(3, 10), rng.randint(3, 10)
        N = lx * ly
        return dict(kind=kind, lx=lx, ly=ly, M=_between(rng, max(N // 2, 8), 2 * N), hidden=_between(rng, 48, 256),
                    chains=_between(rng, 500, 8192), therm=rng.randint(5, 20), samples=_between(rng, 10, 100))
    if kind == "deep_mc_gradient":
        return dict(kind=kind, N=rng.randint(12, 48), m1=_between(rng, 24, 128), m2=_between(rng, 8, 80),
                    chains=_between(rng, 1000, 16384), therm=rng.randint(5, 25), samples=_between(rng, 2, 10))
    if kind == "deep_exact_gradient":
        N = rng.randint(6, 13)
        invariant = N <= 9 and rng.random() < 0.4
        return dict(kind=kind, N=N, m1=2 * N, m2=N, c1=rng.randint(2, N), c2=2 * rng.randint(1, N),
                    precision=rng.choice([32, 64]), invariant=invariant)
    if kind == "sr_step":
        lx, ly = rng.choice([(4, 2), (4, 3), (4, 4), (6, 3), (5, 4), (6, 4)])
        return dict(kind=kind, lx=lx, ly=ly, M=_between(rng, lx * ly, 3 * lx * ly), chains=_between(rng, 1000, 8192),
                    therm=rng.randint(5, 20), samples=rng.randint(2, 8))
    if kind == "distance_gradient":
        N = rng.randint(6, 15)
        return dict(kind=kind, N=N, M=_between(rng, N, 4 * N), precision=rng.choice([32, 64]))
    if kind == "evaluate":
        N = rng.randint(8, 100)
        return dict(kind=kind, N=N, M=_between(rng, max(N // 2, 8), min(2 * N, 200)), n=_between(rng, 50, 20000),
                    precision=rng.choice([32, 32, 64]))
    if kind == "made_train":
        return dict(kind=kind, N=rng.randint(10, 110), hidden=_between(rng, 32, 256), n=_between(rng, 5000, 200000),
                    batch=_between(rng, 1024, 16384), steps=rng.randint(3, 10))
    N = rng.randint(4, 10)
    return dict(kind=kind, N=N, M=_between(rng, N, 2 * N), precision=rng.choice([32, 64]))


# ---------------------------------------------------------------------------
# models and operators, from the seed alone
# ---------------------------------------------------------------------------
def _rounded(z, precision):
    """Parameters that the model's own type holds exactly."""
    return z if precision == 64 else np.asarray(z, np.complex64).astype(complex)


def _rbm(N, M, seed, sigma, precision):
    r = np.random.default_rng(seed)
    b = sigma * (r.normal(size=M) + 1j * r.normal(size=M))
    W = sigma * (r.normal(size=(N, M)) + 1j * r.normal(size=(N, M)))
    return _rounded(b, precision), _rounded(W, precision)


def _psi(b, W, precision):
    N = W.shape[0]
    return R.Psi(np.zeros(N), np.zeros(N), b, W, 1.0, False, True, precision=precision)


#: standard deviation of the real and the imaginary parts of b and W, by lattice: far enough from a flat
#: state that samples, ratios and gradients have structure
def _sigma(N):
    return 0.2 / math.sqrt(N)


def _table(case):
    kind = case["kind"]
    if kind in ("mc_gradient", "learned_gradient"):
        return H.tfim_1d(case["lx"], 1.0, 1.0) if case["ly"] == 1 else H.tfim_2d(case["lx"], case["ly"], 1.0, 3.04)
    if kind == "sr_step":
        return H.heisenberg_2d(case["lx"], case["ly"])
    if kind == "deep_mc_gradient":
        return H.j1j2_chain(case["N"], 1.0, 0.5)
    if kind == "distance_gradient":
        c, t, i = H.tfim_1d(case["N"], 1.0, 1.0)
        return 1j * 0.02 * c, t, i   # psi' follows exp(i dt H) psi
    return H.tfim_1d(case["N"], 1.0, 1.0)


def _deep_layers(case, seed):
    """(connections, biases, weights, final weights) of a two-layer network, N(0, 0.6^2 / fan_in) weights."""
    r = np.random.default_rng(seed)
    N, m = case["N"], [case["m1"], case["m2"]]
    c = [case.get("c1", N), case.get("c2", m[0])]
    precision = case.get("precision", 16)
    conns = [np.asarray(x, np.uint32) for x in deep_connections(N, m, c)]
    W = [_rounded(0.6 / math.sqrt(f) * (r.normal(size=(f, k)) + 1j * r.normal(size=(f, k))), precision) for f, k in zip(c, m)]
    b = [_rounded(0.05 * (r.normal(size=k) + 1j * r.normal(size=k)), precision) for k in m]
    return conns, b, W, np.ones(m[1], complex)


def _random_words(r, n, N):
    w = np.zeros((n, 2), np.uint64)
    w[:, 0] = r.integers(0, 2 ** min(N, 63), size=n, dtype=np.uint64)
    if N >= 64:
        w[:, 0] |= r.integers(0, 2, size=n, dtype=np.uint64) << np.uint64(63)
        if N > 64:
            w[:, 1] = r.integers(0, 2 ** (N - 64), size=n, dtype=np.uint64)
    return w


def _made_params(N, hidden, seed, scale):
    """[W1 (H x N), b1, W2 (N x H), b2] as float32: uniform weights over the square root of the fan-in."""
    r = np.random.default_rng(seed)
    w1 = scale * r.uniform(-1, 1, (hidden, N)) / math.sqrt(N)
    w2 = scale * r.uniform(-1, 1, (N, hidden)) / math.sqrt(hidden)
    deg = 1 + np.arange(hidden) % max(N - 1, 1)
    w1 = np.where(np.arange(N)[None, :] < deg[:, None], w1, 0.0)
    w2 = np.where(deg[None, :] <= np.arange(N)[:, None], w2, 0.0)
    return np.concatenate([w1.ravel(), np.zeros(hidden), w2.ravel(), np.zeros(N)]).astype(np.float32)


def _made_data(case, seed):
    """Recorded configurations with neighbouring spins aligned three times out of four."""
    r = np.random.default_rng(seed + 7)
    n, N = case["n"], case["N"]
    keep = r.random((n, N)) < 0.75
    keep[:, 0] = r.random(n) < 0.5
    up = np.cumsum(~keep, axis=1) % 2 == 0
    words = np.zeros((n, 2), np.uint64)
    for i in range(N):
        words[:, i >> 6] |= up[:, i].astype(np.uint64) << np.uint64(i & 63)
    return words


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, ev=R.ExpectationValue(True))
    if kind == "made_train":
        s.update(words=_made_data(case, seed), made=R.MADE(case["N"], case["hidden"], seed=1),
                 params=_made_params(case["N"], case["hidden"], seed, 1.0), seed=seed)
        return s
    if kind == "evaluate":
        b, W = _rbm(case["N"], case["M"], seed, _sigma(case["N"]), case["precision"])
        s.update(psi=_psi(b, W, case["precision"]), op=R.Operator(*_table(case), True),
                 words=_random_words(np.random.default_rng(seed + 3), case["n"], case["N"]))
        return s
    if kind in ("deep_mc_gradient", "deep_exact_gradient"):
        conns, b, W, final = _deep_layers(case, seed)
        N = case["N"]
        psi = R.PsiDeep(np.zeros(N), np.zeros(N), b, conns, W, final, 1.0, False, True, precision=case.get("precision", 16))
        if case.get("invariant"):
            psi.translational_invariance = True
        s.update(psi=psi, params=psi.params, op=R.Operator(*_table(case), True))
        if kind == "deep_exact_gradient":
            s["ens"] = R.ExactSummation(N, True)
        else:
            s["ens"] = R.MonteCarloLoop(case["chains"] * case["samples"], 1, case["therm"], case["chains"], True, seed=seed)
        return s
    N = case["N"] if "N" in case else case["lx"] * case["ly"]
    precision = case.get("precision", 32)
    # (0.01: the spread of the learned-proposal workload's starting point, near which an untrained network
    # already proposes well)
    b, W = _rbm(N, case["M"], seed, 0.01 if kind == "learned_gradient" else _sigma(N), precision)
    psi = _psi(b, W, precision)
    s.update(psi=psi, params=psi.params)
    if kind != "s_matrix":
        s["op"] = R.Operator(*_table(case), True)
    if kind in ("exact_gradient", "s_matrix"):
        s["ens"] = R.ExactSummation(N, True)
    elif kind == "distance_gradient":
        s["ens"] = R.ExactSummation(N, True)
        psi.normalize(s["ens"])
        b2, W2 = _nearby(b, W, seed, precision)
        s["psi2"] = _psi(b2, W2, precision)
        s["params"] = s["psi2"].params
        s["hs"] = R.HilbertSpaceDistance(N, psi.num_params, True)
    elif kind == "learned_gradient":
        made = R.MADE(N, case["hidden"], params=_made_params(N, case["hidden"], seed, 0.2))
        s["ens"] = R.LearnedMonteCarloLoop(made, case["chains"] * case["samples"], case["therm"], case["chains"], True,
                                           seed=seed)
    else:
        s["ens"] = R.MonteCarloLoop(case["chains"] * case["samples"], 1, case["therm"], case["chains"], True, seed=seed)
        if kind == "sr_step":
            s["ens"].set_total_z_symmetry(0)
    return s


def _nearby(b, W, seed, precision):
    r = np.random.default_rng(seed + 5)
    return (_rounded(b + 0.01 * (r.normal(size=b.shape) + 1j * r.normal(size=b.shape)), precision),
            _rounded(W + 0.01 * (r.normal(size=W.shape) + 1j * r.normal(size=W.shape)), precision))


def _own_type(case, **values):
    """The values in the type that the model computes in."""
    if case.get("precision", 32) == 64:
        return {k: np.asarray(v, complex) for k, v in values.items()}
    return {k: np.asarray(v, np.complex64) for k, v in values.items()}


#: shift of the geometric tensor in an update, and learning rate of the proposal network
EPS, RATE = 1e-2, 1e-4


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "made_train":
        made = s["made"]
        made.params = s["params"]
        made.reset_optimizer()
        # (a network counts its steps for the minibatch draws; a fresh optimiser starts them again)
        losses = made.train(s["words"], case["steps"], batch=case["batch"], lr=RATE, seed=s["seed"])
        return {"losses": losses.astype(np.float32), "params": made.params}
    if kind == "evaluate":
        return _own_type(case, log_psi=R.log_psi_batch(s["psi"], s["words"]),
                         e_loc=R.local_energy_batch(s["psi"], s["op"], s["words"]))
    psi = s["psi"]
    if kind == "distance_gradient":
        s["psi2"].params = s["params"]
        g, d = s["hs"].gradient(psi, s["psi2"], s["op"], False, s["ens"], 1.0)
        return _own_type(case, gradient=g, distance=d)
    psi.params = s["params"]
    if kind == "s_matrix":
        return _own_type(case, S=R.get_S_matrix(psi, s["ens"]))
    if kind == "sr_step":
        x, E = R.sr_update(psi, s["op"], s["ens"], EPS)
        return _own_type(case, update=x, energy=E)
    if kind in ("exact_gradient", "deep_exact_gradient"):
        psi.prefactor = 1.0
        psi.normalize(s["ens"])
    g, E = s["ev"].gradient(psi, s["op"], s["ens"])
    return _own_type(case, gradient=g, energy=E)


# ---------------------------------------------------------------------------
# what a pass cannot do without.  FLOP per hidden unit: 42 for a proposal, 44 for log psi, 50 for a flipped
# neighbour, 91 for the derivative; 8 for a complex multiply-add
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "made_train":
        N, hid, b, steps = case["N"], case["hidden"], case["batch"], case["steps"]
        return {"bytes": 16.0 * case["n"] + 8.0 * (2 * N * hid + hid + N), "flops": 6.0 * steps * b * N * hid}
    N = case["N"] if "N" in case else case["lx"] * case["ly"]
    if kind in ("deep_mc_gradient", "deep_exact_gradient"):
        m1, m2 = case["m1"], case["m2"]
        c1, c2 = case.get("c1", N), case.get("c2", m1)
        forward = 4.0 * c1 * m1 + 8.0 * c2 * m2 + 44.0 * (m1 + m2)
        terms = 2 * N if kind == "deep_mc_gradient" else N
        passes = N if case.get("invariant") else 1
        n = case["chains"] * case["samples"] if kind == "deep_mc_gradient" else 2 ** N
        proposals = case["chains"] * (case["therm"] + case["samples"]) * N if kind == "deep_mc_gradient" else n
        params = c1 * m1 + c2 * m2 + m1 + 2 * m2
        return {"bytes": 32.0 * params, "flops": forward * passes * (proposals + n * (1 + terms)) + n * (forward + 8.0 * params)}
    M = case["M"]
    params = M + N * M
    if kind == "evaluate":
        n = case["n"]
        return {"bytes": n * 64.0 + 16.0 * params, "flops": n * (4.0 * N * M + 44.0 * M + 50.0 * N * M)}
    if kind == "s_matrix":
        P = params
        return {"bytes": 16.0 * params + 16.0 * (2 * N + P) ** 2, "flops": 2.0 ** N * (4.0 * N * M + 91.0 * M + 4.0 * P * P)}
    if kind in ("exact_gradient", "distance_gradient"):
        n, proposals = 2 ** N, 0
    else:
        n = case["chains"] * case["samples"]
        proposals = case["chains"] * (case["therm"] + case["samples"]) * (1 if kind == "learned_gradient" else N)
    terms = 2 * N if kind == "sr_step" else N
    flops = n * (4.0 * N * M + 44.0 * M + 50.0 * terms * M + 91.0 * M + 4.0 * (N + 1) * (M + 1))
    flops += proposals * (4.0 * N * M + 44.0 * M + 4.0 * N * case["hidden"] if kind == "learned_gradient" else 42.0 * M)
    if kind == "exact_gradient":
        flops += n * (4.0 * N * M + 44.0 * M)   # the norm
    if kind == "sr_step":
        # second moments of pairs of spins and pairs of units, and the factorisation
        flops += n * 2.0 * (N * (N + 1) / 2) * M * M + 4.0 * params ** 3 / 3
    return {"bytes": 48.0 * params, "flops": flops}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
_A3, _A2, _A1, _A0 = 3.746646023906276, 7.771429504240965, 10.2180213465, 9.19376335670885
_N0, _N1, _K, _C = 5.49914721954, 2.16564366435, 0.9003320053750442, 0.598139


def _side(z):
    return torch.where(z.real > 0, 1.0, -1.0).to(z.real.dtype)


def _log_cosh(z):
    sg = _side(z)
    w = sg * z
    return _K * w + (_N0 - _N1 * w) / ((((w + _A3) * w + _A2) * w + _A1) * w + _A0) - _C


def _tanh(z):
    sg = _side(z)
    d = (((z + sg * _A3) * z + _A2) * z + sg * 10.218021346543315) * z + _A0
    p = 6.746450656267947 + sg * _K * z
    for c, odd in ((26.632014683761202, 1), (70.82878897882324, 0), (146.36284300074402, 1), (199.24474920889975, 0),
                   (177.6769746361748, 1), (83.68563506532087, 0)):
        p = p * z + (sg * c if odd else c)
    return p * z / (d * d)


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _tensor(x):
    return torch.as_tensor(np.ascontiguousarray(x), device=_device())


def _basis(N):
    k = torch.arange(2 ** N, device=_device())
    return (((k[:, None] >> torch.arange(N, device=_device())) & 1) * 2 - 1).to(torch.float64)


def _exact_local_energy(table, N, lp, spins):
    """E_loc of every basis state from log psi of every basis state."""
    coef, types, idx = table
    k = torch.arange(2 ** N, device=lp.device)
    e = torch.zeros_like(lp)
    for c, ts, js in zip(coef, types, idx):
        el, mask = torch.full((2 ** N,), complex(c), dtype=lp.dtype, device=lp.device), 0
        for t, j in zip(ts, js):
            if j < 0:
                break
            if t in (1, 2):
                mask ^= 1 << int(j)
            if t in (2, 3):
                el = el * spins[:, int(j)]
            if t == 2:
                el = el * -1j
        e = e + el * torch.exp(lp[k ^ mask] - lp)
    return e


def _out(case, **values):
    return {k: (v if v is None else v.cpu().numpy() if isinstance(v, torch.Tensor) else np.asarray(v)) for k, v in values.items()}


def _rbm_exact(N, b, W):
    s = _basis(N)
    th = s.to(torch.complex128) @ _tensor(W) + _tensor(b)
    return s, _log_cosh(th).sum(1), _tanh(th)


def _rbm_rows(coef, s, T):
    """sum_s coef conj(O_k) in parameter order, zero for the axis angles."""
    y = coef[:, None] * T.conj()
    return torch.cat([torch.zeros(2 * s.shape[1], dtype=y.dtype, device=y.device), y.sum(0),
                      (s.to(y.dtype).T @ y).reshape(-1)])


def _probability(lp):
    p = torch.exp(2 * (lp.real - lp.real.max()))
    return p / p.sum()


def _centred(lp, e):
    p = _probability(lp)
    E = (p * e).sum()
    return E, 2 * p * (e - E)


def _exact_made(case, seed):
    N, hid, B, n = case["N"], case["hidden"], case["batch"], case["n"]
    words = _made_data(case, seed)
    x_all = np.stack([(words[:, i >> 6] >> np.uint64(i & 63)) & np.uint64(1) for i in range(N)], axis=1).astype(float)
    x_all = torch.as_tensor(x_all, device=_device())
    flat = _made_params(N, hid, seed, 1.0).astype(float)
    at = [0, hid * N, hid * N + hid, 2 * hid * N + hid, flat.size]
    p = [_tensor(flat[a:z]) for a, z in zip(at, at[1:])]
    p[0], p[2] = p[0].reshape(hid, N), p[2].reshape(N, hid)
    deg = torch.arange(hid, device=_device()) % max(N - 1, 1) + 1
    site = torch.arange(N, device=_device())
    masks = [(site[None, :] < deg[:, None]).double(), None, (deg[None, :] <= site[:, None]).double(), None]
    m, v = [torch.zeros_like(q) for q in p], [torch.zeros_like(q) for q in p]
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    lr, eps = float(np.float32(RATE)), float(np.float32(1e-8))
    losses = []
    for t in range(1, case["steps"] + 1):
        if B == n:
            x = x_all
        else:
            u = (_philox_x(t - 1, np.arange(B), 4, seed).astype(float) + 0.5) * 2.0 ** -32
            x = x_all[_tensor(np.minimum((u * n).astype(np.int64), n - 1))]
        a = x @ p[0].T + p[1]
        h = a.clamp(min=0)
        logit = h @ p[2].T + p[3]
        losses.append(float(-(x * logit - torch.nn.functional.softplus(logit)).sum() / B))
        dl = (torch.sigmoid(logit) - x) / B
        da = (dl @ p[2]) * (a > 0)
        for q, g, mk, mq, vq in zip(p, (da.T @ x, da.sum(0), dl.T @ h, dl.sum(0)), masks, m, v):
            g = g if mk is None else g * mk
            mq.mul_(b1).add_(g, alpha=1 - b1)
            vq.mul_(b2).add_(g * g, alpha=1 - b2)
            q.sub_(lr * (mq / (1 - b1 ** t)) / (torch.sqrt(vq / (1 - b2 ** t)) + eps))
    return _out(case, losses=np.array(losses), params=torch.cat([q.reshape(-1) for q in p]))


def _philox_x(c0, c1, c3, key):
    """First word of Philox4x32-10 of the counters (c0, c1, 0, c3)."""
    lo = np.uint64(0xFFFFFFFF)
    c = [np.full(c1.shape, c0, np.uint64), c1.astype(np.uint64), np.zeros(c1.shape, np.uint64), np.full(c1.shape, c3, np.uint64)]
    k0, k1 = np.uint64(key & 0xFFFFFFFF), np.uint64(key >> 32)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ k0, p1 & lo, (p0 >> np.uint64(32)) ^ c[3] ^ k1, p0 & lo]
        k0, k1 = (k0 + np.uint64(0x9E3779B9)) & lo, (k1 + np.uint64(0xBB67AE85)) & lo
    return c[0]


def _exact_deep(case, seed):
    N = case["N"]
    conns, b, W, final = _deep_layers(case, seed)
    dense = []
    for size_in, cn, w in zip((N, case["m1"]), conns, W):
        d = np.zeros((size_in, w.shape[1]), complex)
        np.add.at(d, (cn.astype(int), np.arange(w.shape[1])[None, :]), w)
        dense.append(_tensor(d))
    b, final = [_tensor(x) for x in b], _tensor(final)

    def forward(x):
        xs, angles = [x], []
        for d, bias in zip(dense, b):
            angles.append(xs[-1] @ d + bias)
            xs.append(_log_cosh(angles[-1]))
        return xs, angles, xs[-1] @ final

    s = _basis(N)
    xs, angles, lp0 = forward(s.to(torch.complex128))
    lp = lp0
    if case["invariant"]:
        lp = sum(forward(torch.roll(s, k, 1).to(torch.complex128))[2] for k in range(N)) / N
    e = _exact_local_energy(_table(case), N, lp, s)
    E, coef = _centred(lp, e)
    delta = [None, final * _tanh(angles[1])]
    delta[0] = (delta[1] @ dense[1].T) * _tanh(angles[0])
    rows = [torch.zeros(2 * N, dtype=lp.dtype, device=lp.device)]
    for layer in range(2):
        y = coef[:, None] * delta[layer].conj()
        G = xs[layer].conj().T @ y
        cn = _tensor(conns[layer].astype(np.int64))
        rows += [y.sum(0), G[cn, torch.arange(cn.shape[1], device=G.device)[None, :]].reshape(-1)]
    # the derivative by a final weight keeps the reference's form, log psi times the unit's value
    rows.append(((coef * lp0.conj())[:, None] * xs[2].conj()).sum(0))
    return _out(case, gradient=torch.cat(rows), energy=E)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mc_gradient", "learned_gradient", "deep_mc_gradient", "sr_step"):
        return None   # the samples are the framework's own
    if kind == "made_train":
        return _exact_made(case, seed)
    if kind == "deep_exact_gradient":
        return _exact_deep(case, seed)
    N, M = case["N"], case["M"]
    b, W = _rbm(N, M, seed, _sigma(N), case["precision"])
    if kind == "evaluate":
        words = _random_words(np.random.default_rng(seed + 3), case["n"], N)
        s = np.stack([(words[:, i >> 6] >> np.uint64(i & 63)) & np.uint64(1) for i in range(N)], axis=1).astype(float) * 2 - 1
        s, w = _tensor(s), _tensor(W)
        lps, es = [], []
        for part in s.split(2000):
            th = part.to(torch.complex128) @ w + _tensor(b)
            lp = _log_cosh(th).sum(1)
            e = -(part * torch.roll(part, -1, 1)).sum(1).to(lp.dtype)
            for i in range(N):
                e = e - torch.exp(_log_cosh(th - 2 * part[:, i:i + 1] * w[i]).sum(1) - lp)
            lps.append(lp)
            es.append(e)
        return _out(case, log_psi=torch.cat(lps), e_loc=torch.cat(es))
    s, lp, T = _rbm_exact(N, b, W)
    if kind == "s_matrix":
        O = torch.cat([torch.zeros((len(s), 2 * N), dtype=T.dtype, device=T.device), T,
                       (s.to(T.dtype)[:, :, None] * T[:, None, :]).reshape(len(s), -1)], dim=1)
        return _out(case, S=O.T @ O.conj() / len(s))
    e = _exact_local_energy(_table(case), N, lp, s)
    if kind == "exact_gradient":
        E, coef = _centred(lp, e)
        return _out(case, gradient=_rbm_rows(coef, s, T), energy=E)
    _, lp2, T2 = _rbm_exact(N, *_nearby(b, W, seed, case["precision"]))
    p = _probability(lp)
    omega, ratio = torch.exp(e + (lp2 - lp).conj()), torch.exp(2 * (lp2 - lp).real)
    om, rm, nrm = (p * omega).sum(), (p * ratio).sum(), (p * torch.exp(2 * e.real)).sum()
    d = torch.sqrt(1 - om.abs() ** 2 / (nrm * rm))
    g = -om.conj() * nrm / (nrm * rm) ** 2 / d * _rbm_rows(p * (rm * omega - ratio * om), s, T2)
    return _out(case, gradient=g, distance=d + 0j)
