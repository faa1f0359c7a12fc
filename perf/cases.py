"""What this framework is used for, as cases that can be timed.

Every case is one call (or one batch) through the public entry points of
rk_amd, with the inputs a caller has in hand.  The kinds:

  solve     rk_amd.solve on device vectors: BRUSS2D, LV pairs or the LV chain,
            with any of the step forms
  host      rk_amd.solver, the reference's solver(t0, te, y0, y, tol) on host
            arrays (what the drop-in library and its driver call)
  ensemble  rk_amd.ensemble.lv_ensemble: many two-component systems, each its
            own adaptive solve
  batch     rk_amd.Batch: uneven BRUSS2D grids and LV chains integrated
            together, results handed back to the host

BRUSS2D starts are the reference's start vector plus one percent of noise on
u, alpha is 2e-3 unless the case says otherwise, the first step is 1e-3 (the
settings of the benchmark).  Large grids are explicit-stability limited (the
step count grows with N squared), so their solves are capped by step_limit,
as the reference's STEP_LIMIT caps its benchmark runs.
"""
import math

import numpy as np
import torch

import rk_amd
from rk_amd.ensemble import lv_ensemble

ALPHA = 2e-3
H0 = 1e-3
DIFF = 1e-3
LV_CONST = (0.1, 0.2, 0.4, 0.2)     # c0, d0, d1, c1


def listed():
    return [
        # the smallest call: a reference-style driver integrating a tiny grid
        # on host arrays, set-up and latency
        dict(name="host_n32", kind="host", N=32, method="DOPRI54", tol=1e-6, te=1.0,
             step_limit=0),
        # the reference's everyday configuration: 128 x 128, the whole
        # interval (336 attempted steps), bound by the time of one small step
        dict(name="bruss_n128", kind="solve", problem="bruss", N=128, method="DOPRI54",
             tol=1e-6, te=4.0, step_limit=0, impl="PipeDls"),
        # a mid-size, odd grid at the tight tolerance, the 8-stage table
        dict(name="bruss_n301_verner65", kind="solve", problem="bruss", N=301,
             method="VERNER65", tol=1e-8, te=0.5, step_limit=0, impl="PipeDls"),
        # an odd grid of the serving range (64..1024), loose tolerance
        dict(name="bruss_n717", kind="solve", problem="bruss", N=717, method="DOPRI54",
             tol=1e-4, te=4.0, step_limit=200, impl="PipeDls"),
        # the headline benchmark's grid: a window of its 19743 steps
        dict(name="bruss_n2000", kind="solve", problem="bruss", N=2000, method="DOPRI54",
             tol=1e-6, te=1.0, step_limit=300, impl="PipeDls"),
        # a grid whose vectors leave the last-level cache
        dict(name="bruss_n4001_verner65", kind="solve", problem="bruss", N=4001,
             method="VERNER65", tol=1e-6, te=1.0, step_limit=60, impl="PipeDls"),
        # the 13-stage table of the benchmark's method matrix
        dict(name="bruss_n1000_dopri87", kind="solve", problem="bruss", N=1000,
             method="DOPRI87", tol=1e-8, te=1.0, step_limit=100, impl="PipeDls"),
        # the full-storage loop order of the reference's seq D
        dict(name="bruss_n1000_form_d", kind="solve", problem="bruss", N=1000,
             method="DOPRI54", tol=1e-6, te=1.0, step_limit=100, impl="D"),
        # independent pairs under one step size: the reference's LV problem
        # at the size of the benchmark (n = 8e6)
        dict(name="lv_pairs_4e6", kind="solve", problem="pairs", N=4000000, method="DOPRI54",
             tol=1e-8, te=20.0, step_limit=0, impl="PipeDls"),
        # a long diffusive chain, the top of the serving range
        dict(name="lv_chain_5e5", kind="solve", problem="chain", N=500000, method="DOPRI54",
             tol=1e-8, te=20.0, step_limit=0, impl="PipeDls"),
        # the benchmark's ensemble: 262144 systems, each with its own steps
        dict(name="ensemble_262144", kind="ensemble", count=262144, method="VERNER65",
             tol=1e-8, te=20.0),
        # what one admission of the server sees: uneven grids and chains with
        # their own tolerances, integrated together
        dict(name="batch_48", kind="batch", grids=36, chains=12, nmin=32, nmax=512,
             mmin=10000, mmax=500000, method="DOPRI54", te=0.5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    r = rng.random()
    if r < 0.45:
        N = _log(rng, 32, 2600)
        method = rng.choice(["DOPRI54", "DOPRI54", "DOPRI54", "VERNER65", "VERNER65", "RKF23",
                             "DOPRI87"])
        # all of [0, te] on small grids, a window of steps on large ones
        limit = 0 if N <= 160 else max(40, min(300, int(3e8 / (N * N))))
        return dict(kind="solve", problem="bruss", N=N, method=method,
                    tol=rng.choice([1e-4, 1e-6, 1e-8]), te=round(rng.uniform(0.5, 4.0), 2),
                    step_limit=limit, impl="PipeDls")
    if r < 0.55:
        return dict(kind="host", N=_log(rng, 16, 200), method=rng.choice(["DOPRI54", "VERNER65"]),
                    tol=rng.choice([1e-4, 1e-6, 1e-8]), te=round(rng.uniform(0.2, 1.0), 2),
                    step_limit=300)
    if r < 0.65:
        return dict(kind="solve", problem="bruss", N=_log(rng, 200, 1200), method="DOPRI54",
                    tol=rng.choice([1e-4, 1e-6]), te=1.0, step_limit=rng.randint(30, 100),
                    impl=rng.choice(["D", "A", "E", "F"]))
    if r < 0.75:
        return dict(kind="solve", problem="pairs", N=_log(rng, 1000, 4000000),
                    method=rng.choice(["DOPRI54", "VERNER65"]),
                    tol=rng.choice([1e-6, 1e-8]), te=round(rng.uniform(4.0, 20.0), 1),
                    step_limit=0, impl="PipeDls")
    if r < 0.85:
        return dict(kind="solve", problem="chain", N=_log(rng, 10000, 1000000),
                    method=rng.choice(["DOPRI54", "VERNER65"]),
                    tol=rng.choice([1e-6, 1e-8]), te=round(rng.uniform(4.0, 20.0), 1),
                    step_limit=0, impl="PipeDls")
    if r < 0.93:
        return dict(kind="ensemble", count=_log(rng, 4096, 262144),
                    method=rng.choice(["DOPRI54", "VERNER65"]), tol=rng.choice([1e-6, 1e-8]),
                    te=round(rng.uniform(4.0, 20.0), 1))
    grids = rng.randint(6, 36)
    return dict(kind="batch", grids=grids, chains=rng.randint(0, 12), nmin=32,
                nmax=rng.randint(128, 512), mmin=10000, mmax=500000, method="DOPRI54",
                te=round(rng.uniform(0.1, 0.5), 2))


# ---- inputs -------------------------------------------------------------------

def _bruss_start_dev(N, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = torch.arange(N, dtype=torch.float64, device="cuda") / float(N - 1)
    y = torch.empty((N, N, 2), dtype=torch.float64, device="cuda")
    y[..., 0] = torch.rand((N, N), generator=g, dtype=torch.float64, device="cuda")
    y[..., 0].mul_(2.0).sub_(1.0).mul_(0.01).add_(0.5 + k[None, :])
    y[..., 1] = 1.0 + 5.0 * k[:, None]
    return y.view(-1)


def _bruss_start_host(N, g):
    k = np.arange(N) / float(N - 1)
    y = np.empty((N, N, 2))
    y[..., 0] = (0.5 + k)[None, :] + 0.01 * g.uniform(-1.0, 1.0, (N, N))
    y[..., 1] = (1.0 + 5.0 * k)[:, None]
    return y.reshape(-1)


def _lv_start_dev(cells, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    y = torch.rand((cells, 2), generator=g, dtype=torch.float64, device="cuda").mul_(0.1)
    y[:, 0].add_(0.2)
    y[:, 1].add_(1.1)
    return y.view(-1)


def _lv_start_host(cells, g):
    y = 0.1 * g.random((cells, 2))
    y[:, 0] += 0.2
    y[:, 1] += 1.1
    return y.reshape(-1)


def _host_rng(seed):
    return np.random.Generator(np.random.Philox(seed))


def _solve_start(case, seed):
    if case["problem"] == "bruss":
        return _bruss_start_dev(case["N"], seed)
    return _lv_start_dev(case["N"], seed)


def _ensemble_inputs(case, seed):
    g = _host_rng(seed)
    prm = np.exp(g.uniform(math.log(0.1), math.log(2.0), (case["count"], 4)))
    y0 = g.uniform(0.5, 2.0, (case["count"], 2))
    return torch.from_numpy(prm).cuda(), torch.from_numpy(y0).cuda()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "solve":
        p = {"bruss": lambda n: rk_amd.Bruss2D(n, ALPHA),
             "pairs": rk_amd.LV,
             "chain": lambda n: rk_amd.LVChain(n, diff=DIFF)}[case["problem"]](case["N"])
        y0 = _solve_start(case, seed)
        return dict(case=case, problem=p, y0=y0, y=torch.empty_like(y0))
    if kind == "host":
        y0 = _bruss_start_host(case["N"], _host_rng(seed))
        return dict(case=case, problem=rk_amd.Bruss2D(case["N"], ALPHA), y0=y0,
                    y=np.empty_like(y0))
    if kind == "ensemble":
        prm, y0 = _ensemble_inputs(case, seed)
        return dict(case=case, params=prm, y0=y0)
    # batch: sizes spread evenly over the ranges (the same in every seed), each
    # instance with its own start, diffusion and tolerance
    g = _host_rng(seed)
    inst = []
    for k in range(case["grids"]):
        N = case["nmin"] + (case["nmax"] - case["nmin"]) * (2 * k + 1) // (2 * case["grids"])
        p = rk_amd.Bruss2D(N, ALPHA * 2.0 ** ((k % 3) - 1))
        inst.append((p, case["te"], _bruss_start_host(N, g), (1e-4, 1e-6, 1e-8)[k % 3]))
    for k in range(case["chains"]):
        M = case["mmin"] + (case["mmax"] - case["mmin"]) * (2 * k + 1) // (2 * case["chains"])
        p = rk_amd.LVChain(M, diff=DIFF)
        inst.append((p, 8.0 * case["te"], _lv_start_host(M, g), (1e-4, 1e-6, 1e-8)[k % 3]))
    return dict(case=case, inst=inst)


# ---- one pass -------------------------------------------------------------------

def _result(y, st):
    return {"y": y, "acc": st.steps_acc, "rej": st.steps_rej, "t": st.t, "h": st.h}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "solve":
        st, _ = rk_amd.solve(state["problem"], case["method"], 0.0, case["te"], state["y0"],
                             state["y"], case["tol"], h0=H0, step_limit=case["step_limit"],
                             impl=case["impl"])
        return _result(state["y"], st)
    if kind == "host":
        st = rk_amd.solver(0.0, case["te"], state["y0"], state["y"], case["tol"],
                           state["problem"], case["method"], h0=H0,
                           step_limit=case["step_limit"])
        return _result(state["y"], st)
    if kind == "ensemble":
        y, acc, rej = lv_ensemble(state["params"], state["y0"], 0.0, case["te"], case["method"],
                                  case["tol"])
        return {"y": y, "acc": acc, "rej": rej}
    with rk_amd.Batch() as b:
        ids = [b.add(p, case["method"], 0.0, te, y0, tol, h0=H0)
               for p, te, y0, tol in state["inst"]]
        while b.run(1 << 20):
            pass
        ys, steps = [], []
        for i in ids:
            st, _ = b.status(i)
            ys.append(b.result(i))
            steps.append((st.steps_acc, st.steps_rej))
            b.remove(i)
    return {"y": ys, "steps": np.array(steps)}


# ---- the tables, for exact() and work() --------------------------------------------

_TABLES = {
    "RKF23": (2, "1/2 1/2 0", "1/6 1/6 4/6", ["1", "1/4 1/4"]),
    "DOPRI54": (5, "35/384 0 500/1113 125/192 -2187/6784 11/84 0",
                "5179/57600 0 7571/16695 393/640 -92097/339200 187/2100 1/40",
                ["1/5", "3/40 9/40", "44/45 -56/15 32/9",
                 "19372/6561 -25360/2187 64448/6561 -212/729",
                 "9017/3168 -355/33 46732/5247 49/176 -5103/18656",
                 "35/384 0 500/1113 125/192 -2187/6784 11/84"]),
    "VERNER65": (6, "3/80 0 4/25 243/1120 77/160 73/700 0 0",
                 "57/640 0 -16/65 1377/2240 121/320 0 891/8320 2/35",
                 ["1/18", "-1/12 1/4", "-2/81 4/27 8/81", "40/33 -4/11 -56/11 54/11",
                  "-369/73 72/73 5380/219 -12285/584 2695/1752",
                  "-8716/891 656/297 39520/891 -416/11 52/27 0",
                  "3015/256 -9/4 -4219/78 5985/128 -539/384 0 693/3328"]),
    "DOPRI87": (8, "14005451/335480064 0 0 0 0 -59238493/1068277825 181606767/758867731 "
                   "561292985/797845732 -1041891430/1371343529 760417239/1151165299 "
                   "118820643/751138087 -528747749/2220607170 1/4",
                "13451932/455176623 0 0 0 0 -808719846/976000145 1757004468/5645159321 "
                "656045339/265891186 -3867574721/1518517206 465885868/322736535 "
                "53011238/667516719 2/45 0",
                ["1/18", "1/48 1/16", "1/32 0 3/32", "5/16 0 -75/64 75/64", "3/80 0 0 3/16 3/20",
                 "29443841/614563906 0 0 77736583/692538347 -28693883/1125000000 "
                 "23124283/1800000000",
                 "16016141/946692911 0 0 61564180/158732637 22789713/633445777 "
                 "545815736/2771057229 -180193667/1043307555",
                 "39632708/573591083 0 0 -433636366/683701615 -421739975/2616292301 "
                 "100302831/723423059 790204164/839813087 800635310/3783071287",
                 "246121993/1340847787 0 0 -37695042795/15268766246 -309121744/1061227803 "
                 "-12992083/490766935 6005943493/2108947869 393006217/1396673457 "
                 "123872331/1001029789",
                 "-1028468189/846180014 0 0 8478235783/508512852 1311729495/1432422823 "
                 "-10304129995/1701304382 -48777925059/3047939560 15336726248/1032824649 "
                 "-45442868181/3398467696 3065993473/597172653",
                 "185892177/718116043 0 0 -3185094517/667107341 -477755414/1098053517 "
                 "-703635378/230739211 5731566787/1027545527 5232866602/850066563 "
                 "-4093664535/808688257 3962137247/1805957418 65686358/487910083",
                 "403863854/491063109 0 0 -5068492393/434740067 -411421997/543043805 "
                 "652783627/914296604 11173962825/925320556 -13158990841/6184727034 "
                 "3936647629/1978049680 -160528059/685178525 248638103/1413531060 0"]),
}


def _row(text):
    return [float(v.split("/")[0]) / float(v.split("/")[1]) if "/" in v else float(v)
            for v in text.split()]


def _table(name):
    order, b, bh, rows = _TABLES[name]
    b, bh = _row(b), _row(bh)
    return order, [[]] + [_row(r) for r in rows], b, [x - z for x, z in zip(b, bh)]


# ---- the values in 64 bits, with plain torch --------------------------------------

def _bruss_rhs(N):
    coef = ALPHA * (N - 1.0) * (N - 1.0)

    def f(y):
        w = y.view(N, N, 2)
        lap = -4.0 * w
        lap[1:] += w[:-1]
        lap[0] += w[1]
        lap[:-1] += w[1:]
        lap[-1] += w[-2]
        lap[:, 1:] += w[:, :-1]
        lap[:, 0] += w[:, 1]
        lap[:, :-1] += w[:, 1:]
        lap[:, -1] += w[:, -2]
        lap *= coef
        u, v = w[..., 0], w[..., 1]
        uuv = u * u * v
        lap[..., 0] += 1.0 + uuv - 4.4 * u
        lap[..., 1] += 3.4 * u - uuv
        return lap.view(-1)
    return f


def _lv_rhs(diff):
    c0, d0, d1, c1 = LV_CONST

    def f(y):
        w = y.view(-1, 2)
        x, z = w[:, 0], w[:, 1]
        out = torch.stack((c0 * x - d0 * x * z, d1 * x * z - c1 * z), dim=1)
        if diff:
            out += diff * (torch.roll(w, 1, 0) + torch.roll(w, -1, 0) - 2.0 * w)
        return out.view(-1)
    return f


def _new_h(h, err, tol, order):
    f = 2.0 if err == 0.0 else 0.9 * (tol / err) ** (1.0 / (order + 1.0))
    return h * min(2.0, max(0.5, f))


def _integrate(f, y, te, tol, limit, table):
    order, A, b, e = table
    t, h, acc, rej = 0.0, H0, 0, 0
    while t < te and (limit <= 0 or acc + rej < limit):
        F = []
        for row in A:
            w = y
            for a, Fi in zip(row, F):
                if a:
                    w = torch.add(w, Fi, alpha=h * a)
            F.append(f(w))
        dy, er = torch.zeros_like(y), torch.zeros_like(y)
        for bi, ei, Fi in zip(b, e, F):
            if bi:
                dy.add_(Fi, alpha=h * bi)
            if ei:
                er.add_(Fi, alpha=h * ei)
        yn = y + dy
        err = float((er.abs() / torch.maximum(yn.abs(), y.abs())).max())
        if err <= tol:
            t, y, acc = t + h, yn, acc + 1
        else:
            rej += 1
        h = min(_new_h(h, err, tol, order), te - t)
    return y, t, h


def _exact_ensemble(case, seed):
    prm, y = _ensemble_inputs(case, seed)
    order, A, b, e = _table(case["method"])
    te, tol = case["te"], case["tol"]
    t = torch.zeros(case["count"], dtype=torch.float64, device="cuda")
    h = torch.full_like(t, 10.0 * tol)
    out, live = y.clone(), torch.arange(case["count"], device="cuda")
    while live.numel():
        c0, d0, d1, c1 = prm.unbind(1)

        def f(w):
            x, z = w[:, 0], w[:, 1]
            return torch.stack((c0 * x - d0 * x * z, d1 * x * z - c1 * z), dim=1)
        F, hc = [], h[:, None]
        for row in A:
            w = y
            for a, Fi in zip(row, F):
                if a:
                    w = w + (hc * a) * Fi
            F.append(f(w))
        dy = sum((hc * bi) * Fi for bi, Fi in zip(b, F) if bi)
        er = sum((hc * ei) * Fi for ei, Fi in zip(e, F) if ei)
        yn = y + dy
        err = (er.abs() / torch.maximum(yn.abs(), y.abs())).amax(1)
        ok = err <= tol
        t = torch.where(ok, t + h, t)
        y = torch.where(ok[:, None], yn, y)
        h = h * (0.9 * (tol / err) ** (1.0 / (order + 1.0))).clamp(0.5, 2.0)
        h = torch.minimum(h, te - t)
        out[live] = y
        keep = t < te
        live, prm, y, t, h = live[keep], prm[keep], y[keep], t[keep], h[keep]
    return {"y": out, "acc": None, "rej": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return None                     # dozens of full solves, one after another
    if kind == "ensemble":
        return _exact_ensemble(case, seed)
    table = _table(case["method"])
    if kind == "host":
        y0 = torch.from_numpy(_bruss_start_host(case["N"], _host_rng(seed))).cuda()
        f = _bruss_rhs(case["N"])
    else:
        y0 = _solve_start(case, seed)
        f = {"bruss": lambda: _bruss_rhs(case["N"]), "pairs": lambda: _lv_rhs(0.0),
             "chain": lambda: _lv_rhs(DIFF)}[case["problem"]]()
    y, t, h = _integrate(f, y0, case["te"], case["tol"], case["step_limit"], table)
    if kind == "host":
        y = y.cpu().numpy()
    return {"y": y, "acc": None, "rej": None, "t": t, "h": h}


# ---- work --------------------------------------------------------------------------

# length of the stable interval on the negative real axis: how far one step of
# a stability-limited solve gets
_STABLE = {"RKF23": 2.5, "DOPRI54": 3.3, "VERNER65": 4.2, "DOPRI87": 5.1}


def _flops(method, rhs):
    """Per component and step: the right-hand side of every stage, a multiply
    and an add for each non-zero coefficient, the error quotient."""
    _, A, b, e = _table(method)
    nz = sum(1 for row in A for a in row if a) + sum(1 for x in b + e if x)
    return len(b) * rhs + 2 * nz + 4


def _bruss_steps(N, alpha, te, method, limit):
    steps = 20 + te * 8.0 * alpha * (N - 1.0) ** 2 / _STABLE[method]
    return min(limit, steps) if limit else steps


def _lv_steps(te, tol, method):
    # smooth oscillation: about the local error's share of a period per step
    order = _TABLES[method][0]
    return 12 + te * 0.25 * (1e-4 / tol) ** (1.0 / (order + 1.0))


def work(case):
    """A step has to read y and write y_new once: 16 bytes per component."""
    kind, m = case["kind"], case["method"]
    todo = []                           # (components, steps, rhs operations)
    if kind == "host" or case.get("problem") == "bruss":
        todo.append((2 * case["N"] ** 2,
                     _bruss_steps(case["N"], ALPHA, case["te"], m, case["step_limit"]), 10))
    elif kind == "solve":
        todo.append((2 * case["N"], _lv_steps(case["te"], case["tol"], m),
                     4 if case["problem"] == "pairs" else 8))
    elif kind == "ensemble":
        n = 2 * case["count"]
        # state stays with the thread: constants, start and result move once
        return {"bytes": 40.0 * n,
                "flops": n * 3 * _lv_steps(case["te"], case["tol"], m) * _flops(m, 4)}
    else:
        for k in range(case["grids"]):
            N = case["nmin"] + (case["nmax"] - case["nmin"]) * (2 * k + 1) // (2 * case["grids"])
            todo.append((2 * N * N, _bruss_steps(N, ALPHA * 2.0 ** ((k % 3) - 1), case["te"], m, 0),
                         10))
        for k in range(case["chains"]):
            M = case["mmin"] + (case["mmax"] - case["mmin"]) * (2 * k + 1) // (2 * case["chains"])
            todo.append((2 * M, _lv_steps(8.0 * case["te"], 1e-6, m), 8))
    return {"bytes": float(sum(16.0 * n * s for n, s, _ in todo)),
            "flops": float(sum(n * s * _flops(m, r) for n, s, r in todo))}
