"""Performance cases of the HELLO hot path on one MI355X.

Each case is one call a user of the framework makes, through its public entry points, on inputs that are on the GPU
beforehand:

* ``pricing``      the optimality check of one hierarchy level: ``ScanExtension.fused_bidir_topk_stats_raw`` (squared
                   Euclidean cost, both directions' candidate lists and the certificate)
* ``chunk``        the same for one query chunk against a resident side (``ResidentSide``, ``pricing_l2sq``)
* ``directional``  the initial assignment scan: ``ScanExtension.initialization_directional_topk_raw``
* ``norm``         the optimality check with an l1 / linf / l2 cost: ``ScanExtension.fused_gcost_bidir_certificate``
* ``norm_init``    the initial assignment scan with such a cost: ``ScanExtension.fused_gcost_topk``
* ``sddmm``        squared Euclidean costs on a CSR support: ``lowrank_csr_costs``
* ``pairs``        costs of a pair list, as every restricted LP starts: ``lowrank_pair_costs`` / ``norm_pair_costs``
* ``lp``           a restricted transport LP: ``NativeRestrictedOTPDLP.solve_restricted``
* ``solve``        a whole solve: ``solve``

``listed`` names the cases, ``draw`` gives more of the same ranges, ``exact`` recomputes a case in plain torch in 64
bits. Duals of the scans are those of a refinement in progress: g small, f the c-transform over a sample of the other
side, so that each row has some ten violated pairs.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "hello-ot_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "hello-ot_amd"))

DEV = "cuda"
NORMS = {"l1": 0, "linf": 1, "l2": 2}


def listed():
    return [
        # the finest level of a small solve (2048 points, d = 32, the quickstart's Brenier problem): launches and
        # latency
        {"name": "pricing_2048_d32", "kind": "pricing", "m": 2048, "n": 2048, "d": 32, "k": 2},
        # a low-dimensional point cloud with unequal, odd sizes
        {"name": "pricing_60001_d4", "kind": "pricing", "m": 60001, "n": 65536, "d": 4, "k": 2},
        # the isolated scan of the benchmark: 131072 x 131072, d = 64, k = 8
        {"name": "pricing_131072_d64_k8", "kind": "pricing", "m": 131072, "n": 131072, "d": 64, "k": 8},
        # a rectangular level's initial assignment (16 best per source point) on 2048 features
        {"name": "directional_d2048_k16", "kind": "directional", "m": 16384, "n": 65536, "d": 2048, "k": 16},
        # one query chunk of a large solve on 8192 features, against a resident side
        {"name": "chunk_8192_d8192", "kind": "chunk", "m": 8192, "n": 163840, "d": 8192, "k": 2},
        # the optimality check of the benchmark's l1 solve (d = 8), one level below its finest size
        {"name": "norm_l1_262144_d8", "kind": "norm", "cost": "l1", "precision": "fp32", "m": 262144, "n": 262144,
         "d": 8, "k": 2},
        # Euclidean cost on 50 principal components, unequal sizes
        {"name": "norm_l2_30000_d50", "kind": "norm", "cost": "l2", "precision": "fp32", "m": 30000, "n": 40961,
         "d": 50, "k": 2},
        # the benchmark's SDDMM: 262144 rows, 16 nonzeros each, d = 256
        {"name": "sddmm_262144_d256", "kind": "sddmm", "m": 262144, "n": 262144, "d": 256, "per_row": 16},
        # the support costs of a level of 65536 points on 2048 features
        {"name": "pairs_d2048", "kind": "pairs", "cost": "l2^2", "precision": "fp64", "m": 65536, "n": 65536, "d": 2048,
         "count": 1500000},
        # the restricted LP of a small level (a few thousand points): launches and latency
        {"name": "lp_4096", "kind": "lp", "n": 4096, "picks": 12, "iterations": 1000},
        # the restricted LP of the benchmark's finest l1 / linf level (524288 points a side, some 12 million edges)
        {"name": "lp_524288", "kind": "lp", "n": 524288, "picks": 14, "iterations": 400},
        # a whole solve: the quickstart's Brenier problem
        {"name": "solve_2048_d32", "kind": "solve", "n": 2048, "d": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    # (squared Euclidean scans below 64 features: clouds of up to 65536 points a side)
    kind = rng.choice(["pricing", "pricing", "chunk", "directional", "norm", "norm", "norm_init", "sddmm", "pairs", "lp",
                       "lp", "solve"])
    while True:
        m, n = _log_int(rng, 700, 140000), _log_int(rng, 700, 140000)
        if kind == "pricing":
            d = _log_int(rng, 2, 8192)
            if m * n * max(d, 32) <= 1 << 40 and (m + n) * d <= 1 << 31 and (d >= 64 or max(m, n) <= 65536):
                return {"kind": kind, "m": m, "n": n, "d": d, "k": rng.choice([1, 2, 2, 4, 8])}
        elif kind == "chunk":
            d = _log_int(rng, 512, 8192)
            m, n = _log_int(rng, 256, 8192), _log_int(rng, 16384, 163840)
            return {"kind": kind, "m": m, "n": n, "d": d, "k": rng.choice([1, 2, 2, 4])}
        elif kind == "directional":
            d = _log_int(rng, 2, 4096)
            if m * n * max(d, 32) <= 1 << 40 and (m + n) * d <= 1 << 31 and (d >= 64 or max(m, n) <= 65536):
                return {"kind": kind, "m": m, "n": n, "d": d, "k": rng.choice([8, 16, 16])}
        elif kind in ("norm", "norm_init"):
            d = _log_int(rng, 2, 100)
            precision = rng.choice(["fp32", "fp32", "fp32", "fp64"])
            if m * n * max(d, 8) <= 1 << 36:
                return {"kind": kind, "cost": rng.choice(["l1", "linf", "l2"]), "precision": precision, "m": m, "n": n,
                        "d": d, "k": rng.choice([1, 2, 2, 4]) if kind == "norm" else 16}
        elif kind == "sddmm":
            d, per_row = _log_int(rng, 4, 2048), rng.randint(3, 24)
            if m * per_row * max(d, 16) <= 1 << 31:
                return {"kind": kind, "m": m, "n": n, "d": d, "per_row": per_row}
        elif kind == "pairs":
            d, count = _log_int(rng, 2, 8192), _log_int(rng, 2000, 8000000)
            if count * max(d, 16) <= 1 << 32 and (m + n) * d <= 1 << 31:
                cost = rng.choice(["l2^2", "l1", "linf", "l2"])
                return {"kind": kind, "cost": cost, "precision": "fp64" if cost == "l2^2" else rng.choice(["fp32", "fp64"]),
                        "m": m, "n": n, "d": d, "count": count}
        elif kind == "lp":
            return {"kind": kind, "n": _log_int(rng, 700, 400000), "picks": rng.randint(5, 14),
                    "iterations": 200 * rng.randint(1, 2)}
        else:
            return {"kind": kind, "n": _log_int(rng, 1100, 4000), "d": _log_int(rng, 5, 64)}


# ----------------------------------------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------------------------------------
def _generator(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFF)
    return g


def _mixture(rows, d, seed, salt):
    """Rows of a 64-component Gaussian mixture (means ~ N(0, 4 I), unit covariance)."""
    g = _generator(seed, salt)
    means = 2.0 * torch.randn(64, d, generator=g, device=DEV)
    out = torch.empty(rows, d, dtype=torch.float32, device=DEV)
    for s in range(0, rows, 32768):
        e = min(rows, s + 32768)
        label = torch.randint(0, 64, (e - s,), generator=g, device=DEV)
        out[s:e] = torch.randn(e - s, d, generator=g, device=DEV) + means[label]
    return out


def _sqnorms(x):
    out = torch.empty(x.shape[0], dtype=torch.float64, device=DEV)
    step = max(1, (1 << 26) // x.shape[1])
    for s in range(0, x.shape[0], step):
        out[s:s + step] = x[s:s + step].double().square().sum(1)
    return out


def _sample(n, seed):
    size = min(n, max(64, min(n // 10, 8192)))
    return torch.randperm(n, device=DEV, generator=_generator(seed, 5))[:size]


def _l2sq_inputs(case, seed):
    m, n, d = case["m"], case["n"], case["d"]
    x, y = _mixture(m, d, seed, 1), _mixture(n, d, seed, 2)
    p, q = _sqnorms(x), _sqnorms(y)
    g = 0.01 * q.mean() * torch.randn(n, dtype=torch.float64, device=DEV, generator=_generator(seed, 3))
    at = _sample(n, seed)
    ys, off = y[at], q[at] - g[at]
    f = torch.empty(m, dtype=torch.float64, device=DEV)
    for s in range(0, m, 4096):
        f[s:s + 4096] = p[s:s + 4096] + (off[None, :] - 2.0 * (x[s:s + 4096] @ ys.T).double()).min(1).values
    return x, y, p, q, f, g


def _norm_tile(x, y, cost, dtype):
    """Dense costs of one block of rows, feature by feature in feature order."""
    acc = torch.zeros(x.shape[0], y.shape[0], dtype=dtype, device=x.device)
    x, yt = x.to(dtype), y.to(dtype).T.contiguous()
    for t in range(x.shape[1]):
        z = x[:, t, None] - yt[t]
        if cost == "l2":
            acc.addcmul_(z, z)
        elif cost == "l1":
            acc.add_(z.abs_())
        else:
            torch.maximum(acc, z.abs_(), out=acc)
    return acc.sqrt_() if cost == "l2" else acc


def _norm_inputs(case, seed):
    """Points uniform in the unit cube, as the benchmark's l1 / linf problems."""
    m, n, d = case["m"], case["n"], case["d"]
    g0 = _generator(seed, 1)
    x = torch.rand(m, d, generator=g0, device=DEV)
    y = torch.rand(n, d, generator=g0, device=DEV)
    g = 0.01 * torch.randn(n, dtype=torch.float64, device=DEV, generator=_generator(seed, 3))
    at = _sample(n, seed)
    ys, gs = y[at], g[at]
    f = torch.empty(m, dtype=torch.float64, device=DEV)
    for s in range(0, m, 16384):
        f[s:s + 16384] = (_norm_tile(x[s:s + 16384], ys, case["cost"], torch.float32).double() - gs[None, :]).min(1).values
    return x, y, f, g


def _lp_inputs(case, seed):
    """A HELLO support: sources and targets on a line, each joined to about `picks` near ones on the other side (some of
    them popular), plus the northwest-corner basis of the shuffled numbering; edges in key order. The count depends on
    the case alone: surplus pairs are dropped at random."""
    n, picks = case["n"], case["picks"]
    gen = _generator(seed, 1)
    place = torch.arange(n, device=DEV).repeat_interleave(picks)

    def near():
        step = torch.empty(place.numel(), dtype=torch.float64, device=DEV).exponential_(1.0 / 30.0, generator=gen)
        sign = torch.randint(0, 2, (place.numel(),), generator=gen, device=DEV) * 2 - 1
        to = (place + (step * sign).long()).clamp_(0, n - 1)
        popular = torch.rand(place.numel(), generator=gen, device=DEV) < 0.25
        return torch.where(popular, torch.div(to, 32, rounding_mode="floor") * 32, to)

    rows, cols = torch.cat((place, near())), torch.cat((near(), place))
    a = 0.5 + torch.rand(n, dtype=torch.float64, generator=gen, device=DEV)
    b = 0.5 + torch.rand(n, dtype=torch.float64, generator=gen, device=DEV)
    a, b = a / a.sum(), b / b.sum()
    number_s = torch.randperm(n, generator=gen, device=DEV)
    number_t = torch.randperm(n, generator=gen, device=DEV)
    ca, cb = a.cumsum(0), b.cumsum(0)
    cuts = torch.cat((ca.new_zeros(1), ca[:-1], cb[:-1], ca.new_ones(1))).sort().values
    mid, flow = 0.5 * (cuts[1:] + cuts[:-1]), (cuts[1:] - cuts[:-1]).clamp_min(0.0)
    basis_r = torch.searchsorted(ca, mid).clamp_max(n - 1)
    basis_c = torch.searchsorted(cb, mid).clamp_max(n - 1)
    basis_key = torch.unique(basis_r * n + basis_c)
    near_key = torch.unique(number_s[rows] * n + number_t[cols])
    near_key = near_key[~torch.isin(near_key, basis_key)]
    keep = torch.randperm(near_key.numel(), generator=gen, device=DEV)[:_lp_edges(case) - basis_key.numel()]
    keys = torch.cat((near_key[keep], basis_key)).sort().values
    rows, cols = torch.div(keys, n, rounding_mode="floor"), keys.remainder(n)
    at_s, at_t = torch.empty_like(number_s), torch.empty_like(number_t)
    at_s[number_s], at_t[number_t] = torch.arange(n, device=DEV), torch.arange(n, device=DEV)
    gap = (at_s[rows] - at_t[cols]).double() / 64.0
    noise = torch.rand(keys.numel(), dtype=torch.float64, generator=gen, device=DEV)
    costs = 0.2 + (gap * gap).clamp_max(4.0) + 0.3 * noise
    x0 = torch.zeros(keys.numel(), dtype=torch.float64, device=DEV)
    x0.index_add_(0, torch.searchsorted(keys, basis_r * n + basis_c), flow)
    y0 = torch.zeros(2 * n, dtype=torch.float64, device=DEV)
    y0[:n].scatter_reduce_(0, rows, costs, "amin", include_self=False)
    return {"rows": rows, "cols": cols, "costs": costs, "a": a, "b": b, "x0": x0, "y0": y0}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("pricing", "chunk", "directional"):
        from hello_ot_amd.kernels.generic_scan import ResidentSide, ScanExtension

        x, y, p, q, f, g = _l2sq_inputs(case, seed)
        if kind == "directional":   # the query side's duals are not known yet
            return {"case": case, "scan": ScanExtension(), "x": x, "y": y, "qb": -p, "db": g - q}
        state = {"case": case, "x": x, "y": y, "p": p, "q": q, "qb": f - p, "db": g - q}
        if kind == "chunk":
            state["side"] = ResidentSide(y)
        else:
            state["scan"] = ScanExtension()
        return state
    if kind in ("norm", "norm_init"):
        from hello_ot_amd.kernels.generic_scan import ScanExtension

        x, y, f, g = _norm_inputs(case, seed)
        return {"case": case, "scan": ScanExtension(), "x": x, "y": y, "f": f, "g": g}
    if kind == "sddmm":
        m, n, d, per_row = case["m"], case["n"], case["d"], case["per_row"]
        gen = _generator(seed, 4)
        x, y = _mixture(m, d, seed, 1), _mixture(n, d, seed, 2)
        keys = torch.arange(m, device=DEV).repeat_interleave(per_row) * n + torch.randint(0, n, (m * per_row,),
                                                                                         generator=gen, device=DEV)
        keys = keys.sort().values   # a column drawn twice in a row stays twice, so every seed has the same count
        rowptr = torch.arange(0, m * per_row + 1, per_row, dtype=torch.int32, device=DEV)
        return {"case": case, "x": x, "y": y, "p": _sqnorms(x), "q": _sqnorms(y), "rowptr": rowptr,
                "col": keys.remainder(n).int()}
    if kind == "pairs":
        m, n, d = case["m"], case["n"], case["d"]
        gen = _generator(seed, 4)
        x, y = _mixture(m, d, seed, 1), _mixture(n, d, seed, 2)
        keys = torch.randint(0, m * n, (case["count"],), generator=gen, device=DEV).sort().values
        state = {"case": case, "x": x, "y": y, "rows": torch.div(keys, n, rounding_mode="floor"), "cols": keys.remainder(n)}
        if case["cost"] == "l2^2":
            state["p"], state["q"] = _sqnorms(x), _sqnorms(y)
        return state
    if kind == "lp":
        from hello_ot_amd.lp import NativeRestrictedOTPDLP

        solver = NativeRestrictedOTPDLP(device=DEV, evaluation_frequency=200, iteration_limit=case["iterations"])
        return {"case": case, "solver": solver, **_lp_inputs(case, seed)}
    # solve: points from N(0, I) and their images under the gradient map x + 2 tanh(x), in another order
    n, d = case["n"], case["d"]
    gen = _generator(seed, 1)
    x = torch.randn(n, d, generator=gen, device=DEV)
    order = torch.randperm(n, generator=gen, device=DEV)
    return {"case": case, "x": x, "y": (x + 2.0 * torch.tanh(x))[order], "order": order}


# ----------------------------------------------------------------------------------------------------------
# one pass
# ----------------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "pricing":
        return state["scan"].fused_bidir_topk_stats_raw(state["x"], state["y"], state["p"], state["q"], state["qb"],
                                                        state["db"], 4096, 4096, 32, case["k"], True, True, False, 0,
                                                        2.0)[:5]
    if kind == "chunk":
        from hello_ot_amd.kernels.generic_scan import pricing_l2sq

        return pricing_l2sq(state["x"], state["y"], state["p"], state["q"], state["qb"], state["db"], case["k"],
                            linf=True, resident=state["side"])
    if kind == "directional":
        return state["scan"].initialization_directional_topk_raw(state["x"], state["y"], state["qb"], state["db"], 4096,
                                                                 4096, case["k"], 2.0)
    if kind == "norm":
        return state["scan"].fused_gcost_bidir_certificate(state["x"], state["y"], state["f"], state["g"], case["k"],
                                                           NORMS[case["cost"]],
                                                           compute_precision=1 if case["precision"] == "fp64" else 0)
    if kind == "norm_init":
        return state["scan"].fused_gcost_topk(state["x"], state["y"], state["g"], case["k"], NORMS[case["cost"]],
                                              compute_precision=1 if case["precision"] == "fp64" else 0)
    if kind == "sddmm":
        from hello_ot_amd.costs.pairs import lowrank_csr_costs

        return lowrank_csr_costs(state["x"], state["y"], state["p"], state["q"], state["rowptr"], state["col"])
    if kind == "pairs":
        from hello_ot_amd.costs.pairs import lowrank_pair_costs, norm_pair_costs

        if case["cost"] == "l2^2":
            return lowrank_pair_costs(state["x"], state["y"], state["p"], state["q"], state["rows"], state["cols"])
        return norm_pair_costs(state["x"], state["y"], state["rows"], state["cols"], NORMS[case["cost"]],
                               precision=case["precision"])
    if kind == "lp":
        r = state["solver"].solve_restricted(rows=state["rows"], cols=state["cols"], costs=state["costs"],
                                             source_mass=state["a"], target_mass=state["b"],
                                             warm_start_primal=state["x0"], warm_start_dual=state["y0"],
                                             tolerance=1e-9)
        return [r.x, r.y, r.obj_val, r.dual_obj_val]
    from hello_ot_amd import SolverOptions, solve

    r = solve(state["x"], state["y"], options=SolverOptions(verbose="off"))
    # the plan as a matrix: how many entries a solver leaves just above zero, and the duals inside the optimal face, are
    # not determined by the problem
    return {"objective": r.objective, "plan": r.solution.to_sparse_matrix().to_dense()}


# ----------------------------------------------------------------------------------------------------------
# the work of one pass, and how far two correct ones may differ
# ----------------------------------------------------------------------------------------------------------
def _lp_edges(case):
    """Edges of a case: the picks of both sides less the pairs both drew, and the basis."""
    return 3 * case["n"] * case["picks"] // 2 + 2 * case["n"] - 1


def work(case):
    kind = case["kind"]
    if kind == "lp":
        # per iteration: read and write the iterate, read its anchor, cost and two endpoints of each edge, and a node's
        # dual, anchor, scale, mass
        e, v = _lp_edges(case), 2 * case["n"]
        return {"bytes": case["iterations"] * (40.0 * e + 56.0 * v), "flops": case["iterations"] * (12.0 * e + 10.0 * v)}
    if kind == "solve":
        # the scans of the finest level: two initial directions and one check
        n, d = case["n"], case["d"]
        return {"bytes": 8.0 * n * d + 8.0 * n * n, "flops": 3 * 2.0 * n * n * d}
    m, n, d = case["m"], case["n"], case["d"]
    sides = 4.0 * (m + n) * d
    if kind in ("pricing", "chunk"):
        return {"bytes": sides + 16.0 * (m + n) + 12.0 * case["k"] * (m + n), "flops": 2.0 * m * n * d}
    if kind == "directional":
        return {"bytes": sides + 8.0 * (m + n) + 12.0 * case["k"] * m, "flops": 2.0 * m * n * d}
    if kind == "norm":
        return {"bytes": sides + 8.0 * (m + n) + 16.0 * case["k"] * (m + n), "flops": 2.0 * m * n * d}
    if kind == "norm_init":
        return {"bytes": sides + 8.0 * n + 16.0 * case["k"] * m, "flops": 2.0 * m * n * d}
    if kind == "sddmm":
        nnz = m * case["per_row"]
        return {"bytes": sides + 8.0 * (m + n) + 4.0 * m + 12.0 * nnz, "flops": 2.0 * nnz * d}
    count = case["count"]
    return {"bytes": min(sides, 8.0 * count * d) + 24.0 * count, "flops": 2.0 * count * d}


def tolerance(case):
    kind = case["kind"]
    if kind in ("pricing", "chunk"):
        # the lists' scores are fp64 (1e-14 off); the certificate's sums come from fp32 costs (up to 2e-8 off)
        return {"rel": 2e-7, "differ": 1e-5}
    if kind == "directional":
        return {"rel": 1e-14, "differ": 1e-5}
    if kind in ("norm", "norm_init"):
        # fp32 costs of up to 100 features: scores up to 7e-7 off, the violations' squares 4e-8
        return {"rel": 3e-6 if case["precision"] == "fp32" else 1e-12, "differ": 1e-5}
    if kind in ("sddmm", "pairs"):
        return {"rel": 4e-7 if case.get("precision") == "fp32" else 1e-14}
    if kind == "lp":
        # hundreds of iterations on sums in another order: 2e-13 off
        return {"rel": 1e-12, "max": 1e-9}
    # the solver stops at 1e-6 of the costs: plans up to 4e-6 off
    return {"rel": 2e-5, "max": 1e-2}


# ----------------------------------------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ----------------------------------------------------------------------------------------------------------
def _best(values, k, dim):
    """The k largest along `dim`, descending (values is overwritten)."""
    v, i = [], []
    for _ in range(k):
        top = values.max(dim)
        v.append(top.values)
        i.append(top.indices)
        values.scatter_(dim, top.indices.unsqueeze(dim), -math.inf)
    return torch.stack(v, 1), torch.stack(i, 1)


def _exact_scan(m, n, k, score, columns):
    """Row (and column) lists and certificate sums of score(s, e) -> (scores, costs) of rows s..e, costs None: none."""
    rv, ri, cv, ci = [], [], None, None
    num = den = count = mx = cmax = 0.0
    step = max(1, min(m, (1 << 28) // n))
    for s in range(0, m, step):
        e = min(m, s + step)
        sig, cost = score(s, e)
        if cost is not None:
            pos = sig.clamp_min(0.0)
            num += float(pos.square_().sum())
            del pos
            count += float((sig > 0).sum())
            mx = max(mx, float(sig.max()))
            cmax = max(cmax, float(cost.max()), -float(cost.min()))
            den += float(cost.square_().sum())
            del cost
        v, i = _best(sig.clone() if columns else sig, min(k, n), 1)
        rv.append(v)
        ri.append(i.int())
        if columns:
            v, i = _best(sig, min(k, e - s), 0)
            i = i + s
            if cv is not None:
                v, i = torch.cat((cv, v), 1), torch.cat((ci, i), 1)
                v, at = torch.sort(v, dim=1, descending=True, stable=True)
                i = i.gather(1, at)
            cv, ci = v[:, :k].contiguous(), i[:, :k].contiguous()
    return torch.cat(rv), torch.cat(ri), cv, None if ci is None else ci.int(), (num, den, count, mx, cmax)


def _exact_lp(case, state):
    """The Halpern-reflected PDHG with degree-sqrt scaling, step 0.998, PID weight restarts and checks every 200
    iterations, on torch tensors."""
    rows, cols, c, x0, y0 = state["rows"], state["cols"], state["costs"], state["x0"], state["y0"]
    n, e = case["n"], rows.numel()
    b = torch.cat((state["a"], state["b"]))
    ends = torch.cat((rows, cols + n))
    root2 = math.sqrt(2.0)

    def gather(node):
        return node[rows] + node[cols + n]

    def sums(edge):
        return torch.zeros(2 * n, dtype=torch.float64, device=c.device).index_add_(0, ends, torch.cat((edge, edge)))

    scale = sums(torch.ones_like(c)).clamp_min(1.0).sqrt()
    ns, bs, cs = root2 * scale, b / scale, c / root2
    x = x0.clamp_min(0.0) * root2
    y = y0 * scale
    ax, ay, px, py = x, y, x, y
    weight = max(float(cs.norm()) / max(float(bs.norm()), 1e-16), 1e-16)
    mass_norm, cost_norm = float(b.norm()), float(c.norm())
    best_weight, error_sum, best_balance = weight, 0.0, math.inf
    initial = last = fixed = math.inf
    total = inner = 0
    while True:
        restart = False
        if total % 200 == 0:
            z = py / scale
            ap = float((sums(px / root2) - b).norm())
            ad = float((gather(z) - c).clamp_min_(0.0).norm())
            rp, rd = ap / (1.0 + mass_norm), ad / (1.0 + cost_norm)
            pobj, dobj = float(c @ (px / root2)), float(b @ z)
            if total >= case["iterations"]:
                return [px / root2, z, pobj, dobj]
            if total == 200:
                restart = True
            elif total > 200:
                restart = inner >= 0.36 * total or fixed <= 0.2 * initial or (fixed <= 0.5 * initial and fixed > last)
            last = fixed
            if restart:
                pd, dd = float((px - ax).norm()), float((py - ay).norm())
                ratio = rd / max(rp, 1e-300)
                if 1e-16 < pd < 1e12 and 1e-16 < dd < 1e12 and 1e-8 < ratio < 1e8:
                    error = math.log(dd) - math.log(pd) - math.log(weight)
                    error_sum = 0.3 * error_sum + error
                    weight *= math.exp(0.99 * error + 0.01 * error_sum)
                else:
                    weight, error_sum = best_weight, 0.0
                if rp > 0 and rd > 0 and abs(math.log10(rd / rp)) < best_balance:
                    best_balance, best_weight = abs(math.log10(rd / rp)), weight
                inner, last = 0, math.inf
                x, y, ax, ay = px, py, px, py
        halpern = (inner + 1) / (inner + 2)
        px = (x - (0.998 / weight) * (cs - gather(y / ns))).clamp_min_(0.0)
        rx = 2.0 * px - x
        py = y - (0.998 * weight) * (sums(rx) / ns - bs)
        ry = 2.0 * py - y
        if restart or (total + 1) % 200 == 0:
            dx, dy = rx - x, ry - y
            fixed = math.sqrt(max(0.0, float(dx @ dx) * weight + float(dy @ dy) / weight
                                  + 2.0 * 0.998 * float(gather(dy / ns) @ dx)))
            if restart:
                initial = fixed
        x, y = halpern * rx + (1.0 - halpern) * ax, halpern * ry + (1.0 - halpern) * ay
        total += 1
        inner += 1


def exact(case, seed):
    kind = case["kind"]
    state = prepare(case, seed)
    if kind in ("pricing", "chunk", "directional"):
        x, yt, qb, db = state["x"].double(), state["y"].double().T.contiguous(), state["qb"], state["db"]

        def score(s, e):
            dot = (x[s:e] @ yt).mul_(2.0)
            cost = None if kind == "directional" else (state["p"][s:e, None] + state["q"][None, :]) - dot
            return dot.add_(qb[s:e, None]).add_(db[None, :]), cost

        rv, ri, cv, ci, st = _exact_scan(case["m"], case["n"], case["k"], score, kind != "directional")
        if kind == "directional":
            return [rv, ri]
        st = (st[0], st[1], st[2], st[4]) if kind == "pricing" else st
        return [rv, ri, cv, ci, torch.tensor(st, dtype=torch.float64)]
    if kind in ("norm", "norm_init"):
        x, y, f, g = state["x"], state["y"], state["f"], state["g"]

        def score(s, e):
            cost = _norm_tile(x[s:e], y, case["cost"], torch.float64)
            if kind == "norm_init":
                return g[None, :] - cost, None
            return (g[None, :] - cost).add_(f[s:e, None]), cost

        rv, ri, cv, ci, st = _exact_scan(case["m"], case["n"], case["k"], score, kind == "norm")
        if kind == "norm_init":
            return [-rv, ri.long()]
        return [rv, ri.long(), cv, ci.long(), st[0], st[1], st[3], st[4], int(st[2])]
    if kind in ("sddmm", "pairs"):
        if kind == "sddmm":
            rows, cols = torch.arange(case["m"], device=DEV).repeat_interleave(case["per_row"]), state["col"].long()
        else:
            rows, cols = state["rows"], state["cols"]
        out = torch.empty(rows.numel(), dtype=torch.float64, device=DEV)
        step = max(1, (1 << 27) // case["d"])
        for s in range(0, rows.numel(), step):
            i, j = rows[s:s + step], cols[s:s + step]
            u, v = state["x"][i].double(), state["y"][j].double()
            cost = case.get("cost", "l2^2")
            if cost == "l2^2":
                out[s:s + step] = (state["p"][i] + state["q"][j]) - 2.0 * (u * v).sum(1)
            elif cost == "l1":
                out[s:s + step] = (u - v).abs().sum(1)
            elif cost == "linf":
                out[s:s + step] = (u - v).abs().max(1).values
            else:
                out[s:s + step] = (u - v).square().sum(1).sqrt()
        return out
    if kind == "lp":
        return _exact_lp(case, state)
    n = case["n"]
    plan = torch.zeros(n, n, dtype=torch.float64, device=DEV)
    plan[state["order"], torch.arange(n, device=DEV)] = 1.0 / n
    gap = state["x"][state["order"]].double() - state["y"].double()
    return {"objective": float(gap.square().sum() / n), "plan": plan}


__all__ = ["draw", "exact", "listed", "prepare", "run", "tolerance", "work"]
