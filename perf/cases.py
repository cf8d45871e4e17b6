"""The work that users have this engine do, as cases that can be timed and checked.

Every case goes through the package's public entry points (cafe5_amd.model and
cafe5_amd.native).  Sizes are those of the repository's own workloads (12, 34,
60 and 100 taxa, bounds 20 to 500, one to 64 parameter points) or lie between
them.  The species tree belongs to the case; families, lambdas and alphas come
from the seed.  exact() repeats each result with plain torch in 64 bits.
"""
import math
import os

import numpy as np
import torch

import cafe5_amd
from cafe5_amd import model, native
from cafe5_amd.workloads import Tree

PATHS = {"plain64": native.PATH_PLAIN64, "batched64": native.PATH_BATCHED64, "batched32": native.PATH_BATCHED32,
         "batched16": native.PATH_BATCHED16}
# per-family bounds of the uneven workloads: the first of these with room for
# the family's largest count
LADDER = (20, 32, 48, 64, 96, 128, 160, 200)
SHAPES = os.path.join(os.path.dirname(os.path.abspath(cafe5_amd.__file__)), "tune_cache.txt")


def listed():
    return [
        # One score of the drop-in model on a table of the examples' size
        # (250 families of 12 mammals): what every CAFE run starts with, and
        # the smallest call, all latency.
        {"name": "score-plain64-250", "op": "infer", "path": "plain64", "taxa": 12, "families": 250, "bound": 116,
         "root": 83},
        # The default path called as a model with the error model and three
        # lambda classes: a mid-sized table, matrices built and inputs
        # uploaded on every call.
        {"name": "score-error-classes-5k", "op": "infer", "path": "batched32", "taxa": 34, "families": 5000,
         "bound": 150, "root": 150, "epsilon": 0.05, "classes": 3},
        # The drop-in model on a whole table under one bound for all families
        # (the reference's rule), where the pruning itself is the time.
        {"name": "score-plain64-10k", "op": "infer", "path": "plain64", "taxa": 34, "families": 10000, "bound": 200,
         "root": 200},
        # One step of a lambda search over a resident base model.
        {"name": "search-base-2k", "op": "plan", "path": "batched32", "taxa": 12, "families": 2000, "bound": 100,
         "root": 100, "points": 1},
        # The headline: a 64-point lambda grid over 20,000 families of uneven
        # sizes, every family's likelihood at every point.
        {"name": "grid-uneven-20k", "op": "plan", "path": "batched32", "taxa": 34, "families": 20000, "bound": 200,
         "root": 200, "points": 64, "uneven": True},
        # The same families in 64-bit arithmetic, as a user checks a grid.
        {"name": "grid-uneven-f64", "op": "plan", "path": "batched64", "taxa": 34, "families": 20000, "bound": 200,
         "root": 200, "points": 16, "uneven": True},
        # The split-FP16 path on its workload: error model, lambda classes, 60
        # taxa, an odd number of families.
        {"name": "search-error-f16-25k", "op": "plan", "path": "batched16", "taxa": 60, "families": 24999,
         "bound": 150, "root": 150, "points": 1, "epsilon": 0.05, "classes": 3},
        # One (lambda, alpha) step of the gamma model's search.
        {"name": "search-gamma-50k", "op": "gamma", "path": "batched32", "taxa": 34, "families": 50000, "bound": 100,
         "root": 100, "cats": 4, "alpha": 0.5, "lambda": 0.003},
        # The same at optimizer scale: 100 taxa, vectors of 501, 8 categories;
        # the largest call.
        {"name": "search-gamma-b500", "op": "gamma", "path": "batched32", "taxa": 100, "families": 16000,
         "bound": 500, "root": 500, "cats": 8, "alpha": 1.5, "lambda": 0.002},
        # Root vectors of simulated families, each with its own bound (the
        # conditional distributions of the p-values).
        {"name": "roots-pvalue-6k", "op": "roots", "path": "plain64", "taxa": 12, "families": 6000, "bound": 160,
         "root": 60},
        # Joint ancestral reconstruction of a whole table, the last step of a
        # run.
        {"name": "reconstruct-20k", "op": "reconstruct", "taxa": 34, "families": 20000, "bound": 200, "root": 200},
        # Transition matrices for a host consumer (get_matrix; simulation draws
        # from their rows), by the reference's closed form.
        {"name": "matrices-host-22", "op": "matrices", "algo": "closed", "taxa": 12, "bound": 200},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# most contraction work of a drawn case (about half of the largest listed one
# of its kind at most)
_MOST = {"plain64": 6e10, "batched64": 5e11, "batched32": 2e12, "batched16": 1e12, "reconstruct": 2.5e10}


def draw(rng):
    op = rng.choice(("infer", "infer", "plan", "plan", "gamma", "roots", "reconstruct", "matrices"))
    if op == "matrices":
        case = {"op": op, "algo": rng.choice(("closed", "recurrence")), "taxa": _log_int(rng, 3, 60),
                "bound": _log_int(rng, 15, 500)}
        while 2 * case["taxa"] * case["bound"] ** 2 > 6e6:
            case["bound"] = case["bound"] * 3 // 4
        return case
    case = {"op": op, "taxa": _log_int(rng, 4, 100), "families": _log_int(rng, 100, 20000),
            "bound": _log_int(rng, 20, 500)}
    case["root"] = rng.choice((case["bound"], max(10, int(case["bound"] * rng.uniform(0.3, 1.0)))))
    if op == "reconstruct":
        case["bound"] = min(case["bound"], 320)
        case["root"] = min(case["root"], case["bound"])
        path = op
    elif op == "roots":
        path = case["path"] = "plain64"
        case["bound"] = max(60, min(case["bound"], 300))
        case["root"] = min(case["root"], 200)
    else:
        path = case["path"] = rng.choice(("plain64", "batched64", "batched32", "batched32", "batched16"))
        if op == "plan":
            case["points"] = _log_int(rng, 1, 64)
        if op == "gamma":
            # categories whose matrices stay away from both ends, so that no
            # family's likelihood vanishes in one of them
            case["taxa"] = min(case["taxa"], 60)
            case["cats"] = rng.randint(2, 8)
            case["alpha"] = round(rng.uniform(0.8, 2.0), 3)
            case["lambda"] = round(math.exp(rng.uniform(math.log(1.5e-3), math.log(4e-3))), 6)
        elif rng.random() < 0.3:
            case["epsilon"] = 0.05
        if op != "gamma" and rng.random() < 0.3 and case["taxa"] >= 8:
            case["classes"] = 3
        if op == "plan" and case["bound"] >= 48 and rng.random() < 0.5:
            case["uneven"] = True
            case["root"] = case["bound"]
    per_family = 2.0 * (case["bound"] + 1) ** 2 * max(1, case["taxa"] - 2) * case.get("points", 1) * case.get("cats", 1)
    while per_family * 60 > _MOST[path]:
        for key in ("points", "cats"):
            if case.get(key, 1) > 2:
                case[key] = case[key] // 2
        case["bound"] = max(60, case["bound"] * 3 // 4)
        case["root"] = min(case["root"], case["bound"])
        per_family = (2.0 * (case["bound"] + 1) ** 2 * max(1, case["taxa"] - 2) * case.get("points", 1)
                      * case.get("cats", 1))
    case["families"] = max(50, min(case["families"], int(_MOST[path] / per_family)))
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _tree(case):
    """(parent, leaf_col, length): a pure-birth tree of height 100, children
    before parents, the root last."""
    taxa = case["taxa"]
    rng = np.random.default_rng(7000 + taxa)
    parent, born, died, active, t = [-1, 0, 0], [0.0, 0.0, 0.0], {0: 0.0}, [1, 2], 0.0
    while len(active) < taxa:
        t += rng.exponential(1.0 / len(active))
        u = active.pop(int(rng.integers(len(active))))
        died[u] = t
        for _ in range(2):
            active.append(len(parent))
            parent.append(u)
            born.append(t)
    end = t + rng.exponential(1.0 / len(active))
    n = len(parent)
    par = np.full(n, -1, dtype=np.int32)
    col = np.full(n, -1, dtype=np.int32)
    length = np.zeros(n)
    for i in range(n):
        at = n - 1 - i
        if parent[i] >= 0:
            par[at] = n - 1 - parent[i]
            length[at] = (died.get(i, end) - born[i]) * 100.0 / end
    interior = np.zeros(n, dtype=bool)
    interior[par[par >= 0]] = True
    col[~interior] = np.arange(int((~interior).sum()))
    return par, col, length


def _inputs(case, seed):
    """Everything a case computes from, as plain numpy arrays."""
    rng = np.random.default_rng((seed, 11, case["taxa"], case["bound"]))
    par, col, length = _tree(case)
    n = len(par)
    x = {"parent": par, "leaf_col": col, "length": length}
    points, classes = case.get("points", 1), case.get("classes", 1)
    jitter = float(rng.uniform(0.97, 1.03))
    if classes > 1:   # random clades with a lambda of their own
        cls = np.zeros(n, dtype=np.int64)
        tops = np.random.default_rng(case["taxa"]).choice(np.flatnonzero((col < 0) & (par >= 0)), classes - 1,
                                                          replace=False)
        for c, top in enumerate(sorted(tops, reverse=True), start=1):
            under = np.zeros(n, dtype=bool)
            under[top] = True
            for i in range(n - 1, -1, -1):
                if par[i] >= 0 and under[par[i]]:
                    under[i] = True
            cls[under] = c
        x["class"] = cls
        x["lambdas"] = np.array([[0.001, 0.004, 0.009]]) * jitter * np.linspace(1.0, 0.8, points)[:, None]
        sim = x["lambdas"][0][cls]
    else:
        if "lambda" in case:
            lam = np.array([case["lambda"] * jitter])
        elif points > 1:
            lam = 1e-4 * 95.0 ** (np.arange(points) / (points - 1)) * jitter
        else:
            lam = np.array([0.002 * jitter])
        x["lambdas"] = lam[:, None]
        sim = np.full(n, case.get("lambda", 0.003 if case.get("uneven") else 0.002))
    if "alpha" in case:
        x["alpha"] = case["alpha"] * float(rng.uniform(0.98, 1.02))
    if case["op"] == "matrices":
        return x
    # families: small roots and a heavy tail (fewer of it where one bound, set
    # by the largest family, holds for all); simulated down the tree by the
    # linear birth-death process
    F, bound = case["families"], case["bound"]
    cap = bound - max(1, bound // 20)
    body = 1 + np.minimum(rng.poisson(3.0, F), 9)
    tail = np.minimum(11 + np.floor(rng.pareto(1.2, F) * 8), 0.75 * bound if case.get("uneven") else 0.5 * bound)
    size0 = np.where(rng.random(F) < (0.85 if case.get("uneven") else 0.97), body, tail.astype(np.int64))
    size = np.zeros((n, F), dtype=np.int64)
    size[n - 1] = np.minimum(size0, min(cap, case["root"]))
    for u in range(n - 2, -1, -1):
        a = sim[u] * length[u] / (1.0 + sim[u] * length[u])
        alive = rng.binomial(size[par[u]], 1.0 - a)
        size[u] = alive + np.where(alive > 0, rng.negative_binomial(np.maximum(alive, 1), 1.0 - a), 0)
    counts = np.zeros((F, int((col >= 0).sum())), dtype=np.int32)
    leaves = np.flatnonzero(col >= 0)
    counts[:, col[leaves]] = np.minimum(size[leaves], cap).T
    x["counts"] = counts
    top = counts.max(axis=1)
    if case.get("uneven"):
        steps = np.array([b for b in LADDER if b < bound] + [bound])
        x["B"] = steps[np.searchsorted(steps, np.minimum(top + np.maximum(5, top // 5), bound))].astype(np.int32)
        x["R"] = x["B"].copy()
    elif case["op"] == "roots":
        x["B"] = np.minimum(bound, top + np.maximum(50, top // 5)).astype(np.int32)
        x["R"] = np.full(F, case["root"], dtype=np.int32)
    else:
        x["B"] = np.full(F, bound, dtype=np.int32)
        x["R"] = np.full(F, case["root"], dtype=np.int32)
    if case.get("epsilon"):
        e = case["epsilon"]
        x["error"] = np.tile([e, 1.0 - 2 * e, e], (bound + 1, 1))
        x["error"][0] = (0.0, 1.0 - e, e)
    return x


def _prior(R):
    return np.full(R, float(np.float32(1.0) / np.float32(R)))


def _key(x, unit):
    return float(int(x * unit)) / unit


def _branch_lambdas(x):
    """(points, nodes) lambda of every branch."""
    return x["lambdas"][:, x["class"]] if "class" in x else np.repeat(x["lambdas"], len(x["parent"]), axis=1)


# ---------------------------------------------------------------------------
# the package's side
# ---------------------------------------------------------------------------
def prepare(case, seed):
    x = _inputs(case, seed)
    n = len(x["parent"])
    tree = Tree(x["parent"], x["leaf_col"], x["length"], ["n%03d" % i for i in range(n)])
    eng = native.Engine(0)
    s = {"op": case["op"], "engine": eng}
    if case["op"] in ("infer", "plan"):
        m = model.BaseModel(eng, tree, x["counts"], x["B"], x["R"], error_model=x.get("error"),
                            path=PATHS[case["path"]])
        s["model"] = m
    if case["op"] == "infer":
        s["lambda"] = x["lambdas"][0]
        s["class"] = x.get("class")
        s["prior"] = _prior
    elif case["op"] == "plan":
        eng.tuning_load(SHAPES)
        keys = native.KeyTable()
        slots = keys.node_slots(tree, _branch_lambdas(x))
        s["lam_q"], s["t_q"] = keys.arrays()
        eng.matrix_reset(s["model"].N, len(s["lam_q"]))
        prior = np.zeros((len(s["model"].buckets), case["root"]))
        for i, (_, R, _) in enumerate(s["model"].buckets):
            prior[i, :R] = _prior(R)
        s["plan"] = eng.plan(slots, prior, s["lam_q"], s["t_q"], path=PATHS[case["path"]])
    elif case["op"] == "gamma":
        eng.tuning_load(SHAPES)
        s["model"] = model.ResidentGammaModel(eng, tree, x["counts"], x["B"], x["R"], case["cats"],
                                              _prior(case["root"]), path=PATHS[case["path"]])
        s["lambda"], s["alpha"] = float(x["lambdas"][0, 0]), x["alpha"]
    else:
        keys = native.KeyTable()
        slots = keys.node_slots(tree, _branch_lambdas(x))
        s["slots"] = slots
        s["lam_q"], s["t_q"] = keys.arrays()
        eng.set_tree(tree)
        eng.matrix_reset(max(case["bound"], case.get("root", 0)) + 1, len(s["lam_q"]))
        if case["op"] == "matrices":
            s["algo"] = native.BUILD_CLOSED_FORM if case["algo"] == "closed" else native.BUILD_RECURRENCE
            return s
        eng.set_families(x["counts"], bound_B=x["B"], bound_R=x["R"])
        eng.matrix_build(s["lam_q"], s["t_q"])
        s["root"], s["bound"] = case["root"], case["bound"]
        if case["op"] == "reconstruct":
            s["prior"] = np.append(_prior(case["root"]), 0.0)
        else:
            s["prior"] = np.tile(_prior(case["root"]), (len(eng.buckets()), 1))
    return s


def run(state):
    op, eng = state["op"], state["engine"]
    if op == "infer":
        m = state["model"]
        total = m.infer_family_likelihoods(state["prior"], state["lambda"] if state["class"] is not None
                                           else float(state["lambda"][0]), state["class"])
        return {"total": total, "lnl": m.results}
    if op == "plan":
        p = state["plan"]
        p.set_keys(state["lam_q"], state["t_q"])
        p.execute()
        r = p.results()
        return {"total": r["total"], "lnl": r["lnl"]}
    if op == "gamma":
        m = state["model"]
        total = m.infer_family_likelihoods(state["lambda"], state["alpha"])
        return {"total": total, "lnl": m.results["lnl"], "cat": m.results["cat"], "post": m.results["post"]}
    if op == "roots":
        return eng.root_vectors(state["slots"], state["prior"], native.PATH_PLAIN64, R=state["root"])
    if op == "reconstruct":
        return eng.reconstruct(state["slots"], state["prior"], state["bound"], state["root"])
    eng.matrix_build(state["lam_q"], state["t_q"], algo=state["algo"])
    return np.stack([eng.matrix_get(k) for k in range(len(state["lam_q"]))])


def work(case):
    """Counts and keys read once, results written once; two flops per matrix
    entry of every contraction (one multiply and one compare in the
    reconstruction) and five per matrix entry built."""
    par, col, _ = _tree(case)
    n, leaves, points = len(par), int((col >= 0).sum()), case.get("points", 1) * case.get("cats", 1)
    size = max(case["bound"], case.get("root", 0)) + 1
    build = 5.0 * points * (n - 1) * size * size
    if case["op"] == "matrices":
        return {"bytes": 8.0 * (n - 1) * (size * size + 2), "flops": build}
    F = case["families"]
    out = {"plan": 8.0 * F * points, "gamma": 8.0 * F * (1 + 2 * case.get("cats", 1)), "infer": 8.0 * F,
           "roots": 8.0 * F * case["root"], "reconstruct": 4.0 * F * n}[case["op"]]
    if case.get("uneven") or case["op"] == "roots":
        x = _inputs(case, 0)
        L, R = x["B"] + 1.0, x["R"].astype(float)
    else:
        L, R = np.full(F, case["bound"] + 1.0), np.full(F, float(case["root"]))
    inner = (col < 0) & (par >= 0)
    under_root = int((inner & (par == n - 1)).sum())
    deep = int(inner.sum()) - under_root
    if case["op"] == "reconstruct":
        return {"bytes": 4.0 * F * leaves + out + 8.0 * (n - 1) * size * size,
                "flops": float(2.0 * np.sum(L * L) * (deep + under_root))}
    flops = points * float(np.sum(2.0 * L * (deep * L + under_root * R) + leaves * L))
    if case["op"] == "roots":   # the matrices are at hand there
        return {"bytes": 4.0 * F * leaves + out + 8.0 * (n - 1) * size * size, "flops": flops}
    return {"bytes": 4.0 * F * leaves + out + 16.0 * points * (n - 1), "flops": flops + build}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _matrices(lam, t, N, dev):
    """(keys, N, N): P(s -> c); row s is row s - 1 convolved with row 1."""
    lt = torch.tensor(lam, dtype=torch.float64, device=dev) * torch.tensor(t, dtype=torch.float64, device=dev)
    a = lt / (1.0 + lt)
    c = torch.arange(N, device=dev, dtype=torch.float64)
    one = (1.0 - a)[:, None] ** 2 * a[:, None] ** torch.clamp(c - 1.0, min=0.0)
    one[:, 0] = a
    shift = torch.arange(N, device=dev)[None, :] - torch.arange(N, device=dev)[:, None]
    step = torch.where(shift >= 0, one[:, shift.clamp(min=0)], torch.zeros((), dtype=torch.float64, device=dev))
    out = torch.zeros(len(lam), N, N, dtype=torch.float64, device=dev)
    out[:, 0, 0] = 1.0
    for s in range(1, N):
        out[:, s:s + 1] = torch.bmm(out[:, s - 1:s], step)
    out[(1.0 - 2.0 * a) <= 0, 1:] = 0.0
    return out


def _root_vectors(x, M, slot, B, R, counts, dev):
    """(R, F) root vectors (sizes 1..R) of families of one bound."""
    par, col = x["parent"], x["leaf_col"]
    n, L = len(par), B + 1
    V = [None] * n
    c = torch.tensor(counts, dtype=torch.int64, device=dev)
    err = torch.tensor(x["error"], dtype=torch.float64, device=dev) if "error" in x else None
    for u in range(n):
        p = par[u]
        if p < 0:
            break
        rows = slice(1, R + 1) if par[p] < 0 else slice(0, L)
        m = M[slot[u]][rows]
        if col[u] >= 0:
            k = c[:, col[u]]
            if err is None:
                f = m[:, k]
            else:
                f = m[:, (k - 1).clamp(min=0)] * err[k, 0] + m[:, k] * err[k, 1] + m[:, k + 1] * err[k, 2]
        else:
            f = m[:, :L] @ V[u]
            V[u] = None
        V[p] = f if V[p] is None else V[p] * f
    return V[n - 1]


def _gamma_rates(K, alpha):
    """Medians of K equal slices of a gamma distribution of mean 1, scaled to
    a mean of 1."""
    q = (2.0 * torch.arange(K, dtype=torch.float64) + 1.0) / (2.0 * K)
    lo, hi = torch.zeros(K, dtype=torch.float64), torch.full((K,), 200.0, dtype=torch.float64)
    shape = torch.full((K,), float(alpha), dtype=torch.float64)
    for _ in range(200):
        mid = 0.5 * (lo + hi)
        below = torch.special.gammainc(shape, mid) < q
        lo, hi = torch.where(below, mid, lo), torch.where(below, hi, mid)
    r = 0.5 * (lo + hi)
    return (r * K / r.sum()).tolist()


def exact(case, seed):
    if case["op"] == "reconstruct":   # states are whole numbers
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x = _inputs(case, seed)
    lams = _branch_lambdas(x)
    if case["op"] == "gamma":
        lams = np.concatenate([lams * r for r in _gamma_rates(case["cats"], x["alpha"])])
    n = len(x["parent"])
    keys, slots = {}, np.zeros(lams.shape, dtype=np.int64)
    for p in range(len(lams)):
        for u in range(n - 1):
            slots[p, u] = keys.setdefault((_key(lams[p, u], 1e9), _key(x["length"][u], 1e3)), len(keys))
    M = _matrices([k[0] for k in keys], [k[1] for k in keys], max(case["bound"], case.get("root", 0)) + 1, dev)
    if case["op"] == "matrices":
        return M.cpu().numpy()
    F, P = case["families"], len(lams)
    if case["op"] == "roots":
        out = np.zeros((F, case["root"]))
    else:
        out = np.zeros((P, F))
    for B, R in sorted({(int(b), int(r)) for b, r in zip(x["B"], x["R"])}):
        at = np.flatnonzero((x["B"] == B) & (x["R"] == R))
        prior = torch.tensor(_prior(R), device=dev)[:, None]
        for p in range(P):
            v = _root_vectors(x, M, slots[p], B, R, x["counts"][at], dev)
            if case["op"] == "roots":
                out[at] = v.T.cpu().numpy()
            elif case["op"] == "gamma":
                out[p, at] = (v * prior).amax(dim=0).cpu().numpy()
            else:
                out[p, at] = (v.log() + prior.log()).amax(dim=0).cpu().numpy()
    if case["op"] == "roots":
        return out
    if case["op"] == "gamma":
        pk = 1.0 / case["cats"]
        cat = out.T * pk
        lnl = np.log(cat.sum(axis=1))
        return {"total": -math.fsum(lnl), "lnl": lnl, "cat": cat, "post": cat * pk / (cat * pk).sum(axis=1)[:, None]}
    if case["op"] == "infer":
        return {"total": -math.fsum(out[0]), "lnl": out[0]}
    return {"total": np.array([-math.fsum(r) for r in out]), "lnl": out}
