"""Learned order selection for the adaptive near quadrature.

The adaptive integrator (triaadap_main, triaintrouts.f:1269-1464) refines a (target,
patch) pair's triangle tree until the children reproduce the parent's moments to epsp,
with one XG rule on every triangle (degree 16 at eps = 1e-6, 55 nodes).  Which rule is
cheapest depends on the pair: a smooth integrand is done with a high degree and no
refinement, a nearly singular one with a lower degree on a deeper tree; measured on the
wavy torus, the cheapest of six degrees per pair needs 0.65 of the kernel evaluations of
the fixed degree.  An 8 -> 64 -> 64 -> 6 MLP, trained on the GPU, predicts that rule
class from eight geometric features of the pair (distance and height over the patch,
nearest node, tolerance, |k| rad, aspect).  Class c runs the same adaptive integrator
with XG degree q0 + (-4, -2, 0, +4, +8, +12)[c] (q0 the reference's degree; class 2 is
the plain rule) and a level cap learned with it; the integrator's own test (children
against parent, one level up) judges every triangle, and a pair whose tree needs a
level past its class's cap is integrated again by the plain integrator.

Labels come from the integrator itself: every adaptive pair is integrated once per class
(forced routing, no cap) and labelled with the class of least cost, the cost being the
pair's own work (node steps on the cached tree, 64-node chunks below it where the
geometry is computed) weighted by unit costs fitted to the measured launch times of the six
classes; the class's level cap is the deepest tree among the training pairs labelled
with it, and its tree cache holds no depth below that cap.

Workflow: ``X, y, idx, info = collect(nq)``, ``params, tinfo = train(X, y)`` (GPU
training, normalisation folded into the first layer), ``lmax = level_caps(y, info)``,
then ``nq.run(selector=params, route_lmax=lmax)``; where ``info["used"]`` holds the plain
class alone, routing does not pay on this surface and ``nq.run()`` is the faster call.
"""
import ctypes as C

import numpy as np

from ._lib import lib
from . import basis
from .layer import _dptr, _torch

NCLASS = 6
NFEAT = 8
FEATURES = ("dist/rad", "height/rad", "nearest node dist/rad", "nearest node height/rad", "nearest node edge",
            "log10 epsp", "|k| rad", "rad^2/area")
DEGREE_OFFSETS = (-4, -2, 0, 4, 8, 12)
PLAIN_CLASS = 2


def nparam():
    return int(lib().fmm3dbie_mlp_nparam())


def class_degree(q0, c):
    """XG degree of rule class c around the plain degree q0 (as the library: not below
    degree 8, where the children-against-parent test stops being a reliable estimate,
    and not above 30, the largest rule in the tables)."""
    q = q0 + DEGREE_OFFSETS[c]
    return min(30, q) if q >= 8 else min(q0, 8)


def xg_size(deg):
    return len(basis.xg_rule(deg)[1])


def plain_degree(kq):
    """The XG degree with kq nodes (the plain rule of a generation)."""
    for d in range(1, 31):
        if xg_size(d) == kq:
            return d
    raise ValueError("no XG rule with %d nodes" % kq)


def forced(c):
    """Parameters whose argmax is class c for every input (all weights zero)."""
    p = np.zeros(nparam(), np.float32)
    p[-NCLASS + c] = 1.0
    return p


def init_params(seed=3):
    """He-normal weights, zero biases (float32, packed W1 b1 W2 b2 W3 b3)."""
    rng = np.random.default_rng(seed)
    parts = []
    for fan_in, fan_out in ((NFEAT, 64), (64, 64), (64, NCLASS)):
        parts.append((rng.standard_normal((fan_out, fan_in)) * np.sqrt(2.0 / fan_in)).ravel())
        parts.append(np.zeros(fan_out))
    p = np.concatenate(parts).astype(np.float32)
    assert p.size == nparam()
    return p


def chunk_rows(norder):
    """Nodes per chunk of the adaptive kernel: 55 at order 6 and above (the LDS of 12
    resident wavefronts per CU), else 64 (quad.hip chunk_rows)."""
    return 55 if norder >= 6 else 64


def per_triangle(norder, kq):
    """Whether the adaptive kernel takes one chunk per triangle for a rule of kq nodes
    (order 6 and above, a triangle filling more than half a chunk: quad.hip step_tris)."""
    cr = chunk_rows(norder)
    return norder >= 6 and cr < 2 * kq <= 2 * cr


def chunks(norder, kq):
    """Chunks of the adaptive kernel for one triangle and for a refinement test with a rule of
    kq nodes: one per triangle (per_triangle), else the nodes of the step in equal
    chunks."""
    if per_triangle(norder, kq):
        return 1, 4
    cr = chunk_rows(norder)
    return -(-kq // cr), -(-4 * kq // cr)


# Cost of a node step on the cached tree in chunks of the subtrees below it: 25 ps per pair and
# step against 2.2 ns per chunk, measured on the deformed sphere of order 6.  Fitted by itself from
# the six launches of a surface the ratio is ill-determined, the steps of a class being nearly a
# cost per pair: 0 to 0.009 on tori, spheres and deformed spheres of orders 2 to 6, both kernels.
# With this one the fitted launch times of orders 4 to 6 are within 10% of the measured ones (16%
# for a Laplace torus), those of orders 2 and 3 within 31%.
STEP_CHUNKS = 0.011


def tile_steps(kq):
    """Node steps of a triangle in the batched levels (4 nodes of 16 targets a step)."""
    return -(-kq // 4)


def collect(nq, stream=None):
    """Features of every adaptive pair (from a plain run) and its label: the rule class
    whose adaptive integration takes the least time.  Every pair is integrated once
    with each class (forced routing, no level cap, every kernel in order on one stream).
    The first levels of the trees are integrated in steps of 4 nodes for 16 targets at a
    time (tile_steps per triangle), the subtrees below them in chunks of at most
    chunk_rows(norder) nodes (chunks() per refinement test; a chunk costs the same whether
    its lanes are all busy or not).  A pair's work is its steps on the cached tree, at
    STEP_CHUNKS chunks each, and its chunks below it (geometry evaluated); the measured times
    of the six launches are fitted by a cost per chunk and a cost per pair, and the label is
    the class of least fitted cost among the classes worth their tree cache and the selector
    itself (open_classes).
    Returns (X (nadap, 8) float32, y (nadap,) int32, CSR entry index of each adaptive pair,
    info with the per-class fitted cost 'cost', kernel evaluations 'evals', deepest levels
    'lev' (6, nadap), launch times 'ms', the fitted unit costs 'unit' (ms per chunk, per
    pair), node counts 'kq', the plain degree 'q0', the classes used 'used', the plain
    rule's tree-cache time for depths 0..2 'ms_tree' and the selector's own time (features,
    inference, bucketing by class) beyond the plain bucketing 'ms_route')."""
    from scipy.optimize import nnls
    from . import layer
    torch = _torch()
    dev = nq.wnear.device
    feat = torch.zeros((nq.nnz, NFEAT), dtype=torch.float32, device=dev)
    side = layer.side_stream_enabled()
    layer.set_side_stream(False)
    try:
        nq.run(stream=stream, want_detail=True, features=feat)
        torch.cuda.synchronize()
        ms_tree = nq.stats["ms_tree"] * 21.0 / max(nq.stats["cache_tris"], 1)  # per depth-0..2 cache
        idx = np.nonzero(nq.stats["cls"] == 1)[0]
        X = feat.cpu().numpy()[idx]
        q0 = plain_degree(nq.stats["kq"])
        kq = np.array([xg_size(class_degree(q0, c)) for c in range(NCLASS)])
        ncached = np.zeros((NCLASS, len(idx)))
        ncomp = np.zeros((NCLASS, len(idx)))
        ccached = np.zeros((NCLASS, len(idx)))
        ccomp = np.zeros((NCLASS, len(idx)))
        lev = np.zeros((NCLASS, len(idx)), np.int32)
        ms = np.zeros(NCLASS)
        route = np.zeros(NCLASS)
        nq.run(stream=stream)
        ms_bucket = nq.stats["ms_select"]
        for c in range(NCLASS):
            sel = torch.as_tensor(forced(c), device=dev)
            for rep in range(2):  # the second run is timed (tables and caches built)
                nq.run(stream=stream, want_detail=True, selector=sel, route_lmax=[20] * NCLASS)
            st = nq.stats
            nref = st["nref"][idx].astype(np.float64)
            unc = st["unc"][idx].astype(np.float64)
            ncached[c] = kq[c] * (1 + 4 * (nref - unc))
            ncomp[c] = kq[c] * 4 * unc
            ccached[c] = tile_steps(kq[c]) * (1 + 4 * (nref - unc))
            ccomp[c] = chunks(nq.norder, kq[c])[1] * unc
            lev[c] = st["lev"][idx]
            ms[c] = st["ms_adap"]
            route[c] = st["ms_select"]
    finally:
        layer.set_side_stream(side)
    # a cost per pair (lists, test, weights: the same for every class) keeps the step costs from
    # absorbing it
    work = STEP_CHUNKS * ccached + ccomp
    unit, _ = nnls(np.stack([work.sum(1), np.full(NCLASS, float(len(idx)))], 1), ms)
    cost = unit[0] * work
    tree = tree_cost(ms_tree, kq, q0)
    fill = np.where(tree > 0.0, fill_cost(nq.npatches, kq, STEP_CHUNKS * unit[0]), 0.0)
    ms_route = max(0.0, float(route.min() - ms_bucket))
    y, used = open_classes(cost, tree + fill, ms_route)
    return X, y, idx, dict(cost=cost, evals=ncached + ncomp, lev=lev, ms=ms, unit=unit, kq=kq, q0=q0,
                           used=used, ms_tree=ms_tree, ms_route=ms_route)


def tree_cost(ms_tree, kq, q0):
    """Time of the tree cache of each routed rule class (depths 0..2, quad.hip), scaled
    from the plain rule's (ms_tree, for depths 0..2) by the node count; 0 for the plain
    rule, whose cache every generation builds."""
    kq = np.asarray(kq, np.float64)
    c = ms_tree * kq / kq[PLAIN_CLASS]
    c[[class_degree(q0, k) == q0 for k in range(NCLASS)]] = 0.0
    return c


def fill_cost(npatches, kq, step):
    """Cost of the partly filled tiles that one more class brings: the batched levels take 16
    targets of a patch and class at a time, so a class leaves half a tile empty at the root
    and at each of its children (5 triangles each), step being the cost per pair and node
    step.  Measured on the wavy torus of order 6 (1536 patches, plain 6.2 ms): classes
    of 79, 112 and 150 nodes beside the plain one 5.75 ms with the first alone, 5.80 with
    two, 6.00 with all three, whose pairs alone would save 0.65, 0.90 and 1.06 ms."""
    return 8.0 * npatches * 25 * step * np.array([tile_steps(int(k)) for k in kq])


def open_classes(cost, cache, route=0.0):
    """Which rule classes to use and each pair's label.  A class other than the plain one
    costs its tree cache and partly filled tiles once per generation (cache[c], same unit as cost);
    starting from the plain class alone, the class whose pairs would save the most
    (sum over pairs of the drop in their least cost, minus its cache) is added while that
    saving is positive.  Routing itself costs route once per generation (the selector): where
    all that is saved does not pay for it, the free classes alone are used.  (Uncharged, a
    torus of 768 patches of order 4 opened a class that took the adaptive part from 0.77 to
    0.94 ms, a sphere of 1728 patches of order 3 one from 0.93 to 1.22 ms.)  Returns (labels: the least-cost used class of every pair, used
    classes as a boolean array)."""
    ncls = cost.shape[0]
    used = np.zeros(ncls, bool)
    used[[c for c in range(ncls) if cache[c] == 0.0] or [PLAIN_CLASS]] = True
    free = used.copy()
    best = cost[used].min(axis=0)
    saved = 0.0
    while True:
        gain = np.array([np.maximum(best - cost[c], 0.0).sum() - cache[c] if not used[c] else -np.inf
                         for c in range(ncls)])
        c = int(np.argmax(gain))
        if not np.isfinite(gain[c]) or gain[c] <= 0.0:
            break
        used[c] = True
        saved += gain[c]
        best = np.minimum(best, cost[c])
    if saved <= route:
        used = free
    masked = np.where(used[:, None], cost, np.inf)
    return np.argmin(masked, axis=0).astype(np.int32), used


def level_caps(y, info):
    """Level cap of each class: the deepest tree among the pairs labelled with it (20,
    the integrator's own cap, for a class without pairs and for the plain class: a pair sent
    back from there would be integrated the same way once more)."""
    caps = np.full(NCLASS, 20, np.int32)
    for c in range(NCLASS):
        m = y == c
        if c != PLAIN_CLASS and m.any():
            caps[c] = max(1, int(info["lev"][c][m].max()))
    return caps


def fold_normalisation(params, mean, std):
    """First layer on raw features: W1' = W1 / std, b1' = b1 - W1' mean."""
    p = np.array(params, np.float32, copy=True)
    W1 = p[:64 * NFEAT].reshape(64, NFEAT).astype(np.float64)
    b1 = p[64 * NFEAT:64 * NFEAT + 64].astype(np.float64)
    W1n = W1 / std[None, :]
    p[:64 * NFEAT] = W1n.ravel().astype(np.float32)
    p[64 * NFEAT:64 * NFEAT + 64] = (b1 - W1n @ mean).astype(np.float32)
    return p


def grad(params, X, y, device="cuda"):
    """Device mean cross-entropy and gradient (the backward kernels), as numpy."""
    torch = _torch()
    dp = torch.as_tensor(np.asarray(params, np.float32), device=device)
    dX = torch.as_tensor(np.ascontiguousarray(X, np.float32), device=device)
    dy = torch.as_tensor(np.ascontiguousarray(y, np.int32), device=device)
    dg = torch.zeros(nparam(), dtype=torch.float32, device=device)
    loss = C.c_float(0.0)
    s = torch.cuda.current_stream()
    rc = lib().fmm3dbie_mlp_grad(_dptr(dp), _dptr(dX), _dptr(dy), len(y), _dptr(dg), C.byref(loss),
                                 C.c_void_p(s.cuda_stream))
    if rc != 0:
        raise RuntimeError("fmm3dbie_mlp_grad failed (status %d)" % rc)
    torch.cuda.synchronize()
    return float(loss.value), dg.cpu().numpy()


def predict(params, X, device="cuda"):
    torch = _torch()
    dp = params if hasattr(params, "is_cuda") else torch.as_tensor(np.asarray(params, np.float32), device=device)
    dX = torch.as_tensor(np.ascontiguousarray(X, np.float32), device=device)
    dc = torch.zeros(len(X), dtype=torch.int32, device=device)
    s = torch.cuda.current_stream()
    rc = lib().fmm3dbie_mlp_predict(_dptr(dp), _dptr(dX), len(X), _dptr(dc), None, C.c_void_p(s.cuda_stream))
    if rc != 0:
        raise RuntimeError("fmm3dbie_mlp_predict failed (status %d)" % rc)
    torch.cuda.synchronize()
    return dc.cpu().numpy()


def train(X, y, n_train=200000, epochs=30, batch=256, lr=3e-3, seed=3, device="cuda"):
    """Train on (at most n_train, sampled with seed) pairs on the GPU.

    Returns (device float32 parameters acting on raw features, info dict with the
    per-epoch loss, train/held-out accuracy and training time)."""
    torch = _torch()
    X = np.asarray(X, np.float32)
    y = np.asarray(y, np.int32)
    n = len(y)
    rng = np.random.default_rng(seed)
    sel = rng.permutation(n)
    tr, ho = sel[:min(n_train, n)], sel[min(n_train, n):]
    ntr = (len(tr) // batch) * batch
    if ntr < batch:
        raise ValueError("need at least %d training pairs, got %d" % (batch, len(tr)))
    mean = X[tr].astype(np.float64).mean(axis=0)
    std = X[tr].astype(np.float64).std(axis=0)
    std[std < 1e-12] = 1.0
    Xn = ((X[tr].astype(np.float64) - mean) / std).astype(np.float32)
    dX = torch.as_tensor(np.ascontiguousarray(Xn), device=device)
    dy = torch.as_tensor(np.ascontiguousarray(y[tr]), device=device)
    dp = torch.as_tensor(init_params(seed), device=device)
    hist = np.zeros(epochs, np.float32)
    s = torch.cuda.current_stream()
    t0 = torch.cuda.Event(enable_timing=True)
    t1 = torch.cuda.Event(enable_timing=True)
    t0.record(s)
    rc = lib().fmm3dbie_mlp_train(_dptr(dp), _dptr(dX), _dptr(dy), len(tr), epochs, batch, lr, seed,
                                  hist.ctypes.data_as(C.c_void_p), C.c_void_p(s.cuda_stream))
    t1.record(s)
    if rc != 0:
        raise RuntimeError("fmm3dbie_mlp_train failed (status %d)" % rc)
    torch.cuda.synchronize()
    params = fold_normalisation(dp.cpu().numpy(), mean, std)
    dpar = torch.as_tensor(params, device=device)
    info = dict(loss=hist.tolist(), ms_train=t0.elapsed_time(t1), n_train=len(tr), n_heldout=len(ho))
    info["acc_train"] = float(np.mean(predict(dpar, X[tr]) == y[tr]))
    info["acc_heldout"] = float(np.mean(predict(dpar, X[ho]) == y[ho])) if len(ho) else None
    return dpar, info
