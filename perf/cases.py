"""Performance cases: the work a user of this library has one MI355X do.

Training on a resident `device.Dataset` (every objective, both gradient
representations and their lattices, narrow and wide data, sampled and not),
prediction with a trained ensemble, an estimator's fit and predict on a host
matrix, and the histogram entry point over device buffers. `listed()` holds
fixed cases, `draw()` gives more of the same ranges.

Binned data is drawn directly: a quantile-binned continuous feature is
uniform over its bins, and the labels are functions of the bins' centers.
"""
import ctypes as C
import math

import numpy as np
import torch

from mojoboost_amd import MojoTreesClassifier, MojoTreesRegressor, _lib, device

_OBJ = {"regression": 0, "binary": 1, "multiclass": 2, "lambdarank": 3}


def listed():
    """Twelve cases, smallest to largest per kind of call."""
    return [
        # a small table trained interactively: every launch's latency counts
        _train("train_small", rows=2_003, features=9, bins=63, leaves=15, trees=20, objective="binary"),
        # regression with the library's default (binary32 gradients) settings
        _train("train_regression", rows=100_000, features=28, bins=255, leaves=31, trees=40,
               objective="regression", quantized=False),
        # the headline workload's full matrix, a part of its trees
        _train("train_large", rows=10_500_000, features=28, bins=255, leaves=255, trees=60, objective="binary"),
        # GOSS on binary32 gradients (the first 10 rounds are not sampled)
        _train("train_goss", rows=4_000_037, features=28, bins=255, leaves=255, trees=30, objective="binary",
               quantized=False, goss=True),
        # wide data: many features of few bins, several feature tiles
        _train("train_wide", rows=200_000, features=1_000, bins=63, leaves=127, trees=30, objective="binary"),
        # ten classes with categorical columns split as sets
        _train("train_multiclass", rows=300_007, features=50, bins=255, leaves=63, trees=5,
               objective="multiclass", classes=10, categorical=10),
        # learning to rank: queries of 1 to some 500 documents
        _train("train_rank", rows=120_000, features=40, bins=255, leaves=63, trees=20, objective="lambdarank",
               quantized=False),
        # the reference's own quantized lattice (int32 pairs), bagged rows and
        # features, missing values
        _train("train_magnitude", rows=1_000_003, features=28, bins=255, leaves=127, trees=20,
               objective="binary", lattice=1, bagging=0.8, feature_fraction=0.8, missing=0.05),
        # scoring a few requests with a trained model
        _predict("predict_small", rows=501, features=28, bins=255, leaves=31, trees=100),
        # scoring a large table with a deep ensemble
        _predict("predict_large", rows=1_000_000, features=28, bins=255, leaves=255, trees=200),
        # an estimator from a host matrix: binning, upload, training, scoring
        _fit("fit_predict", rows=50_000, features=20, leaves=31, trees=50, objective="binary"),
        # one node's histogram from device buffers, nothing allocated
        _histogram("histogram", rows=1_000_000, features=28, bins=255, selected=0.5),
    ]


def draw(rng):
    """A case of the same ranges; `rng` is a random.Random."""
    kind = rng.choice(["train"] * 7 + ["predict"] * 2 + ["fit", "histogram"])
    bins = rng.choice([16, 63, 64, 127, 200, 255, 256])
    leaves = rng.choice([7, 15, 31, 40, 63, 127, 255])
    if kind == "train":
        features = _log(rng, 4, 1_000)
        trees = _log(rng, 5, 40)
        quantized = rng.random() < 0.6
        # bounded so that no drawn case outweighs the largest listed one
        rows = _log(rng, 1_500, min(4_000_000, int(2e9 / (features * trees))))
        objective = rng.choice(["binary", "binary", "regression", "regression", "multiclass", "lambdarank"])
        leaves = min(leaves, 127 if features > 300 else 255)
        if objective == "multiclass":
            return _train(None, rows=min(rows, 400_000), features=min(features, 60), bins=max(bins, 63),
                          leaves=min(leaves, 63), trees=max(1, trees // 6), objective=objective,
                          classes=rng.randint(3, 10), quantized=quantized,
                          categorical=rng.choice([0, min(features, 60) // 5]))
        if objective == "lambdarank":
            return _train(None, rows=min(rows, 200_000), features=min(features, 140), bins=bins,
                          leaves=min(leaves, 63), trees=trees, objective=objective, quantized=False)
        sample = rng.choice(["none", "none", "bagging", "goss"])
        return _train(None, rows=rows, features=features, bins=bins, leaves=leaves, trees=trees,
                      objective=objective, quantized=quantized, goss=sample == "goss",
                      lattice=1 if quantized and rng.random() < 0.3 else 0,
                      bagging=round(rng.uniform(0.5, 0.9), 2) if sample == "bagging" else 1.0,
                      feature_fraction=rng.choice([1.0, 1.0, 0.6]), missing=rng.choice([0.0, 0.0, 0.1]),
                      weighted=rng.random() < 0.2)
    if kind == "predict":
        trees = _log(rng, 10, 200)
        return _predict(None, rows=_log(rng, 200, 1_000_000), features=_log(rng, 5, 200), bins=bins,
                        leaves=leaves, trees=trees, classes=rng.choice([1, 1, 1, 4]) if trees <= 60 else 1)
    if kind == "fit":
        return _fit(None, rows=_log(rng, 1_000, 60_000), features=_log(rng, 5, 40), leaves=min(leaves, 63),
                    trees=_log(rng, 10, 60), objective=rng.choice(["binary", "regression"]))
    return _histogram(None, rows=_log(rng, 1_000, 1_500_000), features=_log(rng, 4, 120), bins=bins,
                      selected=rng.choice([1.0, 0.7, 0.3, 0.05]))


def _log(rng, lo, hi):
    """A whole number, uniform over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(max(lo, hi))))))))


def _named(name, case):
    return {"name": name, **case} if name else case


def _train(name, *, rows, features, bins, leaves, trees, objective, quantized=True, lattice=0, goss=False,
           bagging=1.0, feature_fraction=1.0, missing=0.0, classes=1, categorical=0, weighted=False):
    return _named(name, dict(kind="train", rows=rows, features=features, bins=bins, leaves=leaves, trees=trees,
                             objective=objective, quantized=quantized, lattice=lattice, goss=goss,
                             bagging=bagging, feature_fraction=feature_fraction, missing=missing,
                             classes=classes, categorical=categorical, weighted=weighted))


def _predict(name, *, rows, features, bins, leaves, trees, classes=1):
    return _named(name, dict(kind="predict", rows=rows, features=features, bins=bins, leaves=leaves, trees=trees,
                             classes=classes))


def _fit(name, *, rows, features, leaves, trees, objective):
    return _named(name, dict(kind="fit", rows=rows, features=features, leaves=leaves, trees=trees,
                             objective=objective))


def _histogram(name, *, rows, features, bins, selected):
    return _named(name, dict(kind="histogram", rows=rows, features=features, bins=bins, selected=selected))


# ------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _binned(case, g):
    """(bins uint8 [F, n], scores float32 [n], n_categories or None,
    missing_bin or None), on the GPU: uniform bins per feature, a nonlinear
    score of the first features."""
    n, f, nb = case["rows"], case["features"], case["bins"]
    bins = torch.empty((f, n), dtype=torch.uint8, device="cuda")
    score = torch.zeros(n, device="cuda")
    w = torch.randn(f, generator=g, device="cuda").tolist()
    n_cat = case.get("categorical", 0)
    cards = None
    missing = None
    if n_cat:
        cards = np.zeros(f, np.int32)
        sizes = torch.randint(4, min(64, nb - 1) + 1, (n_cat,), generator=g, device="cuda").tolist()
        cards[f - n_cat:] = sizes
    if case.get("missing", 0.0) > 0.0:
        # the last bin of every third feature is the one reserved for missing
        missing = np.full(f, -1, np.int32)
        missing[::3] = nb - 1
    last = None
    for j in range(f):
        u = torch.rand(n, generator=g, device="cuda")
        if cards is not None and cards[j]:
            b = (u * int(cards[j])).to(torch.uint8) + 1
            effect = torch.randn(int(cards[j]) + 1, generator=g, device="cuda")
            score += effect[b.long()]
        else:
            top = nb - 1 if missing is not None and missing[j] >= 0 else nb
            b = (u * top).clamp_(max=top - 1).to(torch.uint8)
            c = 2.0 * u - 1.0
            if j < 24:
                score += w[j] * (c if last is None else c * last if j % 2 else c.abs())
            last = c
            if missing is not None and missing[j] >= 0:
                gone = torch.rand(n, generator=g, device="cuda") < case["missing"]
                b = torch.where(gone, torch.full_like(b, nb - 1), b)
        bins[j] = b
    return bins, score, cards, missing


def _labels(case, score, g):
    n = score.numel()
    noise = torch.rand(n, generator=g, device="cuda")
    if case["objective"] == "regression":
        return (score + 0.1 * torch.randn(n, generator=g, device="cuda")).double()
    if case["objective"] == "lambdarank":
        rank = torch.argsort(torch.argsort(score + torch.randn(n, generator=g, device="cuda"))) / n
        return (rank > 0.5).double() + (rank > 0.75).double() + (rank > 0.9).double() + (rank > 0.97).double()
    if case.get("classes", 1) > 1:
        z = (score - score.mean()) / score.std() + 0.7 * torch.randn(n, generator=g, device="cuda")
        cdf = 0.5 * (1.0 + torch.erf(z / math.sqrt(2.0 * 1.49)))
        return (cdf * case["classes"]).clamp_(0, case["classes"] - 1).floor().double()
    return (noise < torch.sigmoid(2.0 * (score - score.median()))).double()


def _query_sizes(n, g):
    """Rows per query: log-normal around 60, 1 to 500, in row order."""
    z = torch.randn(n, generator=g, device="cuda")
    sizes = torch.exp(4.1 + 0.8 * z).round().clamp_(1, 500).long()
    ends = torch.cumsum(sizes, 0)
    k = int((ends < n).sum())
    counts = sizes[:k + 1].cpu().numpy().astype(np.int32)
    counts[k] = n - (int(ends[k - 1]) if k else 0)
    return counts


def _train_params(case):
    p = dict(objective=_OBJ[case["objective"]], num_iterations=case["trees"], num_leaves=case["leaves"],
             min_data_in_leaf=20, lambda_l2=1.0, learning_rate=0.1,
             use_quantized_grad=1 if case["quantized"] else 0, feature_fraction=case["feature_fraction"])
    if case["classes"] > 1:
        p["num_class"] = case["classes"]
    if case["lattice"]:
        p["quant_scale_rule"] = case["lattice"]
    if case["goss"]:
        p.update(goss=1, top_rate=0.2, other_rate=0.1)
    if case["bagging"] < 1.0:
        p.update(bagging_fraction=case["bagging"], bagging_freq=1)
    return p


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "train":
        bins, score, cards, missing = _binned(case, g)
        y = _labels(case, score, g).cpu().numpy()
        weights = None
        if case["weighted"]:
            weights = (0.5 + torch.rand(case["rows"], generator=g, device="cuda")).double().cpu().numpy()
        ds = device.Dataset(bins.cpu().numpy(), case["rows"], case["features"], case["bins"], y,
                            missing_bin=missing, n_categories=cards, weights=weights)
        if case["objective"] == "lambdarank":
            ds.set_groups(_query_sizes(case["rows"], g))
        return dict(case=case, ds=ds, params=_train_params(case))
    if kind == "predict":
        # a model trained on other rows of the same distribution
        model = dict(case, rows=60_000, missing=0.0, categorical=0,
                     objective="multiclass" if case["classes"] > 1 else "regression")
        bins, score, _, _ = _binned(model, g)
        y = _labels(model, score, g).cpu().numpy()
        ds = device.Dataset(bins.cpu().numpy(), model["rows"], case["features"], case["bins"], y)
        fit = ds.train(objective=_OBJ[model["objective"]], num_class=case["classes"], num_leaves=case["leaves"],
                       num_iterations=case["trees"])
        ds.free()
        rows, _, _, _ = _binned(dict(case, missing=0.0, categorical=0), g)
        return dict(case=case, fit=fit, bins=rows.cpu().numpy().ravel())
    if kind == "fit":
        n, f = case["rows"], case["features"]
        x = torch.randn((f, n), generator=g, device="cuda", dtype=torch.float64)
        w = torch.randn(f, generator=g, device="cuda", dtype=torch.float64)
        score = (w[:, None] * x).sum(0) / math.sqrt(f) + 0.5 * x[0] * x[1]
        if case["objective"] == "binary":
            y = (torch.rand(n, generator=g, device="cuda") < torch.sigmoid(2.0 * score)).long()
        else:
            y = score + 0.1 * torch.randn(n, generator=g, device="cuda", dtype=torch.float64)
        x = x.cpu().numpy().T  # column-major, as a DataFrame's values are
        return dict(case=case, x=x, y=y.cpu().numpy())
    n, f, nb = case["rows"], case["features"], case["bins"]
    quant_bins = 4
    bins = torch.randint(0, nb, (f, n), generator=g, device="cuda", dtype=torch.uint8) if nb < 256 else \
        torch.randint(0, 256, (f, n), generator=g, device="cuda").to(torch.uint8)
    qg = torch.randint(-quant_bins // 2, quant_bins // 2 + 1, (n,), generator=g, device="cuda", dtype=torch.int8)
    qh = torch.randint(0, quant_bins + 1, (n,), generator=g, device="cuda", dtype=torch.int8)
    rows = None
    if case["selected"] < 1.0:
        keep = torch.rand(n, generator=g, device="cuda") < case["selected"]
        keep[0] = True
        rows = torch.nonzero(keep).ravel().to(torch.int32)
    return dict(case=case, bins=bins, qg=qg, qh=qh, rows=rows, quant_bins=quant_bins,
                out=torch.empty((f, nb, 3), dtype=torch.int32, device="cuda"),
                err=C.create_string_buffer(512))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        fit = state["ds"].train(**state["params"])
        if case["quantized"]:
            return dict(base=fit.base, offsets=fit.off, feature=fit.feature, threshold=fit.threshold, left=fit.left,
                        right=fit.right, default_left=fit.default_left, value=fit.value, gain=fit.gain,
                        count=fit.count, cat_bits=fit.cat_bits.view(np.int64))
        # binary64 sums in no fixed order: splits of equal gain may trade
        # places, the scores they give do not change
        return dict(scores=fit.train_raw())
    if kind == "predict":
        return dict(scores=state["fit"].predict_binned(state["bins"], case["rows"], case["features"]))
    if kind == "fit":
        cls = MojoTreesClassifier if case["objective"] == "binary" else MojoTreesRegressor
        est = cls(n_estimators=case["trees"], num_leaves=case["leaves"]).fit(state["x"], state["y"])
        if case["objective"] == "binary":
            return dict(scores=est.decision_function(state["x"], device="gpu"))
        return dict(scores=est.predict(state["x"], device="gpu"))
    rows = state["rows"]
    rc = _lib.lib().mbh_histogram_noalloc(
        state["bins"].data_ptr(), case["rows"], case["features"], case["bins"], state["qg"].data_ptr(),
        state["qh"].data_ptr(), None if rows is None else rows.data_ptr(), 0 if rows is None else rows.numel(),
        state["quant_bins"], state["out"].data_ptr(), None, torch.cuda.current_stream().cuda_stream,
        state["err"], 512)
    _lib.check(rc, state["err"])
    return dict(histogram=state["out"])


def work(case):
    n, f = case["rows"], case["features"]
    kind = case["kind"]
    if kind == "histogram":
        m = int(n * case["selected"])
        ids = 4 * m if case["selected"] < 1.0 else 0
        return {"bytes": m * (f + 2) + ids + 12 * f * case["bins"], "flops": 2.0 * m * f}
    if kind == "predict":
        k = case["classes"]
        return {"bytes": n * (f + 8 * k) + 20 * case["trees"] * k * (2 * case["leaves"] - 1),
                "flops": 2.0 * n * case["trees"] * k}
    k = case.get("classes", 1)
    # a tree reads its rows' bins once and updates every row's score (and
    # reads its label); a sampled tree's histograms cover its sample
    share = 0.3 if case.get("goss") else case.get("bagging", 1.0)
    per_tree = share * n * f + n * 24
    total = case["trees"] * k * per_tree
    if kind == "fit":
        total += 2 * 8 * n * f
    return {"bytes": total, "flops": 2.0 * share * n * f * case["trees"] * k}


def tolerance(case):
    # integer histograms fix every bit of a quantized fit
    if case["kind"] == "histogram" or (case["kind"] == "train" and case["quantized"]):
        return "exact"
    # each score is a sum of binary64 products in tree order
    if case["kind"] == "predict":
        return {"rel": 1e-13, "max": 1e-12}
    if case.get("goss"):
        # as below, and a score's last bit can move a row across the sample's
        # threshold (measured, two runs: 1.3e-16)
        return {"rel": 1e-5, "max": 1e-2}
    # binary32 gradients, binary64 sums in any order (measured: 3.9e-10
    # against every quantity in binary64, 2.2e-16 between two runs; the rest
    # is room for one row's choice between two splits of nearly equal gain)
    return {"rel": 1e-6, "max": 1e-3}


# ------------------------------------------- 64-bit results, plain torch

def exact(case, seed):
    kind = case["kind"]
    if kind == "predict":
        return _exact_predict(case, seed)
    if kind == "train" and not case["quantized"] and case["objective"] in ("binary", "regression"):
        plain = not (case["goss"] or case["bagging"] < 1.0 or case["feature_fraction"] < 1.0 or case["missing"]
                     or case["weighted"])
        if plain and case["rows"] * case["features"] * case["trees"] * case["leaves"] <= 6e9:
            return _exact_train(case, seed)
    # quantized fits and histograms are whole numbers' sums, compared bit for
    # bit; sampled and ranked fits have no short restatement
    return None


def _exact_predict(case, seed):
    state = prepare(case, seed)
    fit, k = state["fit"], case["classes"]
    bins = torch.from_numpy(state["bins"]).cuda().view(case["features"], case["rows"])
    at_row = torch.arange(case["rows"], device="cuda")
    out = torch.from_numpy(fit.base).cuda().repeat(case["rows"], 1)
    for t in range(fit.n_trees):
        tree = fit.tree(t)
        feature, threshold, left, right, value = (
            torch.from_numpy(np.ascontiguousarray(tree[c])).cuda()
            for c in ("feature", "threshold", "left", "right", "value"))
        at = torch.zeros(case["rows"], dtype=torch.long, device="cuda")
        while True:
            inner = feature[at] >= 0
            if not bool(inner.any()):
                break
            b = bins[feature[at].clamp(min=0).long(), at_row]
            at = torch.where(inner, torch.where(b <= threshold[at], left[at], right[at]).long(), at)
        out[:, t % k] += fit.learning_rate * value[at]
    return dict(scores=out.reshape(-1).cpu().numpy())


def _exact_train(case, seed):
    """Leaf-wise boosting with every quantity in binary64."""
    g = _generator(seed)
    bins, score, _, _ = _binned(case, g)
    y = _labels(case, score, g)
    n, f, nb = case["rows"], case["features"], case["bins"]
    flat = bins.long() + nb * torch.arange(f, device="cuda")[:, None]
    mean = y.mean()
    binary = case["objective"] == "binary"
    raw = torch.full((n,), float(torch.log(mean / (1 - mean)) if binary else mean), dtype=torch.float64,
                     device="cuda")
    lr, l2, min_data, min_hess = 0.1, 1.0, 20, 1e-3

    def histogram(rows, gh):
        idx = flat[:, rows].reshape(-1)
        h = torch.zeros((f * nb, 3), dtype=torch.float64, device="cuda")
        h.index_add_(0, idx, gh[rows].repeat(f, 1))
        return h.view(f, nb, 3)

    def best(h):
        left = torch.cumsum(h, 1)
        total = left[:, -1:, :]
        right = total - left
        ok = (left[..., 2] >= min_data) & (right[..., 2] >= min_data) & (left[..., 1] >= min_hess) & \
            (right[..., 1] >= min_hess)
        gain = left[..., 0] ** 2 / (left[..., 1] + l2) + right[..., 0] ** 2 / (right[..., 1] + l2) - \
            total[..., 0] ** 2 / (total[..., 1] + l2)
        gain = torch.where(ok, gain, torch.full_like(gain, -math.inf)).view(-1)
        v, i = torch.max(gain, 0)
        return float(v), int(i)

    for _ in range(case["trees"]):
        if binary:
            p = torch.sigmoid(raw)
            grad, hess = p - y, p * (1 - p)
        else:
            grad, hess = raw - y, torch.ones_like(raw)
        gh = torch.stack([grad, hess, torch.ones_like(raw)], 1)
        rows = torch.arange(n, device="cuda")
        h = histogram(rows, gh)
        frontier = [(rows, h, *best(h))]
        while len(frontier) < case["leaves"]:
            at = max(range(len(frontier)), key=lambda i: frontier[i][2])
            rows, h, gain, where = frontier[at]
            if not gain > 0.0:
                break
            go_left = bins[where // nb, rows] <= where % nb
            a, b = rows[go_left], rows[~go_left]
            if a.numel() <= b.numel():
                ha = histogram(a, gh)
                hb = h - ha
            else:
                hb = histogram(b, gh)
                ha = h - hb
            frontier[at] = (a, ha, *best(ha))
            frontier.append((b, hb, *best(hb)))
        for rows, _, _, _ in frontier:
            s = gh[rows].sum(0)
            raw[rows] += lr * (-s[0] / (s[1] + l2))
    return dict(scores=raw.cpu().numpy())
