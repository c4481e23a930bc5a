"""The work a user of this package has it do, as cases that can be timed and compared.

A case is one call of the training or serving path through the package's public entry points:

* ``step``     one boosting iteration of an open ``Trainer`` (the tree it adds to the model),
* ``fit``      a whole fit from a row-major float matrix, borders selected on the way,
* ``predict``  raw predictions of a finished model on a host matrix.

Inputs are synthetic, made from the seed alone.  Features of the step cases are standard
normals binned at their own quantiles (what border selection makes of a smooth column), or
mostly one value (a sparse column); targets depend on some of the features, with noise, so
that trees split as they do on real data and leaves differ in size.
"""
import math

import numpy as np
import torch

import catboost_rs_amd as cb

_STEP = dict(kind="step", loss="RMSE", n=100_000, features=50, bins=129, depth=6, classes=1, bootstrap="No",
             weights=False, zeros=0.0, score="Cosine", leaf="Gradient", lr=0.03, ctr=0)


def _step(name=None, **kw):
    c = dict(_STEP, **kw)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # a small table, shallow trees: the launches and their latency are the whole cost
        _step("step small", n=5_000, features=20, bins=33, depth=4),
        # an ordinary regression table
        _step("step regression", lr=0.1),
        # odd sizes, object weights, subsampling, Newton leaves, the L2 score, fewer bins
        _step("step weighted ragged", loss="Logloss", n=777_777, features=77, bins=65, bootstrap="Bernoulli",
              weights=True, score="L2", leaf="Newton"),
        # the package's default benchmark: a large classification table
        _step("step large", loss="Logloss", n=10_000_000, features=200, bins=255, bootstrap="Bayesian"),
        # several classes over dense columns
        _step("step classes", loss="MultiClass", n=300_000, features=60, bins=128, classes=5, leaf="Newton", lr=0.1),
        # many classes over a wide sparse table, deep trees
        _step("step wide sparse", loss="MultiClass", n=1_000_000, features=4096, bins=65, depth=8, classes=10,
              leaf="Newton", zeros=0.7, lr=0.1),
        # ranking by pairs in query groups of 20, scored by pointwise statistics ...
        _step("step pairs", loss="PairLogit", n=1_000_000, features=100, bins=255, leaf="Newton"),
        # ... and by pair statistics
        _step("step pairwise", loss="PairLogitPairwise", n=1_000_000, features=100, bins=255),
        # numbers and categories: 30 float columns and 20 categorical ones as target statistics
        _step("step categories", n=2_000_000, features=30, bins=255, bootstrap="Bernoulli", lr=0.1, ctr=20),
        # a whole short fit from a float matrix: 30 trees, 32 borders
        dict(name="fit", kind="fit", loss="RMSE", n=300_000, features=50, borders=32, depth=6, trees=30),
        # a model answering one small request, and scoring a table
        dict(name="predict request", kind="predict", n=1024, features=50, trees=30, depth=6, classes=1),
        dict(name="predict table", kind="predict", n=500_000, features=100, trees=500, depth=6, classes=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step"] * 5 + ["rank", "rank", "ctr", "fit", "predict"])
    if kind == "fit":
        return dict(kind="fit", loss=rng.choice(["RMSE", "Logloss"]), n=_log(rng, 20_000, 1_000_000),
                    features=_log(rng, 10, 60), borders=rng.choice([15, 32, 64, 128, 254]), depth=rng.randint(4, 7),
                    trees=rng.randint(10, 40))
    if kind == "predict":
        return dict(kind="predict", n=_log(rng, 1, 400_000), features=_log(rng, 5, 120), trees=_log(rng, 10, 500),
                    depth=rng.randint(2, 8), classes=rng.choice([1, 1, 1, 3, 5]))
    if kind == "rank":
        return _step(loss=rng.choice(["PairLogit", "PairLogitPairwise"]), n=20 * _log(rng, 500, 50_000),
                     features=_log(rng, 10, 100), bins=rng.choice([33, 65, 129, 255]), depth=rng.randint(4, 6),
                     leaf="Gradient")
    if kind == "ctr":
        return _step(n=_log(rng, 20_000, 2_000_000), features=_log(rng, 5, 40), bins=rng.choice([65, 129, 255]),
                     depth=rng.randint(4, 7), bootstrap=rng.choice(["No", "Bernoulli"]), lr=0.1, ctr=rng.randint(2, 20))
    if rng.random() < 0.35:
        n = _log(rng, 3_000, 800_000)
        return _step(loss="MultiClass", n=n, features=_log(rng, 8, max(9, min(2000, 40_000_000 // n))),
                     bins=rng.choice([17, 33, 65, 128]), depth=rng.randint(4, 7), classes=rng.choice([2, 3, 5, 7, 10]),
                     leaf="Newton", bootstrap=rng.choice(["No", "Bernoulli"]), zeros=rng.choice([0.0, 0.7]), lr=0.1)
    n = _log(rng, 3_000, 8_000_000)
    return _step(loss=rng.choice(["RMSE", "Logloss", "CrossEntropy"]), n=n,
                 features=_log(rng, 5, max(6, min(1000, 1_200_000_000 // n))), bins=rng.choice([17, 33, 65, 129, 255]),
                 depth=rng.randint(4, 8), bootstrap=rng.choice(["No", "Bayesian", "Bernoulli"]),
                 weights=rng.random() < 0.4, score=rng.choice(["Cosine", "L2"]), leaf=rng.choice(["Gradient", "Newton"]),
                 zeros=rng.choice([0.0, 0.0, 0.7]), lr=0.1)


# ---- inputs -------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1_000_003 + 17)
    return g


def _binned(case, g):
    """u8 bins [F][n] on the host, border counts [F], and the scores [max(1, classes)][n] of
    some of the columns (on the GPU)."""
    n, F, nb, zeros = case["n"], case["features"], case["bins"] - 1, case["zeros"]
    outs = case["classes"] if case["loss"] == "MultiClass" else 1
    used = min(F, 20)
    mix = torch.randn(outs, used, generator=g, device="cuda", dtype=torch.float64)
    score = torch.zeros(outs, n, device="cuda", dtype=torch.float64)
    bins = np.empty((F, n), np.uint8)
    counts = np.full(F, nb, np.uint32)
    step = max(1, min(F, 64_000_000 // n))
    for f0 in range(0, F, step):
        m = min(step, F - f0)
        z = torch.randn(m, n, generator=g, device="cuda")
        u = torch.special.ndtr(z)
        if zeros:   # exact zeros hold most quantiles: a few borders below, a few above, one value between
            half = max(1, int(nb * (1.0 - zeros)) // 2)
            b = torch.clamp((u * 2 - 1).abs() * half, max=half - 1).to(torch.int32)
            b = torch.where(z < 0, half - 1 - b, half + 1 + b)
            off = torch.rand(m, n, generator=g, device="cuda") < zeros
            b = torch.where(off, torch.full_like(b, half), b)
            z = torch.where(off, torch.zeros_like(z), z)
            counts[f0:f0 + m] = 2 * half
        else:
            b = torch.clamp((u * (nb + 1)).to(torch.int32), max=nb)
        torch.from_numpy(bins[f0:f0 + m]).copy_(b.to(torch.uint8))
        if f0 < used:
            k = min(m, used - f0)
            for j in range(k):
                score += mix[:, f0 + j, None] * z[j].double()
    return bins, counts, score / math.sqrt(used)


def _target(case, g, score):
    n = case["n"]
    if case["loss"] == "RMSE":
        return score[0] + 0.3 * torch.randn(n, generator=g, device="cuda", dtype=torch.float64)
    if case["loss"] == "Logloss":
        return (torch.rand(n, generator=g, device="cuda", dtype=torch.float64) < torch.sigmoid(2 * score[0])).double()
    if case["loss"] == "CrossEntropy":
        return torch.sigmoid(2 * score[0] + torch.randn(n, generator=g, device="cuda", dtype=torch.float64))
    noise = torch.randn(score.shape, generator=g, device="cuda", dtype=torch.float64)
    if case["loss"] == "MultiClass":
        return torch.argmax(score + 0.5 * noise, 0).double()
    return torch.clamp(torch.floor(2.5 + 1.5 * (score[0] + 0.5 * noise[0])), 0, 4)   # relevance 0 to 4


def _pairs(case, g, rel):
    """About 10 pairs a query group of 20, better document first."""
    G = case["n"] // 20
    i = torch.randint(0, 20, (G, 13), generator=g, device="cuda")
    j = torch.randint(0, 20, (G, 13), generator=g, device="cuda")
    base = (torch.arange(G, device="cuda") * 20)[:, None]
    ri, rj = rel[base + i], rel[base + j]
    win, los, keep = torch.where(ri > rj, i, j) + base, torch.where(ri > rj, j, i) + base, ri != rj
    return (win[keep].cpu().numpy().astype(np.uint32), los[keep].cpu().numpy().astype(np.uint32),
            np.arange(0, case["n"] + 1, 20, dtype=np.uint32))


def _inputs(case, seed):
    """What a step case's program holds on the host: the Trainer's arguments."""
    g = _generator(seed)
    n = case["n"]
    bins, counts, score = _binned(case, g)
    d = dict(bins=bins, counts=counts, weight=None)
    if case["ctr"]:   # categorical columns, their effect added to the target
        keys = np.empty((case["ctr"], n), np.uint32)
        for j in range(case["ctr"]):
            u = torch.rand(1, generator=g, device="cuda", dtype=torch.float64).item()
            card = int(round(math.exp(math.log(17) + u * math.log(10_000 / 17))))
            cdf = torch.cumsum(1.0 / torch.arange(1, card + 1, device="cuda", dtype=torch.float64) ** 1.1, 0)
            r = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * cdf[-1]
            k = torch.clamp(torch.searchsorted(cdf, r), max=card - 1)
            score[0] += 0.3 * torch.randn(card, generator=g, device="cuda", dtype=torch.float64)[k]
            keys[j] = k.to(torch.int32).cpu().numpy().view(np.uint32)
        d["keys"] = keys
    y = _target(case, g, score)
    if case["loss"].startswith("PairLogit"):
        d["winner"], d["loser"], d["groups"] = _pairs(case, g, y)
    if case["weights"]:
        d["weight"] = (0.5 + 1.5 * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)).cpu().numpy()
    d["target"] = y.cpu().numpy()
    return d


def _params(case):
    return dict(loss=case["loss"], depth=case["depth"], learning_rate=case["lr"], l2_leaf_reg=3.0, score=case["score"],
                leaf_method=case["leaf"], bootstrap_type=case["bootstrap"], subsample=0.66, bagging_temperature=1.0,
                boost_from_average=case["loss"] == "RMSE", random_seed=0, approx_dim=case["classes"])


def _open(case, seed):
    d = _inputs(case, seed)
    kw = _params(case)
    if case["loss"].startswith("PairLogit"):
        kw.update(pairs=(d["winner"], d["loser"]), group_offsets=d["groups"])
    if case["ctr"]:
        two = cb.shuffled_indices(case["n"], int(seed), count=2)
        hashed = [cb.perfect_hash(k) for k in d["keys"]]
        kw["device_ctr"] = cb.DeviceCtr(np.stack([h[0] for h in hashed]), two[0], two[0][two[1]],
                                        d["target"] > np.median(d["target"]), [("Borders", 0.5)],
                                        bucket_counts=[h[1] for h in hashed])
    return cb.Trainer(d["bins"], int(d["counts"].max()) + 1, d["target"], weight=d["weight"], real_folds=d["counts"] + 1, **kw)


def _model(case, seed):
    r = np.random.default_rng(int(seed) * 7 + 5)
    T, D, F, K = case["trees"], case["depth"], case["features"], case["classes"]
    return dict(x=r.standard_normal((F, case["n"]), dtype=np.float32),
                feature=r.integers(0, F, T * D).astype(np.uint32),
                border=r.standard_normal(T * D).astype(np.float32).astype(np.float64),
                split_at=np.arange(0, T * D + 1, D, dtype=np.uint32),
                leaf=0.1 * r.standard_normal((T << D) * K),
                leaf_at=np.arange(0, (T << D) + 1, 1 << D, dtype=np.uint32), bias=r.standard_normal(K))


def prepare(case, seed):
    if case["kind"] == "step":
        return dict(case=case, trainer=_open(case, seed))
    if case["kind"] == "predict":
        return dict(case=case, **_model(case, seed))
    g = _generator(seed)
    x = torch.randn(case["n"], case["features"], generator=g, device="cuda")
    w = torch.randn(case["features"], generator=g, device="cuda", dtype=torch.float64)
    y = _target(case, g, (x.double() @ w)[None] / math.sqrt(case["features"]))
    return dict(case=case, x=x.cpu().numpy(), y=y.cpu().numpy())


# ---- one pass -----------------------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["kind"] == "step":   # the tree is the model's update: its splits and leaf values
        splits, leaves, one_hot = state["trainer"].step()
        return dict(splits=splits, leaves=leaves, one_hot=one_hot)
    if case["kind"] == "predict":
        s = state
        return cb.apply_oblivious(s["x"], s["feature"], s["border"], s["split_at"], s["leaf"], s["leaf_at"],
                                  approx_dim=case["classes"], bias=s["bias"])
    columns = cb.columns_from_rows(state["x"])
    borders = cb.select_borders(columns, case["borders"])
    trainer = cb.Trainer.from_floats(columns, borders, state["y"], loss=case["loss"], depth=case["depth"],
                                     learning_rate=0.1, score="L2")
    try:
        splits, leaves = trainer.fit(case["trees"])
        approx = trainer.approx()
    finally:
        trainer.close()
    return dict(splits=splits, leaves=leaves, approx=approx)


def work(case):
    n, F, D = case["n"], case["features"], case["depth"]
    if case["kind"] == "predict":
        T, K = case["trees"], case["classes"]
        return dict(bytes=4.0 * n * F + 8.0 * n * K + 12.0 * T * D + 8.0 * (T << D) * K, flops=float(n) * T * (D + K))
    # a tree: every row's bins, target and weights read, its approximant updated; each channel of
    # a row added to a cell of each feature, at the first level and, for the smaller child of each
    # split (at best half of the rows), at the others; the best of all borders
    K = case.get("classes", 1)
    cols = F + case.get("ctr", 0)
    B = case["borders"] + 1 if case["kind"] == "fit" else case["bins"]   # a sparse column uses a third of them
    B = B // 3 if case.get("zeros") else B
    tree_bytes = float(n) * cols + 8.0 * n * (2 * K + 1 + bool(case.get("weights")))
    tree_flops = float(n) * cols * (K + 1) * (1 + (D - 1) * 0.25) + 8.0 * cols * B * K * ((1 << D) - 1)
    if case["kind"] == "fit":
        return dict(bytes=4.0 * n * F + 8.0 * n + case["trees"] * tree_bytes, flops=case["trees"] * tree_flops)
    if case["loss"].startswith("PairLogit"):
        tree_bytes += 4.0 * n   # half a pair a row: winner and loser
    return dict(bytes=tree_bytes, flops=tree_flops)


def tolerance(case):
    # splits are whole numbers and the histograms behind them exact sums, so they are the same; leaf
    # values and predictions are 64-bit sums and quotients (4e-16 to 7e-13 off the exact ones here),
    # with several classes the solution of a linear system per leaf (1e-10 off)
    several = case.get("loss") == "MultiClass"
    return dict(rel=4e-10 if several else 4e-12, max=2e-8 if several else 2e-10, differ=0.0)


# ---- the same in plain 64-bit arithmetic ----------------------------------------------------
_MUL = np.uint64(6364136223846793005)


def _mix(x):
    xs = (((x >> np.uint64(18)) ^ x) >> np.uint64(27)).astype(np.uint32)
    rot = (x >> np.uint64(59)).astype(np.uint32)
    return (xs >> rot) | (xs << ((np.uint32(32) - rot) & np.uint32(31)))


class _Rng:
    """The training stream: two 64-bit linear congruential generators with permuted outputs, the
    upper and lower half of every draw (each element of the seeds a stream of its own)."""

    def __init__(self, seed):
        x = np.array(seed, np.uint64, ndmin=1).copy()
        got = []
        for _ in range(6):
            x = x * _MUL + np.uint64(1)
            got.append(_mix(x).astype(np.uint64))
        s1, q1, s2, q2 = got[0] | got[1] << np.uint64(32), got[2], got[3] | got[4] << np.uint64(32), got[5]
        low = np.uint64(0x7FFFFFFF)
        q2 = np.where((q1 & low) == (q2 & low), ~q2 & np.uint64(0xFFFFFFFF), q2)
        self.x, self.c = [s1, s2], [q1 << np.uint64(1) | np.uint64(1), q2 << np.uint64(1) | np.uint64(1)]

    def draw(self):
        for k in range(2):
            self.x[k] = self.x[k] * _MUL + self.c[k]
        return _mix(self.x[0]).astype(np.uint64) << np.uint64(32) | _mix(self.x[1]).astype(np.uint64)

    def run_of(self, n):
        """The next n draws of a single stream (doubling the stretch of known states)."""
        out = []
        for k in range(2):
            a, d = _MUL, np.uint64(1)
            x = self.x[k] * a + self.c[k]
            while x.size < n:
                x = np.concatenate([x, x * a + self.c[k] * d])
                d, a = d * (a + np.uint64(1)), a * a
            out.append(_mix(x[:n]).astype(np.uint64))
        return out[0] << np.uint64(32) | out[1]


def _unit(v):
    return (v >> np.uint64(11)).astype(np.float64) / 9007199254740991.0


def _sample(case):
    """The first tree's sample: (kept, weight) of every row."""
    n = case["n"]
    if case["bootstrap"] == "No":
        return None
    with np.errstate(over="ignore"):
        r = _Rng(0)
        r.draw(), r.draw()
        if case["bootstrap"] == "Bernoulli":
            return (_unit(r.run_of(n)) < float(np.float32(0.66))).astype(np.float64)
        blocks = (n + 999) // 1000
        s = _Rng(r.draw()[0] + np.arange(blocks, dtype=np.uint64))
        for _ in range(10):
            s.draw()
        u = np.stack([_unit(s.draw()) for _ in range(1000)], 1).reshape(-1)[:n].astype(np.float32)
    v = u.view(np.uint32)   # the fast logarithm of the sampler, in its own 32 bits
    m = ((v & np.uint32(0x007FFFFF)) | np.uint32(0x3F000000)).view(np.float32)
    f = np.float32
    y = v.astype(np.float32) * f(1.1920928955078125e-7)
    log = f(0.69314718) * (y - f(124.22551499) - f(1.498030302) * m - f(1.72587999) / (f(0.3520887068) + m))
    return (-log).astype(np.float64)


def _sums(leaf, L, column, B, stats):
    """[L][B] sums of each statistic of one column."""
    at = leaf * B + column
    return [torch.bincount(at, weights=s, minlength=L * B).view(L, B) for s in stats]


def _first_tree(case, d):
    n, F, B, D, K = case["n"], case["features"], int(d["counts"].max()) + 1, case["depth"], case["classes"]
    dev = "cuda"
    y = torch.from_numpy(d["target"]).to(dev)
    w = torch.ones(n, dtype=torch.float64, device=dev) if d["weight"] is None else torch.from_numpy(d["weight"]).to(dev)
    l2 = 3.0 * float(w.mean())
    weight = w
    if case["loss"] == "RMSE":
        der, der2 = [y - y.mean()], -torch.ones_like(y)
    elif case["loss"] in ("Logloss", "CrossEntropy"):
        der, der2 = [y - 0.5], torch.full_like(y, -0.25)
    elif case["loss"] == "MultiClass":
        der = [(y == k).double() - 1.0 / K for k in range(K)]
    else:   # PairLogit: every pair at one half
        pw, pl = (torch.from_numpy(d[k].astype(np.int64)).to(dev) for k in ("winner", "loser"))
        wins, losses = torch.bincount(pw, minlength=n).double(), torch.bincount(pl, minlength=n).double()
        der, der2, weight = [0.5 * (wins - losses)], -0.25 * (wins + losses), wins + losses
    sample = _sample(case)
    s = torch.ones_like(y) if sample is None else torch.from_numpy(sample).to(dev)
    stats = [x * w * s for x in der] + [weight * s]
    bins = torch.from_numpy(d["bins"]).to(dev)
    leaf = torch.zeros(n, dtype=torch.int64, device=dev)
    for level in range(D):
        L, best = 1 << level, (-math.inf, 0, 0)
        for f in range(F):
            nb = int(d["counts"][f])
            h = [torch.cumsum(t, 1) for t in _sums(leaf, L, bins[f].long(), B, stats)]
            num = torch.zeros(B, dtype=torch.float64, device=dev)
            den = torch.full_like(num, 1e-100)
            for k in range(K):
                for side in range(2):
                    a, b = (h[k], h[K]) if side == 0 else (h[k][:, -1:] - h[k], h[K][:, -1:] - h[K])
                    avg = torch.where(b > 0, a / (b + l2), torch.zeros_like(a))
                    num += (avg * a).sum(0)
                    den += (avg * avg * b).sum(0)
            score = (num / den.sqrt() if case["score"] == "Cosine" else num)[:nb].cpu().numpy()
            if score.size and score.max() > best[0]:
                best = (float(score.max()), f, int(np.argmax(score)))
        leaf |= (bins[best[1]].long() > best[2]).long() << level
    L = 1 << D

    def total(x):
        return torch.bincount(leaf, weights=x, minlength=L)

    if case["loss"] == "MultiClass":
        p = 1.0 / K
        W = total(w)
        H = torch.zeros(L, K, K, dtype=torch.float64, device=dev)
        for a in range(K):
            for b in range(K):
                H[:, a, b] = W * (p * p - (p if a == b else 0.0))
        G = torch.stack([total(x * w) for x in der], 1)
        trace = torch.clamp((-torch.diagonal(H, dim1=1, dim2=2)).max(1).values, min=l2)
        adj = torch.clamp(trace.float() * 1.1920928955078125e-7, min=float(np.float32(l2))).double()
        H = H - adj[:, None, None] * torch.eye(K, dtype=torch.float64, device=dev)
        value = torch.linalg.solve((-H).cpu(), G.cpu()).T
    else:
        g = total(der[0] * w)
        if case["leaf"] == "Newton":
            h = -total(der2 * w) + l2
            value = torch.where(h == 0, torch.zeros_like(g), g / h)
        else:
            h = total(weight)
            value = torch.where(h > 0, g / (h + l2), torch.zeros_like(g))
        if case["loss"] == "PairLogit":   # values around zero over the documents
            docs = torch.bincount(leaf, minlength=L)
            value = torch.where(docs > 0, value - (value * docs).sum() / n, torch.zeros_like(value))
        value = value[None].cpu()
    return value.numpy() * float(np.float32(case["lr"]))


def exact(case, seed):
    if case["kind"] == "predict":
        m = _model(case, seed)
        x = torch.from_numpy(m["x"]).to("cuda")
        K, D = case["classes"], case["depth"]
        leaf = torch.from_numpy(m["leaf"]).to("cuda").view(-1, K)
        out = torch.zeros(K, case["n"], dtype=torch.float64, device="cuda")
        for t in range(case["trees"]):
            at = torch.full((case["n"],), t << D, dtype=torch.int64, device="cuda")
            for i in range(D):
                at += (x[int(m["feature"][t * D + i])].double() > m["border"][t * D + i]).long() << i
            out += leaf[at].T
        return (out + torch.from_numpy(m["bias"]).to("cuda")[:, None]).cpu().numpy()
    # None: a fit goes through border selection and many trees, pair statistics solve a linear
    # system for every border, target statistics go row by row through a permutation, and the
    # largest tables take too long a column at a time
    if case["kind"] == "fit" or case["loss"] == "PairLogitPairwise" or case["ctr"]:
        return None
    if float(case["n"]) * case["features"] * case["depth"] * (case["classes"] + 1) > 2.5e9:
        return None
    return dict(splits=None, leaves=_first_tree(case, _inputs(case, seed)), one_hot=None)
