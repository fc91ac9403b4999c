"""The work that users of this package have it do, as cases that can be timed one by one.

Sequences are drawn uniformly over ACGT with 1 % N, packed as the batcher packs them. Sizes come from the benchmark's
configurations (64 to 100 000 sequences of 20 to 500 letters, 1 to 90 models of 16 filters), from the operator benchmark
(8192 sequences, 256 filters) and from the tests (filters of 8 to 32 taps, all three pooling types, both float types,
reverse-complement pairs, the reference's way of scoring windows and mutations).

kind        what a program calls
score       SequenceNet.predict on a resident batch
train       SequenceNet.train_step over the resident minibatches of an epoch
calibrate   ModelGroup.train_step: models of mixed architecture on shared minibatches
layers      the drop-in operators one after another, forward and backward, as the reference's graph drives them
gradients   predict.gen_predictions with back-propagated input gradients, from strings to host arrays
mutations   predict.gen_predictions with finite-difference mutation maps, from strings to host arrays
windows     predict.gen_predictionmaps: every window of long sequences scored, from strings to host arrays
"""
import numpy as np
import torch

from deepbind_amd import kangaroo_smat as ks
from deepbind_amd import predict
from deepbind_amd import smat as sm
from deepbind_amd.model import ModelGroup, SequenceNet


def listed():
    one = dict(models=1, filters=16, rc=False, dropout=0.0)
    return [
        # one trained model scores one small batch: what an interactive user or a service sends per request
        dict(one, name="score_small", kind="score", taps=24, pool="max", hidden=32, loss="nll", count=64, lo=101, hi=101),
        # an ensemble of short-motif models scores a whole array of RNA probes and peaks of mixed lengths
        dict(name="score_ragged", kind="score", models=24, filters=16, rc=False, dropout=0.5, taps=16, pool="all", hidden=32, loss="nll",
             count=20000, lo=30, hi=150),
        # 64 models over 100 000 long sequences: the genome-scale scoring run, and the largest case
        dict(name="score_bulk", kind="score", models=64, filters=16, rc=False, dropout=0.0, taps=24, pool="max", hidden=32, loss="mse",
             count=100000, lo=500, hi=500),
        # one RNA model's final training: short ragged probes, both poolings, no hidden layer
        dict(one, name="train_probes", kind="train", taps=16, pool="all", hidden=0, loss="mse", count=128, batches=8, lo=38, hi=41),
        # one peak model's final training: fixed-length peaks against shuffled ones, dropout
        dict(one, name="train_peaks", kind="train", dropout=0.5, taps=24, pool="max", hidden=32, loss="nll", count=128, batches=8, lo=101, hi=101),
        # hyper-parameter search: 30 random settings x 3 folds trained side by side on shared minibatches
        dict(name="train_calibration", kind="calibrate", draws=30, folds=3, filters=16, taps=24, count=256, batches=4, lo=20, hi=40),
        # an ensemble trained on both strands of whole peaks with long motif detectors
        dict(name="train_paired", kind="train", models=8, filters=16, rc=True, dropout=0.5, taps=32, pool="all", hidden=32, loss="nll",
             count=1024, batches=2, lo=90, hi=200),
        # the reference's own graph, layer by layer, with its operators swapped for this package's
        dict(name="layers_float32", kind="layers", dtype="float32", filters=256, taps=24, pool="all", count=8192, lo=101, hi=101),
        # the same in double precision, which the reference compiles every operator for and its gradient check runs in
        dict(name="layers_float64", kind="layers", dtype="float64", filters=64, taps=24, pool="max", count=1000, lo=60, hi=140),
        # sequence logos: one model's input gradients on a thousand peaks and their reverse strands
        dict(one, name="gradient_maps", kind="gradients", rc=True, taps=24, pool="max", hidden=32, loss="nll", count=1000, lo=101, hi=101),
        # mutation maps: every single-letter change of a handful of sequences
        dict(one, name="mutation_maps", kind="mutations", rc=True, taps=24, pool="max", hidden=32, loss="nll", count=32, lo=60, hi=101),
        # a long sequence searched for its binding sites window by window
        dict(one, name="window_scan", kind="windows", taps=16, pool="all", hidden=0, loss="mse", count=4, lo=900, hi=1100, window=40),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case of the same ranges: sizes spread over their logarithm, capped so that none costs more than the largest listed."""
    kind = rng.choice(("score", "score", "score", "train", "train", "calibrate", "layers", "layers", "gradients", "mutations", "windows"))
    pool = rng.choice(("max", "max", "all", "avg"))
    hidden = rng.choice((0, 32))
    loss = rng.choice(("nll", "mse"))
    rc = rng.random() < 0.3
    dropout = rng.choice((0.0, 0.0, 0.25, 0.5))
    taps = rng.randint(8, 32)
    filters = rng.choice((12, 16, 16, 16))
    lo = _log(rng, 20, 400)
    hi = lo if rng.random() < 0.4 else rng.randint(lo, min(500, 2 * lo))
    net = dict(filters=filters, taps=taps, pool=pool, hidden=hidden, loss=loss, rc=rc, dropout=dropout)
    if kind == "score":
        models, count = _log(rng, 1, 64), _log(rng, 32, 100000)
        return dict(net, kind=kind, models=models, count=count // (2 if rc else 1), lo=lo, hi=hi)
    if kind == "train":
        models, count = _log(rng, 1, 16), _log(rng, 64, 2048)
        return dict(net, kind=kind, models=models, count=count // (2 if rc else 1), batches=rng.randint(2, 8), lo=lo, hi=min(hi, 250) if lo <= 250 else lo)
    if kind == "calibrate":
        return dict(kind=kind, draws=rng.randint(4, 30), folds=3, filters=filters, taps=taps, count=_log(rng, 64, 512), batches=rng.randint(2, 4),
                    lo=min(lo, 101), hi=min(max(hi, lo), 101))
    if kind == "layers":
        double = rng.random() < 0.4
        return dict(kind=kind, dtype="float64" if double else "float32", filters=rng.choice((16, 32, 64, 96) if double else (16, 48, 128, 256)), taps=taps,
                    pool=pool, count=_log(rng, 64, 1000 if double else 8192), lo=min(lo, 101), hi=min(max(hi, lo), 140))
    one = dict(net, models=1)
    if kind == "gradients":
        return dict(one, kind=kind, count=_log(rng, 16, 2000), lo=min(lo, 101), hi=min(max(hi, lo), 140))
    if kind == "mutations":
        return dict(one, kind=kind, count=_log(rng, 1, 128), lo=min(lo, 101), hi=min(max(hi, lo), 101))
    return dict(one, kind=kind, count=rng.randint(1, 8), lo=_log(rng, 100, 1500), hi=1500, window=rng.randint(20, 60))


# ---------------------------------------------------------------------------------------------- inputs
def _plan(case, batch=0):
    """Generator of what belongs to the case and not to its data: sequence lengths, architectures."""
    return np.random.default_rng([case["count"], case["lo"], case["hi"], case["taps"], batch])


def _lengths(case, batch=0):
    return _plan(case, batch).integers(case["lo"], case["hi"] + 1, size=case["count"])


def _pack(gen, case, rc=False, batch=0):
    """Packed batch of random sequences, on the GPU: (X, R). With rc every row is followed by its reverse complement."""
    pad = case["taps"] - 1
    lens = _lengths(case, batch)
    n = lens.repeat(2) if rc else lens
    edges = np.concatenate([[0], np.cumsum(n + pad)])
    X = torch.full((int(edges[-1]) + pad,), 255, dtype=torch.uint8, device="cuda")
    total = int(lens.sum())
    codes = torch.randint(0, 4, (total,), generator=gen, dtype=torch.uint8, device="cuda")
    codes[torch.rand(total, generator=gen, device="cuda") < 0.01] = 255
    start = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)])).cuda()
    lens_d, edges_d = torch.from_numpy(lens).cuda(), torch.from_numpy(edges).cuda()
    step = 2 if rc else 1
    if case["lo"] == case["hi"] and not rc:
        X[:-pad].view(case["count"], -1)[:, pad:] = codes.view(case["count"], -1)
    else:
        row = torch.repeat_interleave(torch.arange(case["count"], device="cuda"), lens_d)
        at = torch.arange(total, device="cuda") - start[row]
        X[edges_d[step * row] + pad + at] = codes
        if rc:
            X[edges_d[2 * row + 2] - 1 - at] = torch.where(codes < 4, 3 - codes, codes)
    R = torch.from_numpy(np.stack([edges[:-1], edges[1:]], axis=1).astype(np.uint32)).cuda()
    return X.view(-1, 1), R


def _strings(rng, case):
    letters = np.frombuffer(b"ACGTN", dtype=np.uint8)
    out = []
    for n in _lengths(case):
        codes = rng.integers(0, 4, size=int(n))
        codes[rng.random(int(n)) < 0.01] = 4
        out.append(letters[codes].tobytes().decode("ascii"))
    return out


def _weights(rng, case, conv, dense):
    """Parameters of a net: filters and dense weights of the given scales, biases a little off zero as training leaves them."""
    k = case["filters"] * (2 if case["pool"] == "all" else 1)
    nm, h, F = case["models"], case["hidden"], case["filters"] * case["models"]
    f = lambda s, *shape: (rng.standard_normal(shape) * s).astype(np.float32)
    p = dict(Wc=f(conv, 4 * case["taps"], F), bc=f(conv, 1, F))
    if h:
        p.update(W1=f(dense, k * nm, h), b1=f(dense, 1, h * nm), W2=f(dense, h * nm, 1), b2=f(dense, 1, nm))
    else:
        p.update(W1=f(dense, k * nm, 1), b1=f(dense, 1, nm))
    return p


def _net(rng, case, conv, dense, **kw):
    net = SequenceNet(case["models"], case["filters"], case["taps"], pool=case["pool"], hidden=case["hidden"], loss=case["loss"],
                      dropout=case["dropout"], reverse_complement=case["rc"], **kw)
    net.set_params(_weights(rng, case, conv, dense))
    return net


def _targets(rng, case, rows, models, loss):
    if loss == "nll":
        y = (rng.random((rows, 1)) < 0.5).astype(np.float32)
    else:
        y = rng.lognormal(0.0, 1.0, size=(rows, 1))
        y = ((y - y.mean()) / y.std()).astype(np.float32)
    return np.repeat(y, models, axis=1)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    state = dict(kind=kind, case=case)
    if kind == "score":
        state["net"] = _net(rng, case, 0.05, 0.05)
        state["X"], state["R"] = _pack(gen, case, case["rc"])
    elif kind == "train":
        state["net"] = _net(rng, case, 0.01, 0.01, rate=0.01, momentum=0.9)
        state["batches"] = []
        for i in range(case["batches"]):
            X, R = _pack(gen, case, case["rc"], batch=i)
            Y = _targets(rng, case, case["count"], case["models"], case["loss"])
            state["batches"].append((X, R, torch.from_numpy(Y.repeat(2, axis=0) if case["rc"] else Y).cuda()))
    elif kind == "calibrate":
        n, folds = case["draws"], case["folds"]
        rep = lambda v: np.repeat(np.asarray(v), folds)
        arch = _plan(case, 96).integers(0, 2, (2, n))
        pools = [("max", "all")[int(v)] for v in arch[0] for _ in range(folds)]
        hiddens = [(0, 32)[int(v)] for v in arch[1] for _ in range(folds)]
        loguniform = lambda lo, hi: np.exp(rng.uniform(np.log(lo), np.log(hi), size=n))
        grp = ModelGroup(pools, hiddens, case["filters"], case["taps"], loss="nll", rate=rep(loguniform(0.0005, 0.05)),
                         momentum=rep(rng.uniform(0.95 ** 0.5, 0.99 ** 0.5, size=n) ** 2), decay_conv=rep(loguniform(1e-15, 1e-3)),
                         decay_full=rep(loguniform(1e-10, 1e-3)), dropout=rep(rng.choice([0.0, 0.0, 0.25, 0.5], size=n)), weight_decay_start=0)
        for g, (idx, net) in enumerate(grp.groups):
            net.init_params(init_conv=rng.uniform(1e-3, 1e-2, len(idx)), init_full=rng.uniform(1e-3, 1e-2, len(idx)), seed=seed + g)
        state["net"], state["batches"] = grp, []
        for i in range(case["batches"]):
            X, R = _pack(gen, case, batch=i)
            Y = _targets(rng, case, case["count"], n * folds, "nll")
            M = (np.arange(case["count"])[:, None] % folds) != (np.arange(n * folds)[None, :] % folds)
            state["batches"].append((X, R, torch.from_numpy(Y).cuda(), torch.from_numpy(M).cuda()))
    elif kind == "layers":
        dtype = getattr(torch, case["dtype"])
        X, R = _pack(gen, case)
        F, k = case["filters"], case["filters"] * (2 if case["pool"] == "all" else 1)
        normal = lambda *s: torch.randn(s, generator=gen, dtype=dtype, device="cuda") * 0.1
        state.update(X=X, R=R, W=normal(4 * case["taps"], F), b=normal(1, F), dP=normal(case["count"], k))
    else:
        state["net"] = _net(rng, case, 0.3, 0.2)
        state["seqs"] = _strings(rng, case)
    return state


# ---------------------------------------------------------------------------------------------- one pass
def _flat(maps):
    return np.concatenate([m for _, m in maps])


def run(state):
    case, kind = state["case"], state["kind"]
    if kind == "score":
        return state["net"].predict(state["X"], state["R"])
    if kind == "train":
        net = state["net"]
        for X, R, Y in state["batches"]:
            net.train_step(X, R, Y)
        return {"P": net.P, "dP": net.dP, "mP": net.mP}
    if kind == "calibrate":
        for X, R, Y, M in state["batches"]:
            state["net"].train_step(X, R, Y, M)
        return [{"P": net.P, "dP": net.dP, "mP": net.mP} for _, net in state["net"].groups]
    if kind == "layers":
        X, R, W, pool = state["X"], state["R"], state["W"], case["pool"]
        Z = sm.zeros((X.numel(), W.shape[1]), dtype=W.dtype)
        ks.corr1ord(W, X, Z, 4)
        A = sm.relu(sm.add_rowvec(Z, state["b"]))
        pooled, argmax = ks.poolrgn(A, R, pool, want_argmax=True)
        dA = sm.zeros_like(A)
        ks.poolrgn_bprop(dA, R, state["dP"], argmax, pool)
        dZ = sm.mul_sign(dA, A)
        db = sm.sum_axis0(dZ)
        dW = torch.zeros_like(W)
        ks.corr1ord_bprop_W(dW, X, dZ, 4)
        dX = sm.zeros((X.numel(), 4), dtype=W.dtype)
        ks.corr1ord_bprop_X(dX, W, dZ, 4)
        return {"Z": Z, "A": A, "pooled": pooled, "dA": dA, "dZ": dZ, "db": db, "dW": dW, "dX": dX}
    if kind == "windows":
        pmaps, _ = predict.gen_predictionmaps(state["net"], state["seqs"], windowsize=case["window"])
        return np.concatenate(pmaps)
    preds, maps = predict.gen_predictions(state["net"], state["seqs"], want_gmaps=True if kind == "gradients" else "finite_diff")
    return {"predictions": preds, "maps": _flat(maps)}


# ---------------------------------------------------------------------------------------------- what it takes at least
def work(case):
    """Bytes: every input read once, every output written once (the layers: each operator's). flops: the scan's gather-adds
    (one per row, filter and tap; the gradients' likewise) and the dense layers' multiply-adds."""
    kind, taps = case["kind"], case["taps"]
    rows = case["count"] * (2 if case.get("rc") else 1)
    mean = 0.5 * (case["lo"] + case["hi"])
    N = rows * (mean + taps - 1)
    if kind == "layers":
        F, size = case["filters"], 8 if case["dtype"] == "float64" else 4
        k = F * (2 if case["pool"] == "all" else 1)
        amap = N * F * size
        # written: Z, Z + b, A, dA, dZ; read: Z, Z + b, A (pooling), dA, A (its gradient), dZ (column sums, dW, dX)
        spread = amap if case["pool"] != "max" else 0.0
        return {"bytes": 13 * amap + spread + 3 * N + N * 4 * size + 2 * rows * k * size, "flops": 3.0 * N * F * taps}
    if kind == "calibrate":
        models, F = case["draws"] * case["folds"], case["filters"] * case["draws"] * case["folds"]
        nparam = F * (4 * taps + 1) + models * (24 * 17 + 17)
        adds = 1.75 * N * F * taps + rows * models * 6 * 24 * 17
        return {"bytes": case["batches"] * (N + rows * (8 + 5 * models)) + 28.0 * nparam, "flops": case["batches"] * adds}
    models, h = case["models"], case["hidden"]
    F, k = case["filters"] * models, case["filters"] * (2 if case["pool"] == "all" else 1)
    head = models * (2 * k * (h or 1) + 2 * h)
    nparam = F * (4 * taps + 1) + models * ((k + 1) * (h or 1) + (h + 1 if h else 0))
    if kind == "score":
        return {"bytes": N + 8 * rows + 4 * nparam + 4 * rows * models, "flops": N * F * taps + rows * head}
    if kind == "train":
        back = rows * F * taps if case["pool"] == "max" else N * F * taps
        return {"bytes": case["batches"] * (N + 8 * rows + 4 * rows * models) + 28.0 * nparam, "flops": case["batches"] * (N * F * taps + back + 3 * rows * head)}
    if kind == "gradients":
        return {"bytes": 2 * rows * mean + 16 * case["count"] * mean + 4 * case["count"], "flops": N * F * taps + rows * F * taps + 2 * rows * head}
    if kind == "mutations":
        # a changed letter moves `taps` rows of the map by one term each, and the pooled maximum with them
        return {"bytes": rows * mean + 16 * case["count"] * mean, "flops": N * F * taps + 4 * rows * mean * (F * taps + head)}
    count = case["count"] * (0.5 * (case["lo"] + case["hi"]) + case["window"] - 1)
    return {"bytes": case["count"] * mean + 4 * count, "flops": count * (2 if case["rc"] else 1) * ((case["window"] + taps - 1) * F * taps + head)}


def tolerance(case):
    """About four times what the path was seen to be off by in float64, or with its sums in another order. What exceeds plain
    round-off comes from decisions that fall the other way when a sum moves by its last bit: a rectifier input that rounds to
    the other side of zero, and, in reverse-complement training, which strand of a pair predicts more."""
    kind = case["kind"]
    if kind == "score":
        return {"rel": 1e-6, "max": 1e-5}                       # seen: 6e-8, 3e-7
    if kind == "train":
        return {"rel": 1e-2, "max": 0.4} if case["rc"] else {"rel": 5e-5, "max": 2e-3}      # seen: 3.5e-3, 0.1; 5e-6 in one pass, 1e-4
    if kind == "calibrate":
        return {"rel": 1e-5, "max": 4e-4}                       # seen: 1.7e-6, 6.7e-5
    if kind == "layers":
        return {"rel": 1e-14, "max": 1e-13} if case["dtype"] == "float64" else {"rel": 5e-5, "max": 0.5}      # seen: 1e-15, 3e-15; 1.3e-5, 0.14
    if kind == "gradients":
        return {"rel": 1e-5, "max": 1e-4}                       # seen: 3e-7, 1e-6, where no rectifier changed sides
    if kind == "mutations":
        return {"rel": 5e-5, "max": 2e-4}                       # seen: 1.7e-5, 5e-5: differences of nearly equal scores
    return {"rel": 2e-6, "max": 1e-5}                           # seen: 3.4e-7, 1.1e-6
