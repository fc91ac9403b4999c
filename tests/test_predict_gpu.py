"""Prediction-time callers on the GPU (scores, gradient maps, mutation maps, window scans) against the oracle."""
import numpy as np
import pytest
import torch

from oracle import deepbind_oracle as orc
from tests.gpu_util import assert_close

pytestmark = pytest.mark.gpu

ACT, GRAD = 1e-5, 1e-4


def _params(rng, m, F, pool, hidden, scale=0.5):
    # dense weights small enough that the logistic output stays away from saturation: two strands that
    # both round to 1.0f would be a tie in float32 but not in the float64 oracle
    k = F * (2 if pool == "all" else 1)
    f = lambda *s: (rng.standard_normal(s) * scale).astype(np.float32)
    p = {"Wc": f(4 * m, F), "bc": f(1, F) * 0.3}
    if hidden:
        p.update(W1=f(k, hidden) * 0.3, b1=f(1, hidden) * 0.2, W2=f(hidden, 1) * 0.3, b2=f(1, 1) * 0.2 - 0.2)
    else:
        p.update(W1=f(k, 1) * 0.2, b1=f(1, 1) * 0.2 - 0.2)
    return p


def _seqs(rng, n, lo, hi, p_n=0.04):
    out = []
    for _ in range(n):
        s = "".join("ACGT"[v] for v in rng.integers(0, 4, int(rng.integers(lo, hi + 1))))
        out.append("".join("N" if rng.random() < p_n else ch for ch in s))
    return out


def _net(p, m, F, pool, hidden, loss, rc, rate):
    from deepbind_amd.model import SequenceNet
    net = SequenceNet(1, F, m, pool=pool, hidden=hidden, loss=loss, dropout=rate, reverse_complement=rc)
    net.set_params(p)
    return net


CASES = [("max", 8, "nll", False, 0.0, 24, 16), ("all", 0, "mse", False, 0.3, 16, 16), ("max", 0, "mse", True, 0.0, 11, 5),
         ("max", 32, "nll", True, 0.5, 24, 16), ("avg", 4, "mse", False, 0.0, 6, 7)]


@pytest.mark.parametrize("pool,hidden,loss,rc,rate,m,F", CASES)
@pytest.mark.parametrize("mode", [False, True, "finite_diff"])
def test_gen_predictions(pool, hidden, loss, rc, rate, m, F, mode):
    from deepbind_amd import predict
    rng = np.random.default_rng(1000 * m + 10 * hidden + int(rc))
    p = _params(rng, m, F, pool, hidden)
    seqs = _seqs(rng, 7, 18, 30)                       # ragged: includes the pad-mutation quirk of short sequences
    out = "logistic" if loss == "nll" else "linear"
    p64 = {k: v.astype(np.float64) for k, v in p.items()}
    Zr, mr = orc.gen_predictions(p64, seqs, pool, hidden, out, dropout_rate=[rate] if rate else None, reverse_complement=rc, want_gmaps=mode)
    net = _net(p, m, F, pool, hidden, loss, rc, rate)
    # two batches, to cover the batch loop
    Z, maps = predict.gen_predictions(net, seqs, want_gmaps=mode, batchsize=4)
    Zr2 = [orc.gen_predictions(p64, seqs[s:s + 4], pool, hidden, out, dropout_rate=[rate] if rate else None, reverse_complement=rc,
                               want_gmaps=mode) for s in (0, 4)]
    Zr = np.vstack([z for z, _ in Zr2])
    assert Z.shape == (len(seqs), 1)
    assert_close(Z, Zr, ACT, "Z")
    if not mode:
        assert maps is None
        return
    mr = sum([mm for _, mm in Zr2], [])
    assert len(maps) == len(mr) == len(seqs)
    scale = max(np.abs(b).max() for _, b in mr) + 1e-30
    for (sa, a), (sb, b) in zip(maps, mr):
        assert sa == sb and a.shape == b.shape
        assert np.abs(a - b).max() <= GRAD * scale, (np.abs(a - b).max(), scale)


@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("stride,want", [(1, True), (1, False), (4, False)])
def test_gen_predictionmaps(rc, stride, want):
    from deepbind_amd import predict
    rng = np.random.default_rng(17)
    m, F, pool, hidden = 8, 6, "max", 5
    p = _params(rng, m, F, pool, hidden)
    p64 = {k: v.astype(np.float64) for k, v in p.items()}
    seqs = _seqs(rng, 3, 25, 40)
    pr, gr = orc.gen_predictionmaps(p64, seqs, pool, hidden, "logistic", reverse_complement=rc, stride=stride, windowsize=12, want_gmaps=want)
    net = _net(p, m, F, pool, hidden, "nll", rc, 0.0)
    pm, gm = predict.gen_predictionmaps(net, seqs, stride=stride, windowsize=12, want_gmaps=want)
    assert len(pm) == len(pr) == 3
    for a, b in zip(pm, pr):
        assert a.shape == b.shape
        assert_close(a, b, ACT, "pmap")
    if want:
        scale = max(np.abs(b).max() for b in gr) + 1e-30
        for a, b in zip(gm, gr):
            assert a.shape == b.shape and np.abs(a - b).max() <= GRAD * scale
    else:
        assert gm is None
    with pytest.raises(ValueError):
        predict.gen_predictionmaps(net, seqs, stride=2, windowsize=12, want_gmaps=True)


@pytest.mark.parametrize("pool,hidden,loss,rc,m,F", [("max", 32, "nll", True, 24, 16), ("all", 40, "nll", False, 32, 17), ("avg", 0, "mse", False, 1, 3),
                                                     ("all", 0, "mse", True, 9, 33), ("max", 5, "mse", False, 17, 64)])
def test_mutation_map_kernel_edges(pool, hidden, loss, rc, m, F):
    """Lengths around a workgroup's 16 letters (one letter to several workgroups, a sequence shorter than its neighbours by more and
    by less than the pad), filters beyond one and two tiles of 16, one tap, hidden units beyond a pass of 16 lanes."""
    from deepbind_amd import _lib, predict
    rng = np.random.default_rng(7 * m + F)
    p = _params(rng, m, F, pool, hidden)
    seqs = ["".join("ACGT"[v] for v in rng.integers(0, 4, n)) for n in (1, 15, 16, 17, 40, 33)]
    seqs[3] = "n" + seqs[3][1:].lower().replace("t", "u")
    out = "logistic" if loss == "nll" else "linear"
    Zr, mr = orc.gen_predictions({k: v.astype(np.float64) for k, v in p.items()}, seqs, pool, hidden, out, reverse_complement=rc,
                                 want_gmaps="finite_diff")
    net = _net(p, m, F, pool, hidden, loss, rc, 0.0)
    assert _lib.dll().dbk_mutation_map_takes(m, F, _lib.str2pooltype[pool], hidden) == 1
    Z, maps = predict.gen_predictions(net, seqs, want_gmaps="finite_diff")
    assert_close(Z, Zr, ACT, "Z")
    scale = max(np.abs(b).max() for _, b in mr)
    for (sa, a), (sb, b) in zip(maps, mr):
        assert sa == sb and a.shape == b.shape
        assert np.abs(a - b).max() <= GRAD * scale, (len(sa), np.abs(a - b).max(), scale)


@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("pool,hidden,m,F", [("max", 0, 2, 16), ("all", 64, 3, 5), ("avg", 17, 5, 16), ("all", 3, 18, 16), ("max", 32, 25, 16), ("all", 0, 33, 4),
                                             ("avg", 9, 64, 2)])
def test_mutation_map_quarters_of_any_number_of_taps(pool, hidden, m, F, rc):
    """A lane scans a quarter of the rows that a letter moves, four, six or eight of them at a time: taps that leave quarters short or empty,
    one more than a multiple, more than one round; sequences shorter than their neighbours, whose changes land in the next one's pad."""
    from deepbind_amd import predict
    rng = np.random.default_rng(11 * m + F)
    p = _params(rng, m, F, pool, hidden)
    seqs = _seqs(rng, 9, 1, 30)
    Zr, mr = orc.gen_predictions({k: v.astype(np.float64) for k, v in p.items()}, seqs, pool, hidden, "logistic", reverse_complement=rc, want_gmaps="finite_diff")
    Z, maps = predict.gen_predictions(_net(p, m, F, pool, hidden, "nll", rc, 0.0), seqs, want_gmaps="finite_diff")
    assert_close(Z, Zr, ACT, "Z")
    scale = max(np.abs(b).max() for _, b in mr)
    for (sa, a), (sb, b) in zip(maps, mr):
        assert sa == sb and np.abs(a - b).max() <= GRAD * scale, (len(sa), np.abs(a - b).max(), scale)


@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("n,length", [(80, 57), (300, 101)])
def test_mutation_maps_do_not_depend_on_how_many_letters_a_workgroup_takes(rc, n, length):
    """Eight and sixteen letters per workgroup (many sequences) give the bits that four do (one sequence): maxima are the same rows' sums."""
    from deepbind_amd import predict
    rng = np.random.default_rng(n)
    net = _net(_params(rng, 24, 16, "max", 32), 24, 16, "max", 32, "nll", rc, 0.0)
    seqs = _seqs(rng, n, length, length)
    Z, maps = predict.gen_predictions(net, seqs, want_gmaps="finite_diff")
    for k in (0, 1, n // 2, n - 1):
        Z1, one = predict.gen_predictions(net, seqs[k:k + 1], want_gmaps="finite_diff")
        assert np.array_equal(Z[k:k + 1], Z1) and np.array_equal(maps[k][1], one[0][1])


@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 12, 13])
def test_mutation_maps_of_few_taps(m, rc):
    """Two rows at a time up to 8 taps, three up to 12: against the oracle with four letters per workgroup, the same bits with eight and sixteen."""
    from deepbind_amd import predict
    rng = np.random.default_rng(40 + m)
    p = _params(rng, m, 16, "max", 32)
    net = _net(p, m, 16, "max", 32, "nll", rc, 0.0)
    seqs = _seqs(rng, 270, 57, 57)
    Z, maps = predict.gen_predictions(net, seqs[:6], want_gmaps="finite_diff")
    Zr, mr = orc.gen_predictions({k: v.astype(np.float64) for k, v in p.items()}, seqs[:6], "max", 32, "logistic", reverse_complement=rc, want_gmaps="finite_diff")
    assert_close(Z, Zr, ACT, "Z")
    scale = max(np.abs(b).max() for _, b in mr)
    for (_, a), (_, b) in zip(maps, mr):
        assert np.abs(a - b).max() <= GRAD * scale
    for n in (130, 270):
        Zn, more = predict.gen_predictions(net, seqs[:n], want_gmaps="finite_diff")
        assert np.array_equal(Zn[:6], Z)
        for (_, a), (_, b) in zip(maps, more):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("pool,hidden,m,F", [("avg", 6, 24, 16), ("all", 0, 9, 33), ("max", 5, 16, 16), ("avg", 0, 1, 4)])
def test_mutation_to_the_letter_that_is_there_is_none(pool, hidden, m, F, rc):
    """Exactly zero at every sequence's own letters, wherever in the sequence the workgroup that scores them begins. (Longer sequences
    first: a shorter one before would have its changes spill into the next.)"""
    from deepbind_amd import predict
    rng = np.random.default_rng(3 * m + F)
    net = _net(_params(rng, m, F, pool, hidden), m, F, pool, hidden, "nll", rc, 0.0)
    seqs = ["".join("ACGT"[v] for v in rng.integers(0, 4, n)) for n in (131, 90, 90, 37, 2)]
    _, maps = predict.gen_predictions(net, seqs, want_gmaps="finite_diff")
    for s, (letters, g) in zip(seqs, maps):
        own = ["ACGT".index(ch) for ch in s]
        assert letters == s and (g[np.arange(len(s)), own] == 0).all()
    assert any((g != 0).any() for _, g in maps)


@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("pool,hidden,m,F,n", [("max", 6, 24, 16, 5), ("max", 0, 9, 33, 70), ("avg", 5, 16, 16, 5), ("all", 8, 32, 16, 300), ("max", 32, 7, 4, 5)])
def test_mutation_between_letters_of_equal_weight_is_none(pool, hidden, m, F, n, rc):
    """A filter that does not tell A from G nor C from T scores a sequence the same, bit for bit, when one takes the other's place: the rows that
    hold the letter are added in one order for all four. (Both strands: the complements are equal as well. Longer sequences first, so that
    no change lands in the next one's pad.)"""
    from deepbind_amd import predict
    rng = np.random.default_rng(5 * m + F)
    p = _params(rng, m, F, pool, hidden)
    W = p["Wc"].reshape(m, 4, F)
    W[:, 2], W[:, 3] = W[:, 0], W[:, 1]
    seqs = sorted(("".join("ACGT"[v] for v in rng.integers(0, 4, int(k))) for k in rng.integers(20, 90, n)), key=len, reverse=True)
    _, maps = predict.gen_predictions(_net(p, m, F, pool, hidden, "nll", rc, 0.0), seqs, want_gmaps="finite_diff")
    for s, (_, g) in zip(seqs, maps):
        twin = ["GTAC".find(ch) for ch in s]
        assert (g[np.arange(len(s)), twin] == 0).all()
    assert all((g != 0).any() for _, g in maps)


@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("hidden,m,F", [(6, 24, 16), (0, 9, 33), (4, 30, 16), (3, 2, 5), (8, 64, 2)])
def test_filters_that_tell_no_letters_apart_have_no_mutations(hidden, m, F, rc):
    """Every window of such a filter has one sum, with unknown letters in it (their mean is the weight that all four have) and where a change
    lands in the pad of the next sequence as well: maps of zeros, bit for bit, by the maximum."""
    from deepbind_amd import predict
    rng = np.random.default_rng(m + F)
    p = _params(rng, m, F, "max", hidden)
    W = p["Wc"].reshape(m, 4, F)
    W[:] = W[:, :1]
    W[1::3] = 0.0
    p["bc"] += 0.5 * np.abs(W[:, 0].sum(axis=0))
    p["b2" if hidden else "b1"] += 5.0                  # (changes count where a score is positive)
    seqs = _seqs(rng, 60, 1, 40, 0.2) + ["N" * 12, "ACGT", "N", "GATTACA" * 5]
    Z, maps = predict.gen_predictions(_net(p, m, F, "max", hidden, "mse", rc, 0.0), seqs, want_gmaps="finite_diff")
    assert np.isfinite(Z).all() and (Z > 0).all()
    for _, g in maps:
        assert (g == 0).all()


@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("m,window,stride", [(1, 2, 1), (24, 20, 3), (8, 65, 7)])
def test_text_and_windows_are_packed_as_on_the_host(rc, m, window, stride):
    from deepbind_amd import _lib, data, predict
    from deepbind_amd.model import SequenceNet
    net = SequenceNet(1, 4, m, reverse_complement=rc)
    every = "".join(chr(c) for c in range(256))
    seqs = ["ACGTUacgtuNn.-", "", every, "G", "TT" * 90]
    X, R = predict._pack(net, predict._Text(seqs))
    Xr, Rr = data.pack_sequences(seqs, m - 1, reverse_complement=rc)
    assert np.array_equal(X.cpu().numpy(), Xr) and np.array_equal(R.cpu().numpy(), Rr)
    text = predict._Text(seqs)
    assert text.strings() == [data.ord2acgt(data.acgt2ord(s)) for s in seqs]
    assert text.strings(np.ones(len(seqs), bool)) == [data.revcomp(data.ord2acgt(data.acgt2ord(s))) for s in seqs]
    # windows: what predict sees, captured instead of scored
    seen = []
    net.predict = lambda X, R, F=None: seen.append((X.cpu().numpy(), R.cpu().numpy())) or torch.zeros((R.shape[0] // (2 if rc else 1), 1))
    predict.gen_predictionmaps(net, seqs, stride=stride, windowsize=window)
    cut = []
    for s in seqs:
        padded = "N" * (window - 1) + s + "N" * (window - 1)
        cut += [padded[i:i + window] for i in range(0, max(1, len(padded) - window + 1), stride)]
    Xr, Rr = data.pack_sequences(cut, m - 1, reverse_complement=rc)
    assert np.array_equal(seen[0][0], Xr) and np.array_equal(seen[0][1], Rr)


@pytest.mark.parametrize("pool,hidden,loss,rc,m,F,nm,lo,hi", [("max", 32, "nll", False, 24, 16, 1, 101, 101), ("all", 0, "mse", True, 32, 16, 3, 0, 40),
                                                              ("avg", 64, "mse", False, 1, 1, 5, 1, 9), ("all", 33, "nll", False, 11, 7, 2, 490, 1100),
                                                              ("max", 1, "mse", True, 64, 12, 1, 60, 70)])
def test_single_launch_scores(pool, hidden, loss, rc, m, F, nm, lo, hi):
    """The one-launch scoring kernel: regions below and above 64 rows on average and beyond one tile of 512, models whose filters and
    pooled features fill no group of 16, hidden units up to a wave; against the oracle's forward pass."""
    from deepbind_amd import _lib, data
    from deepbind_amd.model import SequenceNet
    rng = np.random.default_rng(m + F + nm)
    seqs = _seqs(rng, 9, lo, hi)
    net = SequenceNet(nm, F, m, pool=pool, hidden=hidden, loss=loss, dropout=0.25, reverse_complement=rc)
    params = {name: (rng.standard_normal(shape) * (0.3 if name == "Wc" else 0.2)).astype(np.float32) for name, shape, _ in net.layout}
    net.set_params(params)
    X, R = data.pack_sequences(seqs, m - 1, reverse_complement=rc)
    X[rng.random(len(X)) < 0.02] = 254
    assert _lib.dll().dbk_predict_small_takes(m, nm, F, X.size, len(R), _lib.str2pooltype[pool], hidden) == 1
    got = net.predict(torch.from_numpy(X).cuda(), torch.from_numpy(R).cuda()).cpu().numpy()
    st = orc.model_forward({k: v.astype(np.float64) for k, v in params.items()}, X, R, nm, pool, hidden, out="logistic" if loss == "nll" else "linear",
                           dropout=(np.full(nm, 0.25), None))
    want = st["Zout"]
    if rc:
        want = want.reshape(-1, 2, nm).max(axis=1)
    assert_close(got, want, ACT, "scores")


@pytest.mark.parametrize("pool,hidden,loss,rc,rate,m,F", [("max", 64, "nll", True, 0.5, 24, 16), ("all", 33, "mse", True, 0.0, 32, 16), ("avg", 0, "mse", False, 0.25, 9, 5),
                                                          ("all", 0, "nll", False, 0.0, 2, 1), ("max", 1, "mse", False, 0.0, 64, 13), ("avg", 8, "nll", True, 0.0, 13, 12)])
def test_gradient_map_kernel_edges(pool, hidden, loss, rc, rate, m, F):
    """Regions around 64 rows (a pass of the workgroup) and up to the kernel's 2048, one letter, none, all N (every row of a strand is as large), a
    palindrome (the pair ties); against the oracle and, longest region apart, the layers in place of the kernel: maps differ from
    those by round-off of sums of up to 2 m F terms."""
    from deepbind_amd import _lib, predict
    rng = np.random.default_rng(11 * m + F)
    p = _params(rng, m, F, pool, hidden)
    seqs = ["".join("ACGT"[v] for v in rng.integers(0, 4, n)) for n in (1, max(1, 65 - m), max(1, 66 - m), 130, 2049 - m)] + ["", "N" * 40, "ACGTUACGT"[:4] * 9]
    seqs[3] = "n" + seqs[3][1:].lower().replace("t", "u")
    out = "logistic" if loss == "nll" else "linear"
    net = _net(p, m, F, pool, hidden, loss, rc, rate)
    ptype = _lib.str2pooltype[pool]
    takes = _lib.dll().dbk_gradient_map_takes
    assert takes(m, F, 0, 2049 - m, ptype, hidden) == 1 and takes(m, F, 0, 2050 - m, ptype, hidden) == 0 and takes(1, F, 0, 9, ptype, hidden) == 0
    assert takes(m, 17, 0, 9, ptype, hidden) == 0 and takes(m, F, 0, 9, ptype, 65) == 0 and takes(65, F, 0, 9, ptype, hidden) == 0
    Z, maps = predict.gen_predictions(net, seqs, want_gmaps=True)
    Zr, mr = orc.gen_predictions({k: v.astype(np.float64) for k, v in p.items()}, seqs, pool, hidden, out, dropout_rate=[rate] if rate else None,
                                 reverse_complement=rc, want_gmaps=True)
    assert_close(Z, Zr, ACT, "Z")
    scale = max(np.abs(b).max() for _, b in mr if len(b))
    for (sa, a), (sb, b) in zip(maps, mr):
        assert sa == sb and a.shape == b.shape
        assert len(b) == 0 or np.abs(a - b).max() <= GRAD * scale, (len(sa), np.abs(a - b).max(), scale)
    fused = predict._gradient_maps
    predict._gradient_maps = lambda net, text: None
    try:
        Zl, ml = predict.gen_predictions(net, seqs, want_gmaps=True)
    finally:
        predict._gradient_maps = fused
    assert_close(Z, Zl, ACT, "Z, layer by layer")
    for (sa, a), (sb, b) in zip(maps, ml):
        assert sa == sb and (len(b) == 0 or np.abs(a - b).max() <= GRAD * scale)


@pytest.mark.parametrize("mode", [True, "finite_diff"])
@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("pool,m,F", [("max", 8, 4), ("all", 24, 17), ("avg", 2, 16)])
def test_batches_of_empty_sequences(pool, m, F, rc, mode):
    """No letter in a whole batch - alone, and as what a longer list ends in: scored, with empty maps; by the map kernels and by the layers
    (more than 16 filters have no gradient map kernel)."""
    from deepbind_amd import predict
    rng = np.random.default_rng(m + F)
    p = _params(rng, m, F, pool, 5)
    net = _net(p, m, F, pool, 5, "nll", rc, 0.0)
    p64 = {k: v.astype(np.float64) for k, v in p.items()}
    for seqs, batch in (([""], 2048), (["", ""], 2048), (["ACGT", "GATTACA", ""], 2)):
        Z, maps = predict.gen_predictions(net, seqs, want_gmaps=mode, batchsize=batch)
        Zr = np.vstack([orc.gen_predictions(p64, [s], pool, 5, "logistic", reverse_complement=rc, want_gmaps=False)[0] for s in seqs])
        assert_close(Z, Zr, ACT, "Z")
        assert [g.shape for _, g in maps] == [(len(s), 4) for s in seqs] and maps[-1][0] == ""


@pytest.mark.parametrize("which", ["b2", "W1"])
def test_pairs_whose_scores_do_not_compare(which, monkeypatch):
    """Scores that are not a number - of every strand, or only of strands on which one filter never fires - select neither row of a
    pair: such sequences have no entry among the predictions or the maps, by the one-workgroup kernel as by the layers."""
    from deepbind_amd import predict
    rng = np.random.default_rng(5)
    hidden = 8 if which == "b2" else 0                  # (a hidden unit's rectifier would take such a value for zero)
    p = _params(rng, 8, 4, "max", hidden)
    if which == "b2":
        p["b2"][:] = np.nan
    else:
        p["W1"][0, 0] = np.inf                          # 0 x inf where filter 0 stays at zero
        p["bc"][0, 0] = -2.0
    seqs = _seqs(rng, 40, 10, 14, 0.0)
    net = _net(p, 8, 4, "max", hidden, "nll", True, 0.0)
    Z, maps = predict.gen_predictions(net, seqs, want_gmaps=True)
    monkeypatch.setattr(predict, "_gradient_maps", lambda *a: None)
    Zr, ref = predict.gen_predictions(net, seqs, want_gmaps=True)
    monkeypatch.undo()
    assert len(maps) == len(Z) == len(Zr) == len(ref)
    assert (len(maps) == 0) if which == "b2" else (0 < len(maps) < len(seqs))
    assert [s for s, _ in maps] == [s for s, _ in ref] and np.allclose(Z, Zr, atol=1e-6, equal_nan=True)
    scale = max([np.abs(b[np.isfinite(b)]).max(initial=0.0) for _, b in ref], default=0.0)
    for (_, a), (_, b) in zip(maps, ref):
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[np.isinf(a)], b[np.isinf(b)])
        assert np.abs(a - b)[np.isfinite(a) & np.isfinite(b)].max(initial=0.0) <= GRAD * scale


def test_feature_columns_and_wide_targets():
    """Maps of nets with shared feature columns (absent: zeros) are those of the net without them; a group takes target
    matrices with further columns behind its models' and ones that are not contiguous, and refuses ones with fewer."""
    from deepbind_amd import predict
    from deepbind_amd._lib import DeepbindError
    from deepbind_amd.model import ModelGroup, SequenceNet
    rng = np.random.default_rng(6)
    p = _params(rng, 8, 4, "max", 8)
    seqs = _seqs(rng, 5, 10, 14)
    plain = _net(p, 8, 4, "max", 8, "nll", False, 0.0)
    net = SequenceNet(1, 4, 8, pool="max", hidden=8, loss="nll", feature_columns=2)
    net.set_params(dict(p, W1=np.concatenate([p["W1"], rng.standard_normal((2, 8)).astype(np.float32)])))
    for mode in (True, "finite_diff"):
        (Z, maps), (Zr, ref) = [predict.gen_predictions(n, seqs, want_gmaps=mode) for n in (net, plain)]
        assert_close(Z, Zr, ACT, "predictions")
        assert_close(np.concatenate([g for _, g in maps]), np.concatenate([g for _, g in ref]), GRAD, "maps")
    X, R = [torch.from_numpy(v).cuda() for v in __import__("deepbind_amd.data", fromlist=["data"]).pack_sequences(seqs, 7)]
    Y = rng.random((5, 3)).astype(np.float32)
    wide = torch.from_numpy(np.concatenate([Y, Y + 1], axis=1)).cuda()
    for pools in (["max", "all", "max"], ["max"] * 3):
        out = []
        for t in (wide[:, :3].contiguous(), wide, wide.t().contiguous().t(), wide[:, :3]):
            grp = ModelGroup(pools, [0] * 3, 4, 8, loss="mse", rate=0.05, momentum=0.9)
            for _, n in grp.groups:
                n.init_params(init_conv=0.1, init_full=0.1, seed=3)
            grp.train_step(X, R, t)
            out.append([n.P.cpu().numpy() for _, n in grp.groups])
        for o in out[1:]:
            assert all(np.array_equal(a, b) for a, b in zip(out[0], o))
        with pytest.raises(DeepbindError):
            grp.train_step(X, R, wide[:, :2].contiguous())


@pytest.mark.parametrize("rc", [False, True])
@pytest.mark.parametrize("mode", [False, True, "finite_diff"])
def test_predictions_under_a_default_device(mode, rc):
    """Scores and maps come to the host whatever device a program's new tensors go to by default; the same bits."""
    from deepbind_amd import predict
    rng = np.random.default_rng(12)
    net = _net(_params(rng, 8, 4, "max", 5), 8, 4, "max", 5, "nll", rc, 0.0)
    seqs = _seqs(rng, 6, 10, 20)
    want = predict.gen_predictions(net, seqs, want_gmaps=mode)
    windows = predict.gen_predictionmaps(net, seqs, windowsize=12)[0]
    torch.set_default_device("cuda")
    try:
        got = predict.gen_predictions(net, seqs, want_gmaps=mode)
        again = predict.gen_predictionmaps(net, seqs, windowsize=12)[0]
    finally:
        torch.set_default_device(None)
    assert np.array_equal(got[0], want[0]) and all(np.array_equal(a, b) for a, b in zip(again, windows))
    for (sa, a), (sb, b) in zip(got[1] or [], want[1] or []):
        assert sa == sb and np.array_equal(a, b)
