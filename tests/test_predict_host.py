"""Host side of the prediction-time callers, without a GPU: what is refused, and what is alive when the library is called."""
import types
import weakref

import numpy as np
import pytest
import torch

from deepbind_amd import _lib, predict


def _net(**kw):
    net = dict(ninst=1, m=4, nfilter=2, pool="max", hidden=0, loss="nll", dtype=torch.float32, input_dropout=0.0, use_dropout=True,
               dropout=torch.full((1,), 0.25), reverse_complement=False, device="cpu", mode="fused", nfeat=0,
               p=dict(Wc=torch.zeros(16, 2), bc=torch.zeros(1, 2), W1=torch.zeros(2, 1), b1=torch.zeros(1, 1)))
    net.update(kw)
    return types.SimpleNamespace(**net)


@pytest.fixture
def calls(monkeypatch):
    """The library's calls, recorded in place of being made; every tensor whose address a call takes must be alive when it is made
    (freed before, its memory is another thread's to take while the launch that reads it is not yet on the stream)."""
    taken, made = [], []

    def ptr(t):
        if t is not None:
            taken.append(weakref.ref(t))

    def call(name, *args):
        made.append(name)
        assert all(ref() is not None for ref in taken), "%s was given the address of a tensor that is gone" % name
        taken.clear()

    monkeypatch.setattr(_lib, "ptr", ptr)
    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(_lib, "stream", lambda: None)
    monkeypatch.setattr(torch, "empty", torch.zeros)               # (outputs that no kernel fills: letters that decode)
    return made


@pytest.mark.parametrize("rc", [False, True])
def test_tensors_live_until_the_call_that_reads_them(calls, rc):
    net = _net(reverse_complement=rc, hidden=3)
    net.p.update(W1=torch.zeros(2, 3), b1=torch.zeros(1, 3), W2=torch.zeros(3, 1), b2=torch.zeros(1, 1))
    text = predict._Text(["ACGT", "GGN"])
    assert predict._gradient_maps(net, text) is not None
    X, R = predict._pack(net, text)
    assert predict._mutation_maps(net, X, R, text) is not None
    net.predict = lambda X, R: torch.zeros(R.shape[0], 1)
    predict._score_windows(net, ["ACGT"], [9], 6, 1)
    assert calls == ["dbk_gradient_map", "dbk_pack_text", "dbk_mutation_map", "dbk_pack_windows"]


def test_batches_of_empty_sequences_gather_nothing(calls):
    """A tensor of no elements has no address: what is asked of the library for a batch without a letter names none of them, or takes null."""
    net = _net(nfilter=17, reverse_complement=True)
    net.input_gradients = lambda X, R: (torch.ones(R.shape[0], 1), torch.zeros(X.numel(), 4))
    Z, maps = predict.gen_predictions(net, ["", ""], want_gmaps=True)
    assert calls == ["dbk_pack_text"] and [(s, g.shape) for s, g in maps] == [("", (0, 4))] * 2
    lib, one = _lib.dll(), 1                                       # (a null map is refused where there are letters for it)
    assert lib.dbk_mutation_map(None, one, one, 4, 2, one, 10, one, 1, 4, 0, 0, one, one, None, None, None, 0, 1, one, None) != 0
    assert b"null pointer" in lib.dbk_last_error()


@pytest.mark.parametrize("mode", [False, True, "finite_diff"])
def test_what_is_no_sequence_is_refused(calls, mode):
    """A number is no sequence (bytes(5) would make five letters of it), nor a list of numbers; bytes are one where no reverse complement
    is taken and no window cut."""
    for seqs in ([5], [[65, 67]], [None], ["ACGT", 7]):
        with pytest.raises(TypeError):
            predict.gen_predictions(_net(), seqs, want_gmaps=mode)
    with pytest.raises(TypeError):
        predict.gen_predictions(_net(reverse_complement=True), [b"ACGT"], want_gmaps=mode)
    with pytest.raises(TypeError):
        predict.gen_predictionmaps(_net(), [b"ACGT"], want_gmaps=mode is True)
    assert not calls
    assert predict._Text([b"AC", bytearray(b"g"), np.frombuffer(b"TN", np.uint8), b""]).strings() == ["AC", "G", "TN", ""]


def test_strides_and_windows_below_one(monkeypatch):
    """A stride below one is refused; windows of no letter are scored as they are cut, as many of them as there are."""
    for stride in (0, -1, -7):
        with pytest.raises(ValueError):
            predict.gen_predictionmaps(_net(predict=lambda X, R: torch.zeros(R.shape[0], 1)), ["ACGTACGT"], stride=stride, windowsize=4)
    seen = []
    monkeypatch.setattr(predict, "gen_predictions", lambda net, seqs, **kw: seen.extend(seqs) or (np.arange(len(seqs)).reshape(-1, 1), None))
    pmaps, _ = predict.gen_predictionmaps(_net(), ["ACG", "", "TT"], windowsize=0)
    assert seen == [""] * 8 and [p.tolist() for p in pmaps] == [[0, 1, 2, 3], [4], [5, 6, 7]]
    assert predict.gen_predictionmaps(_net(ninst=2), [])[0] == []


class _Letters(object):
    """So many letters, none of them in memory."""

    def __init__(self, n):
        self.n = n

    def __len__(self):
        return self.n


def test_streams_that_region_bounds_cannot_address_are_refused(calls):
    text = predict._Text(["A"])
    for letters, n, rc in ((2 ** 32, 1, False), (2 ** 32 - 4, 1, False), (2 ** 31 - 5, 2, True)):
        text.bytes, text.lens = _Letters(letters), np.zeros(n, np.int64)
        with pytest.raises(_lib.DeepbindError, match="2\\^32"):
            predict._pack(_net(reverse_complement=rc), text)
    text.bytes = _Letters(2 ** 32)
    with pytest.raises(_lib.DeepbindError, match="2\\^32"):
        text.upload("cpu")
    lib, one = _lib.dll(), 1                                       # (refused for their sizes, before anything is read or launched)
    for strands, nwindow in ((1, 2 ** 32 // 83 + 1), (2, 2 ** 31 // 83 + 1)):
        assert lib.dbk_pack_windows(None, one, one, one, 1, nwindow, 60, 1, 23, strands, one, one) != 0
        assert b"2^32" in lib.dbk_last_error()
    assert lib.dbk_pack_text(None, one, one, 2 ** 27, 32, 1, one, one) != 0 and b"2^32" in lib.dbk_last_error()
    assert lib.dbk_pack_text(None, None, None, 0, 32, 1, None, None) == 0 and lib.dbk_last_error() == b""


@pytest.mark.parametrize("rc", [False, True])
def test_windows_beyond_one_stream_are_cut_on_the_host(rc, monkeypatch):
    """Every batch packs to no more bytes than a stream may have, and together they are the windows the device would cut."""
    net, raws, w, stride = _net(reverse_complement=rc), ["ACGTACGTAA", "", "TTG"], 5, 2
    span = (2 if rc else 1) * (net.m - 1 + w)
    nwin = [len(range(0, max(1, len(s) + w - 1), stride)) for s in raws]
    for most in (1, 3, 6):
        monkeypatch.setattr(predict, "_STREAM_MAX", most * span + net.m - 1)
        seen = []
        monkeypatch.setattr(predict, "gen_predictions", lambda net, seqs, **kw: seen.append(list(seqs)) or (np.array([[hash(s) % 1000] for s in seqs]), None))
        Z = predict._score_windows(net, raws, nwin, w, stride)
        cut = [("N" * (w - 1) + s + "N" * (w - 1))[i:i + w] for s in raws for i in range(0, max(1, len(s) + w - 1), stride)]
        assert sum(seen, []) == cut and all(len(b) <= most for b in seen) and Z.ravel().tolist() == [hash(s) % 1000 for s in cut]


def test_calls_that_fill_the_gpu_are_not_scored_in_one_launch():
    """A workgroup per region and model: one model, or few enough of both; the scan kernel and the head take the rest."""
    takes = _lib.dll().dbk_predict_small_takes
    assert takes(24, 1, 16, 64 * 124 + 23, 64, 0, 32) == 1 and takes(8, 1, 16, 700000, 7000, 0, 0) == 1
    assert takes(8, 16, 8, 128 * 67 + 7, 128, 0, 32) == 1 and takes(8, 16, 8, 129 * 67 + 7, 129, 0, 32) == 0
    assert takes(4, 64, 16, 23020, 1019, 3, 32) == 0 and takes(24, 1, 16, 250001, 2000, 0, 32) == 0
