"""Prediction-time callers of the motif-scan path: scores, gradient maps, finite-difference
mutation maps and sliding-window scans for one trained model.

Mirrors the reference's prediction module (code/libs/kangaroo/kangaroo/predict.py:145-345):
`maskout_revcomp`, `gen_convnet_predictions` and `gen_convnet_predictionmaps`, with the model
evaluation replaced by `SequenceNet` calls. Strings go to the device as they are: packing them, cutting
windows out of them and picking a map's rows are kernels. A mutation map is one launch that re-scans only the
rows a changed letter moves (nets whose shape that kernel does not take re-score the batch once per (position,
base), as the reference does, the stream mutated and the differences collected on the device).
"""
import itertools

import numpy as np
import torch

from . import _lib
from . import data as _data

_RCINDEX = (3, 2, 1, 0)
_STREAM_MAX = 2 ** 32 - 1        # bytes of a packed stream, and letters of a batch: region bounds and text offsets are 32-bit


def maskout_revcomp(Z, reverse_complement):
    """Host version of the pair selection (predict.py:145-164): Z holds fwd,rev,fwd,rev rows; keeps
    the larger of each pair (ties keep fwd). Returns (selected rows, Zmask | None)."""
    if not reverse_complement:
        return Z, None
    Zc = Z.reshape((-1, 2))
    Zmask = np.zeros_like(Zc, dtype=bool)
    Zmask[:, 0] = Zc[:, 0] >= Zc[:, 1]
    Zmask[:, 1] = Zc[:, 0] < Zc[:, 1]
    Zmask = Zmask.reshape((-1, 1))
    return Z[Zmask.ravel()], Zmask


def _finite_diff(net, Xd, Rd, R, Z, dX):
    """Overwrites dX (N, 4, device) with mtZ - Z for every single-base change, the reference's way
    (predict.py:201-240): pass (i, j) sets letter i of EVERY region to base j (reverse rows: the
    mirrored letter to the complement), regions being leading pad + sequence, so passes with i past
    the end of a short sequence write into the pad that follows it exactly as the reference does."""
    rc = net.reverse_complement
    pad = net.m - 1
    a = torch.as_tensor(R[:, 0].astype(np.int64), device=Xd.device)
    b = torch.as_tensor(R[:, 1].astype(np.int64), device=Xd.device)
    length = b - a
    k = torch.arange(len(R), device=Xd.device)
    fwd = (k % 2 == 0) if rc else torch.ones_like(k, dtype=torch.bool)
    # only passes that can reach a reported row matter: i below the longest sequence
    longest = int((R[:, 1].astype(np.int64) - R[:, 0].astype(np.int64)).max()) - pad
    Xflat = Xd.view(-1)
    for i in range(max(longest, 0)):
        live = length > i
        at_f = (pad + a + i)[live & fwd]
        at_r = (b - i - 1)[live & ~fwd]
        for j in range(4):
            mt = Xflat.clone()
            mt[at_f] = j
            if rc:
                mt[at_r] = _RCINDEX[j]
            mtZ = net.predict(mt.view(-1, 1), Rd)       # pair maximum included
            dZ = (mtZ - Z) * torch.clamp(torch.sign(torch.maximum(Z, mtZ)), min=0)
            rows = (live & fwd).nonzero().ravel()
            dX[(pad + a + i)[rows], j] = dZ[(rows // 2) if rc else rows, 0]


class _Text(object):
    """Sequences as the device takes them: their letters end to end, and where each begins. Strings, or anything whose
    buffer holds letters unless `strings` says that only strings will do (reverse complements and windows of a sequence)."""

    def __init__(self, seqs, strings=False):
        try:
            joined = "".join(seqs)           # (also the check that all are strings: a thousand sequences one by one took 75 us)
        except TypeError:
            if strings:
                raise TypeError("sequences must be strings")
            seqs = [s if isinstance(s, str) else np.frombuffer(s, dtype=np.uint8).tobytes().decode("latin-1") for s in seqs]
            joined = "".join(seqs)
        self.bytes = np.frombuffer(joined.encode("latin-1"), dtype=np.uint8)
        self.lens = np.fromiter(map(len, seqs), dtype=np.int64, count=len(seqs))
        self.offsets = np.zeros(len(seqs) + 1, dtype=np.int64)
        np.cumsum(self.lens, out=self.offsets[1:])

    def upload(self, device, *tables):
        """One copy to the device: (offsets, the further uint32 tables, letters)."""
        _lib.require(len(self.bytes) <= _STREAM_MAX, "ValueError: more than 2^32 - 1 letters in one batch")
        words = [np.asarray(t, dtype=np.uint32) for t in (self.offsets,) + tables]
        buf = torch.from_numpy(np.concatenate([w.view(np.uint8) for w in words] + [self.bytes])).to(device)
        out, at = [], 0
        for w in words:
            out.append(buf[at:at + w.nbytes])
            at += w.nbytes
        return out + [buf[at:]]

    def strings(self, reverse=None):
        """The sequences in the packed stream's letters (ACGT, else N); those marked in `reverse` as their reverse complement."""
        fwd = _data.normalize(self.bytes.tobytes())
        n, o = len(fwd), self.offsets.tolist()
        if reverse is None or not reverse.any():
            return [fwd[a:b] for a, b in zip(o[:-1], o[1:])]
        rev = _data.revcomp(fwd)
        return [rev[n - b:n - a] if r else fwd[a:b] for a, b, r in zip(o[:-1], o[1:], reverse.tolist())]


def _pack(net, text):
    """(X, R) of the batch on the device, as data.pack_sequences lays them out."""
    strands, pad, n = (2 if net.reverse_complement else 1), net.m - 1, len(text.lens)
    N = strands * (n * pad + len(text.bytes)) + pad
    _lib.require(N <= _STREAM_MAX, "ValueError: a batch of %d letters packs to more than 2^32 - 1 bytes; score in smaller batches" % len(text.bytes))
    offsets, letters = text.upload(net.device)
    X = torch.empty((N, 1), dtype=torch.uint8, device=net.device)
    R = torch.empty((n * strands, 2), dtype=torch.uint32, device=net.device)
    _lib.call("dbk_pack_text", _lib.stream(), _lib.ptr(letters), _lib.ptr(offsets), n, pad, strands, _lib.ptr(X), _lib.ptr(R))
    return X, R


def _split(maps, text):
    """The sequences' parts of an array, or a string. (Of equal lengths an array's come at once, in half the time.)"""
    if isinstance(maps, np.ndarray) and (text.lens == text.lens[0]).all():
        return list(maps.reshape((len(text.lens), int(text.lens[0])) + maps.shape[1:]))
    o = text.offsets.tolist()
    return [maps[a:b] for a, b in zip(o[:-1], o[1:])]


def _mutation_maps(net, X, R, text):
    """(Z (nseq, 1), [(letters, map (length, 4))]) of the batch, or None when the kernel does not take the net's shape."""
    ptype = _lib.str2pooltype[net.pool]
    if net.dtype != torch.float32 or int(text.lens.max()) > 4 * 65535 or not _lib.dll().dbk_mutation_map_takes(net.m, net.nfilter, ptype, net.hidden):
        return None
    p = net.p
    Wc = p["Wc"] if net.input_dropout <= 0 else p["Wc"] * (1.0 - net.input_dropout)
    scale = (1.0 - net.dropout) if net.use_dropout else None
    n = len(text.lens)
    out = torch.empty(n + 4 * len(text.bytes), dtype=torch.float32, device=net.device)       # (one copy back to the host)
    Z, maps = out[:n], out[n:]
    _lib.call("dbk_mutation_map", _lib.stream(), _lib.ptr(Wc), _lib.ptr(p["bc"]), net.m, net.nfilter, _lib.ptr(X), X.numel(), _lib.ptr(R),
              R.shape[0], int(text.lens.max()), ptype, net.hidden, _lib.ptr(p["W1"]), _lib.ptr(p["b1"]), _lib.ptr(p.get("W2")),
              _lib.ptr(p.get("b2")), _lib.ptr(scale), int(net.loss == "nll"), 2 if net.reverse_complement else 1, _lib.ptr(Z), _lib.ptr(maps))
    host = torch.empty(out.shape, dtype=out.dtype, device="cpu")
    result = host.numpy()
    gmaps = list(zip(text.strings(), _split(result[n:].reshape(-1, 4), text)))               # (cut while the kernel runs, filled by the copy)
    host.copy_(out)
    return result[:n].reshape(-1, 1), gmaps


def _gradient_maps(net, text):
    """(Z (rows, 1), [(letters, map (length, 4)) of the strand mapped]) of the batch, or None when the kernel does not take it."""
    ptype, shortest, longest = _lib.str2pooltype[net.pool], int(text.lens.min()), int(text.lens.max())
    if net.dtype != torch.float32 or net.input_dropout > 0 or not _lib.dll().dbk_gradient_map_takes(net.m, net.nfilter, shortest, longest, ptype, net.hidden):
        return None
    p, n, L = net.p, len(text.lens), len(text.bytes)
    scale = (1.0 - net.dropout) if net.use_dropout else None
    offsets, letters = text.upload(net.device)
    out = torch.empty(4 * n + 17 * L, dtype=torch.uint8, device=net.device)                  # (one copy back to the host)
    Z, maps, strand = out[:4 * n], out[4 * n:4 * n + 16 * L], out[4 * n + 16 * L:]
    _lib.call("dbk_gradient_map", _lib.stream(), _lib.ptr(p["Wc"]), _lib.ptr(p["bc"]), net.m, net.nfilter, _lib.ptr(letters), _lib.ptr(offsets), n,
              shortest, longest, ptype, net.hidden, _lib.ptr(p["W1"]), _lib.ptr(p["b1"]), _lib.ptr(p.get("W2")), _lib.ptr(p.get("b2")),
              _lib.ptr(scale), int(net.loss == "nll"), 2 if net.reverse_complement else 1,
              _lib.ptr(Z), _lib.ptr(maps), _lib.ptr(strand))
    host = torch.empty(out.shape, dtype=out.dtype, device="cpu")
    result = host.numpy()
    cut = _split(result[4 * n:4 * n + 16 * L].view(np.float32).reshape(-1, 4), text)         # (while the kernel runs; filled by the copy)
    host.copy_(out)
    Z = result[:4 * n].view(np.float32).reshape(-1, 1)
    gmaps = list(zip(_split(result[4 * n + 16 * L:].tobytes().decode("ascii"), text), cut))
    keep = Z[:, 0] == Z[:, 0]
    if net.reverse_complement and not keep.all():    # (scores that do not compare select neither row of their pair)
        return Z[keep], [gmap for gmap, k in zip(gmaps, keep) if k]
    return Z, gmaps


def gen_predictions(net, seqs, want_gmaps=False, batchsize=2048):
    """Scores a list of sequence strings with a single-model SequenceNet.

    Returns (predictions (nseq, 1) float32, gmaps). gmaps is None, or a list of
    (sequence string, (len, 4) float32 map): with want_gmaps=True the back-propagated input
    gradient (with reverse complements only the winning strand's entry, whose string is that
    strand's), with want_gmaps="finite_diff" the mutation map of the forward strand. The maps of one
    batch are disjoint parts of one array, written to by nobody else: a program that keeps a few maps of
    many for long copies those, or it keeps their whole batch (up to `batchsize` sequences).
    (reference: predict.py:168-260)"""
    assert net.ninst == 1, "prediction maps are defined for one model at a time"
    rc, pad = net.reverse_complement, net.m - 1
    preds, gmaps = [], ([] if want_gmaps else None)
    for s0 in range(0, len(seqs), batchsize):
        text = _Text(seqs[s0:s0 + batchsize], strings=rc)
        fused = _gradient_maps(net, text) if want_gmaps and want_gmaps != "finite_diff" else None
        if fused is not None:
            preds.append(fused[0])
            gmaps += fused[1]
            continue
        X, R = _pack(net, text)
        if not want_gmaps:
            preds.append(net.predict(X, R).cpu().numpy())
            continue
        fused = _mutation_maps(net, X, R, text) if want_gmaps == "finite_diff" else None
        if fused is not None:
            preds.append(fused[0])
            gmaps += fused[1]
            continue
        Zall, dX = net.input_gradients(X, R)
        Zh, Zmask = maskout_revcomp(Zall.cpu().numpy(), rc)
        preds.append(Zh)
        if want_gmaps == "finite_diff":
            Rh = R.cpu().numpy().astype(np.int64)
            _finite_diff(net, X, R, Rh, torch.from_numpy(Zh).to(net.device), dX)
            dXh = dX.cpu().numpy()
            gmaps += [(s, dXh[a + pad:b].copy()) for s, (a, b) in zip(text.strings(), Rh[::2] if rc else Rh)]
            continue
        maps = torch.empty((len(text.bytes), 4), dtype=dX.dtype, device=dX.device)
        if len(text.bytes):                  # (a batch of empty sequences has no letter to gather for, and no memory for them)
            _lib.call("dbk_gather_maps", _lib.stream(), _lib.dtype_code(dX), _lib.ptr(R), R.shape[0], pad, 2 if rc else 1, _lib.ptr(Zall),
                      _lib.ptr(dX), _lib.ptr(maps))
        pairs = Zmask.reshape(-1, 2) if Zmask is not None else None
        new = zip(text.strings(None if pairs is None else pairs[:, 1]), _split(maps.cpu().numpy(), text))
        gmaps += new if pairs is None else [gmap for gmap, keep in zip(new, pairs.any(axis=1)) if keep]
    return np.vstack(preds), gmaps


def _cut(raws, nwin, windowsize, stride):
    """The windows of the sequences, one after another, as strings."""
    for raw, n in zip(raws, nwin):
        padseq = "N" * (windowsize - 1) + raw + "N" * (windowsize - 1)
        for i in range(n):
            yield padseq[i * stride:i * stride + windowsize]


def _score_windows(net, raws, nwin, windowsize, stride):
    """Predictions of all windows of a few sequences: the windows are cut on the device. (Sequences whose windows pack to
    more than region bounds can say are cut on the host, a batch at a time.)"""
    strands, pad, total = (2 if net.reverse_complement else 1), net.m - 1, int(sum(nwin))
    span = strands * (pad + windowsize)
    if total * span + pad > _STREAM_MAX:
        windows, Z = _cut(raws, nwin, windowsize, stride), []
        most = max(1, min(2 ** 20, (_STREAM_MAX - pad) // span))
        for batch in iter(lambda: list(itertools.islice(windows, most)), []):
            Z.append(gen_predictions(net, batch, batchsize=len(batch))[0])
        return np.vstack(Z)
    text = _Text(raws, strings=True)
    offsets, first, letters = text.upload(net.device, np.concatenate([[0], np.cumsum(nwin)]))
    X = torch.empty((total * strands * (pad + windowsize) + pad, 1), dtype=torch.uint8, device=net.device)
    R = torch.empty((total * strands, 2), dtype=torch.uint32, device=net.device)
    _lib.call("dbk_pack_windows", _lib.stream(), _lib.ptr(letters), _lib.ptr(offsets), _lib.ptr(first), len(raws), total, int(windowsize), int(stride),
              pad, strands, _lib.ptr(X), _lib.ptr(R))
    return net.predict(X, R).cpu().numpy()


def gen_predictionmaps(net, seqs, stride=1, windowsize=20, want_gmaps=False):
    """Sliding-window scan (reference: predict.py:263-345): every sequence is padded with
    windowsize-1 N on both sides and cut into windows of `windowsize` letters every `stride`;
    all windows of up to 32 sequences are scored in one batch. Returns (list of per-sequence
    prediction maps, list of (len+windowsize-1, 4) window-averaged gradient maps | None)."""
    if want_gmaps and stride != 1:
        # the reference's aggregation (predict.py:330-340) slices rows that only line up for stride 1
        raise ValueError("window-averaged gradient maps need stride 1 (got %d)" % stride)
    pmaps, gmaps = [], ([] if want_gmaps else None)
    chunk = 32
    for c0 in range(0, len(seqs), chunk):
        raws = list(seqs[c0:c0 + chunk])
        if want_gmaps or windowsize < 2:         # (one-letter windows have no N around them: an empty sequence's window is empty)
            windows, nwin = [], []
            for raw in raws:
                padseq = "N" * (windowsize - 1) + raw + "N" * (windowsize - 1)
                cut = [padseq[i:i + windowsize] for i in range(0, max(1, len(padseq) - windowsize + 1), stride)]
                windows += cut
                nwin.append(len(cut))
            Z, wmaps = gen_predictions(net, windows, want_gmaps=want_gmaps, batchsize=len(windows))
        else:
            assert net.ninst == 1, "prediction maps are defined for one model at a time"
            if stride < 1:
                raise ValueError("windows are cut every stride letters, at least 1 (got %d)" % stride)
            nwin = [len(range(0, max(1, len(raw) + windowsize - 1), stride)) for raw in raws]
            Z = _score_windows(net, raws, nwin, windowsize, stride)
        edges = np.cumsum([0] + nwin)
        for i, raw in enumerate(raws):
            pmaps.append(Z[edges[i]:edges[i + 1]].ravel().copy())
            if want_gmaps:
                gmap = np.zeros((len(raw) + windowsize - 1, 4), Z.dtype)
                denom = np.zeros_like(gmap)
                for j in range(nwin[i]):
                    dXj = wmaps[edges[i] + j][1][:min(windowsize, (nwin[i] - j) * stride)]
                    gmap[j * stride:j * stride + windowsize] += dXj
                    denom[j * stride:j * stride + windowsize] += 1
                with np.errstate(invalid="ignore", divide="ignore"):
                    gmap /= denom
                gmaps.append(np.nan_to_num(gmap))
    return pmaps, gmaps
