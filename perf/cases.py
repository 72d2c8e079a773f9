"""The work that users of this package have it do, as measurable cases.

Six kinds of call, each through an entry point that a program uses:

* ``fit``        WarpGBM.fit on host arrays, then predictions of held-out rows
                 (the estimator from numpy to numpy; small and mid-sized data);
* ``round``      boosting rounds of the level-wise engine on resident codes
                 (what a fit spends its device time on; regression, eras,
                 softmax classes, feature subsets, any bin count);
* ``histogram``  the histogram operator: ``calls``, one compute_histogram3 for
                 the root and one per node on raw codes, or ``level``, the root
                 and all nodes batched on native codes;
* ``split``      compute_split on per-era histograms;
* ``ingest``     quantile edges and binning of a resident float matrix;
* ``predict``    ensemble inference: ``table``, the flattened-tree operator on
                 raw codes, or ``heap``, the heap predictor on native codes
                 (with the row softmax for class scores).

``listed`` gives the fixed cases, ``draw`` more of the same ranges,
``prepare`` the inputs and handles, ``run`` one pass, ``exact`` the same
outputs in 64 bits by plain torch.  Every operator of the package promises
results that do not depend on launch shape or execution order, so outputs are
compared bit for bit (``tolerance``).
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from warpgbm_amd import WarpGBM, _lib, node_kernel
from warpgbm_amd import device as D

DEV = "cuda:0"
F64 = torch.float64


# --------------------------------------------------------------------------- the cases
def listed():
    return [
        # a small table end to end: launches and host work count, not bytes
        dict(name="fit small", kind="fit", rows=10_000, feats=50, bins=32, depth=5, rounds=20,
             classes=0, eras=1),
        # multiclass training at a mid size: ten trees a round, deep levels of
        # small nodes
        dict(name="fit classes", kind="fit", rows=200_000, feats=100, bins=32, depth=6, rounds=20,
             classes=10, eras=1),
        # the headline table: a million rows by a thousand features, depth 5
        dict(name="round wide", kind="round", rows=1_000_000, feats=1000, bins=32, depth=5,
             rounds=2, classes=0, eras=1, colsample=1.0),
        # era-aware splits on pre-binned features: 500 eras, five bins, depth 8
        dict(name="round eras", kind="round", rows=500_000, feats=2000, bins=5, depth=8, rounds=1,
             classes=0, eras=500, colsample=1.0),
        # ragged sizes, few long eras, many bins, half of the columns per tree
        dict(name="round ragged eras", kind="round", rows=123_457, feats=307, bins=63, depth=6,
             rounds=2, classes=0, eras=7, colsample=0.5),
        # the estimator's default tree shape (10 bins, depth 3) on an ordinary table
        dict(name="round default", kind="round", rows=100_003, feats=200, bins=10, depth=3,
             rounds=8, classes=0, eras=1, colsample=1.0),
        # the reference's growth pattern: a histogram call per node
        dict(name="histogram calls", kind="histogram", how="calls", rows=1_000_000, feats=1000,
             bins=32, nodes=16),
        # the same histograms, batched, on codes in the native layout
        dict(name="histogram level", kind="histogram", how="level", rows=1_000_000, feats=1000,
             bins=32, nodes=16),
        # gains and directions of one node of the 500-era table
        dict(name="split eras", kind="split", eras=500, feats=2000, bins=5),
        # ingestion of the headline table once it is on the device
        dict(name="ingest wide", kind="ingest", rows=1_000_000, feats=1000, bins=32),
        # inference of a regression forest given as flattened trees
        dict(name="predict table", kind="predict", how="table", rows=1_000_000, feats=1000,
             bins=32, depth=5, rounds=100, classes=1),
        # inference of a large multiclass ensemble: 2000 trees of depth 6
        dict(name="predict classes", kind="predict", how="heap", rows=1_000_000, feats=100,
             bins=32, depth=6, rounds=200, classes=10),
    ]


def _log(rng, lo, hi):
    """A whole number whose logarithm is uniform between those of lo and hi."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fit", "round", "round", "histogram", "histogram", "split", "ingest",
                       "predict", "predict"])
    if kind == "fit":
        classes = rng.choice([0, 0, 2, 3, 7])
        return dict(kind="fit", rows=_log(rng, 2_000, 200_000), feats=_log(rng, 8, 100),
                    bins=rng.choice([5, 10, 16, 32, 63]), depth=rng.randint(2, 6),
                    rounds=rng.randint(5, 20), classes=classes,
                    eras=rng.choice([1, 1, 5]) if not classes else 1)
    if kind == "round":
        classes = rng.choice([0, 0, 0, 3, 10])
        eras = 1 if classes else rng.choice([1, 1, 3, 20, 101, 500])
        feats = _log(rng, 10, 2000)
        top = 100_000_000 if classes else 500_000_000
        rows = _log(rng, 5_000 if eras < 100 else 50_000, min(500_000, max(60_000, top // feats)))
        # the widest staging is that of the listed era case: eras * feats * bins
        bins = rng.choice([b for b in (5, 10, 16, 32, 63, 127)
                           if eras == 1 or eras * feats * b <= 5_000_000 or b == 5])
        return dict(kind="round", rows=rows, feats=feats, bins=bins, depth=rng.randint(3, 7),
                    rounds=rng.randint(1, 2), classes=classes, eras=eras,
                    colsample=rng.choice([1.0, 1.0, 0.5]))
    if kind == "histogram":
        rows = _log(rng, 2_000, 1_000_000)
        return dict(kind="histogram", how=rng.choice(["calls", "level"]), rows=rows,
                    feats=_log(rng, 10, 1000), bins=rng.choice([5, 10, 32, 63, 127]),
                    nodes=rng.choice([1, 2, 4, 8, 16]))
    if kind == "split":
        return dict(kind="split", eras=_log(rng, 1, 500), feats=_log(rng, 20, 2000),
                    bins=rng.choice([2, 5, 5, 10]))
    if kind == "ingest":
        feats = _log(rng, 10, 1000)
        return dict(kind="ingest", rows=_log(rng, 2_000, 1_000_000), feats=feats,
                    bins=rng.choice([5, 10, 32, 63, 127]))
    how = rng.choice(["table", "heap"])
    classes = 1 if how == "table" else rng.choice([1, 3, 10])
    depth = rng.randint(3, 6 if how == "table" else 8)
    feats = _log(rng, 20, 1000 if classes == 1 else 300)
    rounds = _log(rng, 10, 100)
    rows = _log(rng, 1_000, 1_000_000 if feats < 500 else 300_000)
    return dict(kind="predict", how=how, rows=rows, feats=feats, bins=rng.choice([5, 10, 32, 127]),
                depth=depth, rounds=rounds, classes=classes)


# --------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * int(seed) + 17)
    return g


def _signal(X, g):
    """A target's signal from up to 20 of the columns of X (float32, roughly
    unit columns): linear terms and one product."""
    k = min(20, X.shape[1])
    w = torch.randn(k, generator=g, device=DEV)
    s = X[:, :k] @ w
    if k > 1:
        s = s + 0.5 * torch.sin(X[:, 0] * X[:, 1])
    return s


def _labels(s, K, g):
    """K classes from a score: noisy quantile buckets of it."""
    s = s + 0.3 * s.std() * torch.randn(s.shape, generator=g, device=DEV)
    cuts = torch.quantile(s[: 1 << 20], torch.linspace(0, 1, K + 1, device=DEV)[1:-1])
    return torch.bucketize(s, cuts)


def _era_ids(case, g):
    """Contiguous eras of uneven length (every row's era, ascending)."""
    n, E = case["rows"], case["eras"]
    era = torch.randint(0, E, (n,), generator=g, device=DEV, dtype=torch.int32)
    return torch.sort(era).values.cpu().numpy()


def _codes8(case, g):
    """Uniform int8 codes [rows, feats], as quantile binning gives."""
    return torch.randint(0, case["bins"], (case["rows"], case["feats"]), generator=g, device=DEV,
                         dtype=torch.int8)


def _fit_inputs(case, seed):
    g = _gen(seed)
    n, hold = case["rows"], max(500, case["rows"] // 10)
    X = torch.randn((n + hold, case["feats"]), generator=g, device=DEV)
    s = _signal(X, g)
    if case["classes"]:
        y = _labels(s, case["classes"], g).cpu().numpy()
    else:
        y = (s + 0.5 * torch.randn(s.shape, generator=g, device=DEV)).cpu().numpy()
    era = _era_ids(case, g) if case["eras"] > 1 else None
    X = X.cpu().numpy()
    return dict(X=X[:n], y=y[:n], era=era, X_new=X[n:])


def _round_inputs(case, seed):
    g = _gen(seed)
    x8 = _codes8(case, g)
    unit = (x8[:, :20].float() - (case["bins"] - 1) / 2) / max(1.0, case["bins"] / 3.5)
    s = _signal(unit, g)
    if case["classes"]:
        target = _labels(s, case["classes"], g).to(torch.int32)
        start = torch.full((case["classes"], case["rows"]), -math.log(case["classes"]),
                           device=DEV)
    else:
        target = s + 0.5 * torch.randn(s.shape, generator=g, device=DEV)
        start = torch.full((case["rows"],), float(target.double().mean()), device=DEV)
    era = _era_ids(case, g) if case["eras"] > 1 else np.zeros(case["rows"], np.int32)
    k = max(1, int(case["colsample"] * case["feats"]))
    sels = [torch.randperm(case["feats"], generator=g, device=DEV, dtype=torch.int32)[:k]
            if k < case["feats"] else
            torch.arange(case["feats"], device=DEV, dtype=torch.int32)
            for _ in range(case["rounds"])]
    return x8, target, start, era, sels


def _hist_inputs(case, seed):
    g = _gen(seed)
    x8 = _codes8(case, g)
    resid = torch.randn(case["rows"], generator=g, device=DEV)
    node = torch.randint(0, case["nodes"], (case["rows"],), generator=g, device=DEV)
    order = torch.argsort(node, stable=True).to(torch.int32)
    seg = torch.zeros(case["nodes"] + 1, dtype=torch.int64, device=DEV)
    seg[1:] = torch.cumsum(torch.bincount(node, minlength=case["nodes"]), 0)
    return x8, resid, order, seg


def _split_inputs(case, seed):
    g = _gen(seed)
    shape = (case["eras"], case["feats"], case["bins"])
    H = torch.randint(0, 400, shape, generator=g, device=DEV).float()
    G = torch.randn(shape, generator=g, device=DEV) * H.sqrt()
    return G, H


def _forest(case, g):
    """Heap tables of random trees: most nodes split, on features some of
    which are used far more often than others; early leaves here and there."""
    H = (1 << (case["depth"] + 1)) - 1
    T = case["rounds"] * case["classes"]
    u = torch.rand((T, H), generator=g, device=DEV)
    feat = (u * u * case["feats"]).to(torch.int32).clamp_(max=case["feats"] - 1)
    bin_ = torch.randint(0, max(1, case["bins"] - 1), (T, H), generator=g, device=DEV,
                         dtype=torch.int32)
    leaf = 0.3 * torch.randn((T, H), generator=g, device=DEV)
    early = torch.rand((T, H), generator=g, device=DEV) < 0.04
    inner = (1 << case["depth"]) - 1
    early[:, 0] = False
    feat[:, inner:] = -1
    feat[early] = -1
    for h in range(1, H):  # below a leaf there is no node
        gone = feat[:, (h - 1) // 2] < 0
        feat[gone, h] = -2
    return feat.contiguous(), bin_, leaf


def _tables(feat, bin_, leaf):
    """The heap tables as flattened trees [T, M, 6] in pre-order (feature, bin,
    left, right, is_leaf, value), empty rows NaN."""
    T, H = feat.shape
    f = feat.cpu().numpy()
    depth = (H + 1).bit_length() - 2
    pos = np.full((T, H), -1, np.int64)   # a node's place in its tree's table
    size = np.zeros((T, H), np.int64)     # nodes under it, itself included
    for h in range(H - 1, -1, -1):
        size[:, h] = f[:, h] != -2
        if 2 * h + 2 < H:
            size[:, h] += np.where(f[:, h] >= 0, size[:, 2 * h + 1] + size[:, 2 * h + 2], 0)
    pos[:, 0] = 0
    for h in range((1 << depth) - 1):
        pos[:, 2 * h + 1] = pos[:, h] + 1
        pos[:, 2 * h + 2] = pos[:, h] + 1 + size[:, 2 * h + 1]
    out = np.full((T, H + 1, 6), np.nan, np.float32)
    b, v = bin_.cpu().numpy(), leaf.cpu().numpy()
    for h in range(H):
        t = np.flatnonzero(f[:, h] >= 0)
        row = pos[t, h]
        out[t, row, 0], out[t, row, 1], out[t, row, 4] = f[t, h], b[t, h], 0
        if 2 * h + 2 < H:
            out[t, row, 2], out[t, row, 3] = pos[t, 2 * h + 1], pos[t, 2 * h + 2]
        t = np.flatnonzero(f[:, h] == -1)
        out[t, pos[t, h], 4], out[t, pos[t, h], 5] = 1, v[t, h]
    return torch.from_numpy(out).to(DEV)


def _predict_inputs(case, seed):
    g = _gen(seed)
    x8 = _codes8(case, g)
    return (x8, *_forest(case, g))


# --------------------------------------------------------------------------- prepare and run
MIN_CHILD, L2, LR = 20, 1e-6, 0.1


class _Rounds:
    """An engine on resident codes with the buffers its rounds write."""

    def __init__(self, case, seed):
        x8, self.target, self.start, era, self.sels = _round_inputs(case, seed)
        codes, _ = D.codes_from_int8(x8, True, case["bins"])
        _, _, order, era_start = D.era_layout(era)
        K = case["classes"]
        T, H, R = max(1, K), (1 << (case["depth"] + 1)) - 1, case["rounds"]
        self.eng = D.Engine(codes, torch.from_numpy(order).to(DEV),
                            torch.from_numpy(era_start).to(DEV), case["bins"], len(era_start) - 1,
                            case["depth"], T, 1 if K else 0, MIN_CHILD, 0.0, L2, LR)
        self.pred = torch.empty_like(self.start)
        z = dict(device=DEV)
        self.rec = [dict(feat=torch.zeros((T, H), dtype=torch.int32, **z),
                         bin=torch.zeros((T, H), dtype=torch.int32, **z),
                         leaf=torch.zeros((T, H), **z),
                         count=torch.zeros((T, H), dtype=torch.int64, **z),
                         gain=torch.zeros((T, H, len(era_start) - 1), **z)) for _ in range(R)]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "fit":
        return dict(case=case, **_fit_inputs(case, seed))
    if kind == "round":
        return dict(case=case, rounds=_Rounds(case, seed))
    if kind == "histogram":
        x8, resid, order, seg = _hist_inputs(case, seed)
        st = dict(case=case, resid=resid, order=order, seg=seg)
        shape = (case["nodes"] + 1, case["feats"], case["bins"])
        st["G"], st["H"] = torch.zeros(shape, device=DEV), torch.zeros(shape, device=DEV)
        if case["how"] == "calls":
            st["x8"] = x8
            st["all_rows"] = torch.arange(case["rows"], dtype=torch.int32, device=DEV)
            st["feats"] = torch.arange(case["feats"], dtype=torch.int32, device=DEV)
            st["era"] = torch.zeros(case["rows"], dtype=torch.int32, device=DEV)
            at = seg.tolist()
            st["node_rows"] = [order[a:b].contiguous() for a, b in zip(at[:-1], at[1:])]
        else:
            st["codes"] = D.codes_from_int8(x8, False, case["bins"])[0]
            st["root_seg"] = torch.tensor([0, case["rows"]], dtype=torch.int64, device=DEV)
        return st
    if kind == "split":
        G, H = _split_inputs(case, seed)
        shape = (case["eras"], case["feats"], case["bins"] - 1)
        return dict(case=case, G=G, H=H, gain=torch.empty(shape, device=DEV),
                    direction=torch.empty(shape, device=DEV))
    if kind == "ingest":
        g = _gen(seed)
        X = torch.randn((case["rows"], case["feats"]), generator=g, device=DEV)
        X[:, 1::7].exp_()  # some long-tailed columns
        X[:, 3::11].round_()  # and some with many equal values
        return dict(case=case, X=X)
    x8, feat, bin_, leaf = _predict_inputs(case, seed)
    st = dict(case=case)
    if case["how"] == "table":
        st.update(x8=x8, table=_tables(feat, bin_, leaf))
    else:
        st.update(codes=D.codes_from_int8(x8, False, case["bins"])[0], feat=feat, bin=bin_,
                  leaf=leaf)
    return st


def run(state):
    return _RUN[state["case"]["kind"]](state, state["case"])


def _run_fit(st, case):
    m = WarpGBM(objective="multiclass" if case["classes"] else "regression",
                num_bins=case["bins"], max_depth=case["depth"], n_estimators=case["rounds"],
                learning_rate=LR, min_child_weight=MIN_CHILD, L2_reg=L2, device=DEV)
    m.fit(st["X"], st["y"], era_id=st["era"])
    out = m.predict_proba(st["X_new"]) if case["classes"] else m.predict(st["X_new"])
    return dict(edges=m.bin_edges, importance=m.per_era_feature_importance_, new=out)


def _run_round(st, case):
    r = st["rounds"]
    r.pred.copy_(r.start)
    for sel, rec in zip(r.sels, r.rec):
        r.eng.round(r.target, r.pred, sel, rec)
    return dict(pred=r.pred, records=r.rec)


def _run_histogram(st, case):
    G, H = st["G"].zero_(), st["H"].zero_()
    n, B, k = case["rows"], case["bins"], case["nodes"]
    if case["how"] == "calls":
        for i, rows in enumerate([st["all_rows"], *st["node_rows"]]):
            node_kernel.compute_histogram3(st["x8"], st["resid"], rows, st["feats"], st["era"],
                                           G[i:i + 1], H[i:i + 1], B)
        return dict(G=G, H=H)
    lib, c = _lib.load(), st["codes"]
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.wgbm_histogram_segments(
        c.rm.data_ptr(), n, c.stride, c.n_feats, st["resid"].data_ptr(), None,
        st["root_seg"].data_ptr(), 1, n, B, _lib.CODES_NATIVE, G[:1].data_ptr(),
        H[:1].data_ptr(), C.c_void_p(stream)), "root")
    _lib.check(lib.wgbm_histogram_segments(
        c.rm.data_ptr(), n, c.stride, c.n_feats, st["resid"].data_ptr(), st["order"].data_ptr(),
        st["seg"].data_ptr(), k, n, B, _lib.CODES_NATIVE, G[1:].data_ptr(), H[1:].data_ptr(),
        C.c_void_p(stream)), "nodes")
    return dict(G=G, H=H)


def _run_split(st, case):
    node_kernel.compute_split(st["G"], st["H"], 0.0, float(MIN_CHILD), L2, st["gain"],
                              st["direction"], 128)
    return dict(gain=st["gain"], direction=st["direction"])


def _run_ingest(st, case):
    edges = D.quantile_edges(st["X"], case["bins"])
    codes = D.bin_matrix(st["X"], edges, with_cm=True)
    return dict(edges=edges, rm=codes.rm, cm=codes.cm)


def _run_predict(st, case):
    if case["how"] == "table":
        out = torch.zeros(case["rows"], device=DEV)
        node_kernel.predict_forest(st["x8"], st["table"], LR, out)
        return out
    out = torch.zeros((case["rows"], case["classes"]), device=DEV)
    D.predict_heap(st["codes"], st["feat"], st["bin"], st["leaf"], case["rounds"],
                   case["classes"], case["depth"], LR, out)
    if case["classes"] > 1:
        D.softmax_rows(out)
    return out


_RUN = dict(fit=_run_fit, round=_run_round, histogram=_run_histogram, split=_run_split,
            ingest=_run_ingest, predict=_run_predict)


# --------------------------------------------------------------------------- work and tolerance
def work(case):
    """Bytes and operations that a pass cannot do without: each input read
    once and each output written once.  Growing a tree needs the codes of
    every row once per tree (class trees share them), and one add of a sum
    and one of a count per row and feature; each further level needs the rows
    of the smaller children only (counted as none: it may be any share)."""
    kind = case["kind"]
    n, F, B = case.get("rows", 0), case.get("feats", 0), case.get("bins", 0)
    if kind == "fit":
        T, hold = max(1, case["classes"]), max(500, n // 10)
        return dict(bytes=4.0 * (n + hold) * F + case["rounds"] * (n * F + 12.0 * n * T),
                    flops=2.0 * case["rounds"] * T * n * F)
    if kind == "round":
        T = max(1, case["classes"])
        k = max(1, int(case["colsample"] * F))
        return dict(bytes=case["rounds"] * (1.0 * n * k + 12.0 * n * T),
                    flops=2.0 * case["rounds"] * T * n * k)
    if kind == "histogram":
        return dict(bytes=2.0 * n * F + 12.0 * n + 8.0 * (case["nodes"] + 1) * F * B,
                    flops=4.0 * n * F)
    if kind == "split":
        cells = 1.0 * case["eras"] * F
        return dict(bytes=8.0 * cells * B + 8.0 * cells * (B - 1), flops=14.0 * cells * B)
    if kind == "ingest":
        return dict(bytes=4.0 * n * F + 2.0 * n * F + 4.0 * F * (B - 1),
                    flops=1.0 * n * F * max(1.0, math.log2(B)))
    T = case["rounds"] * case["classes"]
    return dict(bytes=1.0 * n * F + 4.0 * n * case["classes"] + 12.0 * T * (2 << case["depth"]),
                flops=1.0 * n * T * (case["depth"] + 2))


def tolerance(case):
    """Sums are exact integers of the quantised residuals, split scans
    sequential, trees added in tree order: the package documents every one of
    these results as independent of how it was computed, bit for bit."""
    return "exact"


# --------------------------------------------------------------------------- 64-bit results
def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _cells(codes, key, n_keys, w, B, feats):
    """Sums of w and counts [n_keys, F, B] in float64 over the rows of each
    key (rows of a negative key, and codes outside [0, B), are dropped)."""
    rows = torch.nonzero(key >= 0)[:, 0]
    key, w = key[rows].long(), w[rows].to(F64)
    F = feats.numel()
    G, H = (torch.zeros((n_keys, F, B), dtype=F64, device=DEV) for _ in range(2))
    step = max(1, min(F, 60_000_000 // max(1, rows.numel())))
    for f0 in range(0, F, step):
        c = codes[:, feats[f0:f0 + step].long()][rows].long()
        k = c.shape[1]
        at = (key[:, None] * k + torch.arange(k, device=DEV)[None, :]) * B + c
        at = at.reshape(-1)
        size = n_keys * k * B
        gs = torch.bincount(at, weights=w[:, None].expand(-1, k).reshape(-1), minlength=size)
        hs = torch.bincount(at, minlength=size)
        G[:, f0:f0 + step] = gs.view(n_keys, k, B)
        H[:, f0:f0 + step] = hs.view(n_keys, k, B).to(F64)
    return G, H


def _gains(G, H):
    """Gains and directions [..., B - 1] of the cuts after each bin."""
    Gt, Ht = G.sum(-1, keepdim=True), H.sum(-1, keepdim=True)
    GL, HL = G.cumsum(-1)[..., :-1], H.cumsum(-1)[..., :-1]
    GR, HR = Gt - GL, Ht - HL
    ok = (HL >= MIN_CHILD) & (HR >= MIN_CHILD)
    gain = GL * GL / (HL + L2) + GR * GR / (HR + L2) - Gt * Gt / (Ht + L2)
    way = torch.where(GL / (HL + L2) > GR / (HR + L2), 1.0, -1.0).to(F64)
    zero = torch.zeros((), dtype=F64, device=DEV)
    return torch.where(ok, gain, zero), torch.where(ok, way, zero)


def _grow(codes, resid, era, E, sel, B, depth):
    """One tree in 64 bits: its heap (feature -1 at a leaf and -2 where there
    is no node, cut, leaf value, per-era gains of the cut) and the value that
    it gives each row."""
    n, Hn = codes.shape[0], (1 << (depth + 1)) - 1
    feat = torch.full((Hn,), -2, dtype=torch.int64, device=DEV)
    cut = torch.zeros(Hn, dtype=torch.int64, device=DEV)
    leaf = torch.zeros(Hn, dtype=F64, device=DEV)
    gains = torch.zeros((Hn, E), dtype=F64, device=DEV)
    feat[0] = -1
    at = torch.zeros(n, dtype=torch.int64, device=DEV)
    for d in range(depth + 1):
        first, k = (1 << d) - 1, 1 << d
        live = at >= first  # rows whose node is on this level
        loc = torch.where(live, at - first, torch.full_like(at, -1))
        total = torch.zeros(k + 1, dtype=F64, device=DEV).index_add_(0, loc + 1, resid)[1:]
        count = torch.bincount(loc + 1, minlength=k + 1)[1:]
        leaf[first:first + k] = total / count.clamp(min=1)
        if d == depth:
            break
        key = torch.where(live, loc * E + era, loc)
        top = torch.full((k,), -1.0, dtype=F64, device=DEV)  # agreement and gain of the best cut
        gain = torch.zeros(k, dtype=F64, device=DEV)
        step = max(1, min(sel.numel(), 60_000_000 // (k * E * B)))
        for f0 in range(0, sel.numel(), step):
            G, H = _cells(codes, key, k * E, resid, B, sel[f0:f0 + step])
            g, way = (x.reshape(k, E, -1) for x in _gains(G, H))
            agree = way.sum(1).abs() if E > 1 else torch.zeros_like(g[:, 0])
            crit = g.mean(1)
            best_agree = agree.max(1).values
            crit_ok = torch.where(agree == best_agree[:, None], crit,
                                  torch.full_like(crit, -math.inf))
            c, j = crit_ok.max(1)
            better = (best_agree > top) | ((best_agree == top) & (c > gain))
            top = torch.where(better, best_agree, top)
            gain = torch.where(better, c, gain)
            at_h = torch.arange(first, first + k, device=DEV)[better]
            jb = j[better]
            feat_new, cut_new = sel.long()[f0 + jb // (B - 1)], jb % (B - 1)
            cut[at_h] = cut_new
            gains[at_h] = g[better].gather(2, jb[:, None, None].expand(-1, E, 1))[:, :, 0]
            feat[at_h] = torch.where(feat[at_h] == -2, feat[at_h], feat_new)
            del G, H, g, way
        lvl = torch.arange(first, first + k, device=DEV)
        stop = (feat[lvl] != -2) & ((gain <= 0) | (count == 0))
        feat[lvl[stop]] = -1
        gains[lvl[stop | (feat[lvl] < 0)]] = 0
        split = lvl[feat[lvl] >= 0]
        leaf[split] = 0
        leaf[lvl[feat[lvl] == -2]] = 0
        feat[2 * split + 1] = -1
        feat[2 * split + 2] = -1
        f = feat[at]
        code = codes.gather(1, f.clamp(min=0)[:, None])[:, 0].long()
        at = torch.where(live & (f >= 0), 2 * at + 1 + (code > cut[at]).long(), at)
    return feat, cut, leaf, gains, leaf[at]


def _walk(codes, feat, cut, leaf, depth):
    """The value that a heap-ordered tree gives each row of codes."""
    i = torch.zeros(codes.shape[0], dtype=torch.int64, device=DEV)
    for _ in range(depth):
        f = feat[i]
        code = codes.gather(1, f.clamp(min=0)[:, None])[:, 0].long()
        i = torch.where(f >= 0, 2 * i + 1 + (code > cut[i]).long(), i)
    return leaf[i]


def _residuals(target, pred, K):
    """The trees' targets of one round: pred [max(1, K), n]."""
    if not K:
        return [target.to(F64) - pred[0]]
    p = torch.softmax(pred, 0)
    return [(target == k).to(F64) - p[k] for k in range(K)]


def _affordable(case, most):
    trees = case["rounds"] * max(1, case["classes"])
    return trees * case["depth"] * case["rows"] * case["feats"] <= most


def _era_of_rows(era):
    """Era index of every row (device) and the number of eras."""
    uniq, inv = np.unique(era, return_inverse=True)
    return torch.from_numpy(inv.reshape(-1)).to(DEV), len(uniq)


def _exact_round(case, seed):
    # a split is the largest of thousands of gains: where two differ by less
    # than their rounding the 64-bit tree may take the other one, and all that
    # follows differs
    if not _affordable(case, 1.2e10):
        return None
    x8, target, start, era, sels = _round_inputs(case, seed)
    era_d, E = _era_of_rows(era)
    K = case["classes"]
    pred = start.to(F64).reshape(max(1, K), -1).clone()
    lr, records = float(np.float32(LR)), []
    for sel in sels:
        trees = [_grow(x8, r, era_d, E, sel, case["bins"], case["depth"])
                 for r in _residuals(target, pred, K)]
        for k, tree in enumerate(trees):
            pred[k] += lr * tree[4]
        records.append(dict(feat=None, bin=None, count=None,
                            leaf=torch.stack([t[2] for t in trees]),
                            gain=torch.stack([t[3] for t in trees])))
    return dict(pred=pred if K else pred[0], records=records)


def _quantiles(X, B):
    """Interpolated order statistics of every column, in float64."""
    n, F = X.shape
    rank = torch.linspace(0, 1, B + 1)[1:-1].to(F64) * (n - 1)
    lo, hi = (r.long().clamp(max=n - 1).to(DEV) for r in (rank.floor(), rank.ceil()))
    w = (rank - rank.floor()).to(DEV)
    out = torch.empty((F, B - 1), dtype=F64, device=DEV)
    step = max(1, 100_000_000 // n)
    for f in range(0, F, step):
        s = X[:, f:f + step].t().contiguous().sort(dim=1).values.to(F64)
        a, b = s[:, lo], s[:, hi]
        out[f:f + step] = a + w * (b - a)
    return out


def _exact_fit(case, seed):
    if not _affordable(case, 6e9):
        return None
    d = _fit_inputs(case, seed)
    X, X_new = torch.from_numpy(d["X"]).to(DEV), torch.from_numpy(d["X_new"]).to(DEV)
    y = torch.from_numpy(d["y"]).to(DEV)
    n, B, K, F = case["rows"], case["bins"], case["classes"], case["feats"]
    edges = _quantiles(X, B)

    def codes_of(M):
        # against the edges in the type of the data, as binning compares them
        return torch.stack([torch.bucketize(M[:, f].contiguous(), edges[f].float(), right=True)
                            for f in range(F)], 1).to(torch.int8)

    codes, new = codes_of(X), codes_of(X_new)
    era_d, E = _era_of_rows(d["era"] if d["era"] is not None else np.zeros(n, np.int32))
    if K:
        prior = (torch.bincount(y, minlength=K).to(F64) / n + 1e-10).log()
        out = torch.full((K, new.shape[0]), math.log(1 / K + 1e-10), dtype=F64, device=DEV)
    else:
        prior = y.to(F64).mean()[None]
        out = prior[:, None].repeat(1, new.shape[0])
    pred = prior[:, None].repeat(1, n)
    sel, lr = torch.arange(F, device=DEV), float(np.float32(LR))
    importance = torch.zeros((E, F), dtype=F64, device=DEV)
    for _ in range(case["rounds"]):
        for k, r in enumerate(_residuals(y, pred, K)):
            feat, cut, leaf, gains, value = _grow(codes, r, era_d, E, sel, B, case["depth"])
            pred[k] += lr * value
            out[k] += lr * _walk(new, feat, cut, leaf, case["depth"])
            importance.index_add_(1, feat.clamp(min=0), (gains * (feat >= 0)[:, None]).t())
    return dict(edges=edges, importance=importance,
                new=torch.softmax(out, 0).t() if K else out[0])


def _exact_histogram(case, seed):
    x8, resid, order, seg = _hist_inputs(case, seed)
    at = seg.tolist()
    node = torch.empty(case["rows"], dtype=torch.int64, device=DEV)
    for k, (a, b) in enumerate(zip(at[:-1], at[1:])):
        node[order[a:b].long()] = k
    feats = torch.arange(case["feats"], device=DEV)
    G, H = _cells(x8, node, case["nodes"], resid, case["bins"], feats)
    return dict(G=torch.cat([G.sum(0, keepdim=True), G]), H=torch.cat([H.sum(0, keepdim=True), H]))


def _exact_split(case, seed):
    G, H = _split_inputs(case, seed)
    gain, way = _gains(G.to(F64), H.to(F64))
    return dict(gain=gain, direction=way)


def _exact_ingest(case, seed):
    X = prepare(case, seed)["X"]
    return dict(edges=_quantiles(X, case["bins"]), rm=None, cm=None)


def _exact_predict(case, seed):
    x8, feat, bin_, leaf = _predict_inputs(case, seed)
    K, lr = case["classes"], float(np.float32(LR))
    out = torch.zeros((case["rows"], K), dtype=F64, device=DEV)
    for t in range(feat.shape[0]):
        out[:, t % K] += lr * _walk(x8, feat[t].long(), bin_[t].long(), leaf[t].to(F64),
                                    case["depth"])
    if case["how"] == "table":
        return out[:, 0]
    return torch.softmax(out, 1) if K > 1 else out


_EXACT = dict(fit=_exact_fit, round=_exact_round, histogram=_exact_histogram, split=_exact_split,
              ingest=_exact_ingest, predict=_exact_predict)
