"""Rows drawn from whole (no filter, or typical-p alone) and rows loaded
element by element, through the production route (no probabilities asked
for, which would send every row elsewhere), against the oracle: fp32 and
bf16, sliced and single-slice batches, rows at 16-byte, dword and odd
addresses, masks, NaN, infinities and ties."""
from __future__ import annotations

import numpy as np
import pytest

import cases
from chenxing_amd import workloads as W
from chenxing_amd._lib import FLAG_DEEP, FLAG_SLOW, sample_host
from chenxing_amd.params import RowParams
from oracle import sampler_ref as R
from parity import Tally, compare_rows

pytestmark = pytest.mark.gpu


def _sample(x, prm, hist, hl, u, dtype, label):
    """Device ids and statuses of the rows, compared with the oracle's."""
    bits = W.f32_to_bf16_rne(x) if dtype == "bf16" else x
    rows = W.bf16_to_f32(bits) if dtype == "bf16" else x
    print(f"[gpu] {label} {dtype} B={x.shape[0]} V={x.shape[1]}", flush=True)
    ids, st, _ = sample_host(bits, prm, hist, hl, u, bf16=(dtype == "bf16"))
    lists = None if hist is None else R.hist_rows_to_lists(hist, hl)
    orc = [R.sample_row(rows[b], prm[b], None if lists is None else lists[b], u[b], tie="spread")
           for b in range(x.shape[0])]
    t = compare_rows(ids, st, None, orc, label)
    assert not t.mismatches, t.mismatches[:5]
    return t, st


def _zero_cut(row: np.ndarray) -> float:
    """A typical_p whose cut keeps about half of the row's zeros."""
    P = R.tempered_probs(row.astype(np.float64), 1.0)
    logp = np.log(np.maximum(P, 1e-38))
    dist = np.abs(logp - (P * logp).sum())
    order = np.argsort(dist, kind="stable")
    run = np.cumsum(P[order])
    pos = np.flatnonzero(dist[order] == dist[np.flatnonzero(row == 0.0)[0]])
    j = pos[pos.size // 2]
    return float((run[j - 1] + run[j]) / 2)


def _whole_batch(B, V, seed):
    """Row kinds in turn; returns the logits, parameters and, per row, the
    flags a decided row carries (None: a row the multi-pass path ends)."""
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 2.0, (B, V)).astype(np.float32)
    prm, ends = [], []
    for b in range(B):
        k = b % 13
        kw = [dict(), dict(temperature=0.6), dict(typical_p=0.9), dict(typical_p=0.5, temperature=1.4),
              dict(), dict(typical_p=0.95), dict(typical_p=0.7), dict(typical_p=0.7),
              dict(), dict(typical_p=0.8), dict(), dict(), dict(typical_p=0.6)][k]
        end = "typical" if "typical_p" in kw else "plain"
        if k in (4, 5):                                   # masked ids, and chunks of nothing else
            x[b, rng.choice(V, V // 3, replace=False)] = -np.inf
            x[b, 1024:min(V, 3072)] = -np.inf
            x[b, 7] = 1.0
        elif k in (6, 7):                                 # ties; zeros of both signs at the cut
            x[b] = np.round(x[b] * 8) / 8
            if k == 7:
                zero = np.flatnonzero(x[b] == 0.0)
                x[b, zero[rng.random(zero.size) < 0.5]] = np.float32(-0.0)
                kw = dict(typical_p=_zero_cut(x[b]))
        elif k in (8, 9):                                 # NaN
            x[b, V - 3], end = np.nan, None
        elif k == 10:                                     # +inf
            x[b, V // 2], end = np.inf, None
        elif k in (11, 12):                               # nothing at all
            x[b], end = -np.inf, None
        prm.append(RowParams(**kw))
        ends.append(end)
    return x, prm, rng.random(B), ends


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("B,V", [(26, 50256), (26, 50258), (26, 50257),      # sliced
                                 (13, 9001), (260, 2001), (260, 2004), (13, 300)])
def test_whole_rows(dtype, B, V):
    x, prm, u, ends = _whole_batch(B, V, B + V)
    t, st = _sample(x, prm, None, None, u, dtype, "whole rows")
    assert t.draws >= 8 * (B // 13)
    # bf16 rows an odd number of elements apart have no vector loads: their
    # typical-p rows take the multi-pass path
    typical = FLAG_SLOW if dtype == "bf16" and V % 2 else FLAG_SLOW | FLAG_DEEP
    want = {"plain": 0, "typical": typical}
    # (short rows crowd the typical order's buckets: some are handed back)
    for b, end in enumerate(ends):
        if end == "plain" or (end == "typical" and V > 40000):
            assert int(st[b]) & 0xF00 == want[end], (b, hex(int(st[b])), end)


@pytest.mark.parametrize("dtype,B,V", [("bf16", 24, 30001), ("bf16", 24, 50257), ("bf16", 260, 3001),
                                       ("f32", 24, 5001), ("f32", 260, 1001), ("f32", 24, 8191),
                                       ("f32", 24, 8193), ("bf16", 24, 1002)])
def test_rows_loaded_by_elements(dtype, B, V):
    """Every knob on rows off 16-byte boundaries: bf16 rows at odd addresses
    and short rows (below 8192 elements), element by element; beside them the
    lengths where vector loads take over and one-chunk top-k rows."""
    rng = np.random.default_rng(B * 3 + V)
    H = 300
    x = rng.normal(0, 2.0, (B, V)).astype(np.float32)
    x[np.arange(B), rng.integers(0, V, B)] += np.float32(8.0)
    hist = rng.integers(-50, V + 50, (B, H)).astype(np.int32)
    hl = rng.integers(0, H + 1, B).astype(np.int32)
    hl[::3] = 0                                           # no penalty window
    prm = [RowParams(temperature=float(rng.choice([0.0, 0.6, 1.0, 1.5])),
                     top_k=int(rng.choice([0, 0, 7, 64, 65, 300])),
                     top_p=float(rng.choice([1.0, 0.8, 0.97])),
                     min_p=float(rng.choice([0.0, 0.0, 0.02])),
                     typical_p=float(rng.choice([1.0, 1.0, 1.0, 0.9])),
                     repetition_penalty=float(rng.choice([1.0, 1.3])),
                     presence_penalty=float(rng.choice([0.0, 0.4])),
                     frequency_penalty=float(rng.choice([0.0, 0.2]))) for _ in range(B)]
    t, _ = _sample(x, prm, hist, hl, rng.random(B), dtype, "element loads")
    assert t.boundary == 0


def test_golden_small_rows_without_probabilities():
    """The small golden rows (every knob, ties, -inf, NaN, underflow), ids and
    outcomes only."""
    by_v: dict = {}
    for c in cases.small_sampler_cases():
        by_v.setdefault(c.logits.size, []).append(c)
    total = Tally()
    for V, cs in sorted(by_v.items()):
        H = max(1, max(len(c.hist) for c in cs))
        hist = np.full((len(cs), H), -1, np.int32)
        hl = np.zeros(len(cs), np.int32)
        for b, c in enumerate(cs):
            hist[b, :len(c.hist)] = c.hist
            hl[b] = len(c.hist)
        prm = [RowParams(**{k: c.params[k] for k in (
            "temperature", "top_k", "top_p", "min_p", "typical_p", "repetition_penalty", "n_keep")})
            for c in cs]
        u = np.array([np.random.default_rng(c.params["seed"]).random() for c in cs])
        print(f"[gpu] golden small rows V={V} B={len(cs)}", flush=True)
        ids, st, _ = sample_host(np.stack([c.logits for c in cs]), prm, hist, hl, u)
        orc = [R.sample_row(c.logits, p, c.hist, u[b], tie="spread")
               for b, (c, p) in enumerate(zip(cs, prm))]
        total.merge(compare_rows(ids, st, None, orc, f"V{V}"))
    assert not total.mismatches, total.mismatches[:5]
    assert total.boundary <= 2                            # as in the host emulation
