"""Sampler parity on the GPU: the HIP library against the oracle on the same
inputs and uniforms (rules in tests/parity.py).

Every workload runs twice: with ``out_probs`` (which routes every stochastic
row through the region finisher, so the probabilities can be compared) and
without it (the production route, the one the benchmark times: single-slice
top-k rows are finished inside the fused kernel).  Each is compared with the
oracle in the device's tie order and, for the rate report, in numpy's own
order (what the reference computes)."""
from __future__ import annotations

import functools
import sys

import numpy as np
import pytest

import cases
from chenxing_amd import workloads as W
from chenxing_amd._lib import FLAG_SLOW, ROW_UNSUPPORTED, sample_host
from chenxing_amd.params import RowParams
from oracle import sampler_ref as R
from oracle_pool import oracle_rows_parallel
from parity import REF_BUDGET, Tally, compare_rows

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@functools.lru_cache(maxsize=2)
def _workload(name, **kw):
    return getattr(W, name)(**kw)


def _run(w, want_probs=True):
    _say(f"[gpu] sample {w.name} B={w.B} V={w.V} dtype={w.dtype} probs={want_probs}")
    ids, st, probs = sample_host(w.logits, w.params, w.hist if w.hist.size else None,
                                 w.hist_len, w.u, bf16=(w.dtype == "bf16"), want_probs=want_probs)
    return ids, st, probs


def _check(w, ids, st, probs, label):
    """Device rows against the oracle in both tie orders; returns the tally."""
    pairs = oracle_rows_parallel(w, ties=("spread", "numpy"), keep_probs=probs is not None)
    t = compare_rows(ids, st, probs, [p[0] for p in pairs], label, ref_rows=[p[1] for p in pairs])
    _say(f"    {label}: draws {t.draws}, margin cases {t.boundary}; vs numpy's order: "
         f"{t.ref_diff} differ ({t.ref_diff_tie} tie straddles), {t.ref_straddle} straddle")
    assert not t.mismatches, t.mismatches[:5]
    assert t.boundary <= REF_BUDGET * t.draws + 1e-9 or t.boundary == 0
    return t


def _probs_label(name, want_probs):
    return name + ("+probs" if want_probs else "")


def test_small_batch_config():
    w = W.small_batch()
    for want_probs in (True, False):
        ids, st, probs = _run(w, want_probs)
        t = _check(w, ids, st, probs, _probs_label("small_batch", want_probs))
        assert t.draws == 4


@pytest.mark.parametrize("want_probs", [True, False])
def test_full_penalty_config(want_probs):
    w = _workload("full_penalty")
    ids, st, probs = _run(w, want_probs)
    t = _check(w, ids, st, probs, _probs_label("full_penalty", want_probs))
    assert t.draws == 256 and t.boundary == 0


@pytest.mark.parametrize("want_probs", [True, False])
@pytest.mark.parametrize("greedy", [True, False])
def test_nucleus_config(greedy, want_probs):
    w = _workload("nucleus", greedy=greedy)
    ids, st, probs = _run(w, want_probs)
    t = _check(w, ids, st, probs, _probs_label(w.name, want_probs))
    assert t.rows == 64


def test_hetero_bf16_config_subset():
    """B=96: each row in three slices, probabilities compared."""
    w = W.hetero_bf16(B=96)
    ids, st, probs = _run(w, True)
    _check(w, ids, st, probs, "hetero_bf16[B=96]+probs")


def test_hetero_bf16_config_full_size():
    """B=1024, V=256000 bf16, the workload's own size: one slice per row, so
    the one-wave top-k finish, the FINISH hand-off and the refinement of
    single-slice rows run exactly as the benchmark runs them."""
    w = _workload("hetero_bf16")
    ids, st, probs = _run(w, False)
    t = _check(w, ids, st, None, "hetero_bf16")
    assert t.rows == 1024 and t.boundary == 0


def test_golden_small_rows():
    """Every small golden case (all knobs, ties, -inf, NaN, underflow) through
    the device, one batch per vocabulary size."""
    all_cases = cases.small_sampler_cases()
    by_v: dict = {}
    for c in all_cases:
        by_v.setdefault(c.logits.size, []).append(c)
    total = Tally()
    for V, cs in sorted(by_v.items()):
        B = len(cs)
        x = np.stack([c.logits for c in cs])
        prm = [RowParams(temperature=c.params["temperature"], top_k=c.params["top_k"],
                         top_p=c.params["top_p"], min_p=c.params["min_p"],
                         typical_p=c.params["typical_p"],
                         repetition_penalty=c.params["repetition_penalty"],
                         n_keep=c.params["n_keep"]) for c in cs]
        H = max(1, max(len(c.hist) for c in cs))
        hist = np.full((B, H), -1, np.int32)
        hl = np.zeros(B, np.int32)
        for b, c in enumerate(cs):
            hist[b, :len(c.hist)] = c.hist
            hl[b] = len(c.hist)
        u = np.array([np.random.default_rng(c.params["seed"]).random() for c in cs])
        _say(f"[gpu] golden small rows V={V} B={B}")
        ids, st, probs = sample_host(x, prm, hist, hl, u, want_probs=True)
        orc = [R.sample_row(c.logits, p, c.hist, u[b], tie="spread", keep_probs=True)
               for b, (c, p) in enumerate(zip(cs, prm))]
        total.merge(compare_rows(ids, st, probs, orc, f"V{V}"))
    assert not total.mismatches, total.mismatches[:5]


def _slow_batch(V=50000, seed=3):
    """Rows built to leave the fused path: each needs the multi-pass kernel."""
    rng = np.random.default_rng(seed)
    rows, prms = [], []

    def add(x, **kw):
        rows.append(np.asarray(x, np.float32))
        prms.append(RowParams(**kw))

    add(rng.normal(0, 0.5, V), temperature=1.0, top_p=0.9)            # deep nucleus
    add(rng.normal(0, 2, V), temperature=0.8, top_k=5000)             # k beyond the region
    add(np.zeros(V), temperature=1.0, top_k=10)                       # one tie group
    q = np.round(rng.normal(0, 1, V) * 4) / 4                          # coarse ties
    add(q, temperature=1.0, top_p=0.6)
    add(rng.normal(0, 1, V), temperature=1.0, min_p=0.01)             # wide min-p
    add(rng.normal(0, 2, V), temperature=1.0, typical_p=0.8)          # typical-p
    add(rng.normal(0, 2, V), temperature=0.9, top_k=100, typical_p=0.5)
    bad = rng.normal(0, 2, V)
    bad[123] = np.nan
    add(bad, temperature=1.0, top_k=5)                                 # NaN -> argmax
    add(bad, temperature=1.0)                                          # NaN -> error
    inf = rng.normal(0, 2, V)
    inf[77] = np.inf
    add(inf, temperature=1.0, min_p=0.1)                               # +inf -> argmax
    add(np.full(V, -np.inf), temperature=1.0)                          # all -inf -> error
    add(rng.normal(0, 0.1, V), temperature=0.001, top_k=3)             # underflow -> argmax
    add(rng.normal(0, 0.1, V), temperature=0.001)                      # underflow -> error
    add(rng.normal(0, 1, V), temperature=1.3, top_p=0.999)            # nucleus ~ all
    return np.stack(rows), prms


def test_slow_path_rows():
    x, prm = _slow_batch()
    B = x.shape[0]
    u = np.random.default_rng(11).random(B)
    _say(f"[gpu] slow-path rows B={B} V={x.shape[1]}")
    ids, st, probs = sample_host(x, prm, None, None, u, want_probs=True)
    orc = [R.sample_row(x[b], prm[b], None, u[b], tie="spread", keep_probs=True)
           for b in range(B)]
    t = compare_rows(ids, st, probs, orc, "slow")
    assert not t.mismatches, t.mismatches[:5]
    assert all(int(s) & FLAG_SLOW for s in st[:7])


def test_penalties_long_window_and_unaligned_rows():
    """Penalty windows with n_keep, duplicates and out-of-range ids; rows of
    an odd length, so most start off 16-byte boundaries (read as vectors at
    dword addresses; element loads: test_gpu_whole.py)."""
    rng = np.random.default_rng(5)
    B, V, H = 24, 30001, 3000
    x = rng.normal(0, 2, (B, V)).astype(np.float32)
    hist = rng.integers(-50, V + 50, (B, H)).astype(np.int32)
    hl = rng.integers(0, H + 1, B).astype(np.int32)
    prm = [RowParams(temperature=float(rng.choice([0.0, 0.6, 1.0])), top_k=int(rng.choice([0, 7])),
                     top_p=float(rng.choice([1.0, 0.8])), repetition_penalty=float(rng.choice([1.0, 1.3])),
                     presence_penalty=float(rng.choice([0.0, 0.4])),
                     frequency_penalty=float(rng.choice([0.0, 0.2])),
                     n_keep=int(rng.choice([0, 100, 2000]))) for _ in range(B)]
    u = rng.random(B)
    _say(f"[gpu] penalties B={B} V={V} H={H}")
    ids, st, probs = sample_host(x, prm, hist, hl, u, want_probs=True)
    lists = R.hist_rows_to_lists(hist, hl)
    orc = [R.sample_row(x[b], prm[b], lists[b], u[b], tie="spread", keep_probs=True)
           for b in range(B)]
    t = compare_rows(ids, st, probs, orc, "penalties")
    assert not t.mismatches, t.mismatches[:5]


def test_window_beyond_lds_limit_is_reported():
    rng = np.random.default_rng(6)
    B, V, H = 2, 5000, 5000
    x = rng.normal(0, 1, (B, V)).astype(np.float32)
    hist = rng.integers(0, V, (B, H)).astype(np.int32)
    prm = [RowParams(repetition_penalty=1.2), RowParams(repetition_penalty=1.2, n_keep=100)]
    _say("[gpu] window limit")
    ids, st, _ = sample_host(x, prm, hist, np.full(B, H, np.int32), np.full(B, 0.5))
    assert int(st[0]) & 0xFF == ROW_UNSUPPORTED       # 5000-id window
    assert int(st[1]) & 0xFF != ROW_UNSUPPORTED       # last max(64, 100) ids only


@pytest.mark.parametrize("freq", [0.0, 0.3])
def test_long_windows_on_a_long_vocabulary(freq):
    """4095-id windows (the longest the LDS index holds) at V=256000: the
    fused kernel's layout then needs shorter slices than the batch alone
    would pick; every row must still sample as the oracle does."""
    rng = np.random.default_rng(21)
    B, V, H = 256, 256000, 4095
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(2.0))
    x[np.arange(B), rng.integers(0, V, B)] += np.float32(8.0)
    hist = rng.integers(0, V, (B, H)).astype(np.int32)
    hist[:, : H // 2] = rng.integers(0, 5000, (B, H // 2))       # repeated ids too
    prm = [RowParams(temperature=float(rng.choice([0.0, 0.7, 1.0])),
                     top_k=int(rng.choice([0, 40])), top_p=float(rng.choice([1.0, 0.9])),
                     repetition_penalty=1.2, presence_penalty=0.4, frequency_penalty=freq)
           for _ in range(B)]
    w = W.SampleWorkload(f"long_window_f{freq}", x, "f32", prm, hist,
                         np.full(B, H, np.int32), rng.random(B))
    ids, st, _ = _run(w, False)
    t = _check(w, ids, st, None, w.name)
    assert t.boundary == 0
