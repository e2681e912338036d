"""More full-vocabulary rows in a step than the slices serve (one workgroup each): rows matched on byte
codes kept from the first pass, and every way out of the match into the second pass. Vocabularies on
both sides of the coded range (32,768 .. 262,144 ids, a multiple of four, 16-byte rows), that fill the
codes' turns of 65,536 ids and that do not; rows built for each branch, with the branch's condition
checked on a numpy model of the plan. Every token must pass the oracle's interval check."""
import numpy as np
import pytest

import orc_py as O
import parity_util as P
import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

NB = 66  # above the 64 rows that the slices serve
F32 = np.float32


def plan(l, temp, top_p, u):
    """(nucleus bin, first and last bin of the draw, bins of all elements): the plan over 2048 value bins."""
    m = l.max()
    lo = max(l[np.isfinite(l)].min(), m - F32(48) * max(F32(1), F32(temp)))
    inv = F32(2048) / (m - lo)
    with np.errstate(invalid="ignore"):
        d = (m - l) * inv
        bins = np.where(d < 2047, d, 2047).astype(np.int64)
    w1 = np.bincount(bins, np.exp(l.astype(np.float64) - m), 2048)
    wt = np.bincount(bins, np.exp((l.astype(np.float64) - m) / temp), 2048)
    cb = 2048
    if top_p < 1.0:
        cb = int(np.searchsorted(np.cumsum(w1), top_p * w1.sum()))
    A = wt[:cb].sum()
    B = wt[cb] if cb < 2048 else 0.0
    c = np.cumsum(wt[:min(cb + 1, 2048)])
    dlo, dhi = (min(int(np.searchsorted(c, u * t)), c.size - 1) for t in (A, A + B))
    return cb, dlo, dhi, bins


def spread_row(g, vocab, n, first, last, u, ties=0):
    """n values over bins first .. last of a range of two units, a cluster of equal values near the end of
    the range that holds the nucleus bound, the rest banned: (row, top_p, u)."""
    l = np.full(vocab, -np.inf, F32)
    ids = g.permutation(vocab)
    l[ids[0]], l[ids[1]] = 0.0, -2.0
    l[ids[2:n + 2]] = -2.0 * (first + (last - first) * g.random(n)) / 2048.0
    w = np.exp(l[ids[:n + 2]].astype(np.float64)).sum()
    k = ties or max(1, int(0.4 * w / np.exp(-1.9)))
    l[ids[n + 2:n + 2 + k]] = -1.9
    c = k * np.exp(F32(-1.9).astype(np.float64))
    return l, float(F32((w + 0.5 * c) / (w + c))), u


def make_rows(vocab, seed):
    g = np.random.default_rng(seed)
    L, params, us, seen = [], [], [], dict.fromkeys(["border", "wide", "many", "top", "tail"], 0)
    for b in range(NB):
        kind, temp, top_p, u = b % 8, 1.0, 0.9, float(F32(g.random()))
        if kind == 0:    # nearly all the weight on one id: the draw is in bin 0
            l = g.standard_normal(vocab).astype(F32)
            l[g.integers(vocab)] = 25.0
            temp = 0.8
        elif kind == 1:  # a row as a head gives it
            l = (3.0 * g.standard_normal(vocab)).astype(F32)
            temp, top_p = 0.9, 0.95
        elif kind == 2:  # the draw's bins lie on both sides of bin 512
            l, top_p, u = spread_row(g, vocab, 2000, 420, 600, 0.45)
        elif kind == 3:  # more than 128 pairs of bins
            l, top_p, u = spread_row(g, vocab, 6000, 10, 1800, 0.5)
        elif kind == 4:  # more matches than the list holds, within a few bins
            l, top_p, u = spread_row(g, vocab, 14000, 700, 702, 0.5, ties=3000)
        elif kind == 5:  # no nucleus, the draw near the end of the row's weight
            l = (2.0 * g.standard_normal(vocab)).astype(F32)
            top_p, u, temp = 1.0, 0.9999, 1.2
        elif kind == 6:  # one value everywhere
            l = np.full(vocab, 1.5, F32)
        else:            # the nucleus ends in the bin of the maximum
            l = g.standard_normal(vocab).astype(F32)
            l[g.integers(vocab, size=3)] = [12.0, 11.9999, 11.0]
            top_p = 0.3
        if kind in (2, 3, 4, 5, 0):
            cb, dlo, dhi, bins = plan(l, temp, top_p, u)
            pairs = (dhi >> 1) - (dlo >> 1) + 1
            inside = int(((bins >> 1 >= dlo >> 1) & (bins >> 1 <= dhi >> 1)).sum())
            seen["border"] += kind == 2 and dlo >> 9 != dhi >> 9 and pairs <= 128 and inside <= 8192
            seen["wide"] += kind == 3 and pairs > 128
            seen["many"] += kind == 4 and pairs <= 128 and inside > 8192
            seen["top"] += kind == 0 and dlo == 0
            seen["tail"] += kind == 5 and cb == 2048
        L.append(l)
        params.append((temp, top_p))
        us.append(u)
    assert all(seen.values()), seen
    return np.stack(L), params, np.array(us, F32)


@pytest.mark.parametrize("vocab,shift", [(32764, 0), (32768, 0), (49152, 0), (65536, 0), (65540, 0), (131068, 0), (151936, 0),
                                         (262144, 0), (262148, 0), (32769, 0), (65537, 0), (65536, 1)])
def test_rows_of_one_workgroup_each(vocab, shift):
    z = torch.zeros((vocab, 32), dtype=torch.uint8, device="cuda")
    s = torch.zeros((vocab, 1), dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    h = T.LMHead(z, s, s, None, vocab=vocab, hidden=64, softcap=30.0, on_device=True)
    try:
        logits, params, us = make_rows(vocab, vocab + shift)
        rows = [T.row_default(temperature=t, top_k=0, top_p=p, flags=T.TURBO_ROW_FULL_VOCAB) for t, p in params]
        buf = torch.zeros(NB * vocab + shift, device="cuda")
        lt = buf[shift:].view(NB, vocab)  # off a 16-byte line with shift 1
        lt.copy_(torch.from_numpy(logits))
        ut = torch.from_numpy(us).cuda()  # the call reads its address
        inp, keep = h.make_inputs(NB, rows, uniforms=ut)
        tok = torch.full((NB,), -2, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        h.sample_logits(lt, inp, tok)
        h.sync()
        toks = tok.cpu().numpy()
        assert np.array_equal(lt.cpu().numpy(), logits)
        for b in range(NB):
            p = O.params(temperature=float(F32(params[b][0])), top_p=params[b][1], top_k=0, flags=T.TURBO_ROW_FULL_VOCAB)
            P.draw_check(logits[b], p, float(us[b]), int(toks[b]))
    finally:
        h.close()
