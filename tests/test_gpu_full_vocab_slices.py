"""Full-vocabulary rows beside shortlist and greedy rows in one step, over the slice counts that the
number of such rows and of other rows give (one row, a mix, only such rows, more than the slices
serve), with u = 0, banned and degenerate rows, and repeated calls (the histogram sums must come
back to zero). Every token's interval of the cumulative weights is checked in 64 bits."""
import numpy as np
import pytest

import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,batch,every", [(257, 3, 1), (4099, 1, 1), (32003, 9, 2), (32003, 40, 40),
                                               (8192, 64, 1), (8192, 70, 1), (5000, 256, 8), (65537, 5, 3)])
def test_full_vocab_rows_by_slices(vocab, batch, every):
    g = np.random.default_rng(vocab + batch)
    w = torch.zeros((vocab, 32), dtype=torch.uint8, device="cuda")
    s = torch.zeros((vocab, 1), dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    h = T.LMHead(w, s, s, None, vocab=vocab, hidden=64, softcap=30.0, on_device=True)
    try:
        logits = (g.standard_normal((batch, vocab)) * 3.0).astype(np.float32)
        logits[0, vocab // 2:] = -np.inf
        dead = batch // 2 if batch > 4 else None
        if dead is not None:
            logits[dead] = -np.inf
        us = g.random(batch).astype(np.float32)
        us[0] = 0.0 if batch > 1 else us[0]
        rows = []
        for b in range(batch):
            full = b % every == 0
            rows.append(T.row_default(temperature=0.0 if (not full and b % 3 == 0) else 0.9 + 0.05 * (b % 5),
                                      top_k=0 if full else 20, top_p=0.9 if b % 2 else 1.0,
                                      flags=T.TURBO_ROW_FULL_VOCAB if full else 0))
        lt, ut = torch.from_numpy(logits).cuda(), torch.from_numpy(us).cuda()
        inp, keep = h.make_inputs(batch, rows, uniforms=ut)
        tok = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
        first = None
        for _ in range(3):
            h.sample_logits(lt, inp, tok)
            h.sync()
            got = tok.cpu().numpy().copy()
            if first is None:
                first = got
            assert np.array_equal(got, first)
        assert np.array_equal(lt.cpu().numpy(), logits)
        for b in range(batch):
            if b == dead:
                assert np.uint32(first[b]) == 0xFFFFFFFF
                continue
            r = rows[b]
            if r.temperature <= 0.0:
                assert first[b] == int(np.argmax(logits[b]))
                continue
            if us[b] == 0.0:
                assert first[b] == int(np.argmax(logits[b]))
                continue
            order = np.lexsort((np.arange(vocab), -logits[b]))
            l = logits[b][order].astype(np.float64)
            keepn = vocab if r.top_k == 0 else min(r.top_k, vocab)
            p = np.exp(l - l[0])
            cum = np.cumsum(p) / p.sum()
            cut = keepn
            if r.top_p < 1.0:
                cut = min(keepn, int(np.searchsorted(cum[:keepn], r.top_p)) + 1)
            q = np.exp((l[:cut] - l[0]) / np.float32(r.temperature))
            c = np.cumsum(q)
            # weights relative to 3e-7 (fp32 exponent argument and hardware exp2): the interval of
            # the token, widened by that share of the total on each side
            i = int(np.where(order == first[b])[0][0])
            eps = 1e-6 * c[-1]
            target = float(us[b]) * c[-1]
            lo = c[i - 1] if i else 0.0
            hi = c[min(i, cut - 1)]
            assert i <= cut and lo - eps <= target <= hi + eps, (b, i, cut, lo, target, hi)
    finally:
        h.close()
