"""Sampled rows over vocabularies that the shortlist holds whole (at most 256 ids): with the shortlist
limit at, below and above the vocabulary, lifted (top_k 0) with and without the full-vocabulary flag,
alone in a step and beside a row with a shorter list, through the step and the sampler entry. Every
token must pass the oracle's interval check, and a row's token must not depend on the rows beside it."""
import numpy as np
import pytest

import orc_py as O
import parity_util as P
import synth
import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def row_kinds(vocab):
    flag = T.TURBO_ROW_FULL_VOCAB
    return [dict(top_k=0, top_p=0.9, flags=flag), dict(top_k=0, top_p=1.0, flags=flag), dict(top_k=0, top_p=1.0),
            dict(top_k=min(vocab, 256), top_p=0.8), dict(top_k=256, top_p=0.95), dict(top_k=max(1, vocab // 2), top_p=1.0)]


@pytest.mark.parametrize("entry", ["step", "sample"])
@pytest.mark.parametrize("vocab", [1, 2, 64, 65, 255, 256])
def test_sampled_rows_of_a_vocabulary_within_the_shortlist(vocab, entry):
    hidden, cap = 128, 30.0
    W, S, B, g = synth.make_head(vocab, hidden, vocab)
    h = T.LMHead(W, S, B, g, vocab=vocab, hidden=hidden, softcap=cap)
    kinds = row_kinds(vocab)
    us = (np.arange(len(kinds)) * 0.37 % 1.0 + 0.01).astype(np.float32)
    x = synth.hidden_states(len(kinds), hidden, 7 + vocab)
    given = (synth.normal(vocab + 3, 5, len(kinds) * vocab).reshape(len(kinds), vocab) * 3).astype(np.float32)

    def call(which):
        n = len(which)
        rows = [T.row_default(temperature=0.7 + 0.1 * i, **kinds[i]) for i in which]
        tok = torch.full((n,), -2, dtype=torch.int32, device="cuda")
        dev_rep = torch.zeros((n, T.C.sizeof(T.TurboRowReport)), dtype=torch.uint8, device="cuda")
        u = torch.from_numpy(us[which]).cuda()
        if entry == "step":
            hd = torch.from_numpy(x[which]).cuda()
            lo = torch.empty((n, vocab), device="cuda")
            inp, keep = h.make_inputs(n, rows, hidden=hd, uniforms=u)
            torch.cuda.synchronize()
            h.step(inp, tok, lo, dev_rep)
        else:
            lo = torch.from_numpy(given[which]).cuda()
            inp, keep = h.make_inputs(n, rows, uniforms=u)
            torch.cuda.synchronize()
            h.sample_logits(lo, inp, tok, dev_rep)
        h.sync()
        rep = (T.TurboRowReport * n).from_buffer_copy(dev_rep.cpu().numpy().tobytes())
        toks, lo = tok.cpu().numpy(), lo.cpu().numpy()
        for k, i in enumerate(which):
            # the whole vocabulary is the shortlist, whichever way the row asks for it
            limit = min(kinds[i]["top_k"], vocab) or vocab
            p = O.params(temperature=float(np.float32(0.7 + 0.1 * i)), top_p=kinds[i]["top_p"], top_k=limit)
            assert 0 <= toks[k] < vocab, (i, toks[k])
            P.draw_check(lo[k], p, float(us[i]), int(toks[k]))
            assert rep[k].path == 1, (i, rep[k].path)
        return lo, toks

    try:
        alone = [call([i]) for i in range(len(kinds))]
        call(list(range(5)))                          # five rows, none with a shorter list
        together, toks = call(list(range(len(kinds))))  # and beside one
        if entry == "sample":  # the same logits: the same tokens
            assert [int(t[0]) for _, t in alone] == [int(t) for t in toks]
    finally:
        h.close()
