"""Steps of one and two rows over tables of few tiles: the folded preparation (RMSNorm, history counts)
against the prepared one (hidden rows off by four bytes), bit for bit, on both sides of each line of
tiles per workgroup; logits against the oracle's modifiers on the raw logits; the greedy entry."""
import numpy as np
import pytest

import orc_py as O
import synth
import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,hidden", [(1, 64), (64, 64), (65, 128), (4099, 1600), (768 * 64, 192), (768 * 64 + 1, 192),
                                          (1024 * 64, 64), (1025 * 64, 64), (1536 * 64 + 1, 128), (2047 * 64, 64)])
def test_folded_step_matches_prepared(vocab, hidden):
    W, S, B, g = synth.make_head(vocab, hidden, vocab)
    h = T.LMHead(W, S, B, g, vocab=vocab, hidden=hidden)
    try:
        for batch in (1, 2):
            x = torch.from_numpy(synth.hidden_states(batch, hidden, vocab + 1)).cuda()
            buf = torch.zeros(batch * hidden + 1, device="cuda")
            buf[1:] = x.reshape(-1)
            nh = 700
            hists = np.stack([synth.zipf_ids(nh, vocab + 3, 1.1, 5 + b) for b in range(batch)]).astype(np.uint32)
            lens = np.array([nh, 33][:batch], np.int32)
            rows = [T.row_default(temperature=0.0, repetition_penalty=1.3, presence_penalty=0.2, frequency_penalty=0.1)
                    for _ in range(batch)]
            hd, ld = torch.from_numpy(hists.view(np.int32)).cuda(), torch.from_numpy(lens).cuda()
            got = []
            for src in (x, buf[1:], x):
                inp, keep = h.make_inputs(batch, rows, hidden=src, history=hd, history_len=ld)
                tok = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
                lo = torch.full((batch, vocab), float("nan"), device="cuda")
                torch.cuda.synchronize()
                h.step(inp, tok, lo)
                h.sync()
                got.append((tok.cpu().numpy(), lo.cpu().numpy()))
            xn = torch.empty((batch, hidden), device="cuda")
            raw = torch.empty((batch, vocab), device="cuda")
            t2 = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            h.rms_norm(x, batch, xn)
            h.logits(xn, batch, raw)
            h.greedy(xn, batch, t2)
            h.sync()
            raw, t2 = raw.cpu().numpy(), t2.cpu().numpy()
            for b in range(batch):
                p = O.params(repetition_penalty=1.3, presence_penalty=0.2, frequency_penalty=0.1)
                want = O.apply_modifiers(raw[b], p, 30.0, history=hists[b][:lens[b]])
                for tok, lo in got:
                    assert np.array_equal(lo[b].view(np.uint32), want.view(np.uint32)), (batch, b)
                    assert tok[b] == int(np.argmax(want))
                assert t2[b] == int(np.argmax(raw[b]))
    finally:
        h.close()
