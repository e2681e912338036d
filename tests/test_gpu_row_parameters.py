"""turbo_sample_logits without modifiers, where the logits pass itself carries the row parameters to
device memory: many rows over one and over several workgroups each, every row with parameters of its
own, call after call with others."""
import numpy as np
import pytest

import orc_py as O
import parity_util as P
import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,batch", [(300, 256), (1024, 9), (1025, 200), (4100, 64), (32004, 17), (1, 256), (5000, 1), (5000, 8)])
def test_every_row_keeps_its_own_parameters(vocab, batch):
    z = torch.zeros((vocab, 32), dtype=torch.uint8, device="cuda")
    s = torch.zeros((vocab, 1), dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    h = T.LMHead(z, s, s, None, vocab=vocab, hidden=64, softcap=30.0, on_device=True)
    try:
        g = np.random.default_rng(vocab)
        logits = (2.0 * g.standard_normal((batch, vocab))).astype(np.float32)
        lt = torch.from_numpy(logits).cuda()
        for call in range(20):  # more calls than the staging ring has slots
            rows = [T.row_default(temperature=0.0 if (b + call) % 5 == 0 else 0.5 + 0.05 * ((b + call) % 13),
                                  top_k=1 + (7 * b + call) % min(vocab, 200), top_p=0.5 + 0.5 * ((b + 3 * call) % 8) / 8,
                                  seed=b, counter=call) for b in range(batch)]
            inp, keep = h.make_inputs(batch, rows)
            tok = torch.full((batch,), -2, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            h.sample_logits(lt, inp, tok)
            h.sync()
            toks = tok.cpu().numpy()
            for b in range(batch):
                p = O.params(temperature=float(np.float32(rows[b].temperature)), top_p=float(rows[b].top_p), top_k=rows[b].top_k)
                P.draw_check(logits[b], p, T.row_uniform(rows[b]), int(toks[b]))
    finally:
        h.close()
