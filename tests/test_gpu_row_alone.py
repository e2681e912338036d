"""A row's logits must not depend on the row beside it: steps and logits of one and of two rows give the
same bits over every table size that changes kernels (few tiles, wave pairs, the folded head), for group
counts with whole and partial units of four chunks and for one to sixteen ranges of them."""
import numpy as np
import pytest

import synth
import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,hidden", [(500, 1600), (1024 * 64, 320), (1025 * 64, 64), (1025 * 64 - 3, 128), (1026 * 64, 320),
                                          (1100 * 64, 448), (1536 * 64 + 1, 1152), (1030 * 64, 2816), (1027 * 64, 8192),
                                          (2047 * 64, 192), (2048 * 64, 192)])
def test_one_row_equals_the_same_row_beside_another(vocab, hidden):
    g = torch.Generator(device="cuda")
    g.manual_seed(vocab + hidden)
    w = torch.randint(0, 256, (vocab, hidden // 2), generator=g, device="cuda", dtype=torch.uint8)
    s = (torch.randn((vocab, hidden // 64), generator=g, device="cuda").abs() * 0.004).bfloat16()
    b = (-8.0 * s.float() + 1e-3).bfloat16()
    gamma = (1.0 + 0.02 * torch.randn(hidden, generator=g, device="cuda")).bfloat16()
    torch.cuda.synchronize()
    h = T.LMHead(w, s, b, gamma, vocab=vocab, hidden=hidden, on_device=True)
    try:
        x = torch.from_numpy(synth.hidden_states(2, hidden, 5)).cuda()
        nh = 300
        hist = torch.randint(0, vocab, (2, nh), generator=g, device="cuda", dtype=torch.int32)
        lens = torch.full((2,), nh, dtype=torch.int32, device="cuda")
        rows = [T.row_default(temperature=0.0, repetition_penalty=1.2, frequency_penalty=0.1) for _ in range(2)]

        def step(first, n):
            lo = torch.full((n, vocab), float("nan"), device="cuda")
            tok = torch.full((n,), -1, dtype=torch.int32, device="cuda")
            inp, keep = h.make_inputs(n, rows[:n], hidden=x[first:], history=hist[first:], history_len=lens[first:])
            torch.cuda.synchronize()
            h.step(inp, tok, lo)
            h.sync()
            return lo.cpu().numpy().view(np.uint32), tok.cpu().numpy()

        def logits(first, n):
            lo = torch.full((n, vocab), float("nan"), device="cuda")
            tok = torch.full((n,), -1, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            h.logits(x[first:], n, lo)
            h.greedy(x[first:], n, tok)
            h.sync()
            return lo.cpu().numpy().view(np.uint32), tok.cpu().numpy()

        for call in (step, logits):
            both, toks = call(0, 2)
            for r in range(2):
                one, tok = call(r, 1)
                assert np.array_equal(one[0], both[r]), (call.__name__, r, int((one[0] != both[r]).sum()))
                assert tok[0] == toks[r]
    finally:
        h.close()
