"""Which batches give a row the same bits (turbo_lmhead_step in the header): batches of three to 256
rows over tables past 768 tiles and up to 128; in between, the batches on one side of 1024 products of
tiles and 32-row blocks."""
import numpy as np
import pytest

import synth
import test_gpu_batched_shapes as S
import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles,hidden,groups", [
    (1, 64, [[3, 32, 33, 64, 65, 256]]),
    (128, 448, [[3, 31, 64, 128, 129, 256]]),
    (129, 320, [[3, 32, 224], [225, 256]]),
    (256, 192, [[3, 32, 33, 128], [129, 200, 256]]),
    (501, 1600, [[3, 5, 32, 64], [65, 128, 129, 256]]),
    (768, 128, [[3, 32], [33, 64, 65, 256]]),
    (769, 320, [[3, 32, 33, 64, 65, 128, 129, 256]]),
    (3073, 192, [[3, 33, 64, 65, 256]]),
])
def test_same_bits_over_batches(tiles, hidden, groups):
    vocab = tiles * 64 - 1
    w, s, b = S.make_table(vocab, hidden, tiles)
    gamma = (1.0 + 0.02 * torch.randn(hidden, device="cuda")).bfloat16()
    torch.cuda.synchronize()
    h = T.LMHead(w, s, b, gamma, vocab=vocab, hidden=hidden, softcap=30.0, on_device=True)
    try:
        x = torch.from_numpy(synth.hidden_states(256, hidden, 5)).cuda()
        rows = [T.row_default() for _ in range(256)]
        for group in groups:
            first = None
            for batch in group:
                lo = torch.full((batch, vocab), float("nan"), device="cuda")
                tok = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
                inp, keep = h.make_inputs(batch, rows[:batch], hidden=x)
                torch.cuda.synchronize()
                h.step(inp, tok, lo)
                h.sync()
                got = lo[:3].cpu().numpy().view(np.uint32)
                first = got if first is None else first
                assert np.array_equal(got, first), (batch, int((got != first).sum()))
    finally:
        h.close()
