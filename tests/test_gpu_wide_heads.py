"""The 16-wave workgroup of the 64-column matrix-core head (33 to 64 rows over 3072 tiles or more) where
its last workgroup lies partly past the table: one and fifteen tiles in it, an even and an odd group
count, partial column blocks, and the modifier words it stages for tiles that are not there."""
import numpy as np
import pytest

import orc_py as O
import synth
import test_gpu_batched_shapes as S
import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [3073 * 64 - 5, 3087 * 64])
@pytest.mark.parametrize("in_dim", [128, 192, 320])
def test_last_workgroup_partly_past_the_table(rows, in_dim):
    S.check(rows, in_dim, [33, 48, 64], rows + in_dim)


@pytest.mark.parametrize("groups", [8, 9, 15, 16, 17])
def test_lines_of_the_wide_workgroup(groups):
    """Short rows take it from 2049 tiles and 48 rows on: both sides of the tiles, rows and groups."""
    S.check(2048 * 64, 64 * groups, [64], groups)
    S.check(2049 * 64 - 3, 64 * groups, [47, 48, 64], groups + 1)


@pytest.mark.parametrize("groups", [1, 7, 8, 9, 10, 11])
def test_short_rows_in_one_round(groups):
    """65 to 256 rows over tables of 512 workgroups and one more: few odd groups look two ahead there."""
    S.check(1024 * 64, 64 * groups, [129, 256], groups)
    S.check(2048 * 64 - 7, 64 * groups, [65, 128], groups + 1)
    S.check(2049 * 64, 64 * groups, [65], groups + 2)


@pytest.mark.parametrize("vocab", [3073 * 64 - 5, 3087 * 64])
@pytest.mark.parametrize("hidden,batch", [(128, 48), (192, 33)])
def test_modifiers_in_the_last_workgroup(vocab, hidden, batch):
    """Two steps with different histories: the raw logits with the oracle's modifiers, bit for bit."""
    w, s, b = S.make_table(vocab, hidden, vocab)
    h = T.LMHead(w, s, b, None, vocab=vocab, hidden=hidden, softcap=30.0, on_device=True)
    try:
        x = torch.from_numpy(synth.hidden_states(batch, hidden, 3)).cuda()
        raw = torch.empty((batch, vocab), device="cuda")
        torch.cuda.synchronize()
        h.logits(x, batch, raw)
        h.sync()
        raw = raw.cpu().numpy()
        nh, nb, edge = 400, 30, vocab - 700  # half the ids in the last tiles
        bans = np.zeros((batch, (vocab + 31) // 32), np.uint32)
        bans[::2, -20:] = 0x10010010
        bids = np.stack([np.where(np.arange(nb) % 2, edge + synth.uniform_ids(nb, 700, 7 + r), synth.uniform_ids(nb, vocab, 9 + r))
                         for r in range(batch)]).astype(np.uint32)
        bvals = np.linspace(-3, 3, batch * nb, dtype=np.float32).reshape(batch, nb)
        rows = [T.row_default(repetition_penalty=1.2 if r % 2 else 1.0, presence_penalty=0.3 * (r % 3), frequency_penalty=0.1 * (r % 4))
                for r in range(batch)]
        for step in range(2):
            hists = np.stack([np.where(np.arange(nh) % 2, edge + synth.uniform_ids(nh, 700, 11 * step + r),
                                       synth.uniform_ids(nh, vocab, 13 + 5 * step + r)) for r in range(batch)]).astype(np.uint32)
            hd, bi = torch.from_numpy(hists.view(np.int32)).cuda(), torch.from_numpy(bids.view(np.int32)).cuda()
            bv, bn = torch.from_numpy(bvals).cuda(), torch.from_numpy(bans.view(np.int32)).cuda()
            hl = torch.full((batch,), nh, dtype=torch.int32, device="cuda")
            bc = torch.full((batch,), nb, dtype=torch.int32, device="cuda")
            inp, keep = h.make_inputs(batch, rows, hidden=x, flags=T.TURBO_STEP_NORMED, history=hd, history_len=hl, ban=bn,
                                      bias_ids=bi, bias_values=bv, bias_count=bc)
            tok = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
            lo = torch.full((batch + 1, vocab), 7.0, device="cuda")
            torch.cuda.synchronize()
            h.step(inp, tok, lo)
            h.sync()
            got, toks = lo.cpu().numpy(), tok.cpu().numpy()
            for r in range(batch):
                p = O.params(repetition_penalty=rows[r].repetition_penalty, presence_penalty=rows[r].presence_penalty,
                             frequency_penalty=rows[r].frequency_penalty)
                want = O.apply_modifiers(raw[r], p, 30.0, history=hists[r], bias_ids=bids[r], bias_values=bvals[r], ban=bans[r])
                assert np.array_equal(got[r].view(np.uint32), want.view(np.uint32)), (step, r)
                assert toks[r] == int(np.argmax(want))
            assert np.all(got[batch] == 7.0)  # the row past the batch is untouched
    finally:
        h.close()
