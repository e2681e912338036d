"""turbo_sample_logits's modifier pass over caller logits: vocabularies around its tiles, 16-byte and
scalar rows (odd vocabularies, a base address off by one float), every modifier, ban bits past the
vocabulary, rows without any change. Logits must equal the oracle's modifiers bit for bit, greedy
tokens its argmax."""
import numpy as np
import pytest

import orc_py as O
import synth
import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("vocab,shift", [(1, 0), (3, 0), (63, 0), (64, 0), (66, 0), (1023, 0), (1024, 0), (1024, 1),
                                         (1028, 0), (4099, 0), (32004, 0), (32004, 3)])
def test_modifiers_on_given_logits(vocab, shift):
    bn = 9  # above the rows that ride in the kernel arguments
    base = (synth.normal(vocab + 5, 81, bn * vocab).reshape(bn, vocab) * 6).astype(np.float32)
    base[3] = np.round(base[3])  # repeats of the maximum
    z = torch.zeros((vocab, 32), dtype=torch.uint8, device="cuda")
    s = torch.zeros((vocab, 1), dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    h = T.LMHead(z, s, s, None, vocab=vocab, hidden=64, softcap=30.0, on_device=True)
    try:
        nh, nb = 200, 20
        hists = np.stack([synth.uniform_ids(nh, vocab + 9, vocab + b) for b in range(bn)]).astype(np.uint32)
        lens = np.array([nh, 0, 17, nh, 1, nh, 64, 3, 100], np.int32)
        bids = np.stack([synth.uniform_ids(nb, vocab, 7 + b) for b in range(bn)]).astype(np.uint32)
        bvals = np.linspace(-3, 3, bn * nb, dtype=np.float32).reshape(bn, nb)
        bans = np.zeros((bn, (vocab + 31) // 32), np.uint32)
        if vocab > 2:
            bans[::2, :] = 0x01010101
        if vocab % 32:
            bans[:, -1] |= np.uint32((0xFFFFFFFF << (vocab % 32)) & 0xFFFFFFFF)  # past the vocabulary
        rows = [T.row_default(repetition_penalty=1.2 if b % 2 else 1.0, presence_penalty=0.3 * (b % 3),
                              frequency_penalty=0.1 * (b % 4)) for b in range(bn)]
        buf = torch.zeros(bn * vocab + shift, dtype=torch.float32, device="cuda")
        lt = buf[shift:].view(bn, vocab)
        for kind in ("none", "ban", "history", "all", "all"):
            lt.copy_(dev(base))
            kw = {}
            if kind in ("ban", "all"):
                kw.update(ban=dev(bans.view(np.int32)))
            if kind in ("history", "all"):
                kw.update(history=dev(hists.view(np.int32)), history_len=dev(lens))
            if kind == "all":
                kw.update(bias_ids=dev(bids.view(np.int32)), bias_values=dev(bvals),
                          bias_count=torch.full((bn,), nb, dtype=torch.int32, device="cuda"))
            inp, keep = h.make_inputs(bn, rows, **kw)
            tok = torch.full((bn,), -1, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            h.sample_logits(lt, inp, tok)
            h.sync()
            got, toks = lt.cpu().numpy(), tok.cpu().numpy()
            for b in range(bn):
                p = O.params(repetition_penalty=rows[b].repetition_penalty, presence_penalty=rows[b].presence_penalty,
                             frequency_penalty=rows[b].frequency_penalty)
                m = {}
                if "history" in kw:
                    m.update(history=hists[b][:lens[b]])
                if "bias_ids" in kw:
                    m.update(bias_ids=bids[b], bias_values=bvals[b])
                if "ban" in kw:
                    m.update(ban=bans[b])
                want = O.apply_modifiers(base[b], p, 30.0, **m)
                assert np.array_equal(got[b], want), (kind, b)
                assert toks[b] == int(np.argmax(want)), (kind, b)
    finally:
        h.close()
