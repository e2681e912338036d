"""The work a program asks of this library, as cases that can be timed and compared.

A case is a dict of plain values. `prepare` builds what the caller holds before the call (handles
with their weights, device buffers, sampling rows), `run` makes one pass through the public entry
points of turbo_decode_tail, `exact` gives the same outputs from plain torch in 64 bits.

Kinds
  step     turbo_lmhead_step: final RMSNorm, int4 head, softcap, modifiers, token per row
  logits   turbo_lmhead_logits: the head over already normalised rows (verification of drafted
           tokens, scoring)
  sample   turbo_sample_logits: the sampler over logits the caller computed itself
  matvec   turbo_int4_matvec: one projection of the layer loop
  experts  turbo_int4_matvec_grouped twice: one token's routed experts, gate + up, then down
  refill   turbo_int4_matrix_load of an expert slot's three matrices, then their products
  embed    turbo_lmhead_embed: embedding rows of a prompt or of one decoded token

Shapes are those of the benchmark and the tests (262,144 x 2,816 tied table, 704 / 2,112 / 4,096
projections); the ragged ones are generic.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "turbo-winfare_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import turbo_decode_tail as T  # noqa: E402

V, D = 262144, 2816
CAP, EPS = 30.0, 1e-6
# Sequences whose decode steps take turns over one handle; each pass appends one token to one of
# them, so histories stay close to their starting length however often a state is run.
SEQUENCES = 64
HISTORY_ROOM = 512
EXPERTS, ROUTED = 64, 8


# ---- the cases ---------------------------------------------------------------------------------

def _step(name, **kw):
    c = {"name": name, "kind": "step", "vocab": V, "hidden": D, "batch": 1, "dtype": "f32", "normed": False,
         "sampling": "topk", "top_k": 64, "top_p": 0.95, "temperature": 0.8, "history": 0, "zipf": False,
         "repetition": 1.0, "presence": 0.0, "frequency": 0.0, "ban": 0.0, "bias": 0}
    c.update(kw)
    if name is None:
        del c["name"]
    return c


def listed():
    return [
        # one expert projection on its own: a few microseconds of launch and round trip
        {"name": "matvec_704x2816", "kind": "matvec", "rows": 704, "in_dim": 2816, "batch": 1, "dtype": "f32"},
        # the embedding rows of a 256-token prompt chunk
        {"name": "embed_256", "kind": "embed", "vocab": V, "hidden": D, "tokens": 256},
        # an expert streamed into its slot: three repacks, then its products
        {"name": "expert_refill", "kind": "refill", "inner": 704, "hidden": 2816},
        # the 8 routed experts of one decoded token (16 gate/up products, 8 down products)
        {"name": "experts_8_of_64", "kind": "experts", "inner": 704, "hidden": 2816},
        # a small model's ragged head: odd vocabulary, odd group count, a handful of sequences
        _step("ragged_b5", vocab=32003, hidden=1600, batch=5, sampling="mixed", history=300, repetition=1.1),
        # greedy decoding of one sequence
        _step("greedy_b1", sampling="greedy", top_k=0, top_p=1.0, temperature=0.0),
        # sampled decoding of one sequence, the interactive default
        _step("sampled_b1", history=256, repetition=1.1),
        # scoring eight drafted tokens at once
        {"name": "logits_b8", "kind": "logits", "vocab": V, "hidden": D, "batch": 8, "dtype": "bf16", "softcap": True},
        # a caller with its own head: the sampler alone, under a grammar's ban mask
        {"name": "sample_b16", "kind": "sample", "vocab": V, "batch": 16, "sampling": "mixed", "top_k": 50,
         "top_p": 0.9, "temperature": 0.9, "ban": 0.3},
        # a server's batch of users, each with their own parameters and penalties
        _step("mixed_b32", batch=32, sampling="mixed", history=1024, zipf=True, presence=0.5, frequency=0.3),
        # constrained decoding: ban mask, logit bias and repetition on every row
        _step("constrained_b64", batch=64, top_k=40, top_p=0.9, temperature=0.7, history=2048, repetition=1.15,
              ban=0.05, bias=300),
        # bulk generation: the largest batch, nucleus over the whole vocabulary, 16-bit hidden states
        _step("fullvocab_b256", batch=256, dtype="bf16", normed=True, sampling="full", top_k=0, top_p=0.9,
              temperature=1.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: batches 1 .. 256, vocabularies up to the largest (odd ones
    among them), projections 64 .. 16,384 rows, every sampling mode and modifier."""
    kind = rng.choices(["step", "logits", "sample", "matvec", "experts", "refill", "embed"],
                       [44, 14, 10, 12, 8, 5, 7])[0]
    dtype = rng.choice(["f32", "bf16"])
    if kind == "matvec":
        return {"kind": kind, "rows": _log(rng, 64, 16384), "in_dim": 64 * _log(rng, 4, 128),
                "batch": rng.choice([1, 1, 1, 2, _log(rng, 3, 64)]), "dtype": dtype}
    if kind in ("experts", "refill"):
        return {"kind": kind, "inner": 64 * rng.randint(4, 24), "hidden": 64 * rng.randint(12, 48)}
    full = rng.random() < 0.5
    vocab = V if full else _log(rng, 4099, V)
    hidden = 64 * rng.randint(8, 44 if vocab > V // 2 else 88)
    if kind == "embed":
        return {"kind": kind, "vocab": vocab, "hidden": hidden, "tokens": _log(rng, 1, 4096)}
    if kind == "logits":
        return {"kind": kind, "vocab": vocab, "hidden": hidden, "batch": _log(rng, 1, 128), "dtype": dtype,
                "softcap": rng.random() < 0.75}
    sampling = rng.choices(["greedy", "topk", "mixed", "full"], [15, 40, 30, 15])[0]
    top_k = _log(rng, 1, 256) if sampling in ("topk", "mixed") else 0
    top_p = round(rng.uniform(0.6, 1.0), 3) if sampling != "greedy" else 1.0
    temp = round(rng.uniform(0.4, 1.5), 3) if sampling != "greedy" else 0.0
    ban = round(rng.choice([0.0, 0.0, rng.uniform(0.01, 0.6)]), 3)
    if kind == "sample":
        return {"kind": kind, "vocab": vocab, "batch": _log(rng, 1, 64), "sampling": sampling, "top_k": top_k,
                "top_p": top_p, "temperature": temp, "ban": ban}
    hist = rng.choice([0, _log(rng, 16, 3000), _log(rng, 16, 3000)])
    c = _step(None, vocab=vocab, hidden=hidden, batch=_log(rng, 1, 256), dtype=dtype, normed=rng.random() < 0.3,
              sampling=sampling, top_k=top_k, top_p=top_p, temperature=temp, history=hist, zipf=rng.random() < 0.5,
              ban=ban, bias=rng.choice([0, 0, _log(rng, 1, 1000)]))
    if hist:
        c["repetition"] = rng.choice([1.0, 1.1, 1.3])
        c["presence"] = rng.choice([0.0, 0.5])
        c["frequency"] = 0.25 if c["repetition"] == 1.0 and c["presence"] == 0.0 else 0.0
    return c


# ---- inputs, from the seed alone -----------------------------------------------------------------

def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + what) & 0x7FFFFFFFFFFFFFFF)
    return g


def _randn(shape, g):
    return torch.randn(shape, generator=g, device="cuda")


def _randint(lo, hi, shape, g):
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int32)


def _table(rows, in_dim, g, gamma=False):
    """An affine-int4 table: uniform nibbles, positive scales around 0.004, biases close to -8 scales."""
    w = torch.randint(0, 256, (rows, in_dim // 2), generator=g, device="cuda", dtype=torch.uint8)
    s = (_randn((rows, in_dim // 64), g).abs() * 0.004).bfloat16()
    b = (-8.0 * s.float() + _randn(s.shape, g) * 1e-4).bfloat16()
    n = (1.0 + 0.02 * _randn((in_dim,), g)).bfloat16() if gamma else None
    return w, s, b, n


def _dequant(w, s, b, rows=None, dtype=torch.float64):
    """q * s + b of the given rows (all of them without)."""
    if rows is not None:
        w, s, b = w[rows], s[rows], b[rows]
    q = torch.stack((w & 15, w >> 4), dim=-1).reshape(w.shape[0], -1).to(dtype)
    q = q.reshape(w.shape[0], -1, 64) * s.to(dtype).unsqueeze(-1) + b.to(dtype).unsqueeze(-1)
    return q.reshape(w.shape[0], -1)


def _hidden(batch, table, g):
    """Hidden states that favour some tokens: noise plus a few vocabulary rows, so that a row's
    distribution has a handful of likely tokens over a broad background, from nearly flat to
    nearly decided."""
    w, s, b, _ = table
    rows, in_dim = w.shape[0], w.shape[1] * 2
    k = 24
    ids = _randint(0, rows, (batch * k,), g).long()
    top = 4.0 + 14.0 * torch.rand((batch, 1), generator=g, device="cuda")
    want = top * torch.rand((batch, k), generator=g, device="cuda").sort(dim=1, descending=True).values
    u = _dequant(w, s, b, ids, torch.float32)
    u = (u / u.norm(dim=1, keepdim=True)).reshape(batch, k, in_dim)
    x = _randn((batch, in_dim), g)
    return (x + (u * want.unsqueeze(-1)).sum(dim=1)).contiguous()


def _cast(x, dtype):
    return x.bfloat16().contiguous() if dtype == "bf16" else x.contiguous()


def _code(dtype):
    return T.TURBO_HIDDEN_BF16 if dtype == "bf16" else T.TURBO_HIDDEN_F32


def _rows(c, seed):
    """One sampling row per sequence; "mixed" batches differ per row, as users do."""
    out = []
    for b in range(c["batch"]):
        mode, k, p, t = c["sampling"], c["top_k"], c["top_p"], c["temperature"]
        if mode == "mixed":
            k = (0, max(1, k // 3), max(1, 2 * k // 3), k)[b % 4]
            p = p + (1.0 - p) * ((b * 7) % 16) / 16.0
            t = t * (0.6 + 0.1 * ((b * 5) % 9))
        out.append(T.row_default(temperature=t, top_k=k, top_p=p, seed=(seed + 77 * b) & 0x7FFFFFFF, counter=0,
                                 repetition_penalty=c.get("repetition", 1.0),
                                 presence_penalty=c.get("presence", 0.0), frequency_penalty=c.get("frequency", 0.0),
                                 flags=T.TURBO_ROW_FULL_VOCAB if k == 0 and mode != "greedy" else 0))
    return out


def _histories(c, g):
    """[SEQUENCES][batch][length + room] ids: uniform, or frequent ids repeating (Zipf-like)."""
    shape = (SEQUENCES, c["batch"], c["history"] + HISTORY_ROOM)
    if c["zipf"]:
        u = torch.rand(shape, generator=g, device="cuda")
        ids = torch.exp(u * math.log(c["vocab"])).to(torch.int32) - 1
        return ids.clamp_(0, c["vocab"] - 1)
    return _randint(0, c["vocab"], shape, g)


def _bans(c, g):
    """The mask as one bit per id, and as truth values."""
    vocab = c["vocab"]
    words = (vocab + 31) // 32
    bits = torch.rand((c["batch"], words * 32), generator=g, device="cuda") < c["ban"]
    shifts = torch.arange(32, device="cuda", dtype=torch.int64)
    packed = (bits.reshape(-1, words, 32).long() << shifts).sum(dim=-1)
    packed = torch.where(packed >= 2 ** 31, packed - 2 ** 32, packed).to(torch.int32)
    return packed.contiguous(), bits[:, :vocab]


def _biases(c, g):
    ids = _randint(0, c["vocab"], (c["batch"], c["bias"]), g)
    vals = torch.rand((c["batch"], c["bias"]), generator=g, device="cuda") * 10.0 - 5.0
    return ids.contiguous(), vals.contiguous()


def _given_logits(c, g):
    """Logits as a head gives them: a background and a few likely tokens per row."""
    l = _randn((c["batch"], c["vocab"]), g)
    ids = _randint(0, c["vocab"], (c["batch"], 24), g).long()
    top = 4.0 + 14.0 * torch.rand((c["batch"], 1), generator=g, device="cuda")
    return l.scatter_(1, ids, top * torch.rand(ids.shape, generator=g, device="cuda"))


def _head(table, vocab, hidden, softcap):
    torch.cuda.synchronize()  # the handle reads the arrays on a stream of its own
    return T.LMHead(table[0], table[1], table[2], table[3], vocab=vocab, hidden=hidden, softcap=softcap, eps=EPS,
                    on_device=True)


def _expert_tables(c, g):
    return [_table(c["inner"], c["hidden"], g), _table(c["inner"], c["hidden"], g), _table(c["hidden"], c["inner"], g)]


class State:
    """What the program holds: handles, buffers, and the number of passes so far."""

    def __init__(self, case):
        self.case, self.step = case, 0


def prepare(case, seed):
    c, st = case, State(case)
    kind = c["kind"]
    if kind == "step":
        table = _table(c["vocab"], c["hidden"], _gen(seed, 1), gamma=True)
        st.x = _cast(_hidden(c["batch"], table, _gen(seed, 2)), c["dtype"])
        st.head = _head(table, c["vocab"], c["hidden"], CAP)
        del table
        st.tokens = torch.zeros(c["batch"], dtype=torch.int32, device="cuda")
        st.logits = torch.zeros((c["batch"], c["vocab"]), device="cuda")
        kw, flags = {}, T.TURBO_STEP_NORMED if c["normed"] else 0
        if c["history"]:
            st.history = _histories(c, _gen(seed, 3))
            st.history_len = torch.full((SEQUENCES, c["batch"]), c["history"], dtype=torch.int32, device="cuda")
            kw.update(history=st.history[0], history_len=st.history_len[0])
            flags |= T.TURBO_STEP_APPEND_HISTORY
        if c["ban"]:
            st.ban, _ = _bans(c, _gen(seed, 4))
            kw.update(ban=st.ban)
        if c["bias"]:
            st.bias_ids, st.bias_vals = _biases(c, _gen(seed, 5))
            st.bias_count = torch.full((c["batch"],), c["bias"], dtype=torch.int32, device="cuda")
            kw.update(bias_ids=st.bias_ids, bias_values=st.bias_vals, bias_count=st.bias_count)
        st.inp, st.rows = st.head.make_inputs(c["batch"], _rows(c, seed), hidden=st.x, dtype=_code(c["dtype"]),
                                              flags=flags, **kw)
    elif kind == "logits":
        table = _table(c["vocab"], c["hidden"], _gen(seed, 1))
        x = _hidden(c["batch"], table, _gen(seed, 2))
        st.x = _cast(x * torch.rsqrt(x.square().mean(dim=1, keepdim=True)), c["dtype"])
        st.head = _head(table, c["vocab"], c["hidden"], CAP)
        st.out = torch.zeros((c["batch"], c["vocab"]), device="cuda")
    elif kind == "sample":
        st.head = _head(_table(c["vocab"], 64, _gen(seed, 1)), c["vocab"], 64, CAP)
        st.logits = _given_logits(c, _gen(seed, 2))
        st.tokens = torch.zeros(c["batch"], dtype=torch.int32, device="cuda")
        kw = {}
        if c["ban"]:
            st.ban, _ = _bans(c, _gen(seed, 4))
            kw.update(ban=st.ban)
        st.inp, st.rows = st.head.make_inputs(c["batch"], _rows(c, seed), **kw)
    elif kind == "matvec":
        st.head = _head(_table(c["rows"], c["in_dim"], _gen(seed, 1)), c["rows"], c["in_dim"], 0.0)
        st.x = _cast(_randn((c["batch"], c["in_dim"]), _gen(seed, 2)), c["dtype"])
        st.out = torch.zeros((c["batch"], c["rows"]), device="cuda")
    elif kind == "experts":
        g = _gen(seed, 1)
        st.experts = []
        for _ in range(EXPERTS):
            mats = []
            for t in _expert_tables(c, g):
                m = T.Int4Matrix(t[0].shape[0], t[0].shape[1] * 2)
                m.load_weights(t[0], t[1], t[2], on_device=True)
                mats.append(m)
            st.experts.append(mats)
        g = _gen(seed, 2)
        st.x = _randn((c["hidden"],), g)
        st.h = _randn((ROUTED, c["inner"]), g)
        st.gate_up = torch.zeros((2 * ROUTED, c["inner"]), device="cuda")
        st.down = torch.zeros((ROUTED, c["hidden"]), device="cuda")
        st.x_up, st.x_down = [st.x] * (2 * ROUTED), list(st.h)
        st.out_up, st.out_down = list(st.gate_up), list(st.down)
    elif kind == "refill":
        g = _gen(seed, 1)
        st.slots = [_expert_tables(c, g) for _ in range(4)]  # experts staged in device memory
        st.mats = [T.Int4Matrix(t[0].shape[0], t[0].shape[1] * 2) for t in st.slots[0]]
        g = _gen(seed, 2)
        st.x, st.h = _randn((c["hidden"],), g), _randn((c["inner"],), g)
        st.xs = [st.x, st.x, st.h]
        st.outs = [torch.zeros(t[0].shape[0], device="cuda") for t in st.slots[0]]
    else:
        st.head = _head(_table(c["vocab"], c["hidden"], _gen(seed, 1)), c["vocab"], c["hidden"], CAP)
        st.ids = _randint(0, c["vocab"], (c["tokens"],), _gen(seed, 2))
        st.out = torch.zeros((c["tokens"], c["hidden"]), device="cuda")
    torch.cuda.synchronize()
    return st


# ---- one pass --------------------------------------------------------------------------------------

def _routed(step):
    """The experts the router picks at this step."""
    return [(step * 5 + 8 * j + j * j) % EXPERTS for j in range(ROUTED)]


def run(st):
    c, kind = st.case, st.case["kind"]
    step = st.step
    st.step = step + 1
    if kind == "step":
        for r in st.rows:
            r.counter = step
        out = {"tokens": st.tokens, "logits": st.logits}
        if c["history"]:
            n = step % SEQUENCES
            st.inp.history = st.history.data_ptr() + n * st.history.stride(0) * 4
            st.inp.history_len = st.history_len.data_ptr() + n * st.history_len.stride(0) * 4
            out["history"], out["history_len"] = st.history, st.history_len
        st.head.step(st.inp, st.tokens, st.logits)
        return out
    if kind == "logits":
        st.head.logits(st.x, c["batch"], st.out, dtype=_code(c["dtype"]), softcap=c["softcap"])
        return st.out
    if kind == "sample":
        for r in st.rows:
            r.counter = step
        st.head.sample_logits(st.logits, st.inp, st.tokens)
        return {"tokens": st.tokens, "logits": st.logits}
    if kind == "matvec":
        st.head.matvec(st.x, c["batch"], st.out, dtype=_code(c["dtype"]))
        return st.out
    if kind == "experts":
        picked = [st.experts[e] for e in _routed(step)]
        T.matvec_grouped([m for e in picked for m in e[:2]], st.x_up, st.out_up)
        T.matvec_grouped([e[2] for e in picked], st.x_down, st.out_down)
        return {"gate_up": st.gate_up, "down": st.down}
    if kind == "refill":
        for m, t in zip(st.mats, st.slots[step % len(st.slots)]):
            m.load_weights(t[0], t[1], t[2], on_device=True)
        T.matvec_grouped(st.mats, st.xs, st.outs)
        return st.outs
    st.head.embed(st.ids, c["tokens"], st.out)
    return st.out


# ---- what a pass cannot do without -------------------------------------------------------------------

def _table_bytes(rows, in_dim):
    return rows * in_dim // 2 + rows * (in_dim // 64) * 4


def work(case):
    c, kind = case, case["kind"]
    if kind in ("step", "logits"):
        size = 2 if c["dtype"] == "bf16" else 4
        n = _table_bytes(c["vocab"], c["hidden"]) + c["batch"] * (c["hidden"] * size + c["vocab"] * 4)
        if kind == "step":
            n += c["batch"] * (4 * c["history"] + 8 * c["bias"] + (c["vocab"] // 8 if c["ban"] else 0) + 4)
        return {"bytes": n, "flops": 2 * c["vocab"] * c["hidden"] * c["batch"]}
    if kind == "sample":  # the logits read once; a mask also makes the pass write the banned ones
        n = c["batch"] * (c["vocab"] * 4 + 4)
        if c["ban"]:
            n += c["batch"] * int(c["vocab"] // 8 + 4 * c["ban"] * c["vocab"])
        return {"bytes": n, "flops": 4 * c["batch"] * c["vocab"]}
    if kind == "matvec":
        size = 2 if c["dtype"] == "bf16" else 4
        return {"bytes": _table_bytes(c["rows"], c["in_dim"]) + c["batch"] * (c["in_dim"] * size + c["rows"] * 4),
                "flops": 2 * c["rows"] * c["in_dim"] * c["batch"]}
    if kind in ("experts", "refill"):
        i, h = c["inner"], c["hidden"]
        one = 2 * _table_bytes(i, h) + _table_bytes(h, i)
        if kind == "experts":
            return {"bytes": ROUTED * (one + 4 * (3 * i + h)) + 4 * h, "flops": 6 * ROUTED * i * h}
        return {"bytes": 3 * one + 4 * (3 * i + 2 * h), "flops": 6 * i * h}
    return {"bytes": c["tokens"] * (_table_bytes(1, c["hidden"]) + 4 + 4 * c["hidden"]),
            "flops": 2 * c["tokens"] * c["hidden"]}


def tolerance(case):
    """One and two rows go through exact integer products with 32-bit sums (5e-7 from 64 bits).
    Larger batches go through 16-bit matrix operands with 32-bit sums: rows held in 32 bits are
    rounded to 11 (1.7e-4), normalised bf16 rows are exact there (1.5e-6). Tokens are draws: a
    rounding may move one over the edge between two neighbours."""
    kind = case["kind"]
    if kind == "embed":
        return {"rel": 4e-7, "max": 4e-6}
    if kind == "sample":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.01}
    if kind in ("experts", "refill") or case["batch"] <= 2:
        return {"rel": 3e-6, "max": 1e-4, "differ": 0.01}
    if case["dtype"] == "bf16" and (kind != "step" or case["normed"]):
        return {"rel": 8e-6, "max": 2e-4, "differ": 0.01}
    return {"rel": 7e-4, "max": 1e-2, "differ": 0.01}


# ---- the same in 64 bits -----------------------------------------------------------------------------

def _product(table, x):
    """[batch][rows] = x w^T in 64 bits, a block of rows at a time."""
    w, s, b, _ = table
    rows, out = w.shape[0], torch.empty((x.shape[0], w.shape[0]), dtype=torch.float64, device="cuda")
    for r in range(0, rows, 16384):
        e = min(rows, r + 16384)
        out[:, r:e] = x @ _dequant(w[r:e], s[r:e], b[r:e]).t().contiguous()
    return out


def _penalised(c, l, ids):
    """Repetition per occurrence with its clamp, then presence and frequency, on one row."""
    uniq, count = ids.long().unique(return_counts=True)
    v = l[uniq].clone()
    p, lim = c["repetition"], 0.9999 * CAP
    if p != 1.0:
        for k in range(int(count.max())):
            n = torch.where(v > 0, v / p, v * p).clamp(-lim, lim)
            v = torch.where(count > k, n, v)
    if c["presence"] or c["frequency"]:
        v = v - c["presence"] - c["frequency"] * count.double()
    l[uniq] = v


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "step":
        table = _table(c["vocab"], c["hidden"], _gen(seed, 1), gamma=True)
        x = _cast(_hidden(c["batch"], table, _gen(seed, 2)), c["dtype"]).double()
        if not c["normed"]:
            x = x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + EPS) * table[3].double()
        l = _product(table, x)
        l = CAP * torch.tanh(l / CAP)
        if c["bias"]:
            ids, vals = _biases(c, _gen(seed, 5))
            l.scatter_add_(1, ids.long(), vals.double())
        if c["history"]:
            h = _histories(c, _gen(seed, 3))[0]
            for b in range(c["batch"]):
                _penalised(c, l[b], h[b, : c["history"]])
        if c["ban"]:
            l.masked_fill_(_bans(c, _gen(seed, 4))[1], -math.inf)
        out = {"tokens": None, "logits": l}
        if c["history"]:
            out.update(history=None, history_len=None)
        return out
    if kind == "logits":
        table = _table(c["vocab"], c["hidden"], _gen(seed, 1))
        x = _hidden(c["batch"], table, _gen(seed, 2))
        x = _cast(x * torch.rsqrt(x.square().mean(dim=1, keepdim=True)), c["dtype"])
        l = _product(table, x.double())
        return CAP * torch.tanh(l / CAP) if c["softcap"] else l
    if kind == "sample":
        l = _given_logits(c, _gen(seed, 2)).double()
        if c["ban"]:
            l.masked_fill_(_bans(c, _gen(seed, 4))[1], -math.inf)
        return {"tokens": None, "logits": l}
    if kind == "matvec":
        table = _table(c["rows"], c["in_dim"], _gen(seed, 1))
        return _product(table, _cast(_randn((c["batch"], c["in_dim"]), _gen(seed, 2)), c["dtype"]).double())
    if kind == "experts":
        g = _gen(seed, 1)
        tables = [_expert_tables(c, g) for _ in range(EXPERTS)]
        g = _gen(seed, 2)
        x = _randn((c["hidden"],), g).double().unsqueeze(0)
        h = _randn((ROUTED, c["inner"]), g).double()
        picked = [tables[e] for e in _routed(0)]
        return {"gate_up": torch.cat([_product(t, x) for e in picked for t in e[:2]]),
                "down": torch.cat([_product(e[2], h[j:j + 1]) for j, e in enumerate(picked)])}
    if kind == "refill":
        g = _gen(seed, 1)
        slots = [_expert_tables(c, g) for _ in range(4)]
        g = _gen(seed, 2)
        x, h = _randn((c["hidden"],), g).double().unsqueeze(0), _randn((c["inner"],), g).double().unsqueeze(0)
        return [_product(t, v)[0] for t, v in zip(slots[0], (x, x, h))]
    table = _table(c["vocab"], c["hidden"], _gen(seed, 1))
    ids = _randint(0, c["vocab"], (c["tokens"],), _gen(seed, 2)).long()
    return _dequant(table[0], table[1], table[2], ids) * math.sqrt(c["hidden"])
