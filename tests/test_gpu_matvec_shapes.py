"""The small matrix-vector product at the edges of its shapes: rows and workgroups per tile on both
sides of each line, input sizes whose chunks do not divide among the slots or the waves, one and two
rows, fp32 and bf16, an address off by four bytes, and the same matrices in one grouped launch (bit
for bit the matrix's own call). Reference: the product in 64 bits on the GPU."""
import pytest

import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def make_table(rows, in_dim, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    w = torch.randint(0, 256, (rows, in_dim // 2), generator=g, device="cuda", dtype=torch.uint8)
    s = (torch.randn((rows, in_dim // 64), generator=g, device="cuda").abs() * 0.004).bfloat16()
    b = (-8.0 * s.float() + torch.randn(s.shape, generator=g, device="cuda") * 1e-4).bfloat16()
    torch.cuda.synchronize()
    return w, s, b


def reference(w, s, b, x):
    """The product, and its bound: activations rounded at 2^-22 of their group's largest (21-bit
    integers, |X| <= 2^21), then fp32 roundings of s D + (8 s + b) S over the chunks, the waves and
    the slots (at most one per chunk plus 32)."""
    rows, in_dim = w.shape[0], w.shape[1] * 2
    q = torch.stack((w & 15, w >> 4), dim=-1).reshape(rows, -1, 64).double()
    sd, bd = s.double().unsqueeze(-1), b.double().unsqueeze(-1)
    full = (q * sd + bd).reshape(rows, in_dim)
    xd = x.double()
    want = xd @ full.t().contiguous()
    gmax = xd.abs().reshape(x.shape[0], -1, 64).amax(dim=2, keepdim=True).expand(-1, -1, 64).reshape(x.shape[0], in_dim)
    parts = (((q - 8.0).abs() * sd) + (8.0 * sd + bd).abs()).reshape(rows, in_dim)
    bound = 2.0**-21 * (gmax @ parts.t().contiguous())
    bound = bound + (in_dim / 32 + 32) * 2.0**-24 * 2.0 * (xd.abs() @ parts.t().contiguous())
    return want, bound + 1e-30


@pytest.mark.parametrize("rows,in_dim", [(1, 64), (16, 64), (17, 128), (63, 192), (64, 320), (704, 2816), (4096, 96 * 2),
                                         (4097, 448), (8192, 64), (8193, 576), (65536, 128), (65537, 64), (100, 8192),
                                         (20000, 1088)])
def test_matvec_shapes(rows, in_dim):
    w, s, b = make_table(rows, in_dim, rows + in_dim)
    h = T.LMHead(w, s, b, None, vocab=rows, hidden=in_dim, softcap=0.0, on_device=True)
    m = T.Int4Matrix(rows, in_dim)
    try:
        m.load_weights(w, s, b, on_device=True)
        for batch in (1, 2):
            g = torch.Generator(device="cuda")
            g.manual_seed(batch)
            x = torch.randn((batch, in_dim), generator=g, device="cuda")
            x[0, in_dim // 2:] *= 300.0
            buf = torch.zeros(batch * in_dim + 1, device="cuda")
            buf[1:] = x.reshape(-1)
            outs = [torch.full((batch, rows), float("nan"), device="cuda") for _ in range(3)]
            xb = x.bfloat16()
            torch.cuda.synchronize()
            h.matvec(x, batch, outs[0])
            h.matvec(buf[1:], batch, outs[1])
            h.matvec(xb, batch, outs[2], dtype=T.TURBO_HIDDEN_BF16)
            h.sync()
            assert torch.equal(outs[0], outs[1])
            for o, xin in ((outs[0], x), (outs[2], xb.float())):
                want, bound = reference(w, s, b, xin)
                assert bool(((o.double() - want).abs() <= bound).all()), (rows, in_dim, batch)
            if batch == 1:
                o = torch.full((3, rows), float("nan"), device="cuda")
                torch.cuda.synchronize()
                T.matvec_grouped([m] * 3, [x[0]] * 3, list(o))
                torch.cuda.synchronize()
                for i in range(3):
                    assert torch.equal(o[i], outs[0][0]), i
    finally:
        m.close()
        h.close()


def test_grouped_mixed_shapes():
    """Matrices of different shapes, wave counts and rows per workgroup in one launch, 32 of them."""
    shapes = [(64, 64), (704, 2816), (2816, 704), (5000, 192), (9000, 64), (33, 8192), (130, 1088), (1, 128)] * 4
    mats, xs, outs, refs = [], [], [], []
    for i, (rows, k) in enumerate(shapes):
        t = make_table(rows, k, i)
        m = T.Int4Matrix(rows, k)
        m.load_weights(*t, on_device=True)
        x = torch.randn(k, device="cuda")
        mats.append(m), xs.append(x), outs.append(torch.full((rows,), float("nan"), device="cuda"))
        refs.append(reference(*t, x.unsqueeze(0)))
    torch.cuda.synchronize()
    T.matvec_grouped(mats, xs, outs)
    torch.cuda.synchronize()
    for o, (want, bound) in zip(outs, refs):
        assert bool(((o.double() - want[0]).abs() <= bound[0]).all())
    for m in mats:
        m.close()


def test_grouped_argument_lists():
    """Addresses and tensors mix; a missing or surplus buffer is refused, not read past the list."""
    t = make_table(64, 128, 1)
    m = T.Int4Matrix(64, 128)
    try:
        m.load_weights(*t, on_device=True)
        x, o = torch.randn(128, device="cuda"), torch.zeros((3, 64), device="cuda")
        torch.cuda.synchronize()
        T.matvec_grouped([m, m], [x, x.data_ptr()], [o[0].data_ptr(), o[1]])
        T.matvec_grouped((m,), (x,), (o[2],))
        torch.cuda.synchronize()
        assert torch.equal(o[0], o[1]) and torch.equal(o[0], o[2]) and bool((o[0] != 0).any())
        with pytest.raises(T.TurboError, match="is NULL"):
            T.matvec_grouped([m, m], [x], [o[0], o[1]])
        with pytest.raises(T.TurboError, match="is NULL"):
            T.matvec_grouped([m], [x], [None])
        with pytest.raises(IndexError):
            T.matvec_grouped([m], [x, x], [o[0]])
        T.matvec_grouped([], [], [])
    finally:
        m.close()
    with pytest.raises(T.TurboError, match="null matrix handle"):
        T.matvec_grouped([m], [x], [o[0]])
