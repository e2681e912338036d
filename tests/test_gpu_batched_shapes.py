"""The matrix-core heads (batches above two rows) at the edges of their shapes: every remainder of
the group count by the prefetch depth, tables on both sides of each dispatch line, the last partial
tile, and batches around the column blocks. Reference: the same product in 64 bits on the GPU."""
import pytest

import turbo_decode_tail as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def make_table(rows, in_dim, seed, big=False):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    w = torch.randint(0, 256, (rows, in_dim // 2), generator=g, device="cuda", dtype=torch.uint8)
    s = (torch.randn((rows, in_dim // 64), generator=g, device="cuda").abs() * 0.004).bfloat16()
    if big:
        s[rows // 2, 0] = 0.5  # a scale the denormal dequant cannot hold: the other form runs
    b = (-8.0 * s.float()).bfloat16()
    torch.cuda.synchronize()
    return w, s, b


def dequant(w, s, b):
    q = torch.stack((w & 15, w >> 4), dim=-1).reshape(w.shape[0], -1, 64).double()
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(w.shape[0], -1)


def check(rows, in_dim, batches, seed, big=False):
    """|got - want| <= sum_c |w_c x_c| (2^-10 + D 2^-24) + 2^-21 sum_c |x_c|: weight and activation
    are each rounded once to fp16 (2^-11 relative), products are exact in fp32 and D fp32 additions
    round; a weight below 2^-10 sits on the fp16 subnormal grid (2^-25 of 16 x)."""
    w, s, b = make_table(rows, in_dim, seed, big)
    h = T.LMHead(w, s, b, None, vocab=rows, hidden=in_dim, softcap=0.0, on_device=True)
    try:
        full = dequant(w, s, b)
        for batch in batches:
            g = torch.Generator(device="cuda")
            g.manual_seed(seed + batch)
            x = torch.randn((batch, in_dim), generator=g, device="cuda")
            out = torch.full((batch, rows), float("nan"), device="cuda")
            torch.cuda.synchronize()
            h.logits(x, batch, out, softcap=False)
            h.sync()
            want = x.double() @ full.t().contiguous()
            bound = (x.double().abs() @ full.abs().t().contiguous()) * (2.0**-10 + in_dim * 2.0**-24)
            bound = bound + x.double().abs().sum(dim=1, keepdim=True) * 2.0**-21
            assert bool(((out.double() - want).abs() <= bound).all()), (rows, in_dim, batch)
    finally:
        h.close()


@pytest.mark.parametrize("in_dim", [64, 128, 192, 256, 320, 448])
def test_group_counts_whole_tile_heads(in_dim):
    """G = 1 .. 7 (all remainders by the prefetch depth, G below it) on a table past the split
    head's line, for each column layout of the whole-tile heads."""
    check(769 * 64 - 5, in_dim, [3, 33, 64, 65, 129], 11 * in_dim)


def test_wide_workgroup_line():
    """64 columns on both sides of the 16-wave workgroup's line (3072 tiles), odd group count."""
    check(3071 * 64, 192, [64], 5)
    check(3072 * 64 - 63, 192, [48, 64], 6)


@pytest.mark.parametrize("rows,in_dim", [(1, 64), (63, 128), (64, 192), (65, 448), (4099, 512), (256 * 64, 576),
                                         (256 * 64 + 1, 256), (768 * 64, 320), (512 * 64, 64)])
def test_split_head_shapes(rows, in_dim):
    """The split head: fewer groups than waves, both wave counts, the last tile it serves, a partial
    last tile, and batches on both sides of a column block and of its line (512 x 3 column blocks
    take the whole-tile head)."""
    check(rows, in_dim, [3, 31, 32, 33, 64, 65, 256], rows + in_dim)


def test_split_head_mantissa_dequant():
    """A table with a scale above 1/16 takes the other dequant form."""
    check(130, 320, [3, 40], 9, big=True)
    check(300 * 64, 192, [5, 64], 10, big=True)


def test_split_head_large_activations():
    """Rows whose largest |x| passes 2^11 are stored scaled down and scaled back: a power of two
    applied to a row scales its products exactly."""
    w, s, b = make_table(1000, 704, 3)
    h = T.LMHead(w, s, b, None, vocab=1000, hidden=704, softcap=0.0, on_device=True)
    try:
        x = torch.randn((5, 704), device="cuda")
        x = x / x.abs().amax(dim=1, keepdim=True) * 1500.0  # the largest stays within 2^11
        big = x * 8.0
        big[0] = x[0]
        a, c = torch.empty((5, 1000), device="cuda"), torch.empty((5, 1000), device="cuda")
        torch.cuda.synchronize()
        h.logits(x, 5, a, softcap=False)
        h.logits(big, 5, c, softcap=False)
        h.sync()
        assert torch.equal(a[0], c[0])
        # fp16 rounding is relative, so the scaled rows differ only where 8 x / 2^k / 8 falls among
        # fp16 subnormals: at most 2^-25 per element times the weights
        bound = dequant(w, s, b).abs().sum(dim=1) * 8.0 * 2.0**-20
        assert bool(((c[1:].double() - 8.0 * a[1:].double()).abs() <= bound + 1e-5 * c[1:].double().abs()).all())
    finally:
        h.close()
