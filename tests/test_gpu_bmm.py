"""GPU parity of the attention contractions (through the C ABI): layout_bmm /
bmm bit-equal to the sequential fp32 oracle (the reference's contract,
verify_bmm_layout.py:16-37), channel_select bit-exact."""
import itertools

import pytest
import torch

from oracle import bmm as ob
from oracle.numerics import bits_equal
from tests.helpers import gen

pytestmark = pytest.mark.gpu


def same_bits(got, expect):
    """Bit-equal, except that a NaN result only has to be a NaN (the payload a
    NaN operand leaves depends on the FMA unit's propagation rules)."""
    got, expect = got.cpu().contiguous(), expect.contiguous()
    assert got.shape == expect.shape and got.dtype == expect.dtype
    nan = expect.isnan()
    assert torch.equal(got.isnan(), nan)
    g, e = got.view(torch.int16), expect.view(torch.int16)
    return torch.equal(g[~nan], e[~nan])


@pytest.mark.parametrize("shape", [(4, 400, 32, 400), (4, 64, 400, 400), (2, 17, 9, 23), (3, 5, 37, 1031),
                                   (1, 1, 1, 1)])
def test_bmm_reference_shapes(gpu, shape):
    """verify_bmm_flow.py:15-25: plain and transposed-view operands."""
    from thintnpu_amd import capi
    batch, m, k, n = shape
    g = gen(2026)
    for transposed in (False, True):
        a = (torch.randn(batch, k, m, generator=g).transpose(1, 2) if transposed
             else torch.randn(batch, m, k, generator=g)).half()
        b = (torch.randn(batch, n, k, generator=g).transpose(1, 2) if transposed
             else torch.randn(batch, k, n, generator=g)).half()
        ad = a.contiguous().to(gpu) if not transposed else a.transpose(1, 2).contiguous().to(gpu).transpose(1, 2)
        bd = b.contiguous().to(gpu) if not transposed else b.transpose(1, 2).contiguous().to(gpu).transpose(1, 2)
        got = capi.bmm(ad, bd)
        assert got.shape == (batch, m, n) and got.stride(1) == (n + 15) // 16 * 16
        expect = ob.sequential_bmm(a, b)
        assert bits_equal(got, expect), (shape, transposed)
        torch.testing.assert_close(got.cpu(), torch.bmm(a.float(), b.float()).half(), rtol=0.002, atol=0.002)


@pytest.mark.parametrize("shape", [(2, 19, 33, 23), (1, 1, 600, 257), (3, 5, 37, 1031)])
@pytest.mark.parametrize("ta,tb", list(itertools.product((False, True), repeat=2)))
def test_bmm_strided_offset_views(gpu, shape, ta, tb):
    """verify_bmm_layout.py:42-57: operands are [.., 1:] views (odd storage
    offsets, non-unit row strides) in all four transpose combinations."""
    from thintnpu_amd import capi
    batch, m, k, n = shape
    g = gen(894)
    ac = torch.randn(batch, k, m + 1, generator=g).half() if ta else torch.randn(batch, m, k + 1, generator=g).half()
    bc = torch.randn(batch, n, k + 1, generator=g).half() if tb else torch.randn(batch, k, n + 1, generator=g).half()
    ad, bd = ac.to(gpu), bc.to(gpu)
    a = ad[:, :, 1:].transpose(1, 2) if ta else ad[:, :, 1:]
    b = bd[:, :, 1:].transpose(1, 2) if tb else bd[:, :, 1:]
    ar = ac[:, :, 1:].transpose(1, 2) if ta else ac[:, :, 1:]
    br = bc[:, :, 1:].transpose(1, 2) if tb else bc[:, :, 1:]
    assert bits_equal(capi.bmm(a, b), ob.sequential_bmm(ar, br))


@pytest.mark.parametrize("heads,key,dim,tokens", [(4, 32, 64, 400), (2, 16, 32, 160), (1, 16, 16, 1),
                                                  (3, 48, 80, 37)])
def test_layout_bmm_blocked_heads(gpu, heads, key, dim, tokens):
    """verify_bmm_layout.py:58-85: q^T k and v p^T over split blocked QKV, and
    the blocked output."""
    from thintnpu_amd import capi
    g = gen(894 + tokens)
    source = torch.randn(heads, (2 * key + dim) // 16, tokens, 16, generator=g).half()
    device = source.to(gpu)
    q, k, v = device.split((key // 16, key // 16, dim // 16), 1)
    qr, kr, vr = source.split((key // 16, key // 16, dim // 16), 1)
    got = capi.layout_bmm(q, k, True, False, False)
    assert bits_equal(got, ob.layout_bmm(qr, kr, True, False, False))
    probability = torch.randn(heads, tokens, tokens, generator=g).half()
    pd = probability.to(gpu)
    assert bits_equal(capi.layout_bmm(v, pd, False, True, False), ob.layout_bmm(vr, probability, False, True, False))
    got = capi.layout_bmm(v, pd, False, True, True)
    assert got.shape == (heads, dim // 16, tokens, 16)
    assert bits_equal(got, ob.layout_bmm(vr, probability, False, True, True))


@pytest.mark.parametrize("heads,key,dim,tokens", [(4, 32, 64, 400), (4, 8, 16, 37), (2, 24, 48, 19),
                                                  (8, 3, 6, 19)])
def test_layout_bmm_grouped_and_select(gpu, heads, key, dim, tokens):
    """verify_bmm_layout.py:86-106: head groups over one N=1 blocked QKV tensor,
    channel ranges per head, the grouped blocked output and channel_select."""
    from thintnpu_amd import capi
    group = 2 * key + dim
    logical = torch.randn(heads, group, tokens, generator=gen(heads * 100 + key)).half()
    source = logical.reshape(1, heads * group // 16, 16, tokens).permute(0, 1, 3, 2).contiguous()
    device = source.to(gpu)
    qr, kr, vr = logical.split((key, key, dim), 1)
    got = capi.layout_bmm(device, device, True, False, False, heads, 0, key, key, key)
    assert bits_equal(got, ob.sequential_bmm(qr.transpose(1, 2), kr))
    probability = torch.randn(heads, tokens, tokens, generator=gen(5)).half()
    pd = probability.to(gpu)
    expect = ob.sequential_bmm(vr, probability.transpose(1, 2))
    expect = expect.reshape(1, heads * dim // 16, 16, tokens).permute(0, 1, 3, 2).contiguous()
    got = capi.layout_bmm(device, pd, False, True, True, heads, 2 * key, dim)
    assert bits_equal(got, expect)
    expect = vr.reshape(1, heads * dim // 16, 16, tokens).permute(0, 1, 3, 2).contiguous()
    assert bits_equal(capi.channel_select(device, heads, 2 * key, dim), expect)


def test_summation_order_and_specials(gpu):
    from thintnpu_amd import capi
    # sequential fp32: 2^24 + 1 rounds back to 2^24, so the sum is 0 (exactly 1)
    a = torch.tensor([[[4096., 1., 4096.], [4096., 4096., 1.]]]).half()
    b = torch.tensor([[[4096., 4096.], [1., -4096.], [-4096., 1.]]]).half()
    got = capi.bmm(a.to(gpu), b.to(gpu)).cpu()
    assert bits_equal(got, ob.sequential_bmm(a, b))
    assert got[0, 0, 0].item() == 0.0 and got[0, 1, 1].item() == 1.0
    # fp32 accumulator over a long reduction (an fp16 one stalls at 2048)
    ones = torch.ones(2, 3, 4096).half()
    got = capi.bmm(ones.to(gpu), ones.transpose(1, 2).contiguous().to(gpu)).cpu()
    assert got.eq(4096).all()
    # infinities, NaNs, signed zeros, subnormals and overflow to inf
    vals = torch.tensor([0., -0., float("inf"), -float("inf"), float("nan"), 2 ** -24, -2 ** -24, 65504., -65504.,
                         1., -1., 0.5, 300.]).half()
    g = gen(3)
    a = vals[torch.randint(0, len(vals), (3, 21, 13), generator=g)]
    b = vals[torch.randint(0, len(vals), (3, 13, 70), generator=g)]
    assert same_bits(capi.bmm(a.to(gpu), b.to(gpu)), ob.sequential_bmm(a, b))
    # tiny products: subnormal fp16 results and -0 from negative underflow
    a = torch.full((1, 2, 3), 2 ** -12).half()
    b = torch.tensor([[[2 ** -8, -2 ** -14], [0., 0.], [2 ** -9, -2 ** -20]]]).half()
    got = capi.bmm(a.to(gpu), b.to(gpu))
    assert bits_equal(got, ob.sequential_bmm(a, b))
    assert got[0, 0, 0].item() == 1.5 * 2 ** -20 and got.cpu().view(torch.int16)[0, 0, 1].item() == -32768


@pytest.mark.parametrize("shape", [(1, 63, 17, 65), (1, 64, 31, 64), (5, 129, 33, 127), (300, 3, 5, 7),
                                   (1, 1000, 3, 1), (2, 16, 2048, 16)])
def test_bmm_tile_edges(gpu, shape):
    """Row / column counts around the 64-column tile, a batch of many small
    products, one column, and a reduction over many staging rounds."""
    from thintnpu_amd import capi
    batch, m, k, n = shape
    g = gen(sum(shape))
    a = torch.randn(batch, m, k, generator=g).half()
    b = torch.randn(batch, k, n, generator=g).half()
    assert bits_equal(capi.bmm(a.to(gpu), b.to(gpu)), ob.sequential_bmm(a, b))
    out = torch.full((batch, m, n + 3), 7.0, dtype=torch.float16, device=gpu)
    capi.bmm(a.to(gpu), b.to(gpu), out=out[:, :, 2:2 + n])
    assert bits_equal(out[:, :, 2:2 + n], ob.sequential_bmm(a, b))
    assert out[:, :, :2].cpu().eq(7).all() and out[:, :, 2 + n:].cpu().eq(7).all()


def test_blocked_ungrouped_batch(gpu):
    from thintnpu_amd import capi
    a = torch.randn(3, 2, 9, 16, generator=gen(9)).half()   # 3 images, 32 channels, 9 tokens
    b = torch.randn(3, 9, 40, generator=gen(10)).half()
    got = capi.layout_bmm(a.to(gpu), b.to(gpu), blocked_output=True)
    assert got.shape == (3, 2, 40, 16)
    assert bits_equal(got, ob.layout_bmm(a, b, blocked_output=True))
    # a channel range of a rank-4 operand read transposed (tokens x channels)
    got = capi.layout_bmm(a.to(gpu), a[:, :, :, :].to(gpu), True, False, False, 0, 5, 11, 3, 11)
    assert bits_equal(got, ob.layout_bmm(a, a, True, False, False, 0, 5, 11, 3, 11))


def test_channel_select_views(gpu):
    from thintnpu_amd import capi
    x = torch.randint(-32768, 32768, (1, 6, 23, 16), dtype=torch.int16, generator=gen(4)).view(torch.float16)
    for groups, begin, count in ((3, 0, 16), (3, 5, 16), (2, 7, 8), (6, 1, 8), (1, 0, 96), (4, 10, 4)):
        assert bits_equal(capi.channel_select(x.to(gpu), groups, begin, count),
                          ob.channel_select(x, groups, begin, count))
    # a token-strided view of a larger tensor
    big = torch.randint(-32768, 32768, (1, 6, 50, 16), dtype=torch.int16, generator=gen(5)).view(torch.float16)
    view = big.to(gpu)[:, :, 3::2]
    assert bits_equal(capi.channel_select(view, 2, 7, 8), ob.channel_select(big[:, :, 3::2], 2, 7, 8))


def test_bmm_errors(gpu):
    from thintnpu_amd import capi
    h = lambda *s: torch.zeros(s, dtype=torch.float16, device=gpu)
    cases = [
        (lambda: capi.bmm(h(2, 3, 4), h(2, 5, 6)), "do not match or are empty"),
        (lambda: capi.bmm(h(2, 3, 4), h(3, 4, 6)), "do not match or are empty"),
        (lambda: capi.bmm(h(2, 3, 4), h(2, 4, 0)), "do not match or are empty"),
        (lambda: capi.bmm(h(2, 0, 4), h(2, 4, 6)), "exceeds its group"),  # zero rows: the channel check first
        (lambda: capi.bmm(h(2, 3, 4).float(), h(2, 4, 6)), "FP16 rank-3 or channel-blocked"),
        (lambda: capi.bmm(h(3, 4), h(4, 6)), "FP16 rank-3 or channel-blocked"),
        (lambda: capi.layout_bmm(h(1, 2, 5, 16), h(1, 2, 5, 16), True, False, False, 3), "divisible channels"),
        (lambda: capi.layout_bmm(h(2, 2, 5, 16), h(2, 2, 5, 16), True, False, False, 2), "requires N=1"),
        (lambda: capi.layout_bmm(h(1, 2, 5, 16), h(1, 2, 5, 16), True, False, False, 2, 10, 8, 0, 8),
         "exceeds its group"),
        (lambda: capi.layout_bmm(h(1, 2, 5, 16), h(1, 2, 5, 16), True, False, False, 0, -1), "invalid channel grouping"),
        (lambda: capi.layout_bmm(h(2, 5, 3), h(2, 3, 4), blocked_output=True), "C0-aligned channels"),
        (lambda: capi.channel_select(h(2, 2, 5, 16), 2, 0, 8), "N=1 FP16 blocked"),
        (lambda: capi.channel_select(h(1, 2, 5, 16), 3, 0, 8), "valid equal groups"),
        (lambda: capi.channel_select(h(1, 2, 5, 16), 2, 10, 8), "valid equal groups"),
        (lambda: capi.channel_select(h(1, 2, 5, 16), 2, 0, 4), "C0-aligned total output"),
    ]
    for fn, text in cases:
        with pytest.raises(capi.ThinError, match=text):
            fn()
    with pytest.raises(capi.ThinError, match="out must be"):
        capi.bmm(h(2, 3, 4), h(2, 4, 6), out=h(2, 3, 5))


@pytest.mark.parametrize("key", [80, 128, 528])
def test_streamed_long_reductions(gpu, key):
    """q^T k with K = key channels: the streamed-column kernel's 64-step
    staging rounds (K > 64), several vector rounds, a partial last round, and
    (K = 528) two rounds of staged rows."""
    from thintnpu_amd import capi
    heads, tokens = 2, 70
    source = torch.randn(heads, 2 * key // 16, tokens, 16, generator=gen(key)).half()
    q, k = source.to(gpu).split((key // 16, key // 16), 1)
    qr, kr = source.split((key // 16, key // 16), 1)
    assert bits_equal(capi.layout_bmm(q, k, True, False, False), ob.layout_bmm(qr, kr, True, False, False))


@pytest.mark.parametrize("k", [21, 77])
def test_streamed_reduction_tail(gpu, k):
    """Columns contiguous along k at a 24-element stride with K % 8 != 0: the
    streamed kernel's whole vectors plus its scalar tail."""
    from thintnpu_amd import capi
    batch, m, n = 2, 9, 70
    pitch = (k + 7) // 8 * 8 + 8
    a = torch.randn(batch, m, k, generator=gen(k)).half()
    store = torch.randn(batch, n, pitch, generator=gen(k + 1)).half()
    b = store[:, :, :k].transpose(1, 2)          # [batch, k, n], column stride `pitch`
    bd = store.to(gpu)[:, :, :k].transpose(1, 2)
    assert bits_equal(capi.bmm(a.to(gpu), bd), ob.sequential_bmm(a, b))


def _operand(form, batch, rows, k, g, device):
    """Logical [batch, rows, k] fp16 operand stored with steps adjacent, with rows
    adjacent (both at odd pitches and offsets), or with neither."""
    if form == "steps":
        t = torch.randn(batch, rows, k + 3, generator=g).half()
        return t[:, :, 1:1 + k], t.to(device)[:, :, 1:1 + k]
    if form == "rows":
        t = torch.randn(batch, k, rows + 5, generator=g).half()
        return t[:, :, 3:3 + rows].transpose(1, 2), t.to(device)[:, :, 3:3 + rows].transpose(1, 2)
    t = torch.randn(batch, rows, 2 * k, generator=g).half()
    return t[:, :, ::2], t.to(device)[:, :, ::2]


@pytest.mark.parametrize("batch,m,n,k", [(*shape, k) for shape in ((2, 33, 31), (1, 47, 100), (130, 66, 70), (1, 1472, 1470))
                                         for k in (1, 31, 32, 34, 64, 67, 130, 259)
                                         if shape[0] * shape[1] * shape[2] * k <= 130 * 66 * 70 * 130])
@pytest.mark.parametrize("fa,fb", [("steps", "steps"), ("rows", "rows"), ("steps", "rows"), ("rows", "steps"),
                                   ("neither", "rows"), ("steps", "neither")])
def test_bmm_load_forms(gpu, batch, m, n, k, fa, fb):
    """Every pair of operand load forms at both tile sizes (the last two shapes
    give 512 or more 64 x 64 tiles), with partial row tiles, reductions around
    the 32, 64 and 128-step chunks and remainders of 4 and 8 steps, operands at
    2-byte alignment: the bits of the sequential sum.  (The largest shapes only
    as far as the oracle is quick.)"""
    from thintnpu_amd import capi
    g = gen(batch * 7 + m + k)
    a, ad = _operand(fa, batch, m, k, g, gpu)
    b, bd = _operand(fb, batch, n, k, g, gpu)
    got = capi.bmm(ad, bd.transpose(1, 2))
    assert bits_equal(got, ob.sequential_bmm(a, b.transpose(1, 2)))


@pytest.mark.parametrize("c0,key,tokens", [(8, 24, 70), (32, 64, 33), (24, 48, 40), (16, 48, 1100)])
def test_blocked_widths(gpu, c0, key, tokens):
    """q^T k over operands blocked by 8, 32 (loaded in runs) and 24 (gathered)
    channels, and over enough tokens for several tiles a block."""
    from thintnpu_amd import capi
    source = torch.randn(2, 2 * key // c0, tokens, c0, generator=gen(c0 + key)).half()
    q, k = source.to(gpu).split((key // c0, key // c0), 1)
    qr, kr = source.split((key // c0, key // c0), 1)
    assert bits_equal(capi.layout_bmm(q, k, True, False, False), ob.layout_bmm(qr, kr, True, False, False))
    # a range of channels that starts inside a block
    got = capi.layout_bmm(q, k, True, False, False, 0, 4, 20, 4, 20)
    assert bits_equal(got, ob.layout_bmm(qr, kr, True, False, False, 0, 4, 20, 4, 20))


def _blocked(batch, channels, tokens, c0, g):
    """[batch, C1, tokens, c0] of `channels` channels, the blocks filled up with NaN."""
    x = torch.randn(batch, (channels + c0 - 1) // c0, tokens, c0, generator=g).half()
    x[:, -1, :, (channels - 1) % c0 + 1:] = float("nan")
    return x


@pytest.mark.parametrize("c0", [8, 16, 32])
@pytest.mark.parametrize("origin", [0, 8])
def test_blocked_step_tails(gpu, c0, origin):
    """Reductions over blocked channels whose count is no multiple of 8: the
    steps after the last whole run of 8 lie in their own block, not behind the
    run before them.  q^T k, one blocked and one plain operand either way
    round, heads of one tensor, and 512 or more 64 x 64 tiles."""
    from thintnpu_amd import capi
    for count in (9, 12, 17, 20, 23, 33, 36, 39, 131):
        g = gen(c0 * 1000 + count)
        for batch, tokens in ((2, 41), (130, 70)):
            x, y = _blocked(batch, origin + count, tokens, c0, g), _blocked(batch, origin + count, tokens, c0, g)
            xd, yd = x.to(gpu), y.to(gpu)
            args = (True, False, False, 0, origin, count, origin, count)
            assert bits_equal(capi.layout_bmm(xd, yd, *args), ob.layout_bmm(x, y, *args)), count
        plain = torch.randn(130, 37, count, generator=g).half()
        args = (False, False, False, 0, 0, -1, origin, count)
        assert bits_equal(capi.layout_bmm(plain.to(gpu), yd, *args), ob.layout_bmm(plain, y, *args)), count
        right = plain.transpose(1, 2)
        args = (True, False, False, 0, origin, count)
        assert bits_equal(capi.layout_bmm(xd, plain.to(gpu).transpose(1, 2), *args), ob.layout_bmm(x, right, *args)), count
        group = (origin + count + 31) // 32 * 32
        heads = _blocked(1, 3 * group, 50, c0, g)
        args = (True, False, False, 3, origin, count, origin, count)
        assert bits_equal(capi.layout_bmm(heads.to(gpu), heads.to(gpu), *args), ob.layout_bmm(heads, heads, *args)), count


@pytest.mark.parametrize("c0", [8, 24, 40, 64, 128])
@pytest.mark.parametrize("channels", [20, 100])
def test_blocked_axis_forms(gpu, c0, channels):
    """Channel blocks of widths that do and do not divide a chunk of steps or
    a tile of rows, as rows of either operand (the last run of rows partial)
    and as steps, with one tile a block and several."""
    from thintnpu_amd import capi
    g = gen(c0 + channels)
    for batch, tokens in ((2, 131), (2, 24), (450, 24)):
        x = _blocked(batch, channels, tokens, c0, g)
        rows = torch.randn(batch, tokens, 70, generator=g).half()
        args = (False, False, False, 0, 0, channels)
        assert bits_equal(capi.layout_bmm(x.to(gpu), rows.to(gpu), *args), ob.layout_bmm(x, rows, *args))
        rows = torch.randn(batch, 70, tokens, generator=g).half()
        args = (False, True, False, 0, 0, -1, 0, channels)
        assert bits_equal(capi.layout_bmm(rows.to(gpu), x.to(gpu), *args), ob.layout_bmm(rows, x, *args))
    args = (True, False, False, 0, 0, channels, 0, channels)
    for batch, tokens in ((2, 131), (130, 70)):
        x = _blocked(batch, channels, tokens, c0, g)
        assert bits_equal(capi.layout_bmm(x.to(gpu), x.to(gpu), *args), ob.layout_bmm(x, x, *args))


@pytest.mark.parametrize("batch", [2, 500, 520])
@pytest.mark.parametrize("rows,k", [(9, 131), (23, 20), (33, 20), (49, 40), (63, 130)])
def test_partial_rows(gpu, batch, rows, k):
    """Row-contiguous operands of one tile that ends in a partial run of 8, on
    both sides of the batch from which 64 x 64 tiles fill the device."""
    from thintnpu_amd import capi
    a = torch.randn(batch, k, rows, generator=gen(rows)).half().transpose(1, 2)
    b = torch.randn(batch, k, rows, generator=gen(k)).half()
    ad = a.transpose(1, 2).contiguous().to(gpu).transpose(1, 2)
    assert bits_equal(capi.bmm(ad, b.to(gpu)), ob.sequential_bmm(a, b))


@pytest.mark.parametrize("batch,m,n", [(3, 1, 5), (2, 40, 70), (700, 8, 65), (650, 16, 33), (650, 17, 33), (2100, 5, 70)])
def test_columns_in_vectors(gpu, batch, m, n):
    """Columns of b in aligned vectors along k, at sizes on both sides of the
    choice between chains of fmas and matrix tiles: one to four rows a wave,
    reductions around the staging rounds, rows of a adjacent (gathered below
    8, which leaves the tiled chains) or not, columns a line apart or not."""
    from thintnpu_amd import capi
    for k in (1, 8, 21, 32, 33, 40, 64, 77, 136, 520, 528):
        entries = batch if batch * m * n * k <= 700 * 16 * 65 * 136 else 2
        g = gen(batch + m + n + k)
        store = torch.randn(entries, n, (k + 7) // 8 * 8, generator=g).half()
        b, bd = store[:, :, :k].transpose(1, 2), store.to(gpu)[:, :, :k].transpose(1, 2)
        a = torch.randn(entries, m, k, generator=g).half()
        expect = ob.sequential_bmm(a, b)
        assert bits_equal(capi.bmm(a.to(gpu), bd), expect), k
        rows = a.transpose(1, 2).contiguous().to(gpu).transpose(1, 2)
        assert bits_equal(capi.bmm(rows, bd), expect), k


@pytest.mark.parametrize("batch,m,n", [(2, 40, 70), (130, 66, 70)])
@pytest.mark.parametrize("k", [20, 40, 67, 140])
def test_specials_in_matrix_tiles(gpu, batch, m, n, k):
    """Infinities, NaN, signed zeros, subnormals and the largest values among
    ordinary ones, in both tile sizes of the short and the long reduction, with
    operands loaded along steps and along rows."""
    from thintnpu_amd import capi
    vals = torch.tensor([0., -0., float("inf"), -float("inf"), float("nan"), 2 ** -24, -2 ** -24, 3 * 2 ** -20, 65504.,
                         -65504.]).half()
    g = gen(batch + k)

    def operand(*shape):
        x = torch.randn(shape, generator=g).half()
        special = vals[torch.randint(0, len(vals), shape, generator=g)]
        return torch.where(torch.rand(shape, generator=g) < 0.5 / k, special, x)

    a, b = operand(batch, m, k), operand(batch, k, n)
    expect = ob.sequential_bmm(a, b)
    assert expect.isnan().any() and expect.isinf().any() and expect.isfinite().any()
    for ta in (False, True):
        ad = a.transpose(1, 2).contiguous().to(gpu).transpose(1, 2) if ta else a.to(gpu)
        for tb in (False, True):
            bd = b.transpose(1, 2).contiguous().to(gpu).transpose(1, 2) if tb else b.to(gpu)
            assert same_bits(capi.bmm(ad, bd), expect), (ta, tb)
    # sums that stay subnormal, and -0 from negative underflow
    a, b = (torch.randn(batch, m, k, generator=g) * 2 ** -12).half(), (torch.randn(batch, k, n, generator=g) * 2 ** -11).half()
    expect = ob.sequential_bmm(a, b)
    assert (expect.view(torch.int16) == -32768).any()
    assert bits_equal(capi.bmm(a.to(gpu), b.to(gpu)), expect)


@pytest.mark.parametrize("entries,m,k,pitch,step", [(24, 17, 8, 8, 1), (24, 17, 72, 72, 1), (24, 1, 40, 72, 1),
                                                    (26, 1, 8, 8, 1), (24, 1, 8, 16, 2)])
def test_more_products_than_a_launch(gpu, entries, m, k, pitch, step):
    """A batch beyond the 2^32 threads of one launch, for each kernel: matrix
    tiles of a short and a long reduction, chains over tiles and columns, the
    gather.  a is a window that slides along one vector, so the sums are those
    of a correlation, formed step by step on the device."""
    from thintnpu_amd import capi
    batch = (1 << entries) + 1
    g = torch.Generator(device=gpu).manual_seed(5)
    line = torch.randn(batch + m + step * k, generator=g, device=gpu, dtype=torch.float16)
    a = line.as_strided((batch, m, k), (1, 1, step))
    b = torch.randn(1, 1, pitch, generator=g, device=gpu, dtype=torch.float16)[:, :, :step * k:step]
    acc = torch.zeros(batch + m - 1, device=gpu)
    for i in range(k):
        acc += line[i * step:i * step + batch + m - 1].float() * b[0, 0, i].float()
    out = torch.full((batch, m, 1), 7.0, device=gpu, dtype=torch.float16)
    capi.bmm(a, b.expand(batch, 1, k).transpose(1, 2), out=out)
    expect = acc.half().view(torch.int16).unfold(0, m, 1)
    assert torch.equal(out[:, :, 0].view(torch.int16), expect)


@pytest.mark.parametrize("heads,tokens", [(8, 24), (4, 16), (300, 72)])
def test_blocked_output_of_few_channels(gpu, heads, tokens):
    """v p^T of 16 channels a head into the blocked layout, heads of one tensor
    and one tensor a head, at sizes that take the chains of fmas."""
    from thintnpu_amd import capi
    g = gen(heads + tokens)
    p = torch.randn(heads, tokens, tokens, generator=g).half()
    x = torch.randn(1, heads, tokens, 16, generator=g).half()
    args = (False, True, True, heads, 0, 16)
    assert bits_equal(capi.layout_bmm(x.to(gpu), p.to(gpu), *args), ob.layout_bmm(x, p, *args))
    x = x.transpose(0, 1).contiguous()
    args = (False, True, True)
    assert bits_equal(capi.layout_bmm(x.to(gpu), p.to(gpu), *args), ob.layout_bmm(x, p, *args))


@pytest.mark.parametrize("heads,tokens", [((1 << 24) + 16, 1), ((1 << 26) + 16, 8)])
def test_more_heads_than_a_launch(gpu, heads, tokens):
    """The same beyond one launch, a channel a head into blocks of 16 heads:
    gathered elements, and chains."""
    from thintnpu_amd import capi
    g = torch.Generator(device=gpu).manual_seed(7)
    x = torch.randn(1, heads // 16, tokens, 16, generator=g, device=gpu, dtype=torch.float16)
    b = torch.randn(heads, 1, tokens, generator=g, device=gpu, dtype=torch.float16)
    out = torch.full((1, heads // 16, 1, 16), 7.0, device=gpu, dtype=torch.float16)
    capi.layout_bmm(x, b.transpose(1, 2), False, False, True, heads, 0, 1, out=out)
    acc = torch.zeros(heads, device=gpu)
    for t in range(tokens):
        acc += x[0, :, t].reshape(-1).float() * b[:, 0, t].float()
    assert torch.equal(out.reshape(-1).view(torch.int16), acc.half().view(torch.int16))
