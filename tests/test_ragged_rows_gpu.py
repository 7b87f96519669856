"""Rows at any alignment through the row kernels: the lanes at the two ends of a row share columns with their
neighbours, and one-wave rows leave through LDS in accesses aligned to cache lines.

Against the fp32 expression, at the edges of the kernels' ranges (a last lane of 1 to 8 columns, a row end in the first lane
of a chunk, the limits of the shapes), with tensors that begin at any element of a 16-byte slot, with a last block that is
not full, in place, and with guard elements around every output: nothing outside of it is written.  The sums of a
row are taken over the same terms in the same order whatever is folded in: zero slopes, a zero bias and dropout give
the plain kernels' bits.
"""
import pytest
import torch

from gpt_neox_amd import _lib
from oracle import torch_ref as R
from bars import TOL, assert_grad

pytestmark = pytest.mark.gpu

GUARD = 64  # elements in front of and behind every output
SCALE = 0.125
# the limits of the shapes (1536 / 2048: chunks; 1856: two waves) and row ends in every place of a lane; the shapes that want
# many rows: test_staged_rows_of_many_rows and what follows it
COLUMNS = [513, 520, 527, 671, 673, 943, 945, 1001, 1018, 1023, 1024, 1025, 1031, 1201, 1535, 1536, 1537, 1855, 1857, 2047, 2049, 4097]


def at(offset, shape, dtype, device, fill=None, gen=None, std=1.0):
    """A tensor that begins `offset` elements behind a 128-byte boundary, and the storage around it."""
    n = 1
    for d in shape:
        n *= d
    store = torch.full((GUARD + offset + n + GUARD,), 7.0, dtype=dtype, device=device)
    t = store[GUARD + offset : GUARD + offset + n].view(shape)
    if gen is not None:
        t.normal_(0.0, std, generator=gen)
    elif fill is not None:
        t.copy_(fill)
    return t, store


def guarded(t, store):
    lead = t.storage_offset()
    return bool((store[:lead] == 7.0).all()) and bool((store[lead + t.numel() :] == 7.0).all())


@pytest.mark.parametrize("sk", COLUMNS)
@pytest.mark.parametrize("offsets", [(0, 0), (1, 0), (3, 5), (8, 1)])
def test_ragged_rows(device, sk, offsets):
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    dtype = (torch.float16, torch.bfloat16)[(sk + offsets[0]) % 2]
    code = _lib.dtype_code(dtype)
    gen = torch.Generator(device=device).manual_seed(sk)
    b, heads, sq = 3, 1, 5  # fifteen rows: the last block of four is not full
    rows = b * heads * sq
    shape = (b, heads, sq, sk)
    i, o = offsets
    x, _ = at(i, shape, dtype, device, gen=gen, std=8.0)
    g, _ = at(i, shape, dtype, device, gen=gen)
    # causal rows of the full length: the last rows of a taller matrix
    tall = (1, 1, sk, sk)
    causal = torch.ones(sk, sk, dtype=torch.bool, device=device).triu_(1).view(tall)
    xt, _ = at(i, tall, dtype, device, gen=gen, std=8.0)
    gt, _ = at(i, tall, dtype, device, gen=gen)
    lens = torch.tensor([sk, sk - 3, max(1, sk // 3)], device=device)
    mask = (torch.arange(sk, device=device).view(1, 1, 1, sk) >= lens.view(b, 1, 1, 1)).expand(b, 1, sq, sk).contiguous()
    mask[0, 0, 1] = True  # a row without a visible key
    mask[0, 0, 2, ::3] = True

    def forward(call, want_shape, inplace_of=None):
        if inplace_of is None:
            y, store = at(o, want_shape, dtype, device)
        else:
            y, store = at(i, want_shape, dtype, device, fill=inplace_of)
        _lib.check(call(y))
        assert guarded(y, store), (sk, offsets)
        return y

    cases = {
        "causal": (xt, gt, causal, lambda y, src: lib.neox_causal_softmax_fwd(y.data_ptr(), src.data_ptr(), SCALE, 1, sk, sk, code, stream)),
        "mask": (x, g, mask, lambda y, src: lib.neox_masked_softmax_fwd(
            y.data_ptr(), src.data_ptr(), mask.data_ptr(), SCALE, b, heads, sq, sk, b, code, stream)),
    }
    for kind, (src, grad, hidden, call) in cases.items():
        y = forward(lambda y: call(y, src), src.shape)
        ref = R.softmax_fp32(src.cpu(), hidden.cpu(), SCALE).to(device)
        assert (y.float() - ref).abs().max().item() <= TOL[dtype], (kind, sk, offsets)
        seen = hidden.all(-1, keepdim=True)
        assert (y[hidden.expand_as(y) & ~seen.expand_as(y)] == 0).all(), kind
        inplace = forward(lambda y: call(y, y), src.shape, inplace_of=src)
        if sk % 8 != 0 or i % 8 != 0 or o % 8 == 0:  # (else in place is aligned: another kernel, sums in another order)
            assert torch.equal(inplace, y), kind
        assert (inplace.float() - ref).abs().max().item() <= TOL[dtype], (kind, sk, offsets)
        dx, store = at(o, src.shape, dtype, device)
        same, same_store = at(i, src.shape, dtype, device, fill=grad)
        for out, dy in ((dx, grad), (same, same)):
            if kind == "causal":
                _lib.check(lib.neox_causal_softmax_bwd(out.data_ptr(), dy.data_ptr(), y.data_ptr(), SCALE, 1, sk, sk, code, stream))
            else:
                _lib.check(lib.neox_masked_softmax_bwd(out.data_ptr(), dy.data_ptr(), y.data_ptr(), SCALE, rows, sk, code, stream))
        assert guarded(dx, store) and guarded(same, same_store), (kind, sk, offsets)
        assert torch.equal(dx, same), kind
        yf, gf = y.float(), grad.float()
        auto = SCALE * yf * (gf - (gf * yf).sum(-1, keepdim=True))
        assert_grad(dx, auto, dtype, (kind, sk, offsets), y=y, g=grad, scale=SCALE)

        # what is folded in leaves the sums as they are
        shape4 = tuple(src.shape)
        zero_bias, slopes = torch.zeros(shape4, dtype=dtype, device=device), torch.zeros(shape4[1], device=device)
        for fold in ("alibi", "bias", "dropout"):
            z, zs = at(o, src.shape, dtype, device)
            extra = (slopes.data_ptr() if fold == "alibi" else None, zero_bias.data_ptr() if fold == "bias" else None, shape4[0])
            p = 0.25 if fold == "dropout" else 0.0
            drop, ds = at(o, src.shape, dtype, device)
            if fold == "dropout":
                if kind == "causal":
                    _lib.check(lib.neox_causal_softmax_dropout_fwd(drop.data_ptr(), z.data_ptr(), src.data_ptr(), *extra, SCALE, p, 5, 0, None,
                                                                   *shape4, code, stream))
                else:
                    _lib.check(lib.neox_masked_softmax_dropout_fwd(drop.data_ptr(), z.data_ptr(), src.data_ptr(), mask.data_ptr(), *extra,
                                                                   SCALE, p, 5, 0, None, *shape4, b, code, stream))
                keep = torch.empty(src.numel(), dtype=torch.uint8, device=device)
                _lib.check(lib.neox_dropout_keep_mask(keep.data_ptr(), p, 5, 0, None, src.numel(), stream))
                assert torch.equal(drop, torch.where(keep.view(src.shape).bool(), (y.float() * (1.0 / 0.75)).to(dtype), 0)), kind
            elif kind == "causal":
                if fold == "alibi":
                    _lib.check(lib.neox_causal_softmax_alibi_fwd(z.data_ptr(), src.data_ptr(), extra[0], SCALE, *shape4, code, stream))
                else:
                    _lib.check(lib.neox_causal_softmax_bias_fwd(z.data_ptr(), src.data_ptr(), extra[1], None, SCALE, *shape4, shape4[0], code, stream))
            elif fold == "alibi":
                _lib.check(lib.neox_masked_softmax_alibi_fwd(z.data_ptr(), src.data_ptr(), mask.data_ptr(), extra[0], SCALE, *shape4, b, code, stream))
            else:
                _lib.check(lib.neox_masked_softmax_bias_fwd(z.data_ptr(), src.data_ptr(), mask.data_ptr(), extra[1], None, SCALE, *shape4, b,
                                                            shape4[0], code, stream))
            assert guarded(z, zs) and guarded(drop, ds), (kind, fold, sk)
            assert torch.equal(z, y), (kind, fold, sk, offsets)


class Written:
    """Calls that write guarded outputs: every element of each is written, nothing around it is."""

    def __init__(self, dtype, device, what):
        self.dtype, self.device, self.what = dtype, device, what

    def __call__(self, call, shape, offset, fill=None, outputs=1):
        outs = [at(offset, shape, self.dtype, self.device, fill=fill) for _ in range(outputs)]
        _lib.check(call(*(t for t, _ in outs)))
        for t, store in outs:
            assert guarded(t, store), self.what
            assert not (t == 7.0).any(), self.what  # no probability, and no gradient of these sizes, is 7
        return outs[0][0] if outputs == 1 else [t for t, _ in outs]


def check_backward(written, run, y, g, offsets, dtype):
    """dx into a tensor of its own and over the gradient: the same bits, within the bar of the closed form."""
    i, o = offsets
    dx = written(lambda dx: run(dx, g), g.shape, o)
    assert torch.equal(written(lambda t: run(t, t), g.shape, i, fill=g), dx), written.what
    yf, gf = y.float(), g.float()
    assert_grad(dx, SCALE * yf * (gf - (gf * yf).sum(-1, keepdim=True)), dtype, written.what, y=y, g=g, scale=SCALE)


# as many rows as it takes for the results to leave through LDS, and one case on the other side of each limit: of two chunks in the
# backward pass (from 672 columns on 8192 rows of an even and 28672 of an odd length, 18432 from 768) and in the forward pass (from 944
# columns on 65536, 32768 from 1022), and of two waves per row in the backward pass (8192, 2049 to 2304 columns); the last block is not full
@pytest.mark.parametrize("sk,sq", [(671, 13655), (673, 13655), (673, 6145), (767, 6145), (769, 6145), (1023, 6143), (943, 21847),
                                   (945, 21847), (1001, 21847), (1001, 21845), (673, 9557), (721, 9559), (722, 2729), (722, 2731),
                                   (1021, 10923), (1022, 10921), (1022, 10923), (1535, 2731), (2047, 2731), (2051, 2731),
                                   (2303, 2731)])
@pytest.mark.parametrize("offsets", [(0, 0), (1, 0), (3, 5), (8, 1)])
def test_staged_rows_of_many_rows(device, sk, sq, offsets):
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    dtype = (torch.float16, torch.bfloat16)[(sk // 2 + offsets[0]) % 2]
    code, gen = _lib.dtype_code(dtype), torch.Generator(device=device).manual_seed(sk)
    b = 3
    shape, (i, o) = (b, 1, sq, sk), offsets
    x, _ = at(i, shape, dtype, device, gen=gen, std=8.0)
    g, _ = at(i, shape, dtype, device, gen=gen)
    lens = torch.tensor([sk, sk - 3, sk // 3], device=device)
    mask = (torch.arange(sk, device=device).view(1, 1, 1, sk) >= lens.view(b, 1, 1, 1)).expand(shape).contiguous()
    mask[0, 0, 1] = True  # a row without a visible key
    written = Written(dtype, device, (sk, offsets))

    def forward(y, src):
        return lib.neox_masked_softmax_fwd(y.data_ptr(), src.data_ptr(), mask.data_ptr(), SCALE, b, 1, sq, sk, b, code, stream)

    y = written(lambda y: forward(y, x), shape, o)
    assert (y.float() - R.softmax_fp32(x, mask, SCALE)).abs().max().item() <= TOL[dtype]
    assert torch.equal(written(lambda t: forward(t, t), shape, i, fill=x), y)
    check_backward(written, lambda dx, dy: lib.neox_masked_softmax_bwd(dx.data_ptr(), dy.data_ptr(), y.data_ptr(), SCALE, b * sq, sk, code, stream),
                   y, g, offsets, dtype)


# causal rows likewise: for two chunks in the forward pass 64000 of an odd and 45000 of an even length (from 944 columns on), in the backward
# pass 81920 and 49152 (672), 45056 and 32768 (760), 27648 (896) and 20480 (960); 6400 for the two outputs of dropout, 4608 for two staged waves per row in the backward pass
@pytest.mark.parametrize("sk,n", [(725, 137), (905, 46), (1001, 131), (1001, 129), (673, 121), (673, 122), (674, 73), (769, 58),
                                  (769, 59), (802, 41), (905, 30), (905, 31), (969, 21), (969, 22), (1001, 63), (1001, 65),
                                  (1002, 44), (1002, 45), (1301, 5), (1601, 5), (1855, 5), (2051, 3), (3071, 3)])
@pytest.mark.parametrize("offsets", [(0, 0), (1, 0), (3, 5), (8, 1)])
def test_staged_causal_rows_of_many_rows(device, sk, n, offsets):
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    dtype = (torch.float16, torch.bfloat16)[(sk // 2 + offsets[0]) % 2]
    code, gen = _lib.dtype_code(dtype), torch.Generator(device=device).manual_seed(sk)
    shape, (i, o) = (n, sk, sk), offsets
    x, _ = at(i, shape, dtype, device, gen=gen, std=8.0)
    g, _ = at(i, shape, dtype, device, gen=gen)
    hidden = torch.ones(sk, sk, dtype=torch.bool, device=device).triu_(1)
    written = Written(dtype, device, (sk, offsets))
    y = written(lambda y: lib.neox_causal_softmax_fwd(y.data_ptr(), x.data_ptr(), SCALE, n, sk, sk, code, stream), shape, o)
    assert (y.float() - R.softmax_fp32(x[None], hidden[None, None], SCALE)[0]).abs().max().item() <= TOL[dtype]
    assert torch.equal(written(lambda t: lib.neox_causal_softmax_fwd(t.data_ptr(), t.data_ptr(), SCALE, n, sk, sk, code, stream), shape, i, fill=x), y)

    def dropped(drop, z):
        return lib.neox_causal_softmax_dropout_fwd(drop.data_ptr(), z.data_ptr(), x.data_ptr(), None, None, 0, SCALE, 0.25, 5, 0, None,
                                                   1, n, sk, sk, code, stream)

    drop, z = written(dropped, shape, o, outputs=2)
    keep = torch.empty(x.numel(), dtype=torch.uint8, device=device)
    _lib.check(lib.neox_dropout_keep_mask(keep.data_ptr(), 0.25, 5, 0, None, x.numel(), stream))
    assert torch.equal(z, y)
    assert torch.equal(drop, torch.where(keep.view(shape).bool(), (y.float() * (1.0 / 0.75)).to(dtype), 0))
    check_backward(written, lambda dx, dy: lib.neox_causal_softmax_bwd(dx.data_ptr(), dy.data_ptr(), y.data_ptr(), SCALE, n, sk, sk, code, stream),
                   y, g, offsets, dtype)


# aligned rows that are no whole cache lines, 32768 and more of them: the same kernels.  The last block is not full where rows
# are not a multiple of the length (mask tensor with known row ends)
@pytest.mark.parametrize("sk", [840, 1000, 1032, 1544, 2040])
@pytest.mark.parametrize("offsets", [(0, 0), (8, 24)])
def test_aligned_rows_through_lds(device, sk, offsets):
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    dtype = (torch.float16, torch.bfloat16)[(sk // 8 + offsets[0]) % 2]
    code, gen = _lib.dtype_code(dtype), torch.Generator(device=device).manual_seed(sk)
    sq = 32769
    shape, (i, o) = (1, 1, sq, sk), offsets
    x, _ = at(i, shape, dtype, device, gen=gen, std=8.0)
    g, _ = at(i, shape, dtype, device, gen=gen)
    lens = sk - torch.arange(sq, device=device, dtype=torch.int32) % 37
    mask = (torch.arange(sk, device=device).view(1, sk) >= lens.view(sq, 1)).view(shape)
    written = Written(dtype, device, (sk, offsets))

    def forward(y, src):
        return lib.neox_masked_softmax_ends_fwd(None, y.data_ptr(), src.data_ptr(), mask.data_ptr(), lens.data_ptr(), None, None, 0, SCALE, 0.0,
                                                0, 0, None, 1, 1, sq, sk, 1, code, stream)

    y = written(lambda y: forward(y, x), shape, o)
    assert (y.float() - R.softmax_fp32(x, mask, SCALE)).abs().max().item() <= TOL[dtype]
    assert torch.equal(written(lambda t: forward(t, t), shape, i, fill=x), y)
    check_backward(written, lambda dx, dy: lib.neox_masked_softmax_ends_bwd(dx.data_ptr(), dy.data_ptr(), y.data_ptr(), lens.data_ptr(), SCALE, 0,
                                                                            0.0, 0, 0, None, 1, 1, sq, sk, 1, code, stream), y, g, offsets, dtype)


# the backward pass with dropout ends a row of an even length by the range check, one of an odd length by a lane that is moved
# back: one to sixteen waves per row, fifteen full rows or a causal matrix
@pytest.mark.parametrize("sk", [514, 516, 517, 804, 1020, 1022, 1030, 1031, 1604, 2052, 4100, 4102, 8204, 16386])
@pytest.mark.parametrize("offsets", [(0, 0), (1, 0), (3, 5), (8, 1)])
def test_dropout_backward_of_even_rows(device, sk, offsets):
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    dtype = (torch.float16, torch.bfloat16)[(sk // 2 + offsets[0]) % 2]
    code, gen = _lib.dtype_code(dtype), torch.Generator(device=device).manual_seed(sk)
    i, o = offsets
    written = Written(dtype, device, (sk, offsets))
    for causal, shape in ((False, (15, sk)), (True, (sk, sk))):
        if causal and sk > 4100:
            continue
        probs = torch.empty(shape, device=device).normal_(0.0, 2.0, generator=gen)
        if causal:
            probs = probs.masked_fill(torch.ones(shape, dtype=torch.bool, device=device).triu_(1), float("-inf"))
        y, _ = at(i, shape, dtype, device, fill=torch.softmax(probs, -1))
        g, _ = at(i, shape, dtype, device, gen=gen)
        keep = torch.empty(g.numel(), dtype=torch.uint8, device=device)
        _lib.check(lib.neox_dropout_keep_mask(keep.data_ptr(), 0.25, 5, 0, None, g.numel(), stream))
        gf, yf = torch.where(keep.view(shape).bool(), g.float() * (1.0 / 0.75), 0), y.float()

        def backward(dx, dy):
            if causal:
                return lib.neox_causal_softmax_dropout_bwd(dx.data_ptr(), dy.data_ptr(), y.data_ptr(), SCALE, 0.25, 5, 0, None, 1, *shape, code, stream)
            return lib.neox_masked_softmax_dropout_bwd(dx.data_ptr(), dy.data_ptr(), y.data_ptr(), SCALE, 0.25, 5, 0, None, *shape, code, stream)

        dx = written(lambda dx: backward(dx, g), shape, o)
        assert_grad(dx, SCALE * yf * (gf - (gf * yf).sum(-1, keepdim=True)), dtype, (sk, offsets, causal), y=y, g=gf, scale=SCALE)
        assert torch.equal(written(lambda t: backward(t, t), shape, i, fill=g), dx)


@pytest.mark.parametrize("sk", [513, 1001, 1201, 1999, 3001])
def test_one_ragged_row(device, sk):
    # a single row: the lanes at its ends have no neighbouring row to share anything with
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=device).manual_seed(sk)
    x, _ = at(1, (1, 1, 1, sk), torch.float16, device, gen=gen, std=8.0)
    mask = torch.zeros(1, 1, 1, sk, dtype=torch.bool, device=device)
    mask[..., sk // 2 : sk // 2 + 9] = True
    y, store = at(1, x.shape, torch.float16, device)
    _lib.check(lib.neox_masked_softmax_fwd(y.data_ptr(), x.data_ptr(), mask.data_ptr(), SCALE, 1, 1, 1, sk, 1, _lib.NEOX_F16, stream))
    assert guarded(y, store)
    ref = R.softmax_fp32(x.cpu(), mask.cpu(), SCALE).to(device)
    assert (y.float() - ref).abs().max().item() <= TOL[torch.float16]
