"""Kernel shapes that depend on how many rows a call has, each side of the limits: the first and the last matrices of a call
against the fp32 expression, and bits that must not depend on the shape (a row-end hint, the dropped probabilities' undropped
twin) against each other.
"""
import pytest
import torch

from gpt_neox_amd import _lib
from gpt_neox_amd.fused_kernels import scaled_masked_softmax_cuda as masked_ext
from oracle import torch_ref as R
from bars import TOL, assert_grad

pytestmark = pytest.mark.gpu

SCALE = 0.125
DTYPES = [torch.float16, torch.bfloat16]


def unwritten(like):
    """An output that holds what no kernel writes: every store has to be this call's own."""
    return torch.full_like(like, 7.0)


def normal(shape, dtype, device, seed, std=1.0):
    return torch.empty(shape, dtype=dtype, device=device).normal_(0.0, std, generator=torch.Generator(device=device).manual_seed(seed))


def check(x, y, g, dx, hidden, dtype, what):
    """x, y, g, dx: [batches, s, s] (dx may be None); hidden: [s, s]."""
    for i in {0, x.shape[0] // 2, x.shape[0] - 1}:
        ref = R.softmax_fp32(x[i][None, None], hidden[None, None], SCALE)[0, 0]
        assert (y[i].float() - ref).abs().max().item() <= TOL[dtype], (what, i)
        assert (y[i][hidden] == 0).all(), (what, i)
        if dx is not None:
            yf, gf = y[i].float(), g[i].float()
            auto = SCALE * yf * (gf - (gf * yf).sum(-1, keepdim=True))
            assert_grad(dx[i], auto, dtype, (what, i), y=y[i], g=g[i], scale=SCALE)
            assert (dx[i][hidden] == 0).all(), (what, i)


# rows of three to seven chunks and more, bands of two chunks and more, 8192 rows and more or fewer
@pytest.mark.parametrize("s,w,batches", [(1152, 288, 29), (1152, 288, 2), (1152, 576, 1), (1472, 368, 6), (2048, 384, 4),
                                         (2048, 600, 1), (2048, 1024, 1), (2560, 256, 4), (2560, 700, 1), (2560, 1600, 1),
                                         (3072, 600, 3), (3072, 600, 2), (3072, 1400, 3), (3584, 1200, 3), (3584, 1792, 1),
                                         (4096, 200, 2), (4096, 200, 1), (4096, 600, 1), (4096, 700, 2), (4096, 1100, 1),
                                         (4096, 2600, 1), (4608, 400, 2), (4616, 400, 2), (1504, 200, 6), (1504, 300, 6),
                                         (2816, 200, 3), (9216, 200, 1), (6144, 3000, 1), (8192, 256, 1), (8192, 1600, 1)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_sliding_window_shapes_by_rows(device, s, w, batches, dtype):
    lib, stream, code = _lib.lib(), torch.cuda.current_stream().cuda_stream, _lib.dtype_code(dtype)
    x, g = normal((batches, s, s), dtype, device, s, 8.0), normal((batches, s, s), dtype, device, w)
    y, dx = unwritten(x), unwritten(x)
    _lib.check(lib.neox_sliding_window_softmax_fwd(y.data_ptr(), x.data_ptr(), SCALE, batches, s, s, w, code, stream))
    _lib.check(lib.neox_sliding_window_softmax_bwd(dx.data_ptr(), g.data_ptr(), y.data_ptr(), SCALE, batches, s, s, w, code, stream))
    check(x, y, g, dx, R.get_attn_mask(s, device, sliding_window_width=w)[0, 0], dtype, (s, w))


# 513-1024 columns with the loads in front or not; above 1024, 2048 and 4096 columns in the backward pass; rows that are no whole
# cache lines, 32768 of them or fewer; odd rows, 2048 / 4608 / 6400 / 8192 of them or fewer
@pytest.mark.parametrize("s,batches", [(576, 1), (888, 6), (1024, 5), (1088, 5), (1088, 4), (1088, 16), (1088, 17), (1088, 33),
                                       (1088, 34), (1088, 18), (1088, 19), (1184, 15), (1184, 16), (1184, 31), (1184, 32),
                                       (1304, 29), (2112, 3), (2112, 2), (2112, 5), (2824, 4), (2848, 3), (2848, 4), (2944, 4),
                                       (3072, 3), (4160, 1), (5136, 1), (5696, 1), (5704, 1), (520, 64), (520, 63), (1000, 33),
                                       (1032, 32), (1416, 24), (1480, 23), (1488, 23), (2056, 16), (3064, 11), (1001, 9), (1001, 8),
                                       (1301, 5), (1301, 4), (1601, 2), (1601, 1), (1801, 4), (1801, 3), (1801, 2), (2051, 3),
                                       (2051, 2), (4101, 1)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_causal_shapes_by_rows(device, s, batches, dtype):
    lib, stream, code = _lib.lib(), torch.cuda.current_stream().cuda_stream, _lib.dtype_code(dtype)
    x, g = normal((batches, s, s), dtype, device, s, 8.0), normal((batches, s, s), dtype, device, s + 1)
    y, dx, z, drop = (unwritten(x) for _ in range(4))
    _lib.check(lib.neox_causal_softmax_fwd(y.data_ptr(), x.data_ptr(), SCALE, batches, s, s, code, stream))
    _lib.check(lib.neox_causal_softmax_bwd(dx.data_ptr(), g.data_ptr(), y.data_ptr(), SCALE, batches, s, s, code, stream))
    hidden = torch.ones(s, s, dtype=torch.bool, device=device).triu_(1)
    check(x, y, g, dx, hidden, dtype, s)
    # with dropout: the same undropped bits, and the gradient of what was kept
    _lib.check(lib.neox_causal_softmax_dropout_fwd(drop.data_ptr(), z.data_ptr(), x.data_ptr(), None, None, 0, SCALE, 0.25, 7, 0, None,
                                                   1, batches, s, s, code, stream))
    assert torch.equal(z, y)
    keep = torch.empty(x.numel(), dtype=torch.uint8, device=device)
    _lib.check(lib.neox_dropout_keep_mask(keep.data_ptr(), 0.25, 7, 0, None, x.numel(), stream))
    keep = keep.view(x.shape).bool()
    assert torch.equal(drop, torch.where(keep, (y.float() * (1.0 / 0.75)).to(dtype), 0))
    dx.fill_(7.0)
    _lib.check(lib.neox_causal_softmax_dropout_bwd(dx.data_ptr(), g.data_ptr(), y.data_ptr(), SCALE, 0.25, 7, 0, None, batches, s, s, code, stream))
    for i in {0, batches - 1}:
        yf, gf = y[i].float(), torch.where(keep[i], g[i].float() * (1.0 / 0.75), 0)
        assert_grad(dx[i], SCALE * yf * (gf - (gf * yf).sum(-1, keepdim=True)), dtype, (s, i), y=y[i], g=gf, scale=SCALE)
    # slopes of zero: the same sums
    slopes = torch.zeros(batches, device=device)
    z.fill_(7.0)
    _lib.check(lib.neox_causal_softmax_alibi_fwd(z.data_ptr(), x.data_ptr(), slopes.data_ptr(), SCALE, 1, batches, s, s, code, stream))
    assert torch.equal(z, y)


@pytest.mark.parametrize("s,heads", [(840, 20), (1000, 17), (1032, 16), (1544, 11), (2040, 9), (1001, 17), (2112, 4), (2112, 1), (4160, 1), (2051, 4), (2051, 1)])
def test_row_ends_of_many_rows(device, s, heads):
    # two samples, the second one padded: the hint changes what is fetched and may change the kernel, never the bits
    dtype, b = DTYPES[s % 2], 2
    x, g = normal((b, heads, s, s), dtype, device, s, 8.0), normal((b, heads, s, s), dtype, device, s + 1)
    lens = torch.tensor([s, s // 3], device=device)
    mask = (torch.arange(s, device=device).view(1, 1, 1, s) >= lens.view(b, 1, 1, 1)).expand(b, 1, s, s).contiguous()
    ends = masked_ext.scan_mask(mask)[1]
    y = masked_ext.forward(x, mask, SCALE)
    assert torch.equal(masked_ext.forward(x, mask, SCALE, row_end=ends), y)
    hinted = masked_ext.backward(g.clone(), y, SCALE, row_end=ends)
    assert torch.equal(masked_ext.backward(g.clone(), y, SCALE), hinted)
    for i in range(b):
        check(x[i], y[i], g[i], hinted[i], mask[i, 0], dtype, (s, heads, i))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("s,heads", [(1301, 5), (1301, 2), (1601, 4), (1601, 2)])
def test_features_of_one_wave_rows(device, s, heads, dtype):
    # every combination of what folds into the causal forward pass, 6400 rows or fewer: zero slopes and a zero bias give the
    # plain bits, and the dropped output follows from them
    lib, stream, code = _lib.lib(), torch.cuda.current_stream().cuda_stream, _lib.dtype_code(dtype)
    x = normal((1, heads, s, s), dtype, device, s, 8.0)
    y, z, drop = (unwritten(x) for _ in range(3))
    _lib.check(lib.neox_causal_softmax_fwd(y.data_ptr(), x.data_ptr(), SCALE, heads, s, s, code, stream))
    slopes, bias = torch.zeros(heads, device=device), torch.zeros_like(x)
    keep = torch.empty(x.numel(), dtype=torch.uint8, device=device)
    _lib.check(lib.neox_dropout_keep_mask(keep.data_ptr(), 0.25, 9, 0, None, x.numel(), stream))
    want = torch.where(keep.view(x.shape).bool(), (y.float() * (1.0 / 0.75)).to(dtype), 0)
    for sl in (None, slopes.data_ptr()):
        for bi in (None, bias.data_ptr()):
            z.fill_(7.0)
            if bi is not None:
                _lib.check(lib.neox_causal_softmax_bias_fwd(z.data_ptr(), x.data_ptr(), bi, sl, SCALE, 1, heads, s, s, 1, code, stream))
                assert torch.equal(z, y)
            z.fill_(7.0)
            drop.fill_(7.0)
            _lib.check(lib.neox_causal_softmax_dropout_fwd(drop.data_ptr(), z.data_ptr(), x.data_ptr(), sl, bi, 1 if bi else 0, SCALE, 0.25, 9, 0,
                                                           None, 1, heads, s, s, code, stream))
            assert torch.equal(z, y) and torch.equal(drop, want)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("s,batches", [(1301, 7), (1301, 1), (1601, 6), (1601, 1), (2051, 4), (2112, 1), (4160, 1), (5632, 1), (5633, 1)])
def test_full_row_backward_by_rows(device, s, batches, dtype):
    # plain and with dropout, 8192 rows or fewer
    lib, stream, code = _lib.lib(), torch.cuda.current_stream().cuda_stream, _lib.dtype_code(dtype)
    y = torch.softmax(normal((batches, s, s), torch.float32, device, s, 2.0), -1).to(dtype)
    g, dx = normal((batches, s, s), dtype, device, s + 1), unwritten(y)
    keep = torch.empty(g.numel(), dtype=torch.uint8, device=device)
    _lib.check(lib.neox_dropout_keep_mask(keep.data_ptr(), 0.25, 3, 0, None, g.numel(), stream))
    kept = torch.where(keep.view(g.shape).bool(), g.float() * (1.0 / 0.75), 0)
    for p, gf in ((0.0, g.float()), (0.25, kept)):
        dx.fill_(7.0)
        if p:
            _lib.check(lib.neox_masked_softmax_dropout_bwd(dx.data_ptr(), g.data_ptr(), y.data_ptr(), SCALE, p, 3, 0, None, batches * s, s, code, stream))
        else:
            _lib.check(lib.neox_masked_softmax_bwd(dx.data_ptr(), g.data_ptr(), y.data_ptr(), SCALE, batches * s, s, code, stream))
        for i in {0, batches - 1}:
            yf = y[i].float()
            assert_grad(dx[i], SCALE * yf * (gf[i] - (gf[i] * yf).sum(-1, keepdim=True)), dtype, (s, p, i), y=y[i], g=gf[i], scale=SCALE)
