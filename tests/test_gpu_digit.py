"""The digit kernels (exact products on the 8-bit matrix cores) at the edges of
their tiles, slices and groups, against 64-bit sums.

An output sums K products whose activations are fixed point to 2^-30 of their
chunk's (or vector's) largest magnitude, or as they are, and ceil(K / 128) chunk sums
rounded to fp32: the bound is that rounding over the sum of the chunks'
magnitudes, plus the FWHT's 10 roundings where the call rotates."""
import numpy as np
import pytest
import torch

import lutmac_amd as L
from lutmac_amd import synth

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def fwht64(x):
    y = x.reshape(-1, 256).astype(np.float64).copy()
    h = 1
    while h < 256:
        y = y.reshape(-1, 256 // (2 * h), 2, h)
        y = np.stack([y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]], axis=2).reshape(-1, 256)
        h *= 2
    return y.reshape(x.shape) / 16


def check(fmt, planes, scales, rows, cols, group, x, y, rotate, bias=None):
    """y [batch, rows] of x [batch, cols] within the derived bound (cols a multiple of 256 when rotating)."""
    W = synth.dequant_f64(fmt, planes, scales, rows, cols, group)
    xr = fwht64(x) if rotate else x.astype(np.float64)
    ref = xr @ W.T
    mag = np.abs(xr) @ np.abs(W).T
    big = np.abs(xr).max(axis=1, keepdims=True) * np.abs(W).sum(axis=1)[None, :]
    chunks = -(-cols // 128) + 18 * L.STAGES[fmt]     # the running sum, the wave and slice sums, scales and joins
    bound = (chunks + (20 if rotate else 0)) * EPS * mag + 2.0 ** -29 * big
    if rotate:
        bound = bound + 10 * EPS * np.abs(x).sum(axis=1, keepdims=True) * np.abs(W).max()
    if bias is not None:
        ref = ref + bias
        bound = bound + EPS * np.abs(ref)
    err = np.abs(y - ref)
    worst = float((err - bound).max())
    assert worst <= 0, (L.FORMAT_NAMES[fmt], rows, cols, x.shape[0], worst, float(err.max()))


def make(fmt, rows, cols, seed, group=128):
    planes, scales, g = synth.make_weights(fmt, rows, cols, seed=seed, group=group)
    return planes, scales, g, L.Weight.from_planes(fmt, planes, scales, rows, cols, g)


def vectors(batch, cols, seed):
    return np.stack([synth.make_activations(cols, seed=seed + i, outliers=True) for i in range(batch)])


# 1..4 vectors take one launch (the 1-3 bit formats from 2), more the split
# vectors: quads and groups of quads partly filled, rows past the last tile,
# a K of one 256-chunk, of more waves than chunks, and of several rounds.
@pytest.mark.parametrize("fmt", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("rows,cols", [(1, 256), (65, 768), (300, 2048), (130, 8960)])
@pytest.mark.parametrize("batch", [1, 2, 4, 5, 9, 17])
def test_digit_linear(cuda, fmt, rows, cols, batch):
    planes, scales, g, w = make(fmt, rows, cols, seed=rows + cols + fmt)
    x = vectors(batch, cols, seed=batch)
    bias = np.random.default_rng(3).standard_normal(rows).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    y = w.linear(xd, bias=torch.from_numpy(bias).cuda()).cpu().numpy().reshape(batch, rows)
    check(fmt, planes, scales, rows, cols, g, x, y, rotate=fmt in (1, 2, 3, 4), bias=bias)
    w.close()


# From 8192 rows a workgroup takes two row tiles, if its waves have a thread for
# each output of 4 vectors, and from 10240 rows and 2048 columns four.
@pytest.mark.parametrize("fmt", [1, 3, 6, 7])
@pytest.mark.parametrize("rows,cols", [(8190, 256), (8190, 512), (10230, 2048)])
@pytest.mark.parametrize("batch", [3, 4])
def test_digit_many_rows(cuda, fmt, rows, cols, batch):
    planes, scales, g, w = make(fmt, rows, cols, seed=cols + fmt)
    x = vectors(batch, cols, seed=batch)
    y = torch.full((batch, rows), torch.nan, device="cuda")
    w.linear(torch.from_numpy(x).cuda(), y=y)
    check(fmt, planes, scales, rows, cols, g, x, y.cpu().numpy(), rotate=fmt in (1, 2, 3, 4))
    w.close()


# Split vectors: one case per tile size of the rows kernel (1, 2, 4 quads, 1 or
# 2 row tiles), then of the tile kernel (4 quads and halves of k, even and
# uneven; 4 quads; 8 quads), last row and vector groups partly filled, and a
# group scale of three chunks.
@pytest.mark.parametrize("fmt", [1, 3, 4, 6, 7])
@pytest.mark.parametrize("rows,cols,batch,group", [
    (2040, 512, 13, 128), (2600, 768, 9, 384), (4090, 512, 13, 128), (4090, 512, 30, 128),
    (2040, 512, 353, 128), (6100, 768, 129, 384), (16380, 512, 70, 128), (16380, 512, 125, 128)])
def test_digit_tiles(cuda, fmt, rows, cols, batch, group):
    planes, scales, g, w = make(fmt, rows, cols, seed=7 + fmt, group=group)
    x = vectors(batch, cols, seed=50)
    y = w.gemv(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, rows)
    check(fmt, planes, scales, rows, cols, g, x, y, rotate=False)
    w.close()


# A handful of rows over a long K: the k-slices of a row block are summed by
# its last workgroup, whose ticket is back at zero for the next call.
def test_digit_slices_repeat(cuda):
    planes, scales, g, w = make(L.FMT_INT4, 200, 8192, seed=1)
    x = vectors(6, 8192, seed=2)
    xd = torch.from_numpy(x).cuda()
    first = w.gemv(xd).cpu().numpy()
    check(L.FMT_INT4, planes, scales, 200, 8192, g, x, first.reshape(6, 200), rotate=False)
    for _ in range(3):
        assert np.array_equal(w.gemv(xd).cpu().numpy().view(np.uint32), first.view(np.uint32))
    w.close()


# Activations far from 1 (the fixed point follows the exponent), all zero, and
# not finite: such a vector gives NaN in every row, the others are untouched.
@pytest.mark.parametrize("batch", [1, 3, 6])
def test_digit_ranges(cuda, batch):
    rows, cols = 96, 512
    planes, scales, g, w = make(L.FMT_INT4, rows, cols, seed=5)
    base = vectors(batch, cols, seed=9)
    for factor in (2.0 ** 100, 2.0 ** -90):
        x = (base * np.float32(factor)).astype(np.float32)
        y = w.gemv(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, rows)
        check(L.FMT_INT4, planes, scales, rows, cols, g, x, y, rotate=False)
    assert not w.gemv(torch.zeros(batch * cols, device="cuda")).any()
    for bad in (float("inf"), float("nan")):
        x = base.copy()
        x[0, 77] = bad
        y = w.gemv(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, rows)
        assert np.isnan(y[0]).all()
        if batch > 1:
            check(L.FMT_INT4, planes, scales, rows, cols, g, x[1:], y[1:], rotate=False)
    w.close()


# x of any 4-byte alignment and a column count that is no multiple of 4
def test_digit_unaligned(cuda):
    rows, cols, batch = 70, 1000, 7
    planes, scales, g, w = make(L.FMT_INT8, rows, cols, seed=6)
    x = vectors(batch, cols, seed=3)
    buf = torch.empty(batch * cols + 1, device="cuda")
    buf[1:] = torch.from_numpy(x.ravel()).cuda()
    y = w.gemv(buf[1:]).cpu().numpy().reshape(batch, rows)
    check(L.FMT_INT8, planes, scales, rows, cols, g, x, y, rotate=False)
    w.close()


# Captured and replayed with eager calls between, one shape of each kernel
@pytest.mark.parametrize("rows,cols,batch", [(512, 2048, 1), (512, 2048, 4), (512, 8192, 16), (2048, 512, 400)])
def test_digit_graph(cuda, rows, cols, batch):
    planes, scales, g, w = make(L.FMT_INT4, rows, cols, seed=8)
    x = torch.randn(batch * cols, device="cuda")
    eager = w.gemv(x).clone()
    out = torch.empty_like(eager)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        w.gemv(x, out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        w.gemv(x)
        torch.cuda.synchronize()
    w.close()


# The digits' products with codes read from the planes (no handle, so no code
# copy; 8 bits: one vector of a handle too): the handle's bits, for one and two
# row tiles, one and more 256-chunks per wave, the last of them alone.
@pytest.mark.parametrize("fmt", [L.FMT_INT4, L.FMT_INT8])
@pytest.mark.parametrize("rows,cols", [(70, 256), (300, 2560), (8190, 1000), (130, 8960), (65, 16640)])
@pytest.mark.parametrize("batch", [1, 3])
def test_digit_codes_from_planes(cuda, fmt, rows, cols, batch):
    planes, scales, g, w = make(fmt, rows, cols, seed=rows + cols)
    tiles = torch.from_numpy(L.tile_planes(fmt, planes, rows, cols)).cuda()
    sc = torch.from_numpy(L.tile_scales(fmt, scales, rows, cols, g)).cuda()
    x = torch.from_numpy(vectors(batch, cols, seed=rows)).cuda()
    y = torch.full((batch * rows,), torch.nan, device="cuda")
    L.gemv_tiles_noalloc(fmt, tiles, sc, rows, cols, g, x, y, batch)
    a = w.gemv(x)
    assert torch.equal(y, a)
    check(fmt, planes, scales, rows, cols, g, x.cpu().numpy(), a.cpu().numpy().reshape(batch, rows), rotate=False)
    w.close()


# One channel far above the rest, which the rows have no weight for (the planes'
# code of 0 in its columns): what it leaves of the other channels counts in full.
# An output is then off by the rounding of its own terms alone, each 128-chunk's
# fixed point relative to that chunk's largest.
def zero_columns(fmt, planes, cols):
    """The code of weight 0 in these columns of canonical planes."""
    one = {L.FMT_TERNARY: 1, L.FMT_INT4: 3}.get(fmt)      # the one plane whose bit is set there
    for k in cols:
        bit = 1 << (7 - k % 8)
        planes[:, :, k // 8] &= 255 - bit
        if one is not None:
            planes[one, :, k // 8] |= bit
    return planes


SPIKES = [2.0 ** 10, 2.0 ** 20, 1e10]


@pytest.mark.parametrize("fmt", [L.FMT_TERNARY, L.FMT_INT4, L.FMT_INT8])
@pytest.mark.parametrize("spike", SPIKES)
@pytest.mark.parametrize("rows,cols,batch", [(2050, 512, 1), (2050, 512, 3), (1030, 1024, 11), (16380, 512, 70),
                                             (6100, 1280, 129)])
def test_digit_far_channel_in_another_chunk(cuda, fmt, spike, rows, cols, batch):
    planes, scales, g = synth.make_weights(fmt, rows, cols, seed=rows + fmt, group=128)
    zero_columns(fmt, planes, range(128, 256))
    w = L.Weight.from_planes(fmt, planes, scales, rows, cols, g)
    x = np.random.default_rng(batch).standard_normal((batch, cols)).astype(np.float32)
    x[:, 200] = spike
    y = w.gemv(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, rows)
    W = synth.dequant_f64(fmt, planes, scales, rows, cols, g)
    err = np.abs(y - x.astype(np.float64) @ W.T)
    xc, wc = np.abs(x).reshape(batch, -1, 128), np.abs(W).reshape(rows, -1, 128)
    big = xc.max(axis=2) @ wc.sum(axis=2).T
    bound = (cols // 128 + 18) * EPS * (np.abs(x).astype(np.float64) @ np.abs(W).T) + 2.0 ** -30 * big
    assert (err <= bound).all(), float((err / bound).max())
    w.close()


# The same within the channel's own chunk: the others are either rounded to
# 2^-31 of a power of two less than 2^8 above most lanes' largest, or kept as
# they are.  So the bound holds no term of the far channel.
@pytest.mark.parametrize("fmt", [L.FMT_TERNARY, L.FMT_INT4, L.FMT_INT8])
@pytest.mark.parametrize("spike", SPIKES)
@pytest.mark.parametrize("rows,cols,batch", [(2050, 512, 1), (70, 8960, 1), (2050, 512, 3), (10230, 2048, 4),
                                             (1030, 1024, 11), (130, 8192, 22), (16380, 512, 70), (6100, 1280, 129)])
def test_digit_far_channel(cuda, fmt, spike, rows, cols, batch):
    planes, scales, g = synth.make_weights(fmt, rows, cols, seed=rows + fmt, group=128)
    zero_columns(fmt, planes, [200, 511])
    w = L.Weight.from_planes(fmt, planes, scales, rows, cols, g)
    x = np.random.default_rng(batch).standard_normal((batch, cols)).astype(np.float32)
    rest = np.abs(x).max()
    x[::2, 200] = spike      # a vector with and one without, in the same quad
    x[:, 511] = -3.0 * spike
    y = w.gemv(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, rows)
    W = synth.dequant_f64(fmt, planes, scales, rows, cols, g)
    err = np.abs(y - x.astype(np.float64) @ W.T)
    mag = np.abs(x).astype(np.float64) @ np.abs(W).T
    # a chunk kept as it is adds 32 products a lane and four lanes in fp32
    bound = (cols // 128 + 18 + 34) * EPS * mag + 2.0 ** -31 * 2.0 ** 8 * rest * np.abs(W).sum(axis=1)
    assert (err <= bound).all(), float((err / bound).max())
    # the error of fp32 sums of the same terms, which the far channel is none of
    fp32 = np.linalg.norm(y - x.astype(np.float64) @ W.T) / np.linalg.norm(x.astype(np.float64) @ W.T)
    assert fp32 < 3e-7, fp32
    w.close()


# Activations below the smallest power the fixed point can be relative to (2^-97)
# are multiplied in fp32: all of them (2^-112), or those of one chunk.
@pytest.mark.parametrize("rows,cols,batch", [(96, 512, 1), (96, 512, 3), (96, 512, 6), (16380, 512, 70)])
def test_digit_tiny(cuda, rows, cols, batch):
    planes, scales, g, w = make(L.FMT_INT4, rows, cols, seed=5)
    x = (vectors(batch, cols, seed=9) * np.float32(2.0 ** -112)).astype(np.float32)
    y = w.gemv(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, rows)
    ref = x.astype(np.float64) @ synth.dequant_f64(L.FMT_INT4, planes, scales, rows, cols, g).T
    # sums of `cols` terms, and 2^-149 for each product and sum that may be subnormal
    mag = np.abs(x).astype(np.float64) @ np.abs(synth.dequant_f64(L.FMT_INT4, planes, scales, rows, cols, g)).T
    assert (np.abs(y - ref) <= (cols // 128 + 52) * EPS * mag + 2 * cols * 2.0 ** -149).all()
    x[:, 128:256] = vectors(batch, cols, seed=10)[:, :128]
    y = w.gemv(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, rows)
    check(L.FMT_INT4, planes, scales, rows, cols, g, x, y, rotate=False)
    w.close()


# A last chunk of few columns: 8 beside outliers elsewhere, which make no vector
# far, and 8 of which one is far above the others.
@pytest.mark.parametrize("rows,cols,batch", [(70, 1032, 1), (70, 1032, 3), (70, 1032, 9), (16380, 520, 70), (16380, 8, 70),
                                             (70, 8, 2), (70, 8, 1), (70, 8, 7)])
def test_digit_short_last_chunk(cuda, rows, cols, batch):
    planes, scales, g = synth.make_weights(L.FMT_INT4, rows, cols, seed=6, group=128)
    zero_columns(L.FMT_INT4, planes, [cols - 3])
    w = L.Weight.from_planes(L.FMT_INT4, planes, scales, rows, cols, g)
    W = synth.dequant_f64(L.FMT_INT4, planes, scales, rows, cols, g)
    x = vectors(batch, cols, seed=11)
    y = w.gemv(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, rows)
    check(L.FMT_INT4, planes, scales, rows, cols, g, x, y, rotate=False)
    x[:, cols - 3] = 1e10
    y = w.gemv(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, rows)
    rest = np.abs(np.delete(x, cols - 3, axis=1)).max()
    mag = np.abs(x).astype(np.float64) @ np.abs(W).T
    bound = (cols // 128 + 53) * EPS * mag + 2.0 ** -31 * 2.0 ** 8 * rest * np.abs(W).sum(axis=1)
    assert (np.abs(y - x.astype(np.float64) @ W.T) <= bound).all()
    w.close()
