"""The network's convolution kernels at the edges of their tiles (image sides and
channel counts that leave remainders, one pixel, one and several patches per
block; every tile shape and the direct kernel), each against a plain float64 product
of the same bf16 operands.
Tolerances are the rounding bound of an fp32 sum of n products in any order,
n 2^-23 sum |a b|, and half a bf16 step for bf16 results."""
import numpy as np
import pytest

from oracle.unet_ref import bf16
from fvmic2d_amd.lib import Context
from fvmic2d_amd.unet import Buf, UNet, bind, from_bf16_bits, to_bf16_bits

pytestmark = pytest.mark.gpu


def _dev(ctx, a, dtype):
    b = Buf(ctx, a.shape, dtype)
    b.set(to_bf16_bits(a) if dtype == np.uint16 else a)
    return b


def _taps(x, K):
    """x (B, H, W, C) -> list over taps of x shifted by the tap's offset, zero outside."""
    h = K // 2
    p = np.pad(x, ((0, 0), (h, h), (h, h), (0, 0)))
    H, W = x.shape[1:3]
    return [p[:, t // K:t // K + H, t % K:t % K + W] for t in range(K * K)]


SHAPES = [(1, 1, 1, 16, 16, 3), (1, 5, 16, 16, 32, 3), (2, 16, 16, 32, 16, 1), (1, 17, 33, 48, 48, 3),
          (3, 15, 9, 32, 64, 3), (1, 16, 20, 96, 32, 3), (2, 40, 35, 16, 16, 3), (1, 8, 8, 256, 128, 3),
          (5, 33, 18, 64, 16, 1)]
# The shapes above are too few pixels for any but the smallest tile; these reach one
# kernel each (tile rows, channel tiles, wavefronts side by side of the dispatch), with
# image sides and output channels that leave remainders.
TILES = {
    "3x3 rows 4, 2 x 2": (33, 17, 19, 32, 80, 3), "3x3 rows 2, 2 x 2": (33, 17, 19, 64, 80, 3),
    "3x3 rows 1, 2 x 2": (24, 9, 19, 96, 80, 3), "3x3 rows 4, 2 x 1": (64, 17, 19, 32, 48, 3),
    "3x3 rows 2, 2 x 1": (64, 9, 19, 96, 48, 3), "3x3 rows 4, 1 x 1": (130, 17, 19, 32, 16, 3),
    "3x3 rows 1, 1 x 2": (20, 7, 19, 64, 48, 3), "3x3 many slabs": (7, 21, 19, 640, 144, 3),
    "3x3 direct": (2, 9, 11, 768, 48, 3),
    "1x1 rows 4, 2 x 2": (33, 17, 19, 48, 80, 1), "1x1 rows 2, 2 x 2": (33, 9, 19, 160, 80, 1),
    "1x1 rows 1, 2 x 2": (24, 9, 19, 224, 80, 1), "1x1 rows 4, 2 x 1": (66, 17, 19, 64, 48, 1),
    "1x1 rows 2, 2 x 1": (66, 9, 19, 160, 48, 1), "1x1 rows 4, 1 x 1": (130, 17, 19, 16, 16, 1),
    "1x1 rows 1, 1 x 2": (20, 7, 19, 64, 48, 1), "1x1 direct, many slabs": (40, 17, 19, 528, 80, 1),
    "1x1 direct, large image": (1, 259, 257, 32, 80, 1),
}


def _operands(shape, seed=0):
    B, H, W, ci, co, K = shape
    r = np.random.default_rng(seed)
    X = bf16(r.standard_normal((B, H, W, ci)).astype(np.float32))
    Wt = bf16((r.standard_normal((K * K, co, ci)) / np.sqrt(K * K * ci)).astype(np.float32))
    dY = bf16(r.standard_normal((B, H, W, co)).astype(np.float32))
    return X, Wt, dY


@pytest.mark.parametrize("shape", SHAPES)
def test_weight_gradient(shape):
    print("CASE wgrad", shape, flush=True)
    B, H, W, ci, co, K = shape
    X, _, dY = _operands(shape)
    ctx, lib = Context(), bind()
    dX, ddY = _dev(ctx, X, np.uint16), _dev(ctx, dY, np.uint16)
    dW, db = Buf(ctx, (K * K, co, ci), np.float32), Buf(ctx, (co,), np.float32)
    ws = Buf(ctx, (lib.fvm_nn_wgrad_workspace(B, H, W, ci, co, K) // 4,), np.float32)
    assert lib.fvm_nn_conv_wgrad(ctx.h, dX.ptr, ddY.ptr, B, H, W, ci, co, K, ws.ptr, dW.ptr, db.ptr) == 0
    flat = dY.reshape(-1, co).astype(np.float64)
    n = flat.shape[0]
    got = dW.get()
    for t, x in enumerate(_taps(X, K)):
        x = x.reshape(-1, ci).astype(np.float64)
        assert np.all(np.abs(got[t] - flat.T @ x) <= n * 2.0 ** -23 * (np.abs(flat).T @ np.abs(x)) + 1e-30), t
    assert np.all(np.abs(db.get() - flat.sum(0)) <= n * 2.0 ** -23 * np.abs(flat).sum(0) + 1e-30)


def test_weight_gradient_takes_any_even_address():
    """Operands that start between 16-byte boundaries, as views of a larger array may."""
    print("CASE wgrad unaligned", flush=True)
    B, H, W, ci, co, K = shape = (1, 9, 10, 16, 16, 3)
    X, _, dY = _operands(shape, 3)
    ctx, lib = Context(), bind()
    outs = []
    for off in (0, 1):
        dX, ddY = Buf(ctx, (X.size + 8,), np.uint16), Buf(ctx, (dY.size + 8,), np.uint16)
        for buf, a in ((dX, X), (ddY, dY)):
            full = np.zeros(a.size + 8, np.uint16)
            full[off:off + a.size] = to_bf16_bits(a).ravel()
            buf.set(full)
        n = K * K * co * ci
        dW, db = Buf(ctx, (n + 4,), np.float32), Buf(ctx, (co + 4,), np.float32)
        ws = Buf(ctx, (lib.fvm_nn_wgrad_workspace(B, H, W, ci, co, K) // 4 + 4,), np.float32)
        assert lib.fvm_nn_conv_wgrad(ctx.h, dX.ptr + 2 * off, ddY.ptr + 2 * off, B, H, W, ci, co, K, ws.ptr + 4 * off,
                                     dW.ptr + 4 * off, db.ptr + 4 * off) == 0
        outs.append((dW.get()[off:off + n], db.get()[off:off + co]))
    assert np.array_equal(outs[0][0], outs[1][0]) and np.array_equal(outs[0][1], outs[1][1])


def _check_bf16(got, ref, bound):
    assert np.all(np.abs(got - ref) <= bound + 2.0 ** -8 * (np.abs(ref) + bound)), np.abs(got - ref).max()


@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_forward(shape, relu):
    print("CASE conv", shape, relu, flush=True)
    B, H, W, ci, co, K = shape
    X, Wt, _ = _operands(shape, 1)
    b = np.random.default_rng(2).standard_normal(co).astype(np.float32)
    ctx, lib = Context(), bind()
    dX, dW, dB = _dev(ctx, X, np.uint16), _dev(ctx, Wt, np.uint16), _dev(ctx, b, np.float32)
    Y, Yf = Buf(ctx, (B, H, W, co), np.uint16), Buf(ctx, (B, H, W, co), np.float32)
    real = co - 5
    assert lib.fvm_nn_conv_fwd(ctx.h, dX.ptr, dW.ptr, dB.ptr, B, H, W, ci, co, K, relu, real, Y.ptr, Yf.ptr) == 0
    ref, mag = np.zeros((B, H, W, co)), np.zeros((B, H, W, co))
    for t, x in enumerate(_taps(X, K)):
        w = Wt[t].astype(np.float64).T
        ref += x.astype(np.float64) @ w
        mag += np.abs(x) @ np.abs(w)
    ref, mag = ref + b, mag + np.abs(b)
    if relu:
        ref = np.maximum(ref, 0.0)
    ref[..., real:], mag[..., real:] = 0.0, 0.0
    bound = (K * K * ci + 1) * 2.0 ** -23 * mag
    assert np.all(np.abs(Yf.get() - ref) <= bound)
    _check_bf16(from_bf16_bits(Y.get()), ref, bound)


@pytest.mark.parametrize("shape", SHAPES)
def test_data_gradient(shape):
    print("CASE dgrad", shape, flush=True)
    B, H, W, ci, co, K = shape
    _, Wt, dY = _operands(shape, 4)
    ctx, lib = Context(), bind()
    ddY, dW = _dev(ctx, dY, np.uint16), _dev(ctx, Wt, np.uint16)
    scratch, dX = Buf(ctx, (K * K * co * ci,), np.uint16), Buf(ctx, (B, H, W, ci), np.uint16)
    assert lib.fvm_nn_conv_dgrad(ctx.h, ddY.ptr, dW.ptr, scratch.ptr, B, H, W, ci, co, K, dX.ptr) == 0
    ref, mag = np.zeros((B, H, W, ci)), np.zeros((B, H, W, ci))
    for t, y in enumerate(_taps(dY, K)):
        w = Wt[K * K - 1 - t].astype(np.float64)
        ref += y.astype(np.float64) @ w
        mag += np.abs(y) @ np.abs(w)
    _check_bf16(from_bf16_bits(dX.get()), ref, K * K * co * 2.0 ** -23 * mag)


@pytest.mark.parametrize("tile", TILES)
def test_forward_of_each_tile(tile):
    test_forward(TILES[tile], 1)


@pytest.mark.parametrize("tile", TILES)
def test_data_gradient_of_each_tile(tile):
    B, H, W, ci, co, K = TILES[tile]
    test_data_gradient((B, H, W, co, ci, K))    # the kernel's input is the layer's output


@pytest.mark.parametrize("tile", ["3x3 rows 1, 2 x 2", "3x3 many slabs", "1x1 rows 1, 2 x 2", "3x3 rows 4, 2 x 2"])
def test_weight_gradient_of_wide_layers(tile):
    test_weight_gradient(TILES[tile])


@pytest.mark.parametrize("tile", TILES)
def test_an_image_alone_gives_the_same_bits(tile):
    """The order of an output's sums does not depend on the tile, so the last image
    of a batch comes out alike by itself, where fewer pixels take a smaller one."""
    print("CASE conv alone", tile, flush=True)
    B, H, W, ci, co, K = TILES[tile]
    X, Wt, _ = _operands(TILES[tile], 6)
    ctx, lib = Context(), bind()
    dW, b = _dev(ctx, Wt, np.uint16), _dev(ctx, np.random.default_rng(7).standard_normal(co).astype(np.float32), np.float32)
    out = []
    for x in (X, X[-1:]):
        dX, Yf = _dev(ctx, x, np.uint16), Buf(ctx, (len(x), H, W, co), np.float32)
        assert lib.fvm_nn_conv_fwd(ctx.h, dX.ptr, dW.ptr, b.ptr, len(x), H, W, ci, co, K, 0, co, None, Yf.ptr) == 0
        out.append(Yf.get()[-1])
    assert np.array_equal(*out)


def _layerwise(net, X, dout):
    """forward and backward through the layer entry points, one call per layer."""
    ctx, lib, L, ch = net.ctx, net.lib, net.L, net.ch
    B, H, W, _ = X.shape
    keep = []

    def buf(h, w, c):
        keep.append(Buf(ctx, (B, h, w, c), np.uint16))
        return keep[-1]

    def call(fn, *a):
        assert getattr(lib, fn)(ctx.h, *a) == 0, fn

    def size(i):
        return H >> i, W >> i

    def conv(name, x, i):
        e = net.p[name]
        y = buf(*size(i), e["co"])
        call("fvm_nn_conv_fwd", x.ptr, e["wb"].ptr, e["b"].ptr, B, *size(i), e["ci"], e["co"], 3, 1, e["co"], y.ptr, None)
        return y

    def grad(name, x, dy, i, need=True):
        e = net.p[name]
        call("fvm_nn_conv_wgrad", x.ptr, dy.ptr, B, *size(i), e["ci"], e["co"], e["K"], net.A["work"].ptr, e["gw"].ptr,
             e["gb"].ptr)
        if need:
            dx, scratch = buf(*size(i), e["ci"]), Buf(ctx, e["wb"].shape, np.uint16)
            call("fvm_nn_conv_dgrad", dy.ptr, e["wb"].ptr, scratch.ptr, B, *size(i), e["ci"], e["co"], e["K"], dx.ptr)
            return dx

    def relu(y, dy):
        dz = buf(*y.shape[1:])
        call("fvm_nn_relu_bwd", int(np.prod(y.shape)), y.ptr, dy.ptr, dz.ptr)
        return dz
    x, h, e, cat, dh, d = {}, {}, {}, {}, {}, {}
    x[0] = X
    for i in range(L):
        h[i] = conv("e%d_1" % i, x[i], i)
        e[i] = conv("e%d_2" % i, h[i], i)
        if i < L - 1:
            x[i + 1] = buf(*size(i + 1), ch[i])
            call("fvm_nn_pool_fwd", e[i].ptr, B, *size(i), ch[i], x[i + 1].ptr)
    d[L - 1] = e[L - 1]
    for i in range(L - 2, -1, -1):
        cc = ch[i + 1] + ch[i]
        cat[i] = buf(*size(i), cc)
        call("fvm_nn_up_fwd", d[i + 1].ptr, B, *size(i + 1), ch[i + 1], cat[i].ptr, cc, 0)
        call("fvm_nn_copy_channels", e[i].ptr, B * (H >> i) * (W >> i), ch[i], ch[i], 0, cat[i].ptr, cc, ch[i + 1])
        dh[i] = conv("d%d_1" % i, cat[i], i)
        d[i] = conv("d%d_2" % i, dh[i], i)
    o = net.p["out"]
    out = Buf(ctx, (B, H, W, net.cout), np.float32)
    call("fvm_nn_conv_fwd", d[0].ptr, o["wb"].ptr, o["b"].ptr, B, H, W, o["ci"], o["co"], 1, 0, net.cout_real, None, out.ptr)
    g = grad("out", d[0], dout, 0)
    skip = {}
    for i in range(L - 1):
        g = grad("d%d_2" % i, dh[i], relu(d[i], g), i)
        dcat = grad("d%d_1" % i, cat[i], relu(dh[i], g), i)
        cc, skip[i], g = ch[i + 1] + ch[i], buf(*size(i), ch[i]), buf(*size(i + 1), ch[i + 1])
        call("fvm_nn_copy_channels", dcat.ptr, B * (H >> i) * (W >> i), ch[i], cc, ch[i + 1], skip[i].ptr, ch[i], 0)
        call("fvm_nn_up_bwd", dcat.ptr, B, *size(i + 1), ch[i + 1], cc, 0, g.ptr)
    skip[L - 1] = g
    for i in range(L - 1, -1, -1):
        if i < L - 1:
            call("fvm_nn_add_channels", g.ptr, B * (H >> i) * (W >> i), ch[i], ch[i], 0, skip[i].ptr)
        g = grad("e%d_2" % i, h[i], relu(e[i], skip[i]), i)
        dx = grad("e%d_1" % i, x[i], relu(h[i], g), i, i > 0)
        if i > 0:
            g = buf(*size(i - 1), ch[i - 1])
            call("fvm_nn_pool_bwd", dx.ptr, B, *size(i - 1), ch[i - 1], g.ptr)
    return out.get()


class _Same(int):
    """As many channels on every level (levels of their own size would be gigabytes)."""

    def __mul__(self, factor):
        return int(self)


# the fourth: 768 concatenated channels, which the direct kernel reads from both
# parents; then its data gradients through a ReLU, 3x3 and 1x1; then deep ones, to the
# most levels there are
@pytest.mark.parametrize("L,base,B,H,W", [(2, 16, 2, 6, 14), (2, 48, 1, 10, 18), (4, 16, 3, 24, 40), (4, 64, 1, 8, 16),
                                          (5, 64, 1, 16, 32), (1, 64, 1, 256, 272),
                                          (9, _Same(16), 1, 256, 256), (12, _Same(16), 1, 2048, 2048)])
def test_whole_passes_equal_the_layers(L, base, B, H, W):
    """The one-call passes, which fuse the copies, the concatenation and the ReLU
    passes into the kernels beside them, are bitwise the layer-by-layer ones."""
    print("CASE unet passes", L, base, B, H, W, flush=True)
    net = UNet(Context(), levels=L, base=base, seed=3)
    r = np.random.default_rng(5)
    X = np.zeros((B, H, W, net.cin), np.float32)
    X[..., :5] = r.standard_normal((B, H, W, 5))
    T = r.standard_normal((B, H, W, 3)).astype(np.float32)
    dX, dT = _dev(net.ctx, X, np.uint16), _dev(net.ctx, T, np.float32)
    out = net.forward(dX).get()
    dX.zero()       # the caller may reuse its input before the backward pass
    net.loss(dT)
    net.backward()
    grads = net.grads_numpy()
    assert np.array_equal(out, _layerwise(net, _dev(net.ctx, X, np.uint16), net.A["dout"]))
    for name, (gw, gb) in net.grads_numpy().items():
        assert np.array_equal(grads[name][0], gw) and np.array_equal(grads[name][1], gb), name


def test_more_levels_than_there_are_places():
    """Refused before anything is allocated."""
    with pytest.raises(ValueError):
        UNet(levels=13, base=16)
