"""The learned Stokes initial guess: a U-Net run by the hand-written gfx950
kernels of csrc/unet.hip (bf16 activations and weights, fp32 accumulation on
the matrix cores, fp32 Adam master weights).

Architecture (levels L, base channels c): encoder level i has two 3x3
conv+ReLU layers with c*2^i channels and a 2x2 average pool between levels;
decoder level i upsamples (nearest, x2), concatenates the encoder skip and
applies two 3x3 conv+ReLU layers with c*2^i channels; a 1x1 convolution maps
to the output channels.  Tensors are NHWC; channel counts are padded to
multiples of 16 (the input's 5 fields and the output's 3 fields sit in the
first channels, the rest are zero).
"""
import ctypes as C

import numpy as np

from .lib import Context, load

P = C.c_void_p
I32 = C.c_int32
I64 = C.c_int64
F = C.c_float

_SIGS = {
    "fvm_nn_mfma_selftest": [P, P, P, P],
    "fvm_nn_conv_fwd": [P, P, P, P, I32, I32, I32, I32, I32, I32, I32, I32, P, P],
    "fvm_nn_conv_dgrad": [P, P, P, P, I32, I32, I32, I32, I32, I32, P],
    "fvm_nn_wgrad_workspace": [I32, I32, I32, I32, I32, I32],
    "fvm_nn_conv_wgrad": [P, P, P, I32, I32, I32, I32, I32, I32, P, P, P],
    "fvm_nn_relu_bwd": [P, I64, P, P, P],
    "fvm_nn_pool_fwd": [P, P, I32, I32, I32, I32, P],
    "fvm_nn_pool_bwd": [P, P, I32, I32, I32, I32, P],
    "fvm_nn_up_fwd": [P, P, I32, I32, I32, I32, P, I32, I32],
    "fvm_nn_up_bwd": [P, P, I32, I32, I32, I32, I32, I32, P],
    "fvm_nn_copy_channels": [P, P, I64, I32, I32, I32, P, I32, I32],
    "fvm_nn_add_channels": [P, P, I64, I32, I32, I32, P],
    "fvm_nn_mse": [P, P, P, P, I64, I32, I32, F, P, P, P],
    "fvm_nn_adam": [P, I64, P, P, P, P, P, F, F, F, F, I32, F],
    "fvm_nn_f32_to_bf16": [P, I64, P, P],
    "fvm_nn_unet_forward": [P, P, P],
    "fvm_nn_unet_backward": [P, P],
    "fvm_nn_adam_all": [P, I32, P, P, P, P, P, P, P, F, F, F, F, I32],
}
LEVELS = 12     # of csrc/unet.hip; the weights of more fit no card


class fvm_unet(C.Structure):
    """A network on one batch shape, for the whole-pass calls (csrc/unet.hip)."""
    _fields_ = ([(n, I32) for n in ("levels", "B", "H", "W", "cin", "cout", "cout_real")] + [("ch", I32 * LEVELS)] +
                [(n, P * (4 * LEVELS)) for n in ("wb", "b", "gw", "gb")] +
                [(n, P * LEVELS) for n in ("x", "h", "e", "dh", "d")] + [("out", P)] +
                [(n, P * LEVELS) for n in ("dx", "g1", "g2", "gdh", "gd", "dcat")] + [("dout", P), ("work", P)])


def bind():
    lib = load()
    for n, a in _SIGS.items():
        f = getattr(lib, n)
        f.argtypes = a
        f.restype = C.c_size_t if n == "fvm_nn_wgrad_workspace" else C.c_int
    return lib


def to_bf16_bits(x):
    """float32 -> bfloat16 bit patterns (round to nearest even)."""
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) & 0xFFFF).astype(np.uint16)


def from_bf16_bits(h):
    return (np.asarray(h, dtype=np.uint16).astype(np.uint32) << 16).view(np.float32)


class Buf:
    """A device allocation holding a numpy-typed array (bf16 held as uint16)."""

    def __init__(self, ctx, shape, dtype):
        self.ctx, self.shape, self.dtype = ctx, tuple(shape), np.dtype(dtype)
        self.nbytes = max(1, int(np.prod(self.shape)) * self.dtype.itemsize)
        self.ptr = ctx.alloc(self.nbytes)
        self.zero()

    def zero(self):
        self.ctx.call("fvm_memset", P(self.ptr), 0, self.nbytes)

    def set(self, a):
        a = np.ascontiguousarray(a, dtype=self.dtype)
        assert a.size == int(np.prod(self.shape)), (a.shape, self.shape)
        self.ctx.htod(self.ptr, a)

    def get(self):
        return self.ctx.dtoh(self.ptr, self.shape, self.dtype)

    def __del__(self):
        try:
            self.ctx.free(self.ptr)
        except Exception:
            pass


def _pad16(c):
    return (c + 15) // 16 * 16


class UNet:
    """Parameters, activations and the layer sequence of the learned guess."""

    def __init__(self, ctx=None, levels=4, base=32, cin=5, cout=3, seed=0):
        if not 1 <= levels <= LEVELS:
            raise ValueError("UNet: 1 to %d levels" % LEVELS)
        self.ctx = ctx or Context()
        self.lib = bind()
        self.L, self.c = levels, base
        self.cin_real, self.cout_real = cin, cout
        self.cin, self.cout = _pad16(cin), _pad16(cout)
        self.arch = (levels, base, self.cin, self.cout, cout)
        rng = np.random.default_rng(seed)
        self.layers = []  # (name, K, Cin, Cout, relu)
        ch = [base * 2 ** i for i in range(levels)]
        prev = self.cin
        for i in range(levels):
            self.layers.append(("e%d_1" % i, 3, prev, ch[i], True))
            self.layers.append(("e%d_2" % i, 3, ch[i], ch[i], True))
            prev = ch[i]
        for i in range(levels - 2, -1, -1):
            self.layers.append(("d%d_1" % i, 3, ch[i + 1] + ch[i], ch[i], True))
            self.layers.append(("d%d_2" % i, 3, ch[i], ch[i], True))
        self.layers.append(("out", 1, ch[0], self.cout, False))
        self.ch = ch
        self.p = {}
        for name, K, ci, co, relu in self.layers:
            fan_in = K * K * ci
            W = (rng.standard_normal((K * K, co, ci)) * np.sqrt(2.0 / fan_in)).astype(np.float32)
            if name == "e0_1":
                W[:, :, self.cin_real:] = 0.0
            if name == "out":
                W *= 0.1
                W[:, self.cout_real:, :] = 0.0
            b = np.zeros(co, np.float32)
            ent = {"K": K, "ci": ci, "co": co, "relu": relu,
                   "w": Buf(self.ctx, W.shape, np.float32), "wb": Buf(self.ctx, W.shape, np.uint16),
                   "b": Buf(self.ctx, (co,), np.float32),
                   "gw": Buf(self.ctx, W.shape, np.float32), "gb": Buf(self.ctx, (co,), np.float32),
                   "mw": Buf(self.ctx, W.shape, np.float32), "vw": Buf(self.ctx, W.shape, np.float32),
                   "mb": Buf(self.ctx, (co,), np.float32), "vb": Buf(self.ctx, (co,), np.float32)}
            ent["w"].set(W)
            ent["wb"].set(to_bf16_bits(W))
            ent["b"].set(b)
            self.p[name] = ent
        self.adam_step = 0
        self.shape = None

    # ---- parameters as numpy (tests, checkpoints) ----
    def params_numpy(self):
        return {k: (v["w"].get(), v["b"].get()) for k, v in self.p.items()}

    def grads_numpy(self):
        return {k: (v["gw"].get(), v["gb"].get()) for k, v in self.p.items()}

    def load_params(self, params):
        for k, (W, b) in params.items():
            self.p[k]["w"].set(W)
            self.p[k]["wb"].set(to_bf16_bits(W))
            self.p[k]["b"].set(b)

    # ---- buffers for one batch shape ----
    def _alloc(self, B, H, W):
        if self.shape == (B, H, W):
            return
        assert H % 2 ** (self.L - 1) == 0 and W % 2 ** (self.L - 1) == 0, "H, W must divide by 2^(L-1)"
        ctx = self.ctx
        self.shape = (B, H, W)
        bf = np.uint16
        self.A = {}
        for i in range(self.L):
            h, w = H >> i, W >> i
            cin = self.cin if i == 0 else self.ch[i - 1]
            for n, c in (("x", cin), ("h", self.ch[i]), ("e", self.ch[i]), ("g1_", self.ch[i]), ("g2_", self.ch[i]),
                         ("dx", cin)):
                self.A["%s%d" % (n, i)] = Buf(ctx, (B, h, w, c), bf)
        for i in range(self.L - 1):
            h, w = H >> i, W >> i
            for n, c in (("dh", self.ch[i]), ("d", self.ch[i]), ("gdh", self.ch[i]), ("gd", self.ch[i]),
                         ("dcat", self.ch[i + 1] + self.ch[i])):
                self.A["%s%d" % (n, i)] = Buf(ctx, (B, h, w, c), bf)
        self.A["out"] = Buf(ctx, (B, H, W, self.cout), np.float32)
        self.A["dout"] = Buf(ctx, (B, H, W, self.cout), bf)
        ws = max(self.lib.fvm_nn_wgrad_workspace(B, H >> self._lvl(n), W >> self._lvl(n), ci, co, K)
                 for n, K, ci, co, _ in self.layers)
        self.A["work"] = Buf(ctx, (ws // 4 + 1,), np.float32)
        npix = B * H * W
        self.A["lossw"] = Buf(ctx, ((npix * self.cout + 255) // 256 + 1,), np.float32)
        self.A["loss"] = Buf(ctx, (1,), np.float32)
        self._describe(B, H, W)

    def _describe(self, B, H, W):
        u = fvm_unet(self.L, B, H, W, self.cin, self.cout, self.cout_real)
        for i, c in enumerate(self.ch):
            u.ch[i] = c
        for i in range(self.L):
            for n in ("x", "h", "e", "dx"):
                getattr(u, n)[i] = self.A["%s%d" % (n, i)].ptr
            u.g1[i], u.g2[i] = self.A["g1_%d" % i].ptr, self.A["g2_%d" % i].ptr
        for i in range(self.L - 1):
            for n in ("dh", "d", "gdh", "gd", "dcat"):
                getattr(u, n)[i] = self.A["%s%d" % (n, i)].ptr
        u.out, u.dout, u.work = self.A["out"].ptr, self.A["dout"].ptr, self.A["work"].ptr
        self.desc = u

    def _point(self, *pairs):
        """The parameters' current buffers into the description."""
        for k, (name, *_) in enumerate(self.layers):
            e = self.p[name]
            for field, key in pairs:
                getattr(self.desc, field)[k] = e[key].ptr

    def _lvl(self, name):
        return 0 if name == "out" else int(name[1])

    def _call(self, fn, *a):
        rc = getattr(self.lib, fn)(self.ctx.h, *a)
        if rc != 0:
            self.ctx._check(rc)

    # ---- forward ----
    def forward(self, X):
        """X: Buf (B, H, W, cin) bf16 -> self.A['out'] (fp32, B H W cout)."""
        B, H, W, _ = X.shape
        self._alloc(B, H, W)
        self._point(("wb", "wb"), ("b", "b"))
        self._call("fvm_nn_unet_forward", C.byref(self.desc), P(X.ptr))
        return self.A["out"]

    # ---- loss ----
    def loss(self, T, mask=None):
        """Masked MSE over the real output channels against T (Buf fp32, B H W creal);
        leaves d(loss)/d(out) in A['dout'] and returns the loss (synchronises)."""
        B, H, W = self.shape
        npix = B * H * W
        self._call("fvm_nn_mse", P(self.A["out"].ptr), P(T.ptr), P(mask.ptr) if mask is not None else None,
                   I64(npix), self.cout, self.cout_real, F(1.0 / (npix * self.cout_real)), P(self.A["dout"].ptr),
                   P(self.A["lossw"].ptr), P(self.A["loss"].ptr))
        return float(self.A["loss"].get()[0])

    # ---- backward ----
    def backward(self):
        """Every parameter's gradient (gw, gb) from A['dout'], which loss() left."""
        self._point(("wb", "wb"), ("gw", "gw"), ("gb", "gb"))
        self._call("fvm_nn_unet_backward", C.byref(self.desc))

    # ---- optimizer ----
    def adam(self, lr=1e-3, b1=0.9, b2=0.999, eps=1e-8, wd=0.0):
        self.adam_step += 1
        e = self.p.values()
        t = [(x["w"], x["gw"], x["mw"], x["vw"], x["wb"].ptr) for x in e] + \
            [(x["b"], x["gb"], x["mb"], x["vb"], None) for x in e]
        n = len(t)
        sizes = (I64 * n)(*(int(np.prod(x[0].shape)) for x in t))
        tables = [(P * n)(*(x[k].ptr for x in t)) for k in range(4)] + [(P * n)(*(x[4] for x in t))]
        decay = (F * n)(*([wd] * len(self.layers) + [0.0] * len(self.layers)))
        self._call("fvm_nn_adam_all", n, sizes, *tables, decay, F(lr), F(b1), F(b2), F(eps), self.adam_step)
