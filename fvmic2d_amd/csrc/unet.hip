// Learned initial guess for the Stokes solve: the U-Net's layers as hand-written
// gfx950 kernels.  Activations are NHWC bfloat16 ([B][H][W][C], C fastest),
// weights bfloat16 [tap][Cout][Cin] (tap = ky*K + kx) with fp32 master copies
// for the optimizer; every product accumulates in fp32 on gfx950's double-K
// bf16 matrix instruction (v_mfma_f32_16x16x32_bf16: K = 32 per issue, twice
// the CDNA3 16x16x16 shape).  There is no reference counterpart: the
// reference's only initial guess is initialPressureGuess.c.
//
// MFMA 16x16x32 bf16 operand layout (one wavefront): lane l supplies
//   A: row m = l % 16, k = 8*(l/16) .. 8*(l/16)+7   (eight bf16, one 16-byte load)
//   B: col n = l % 16, k = 8*(l/16) .. 8*(l/16)+7
// and receives D[m = 4*(l/16) + i][n = l % 16], i = 0..3 (four fp32).
// fvm_nn_mfma_selftest checks this layout against a host product.
#include <hip/hip_bf16.h>

#include "fvm_internal.h"

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

namespace {

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// round to nearest even (finite values; NaN stays NaN)
__device__ __forceinline__ uint16_t f2bf(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  const uint32_t r = u + 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(r >> 16);
}

__device__ __forceinline__ f4 mfma32(bf8 a, bf8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// eight bf16 one by one (the self-test's operands)
struct Bf8Builder {
  uint16_t h[8];
  __device__ __forceinline__ bf8 get() const {
    uint4 u;
    u.x = (uint32_t)h[0] | ((uint32_t)h[1] << 16);
    u.y = (uint32_t)h[2] | ((uint32_t)h[3] << 16);
    u.z = (uint32_t)h[4] | ((uint32_t)h[5] << 16);
    u.w = (uint32_t)h[6] | ((uint32_t)h[7] << 16);
    return __builtin_bit_cast(bf8, u);
  }
};

// ---- MFMA layout self-test: D(16x16) = A(16x32) B(32x16) ---------------------
__global__ void __launch_bounds__(64) k_mfma_selftest(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                                                      float *__restrict__ D) {
  const int l = threadIdx.x;
  const int m = l % 16, kg = l / 16;
  Bf8Builder a, b;
  for (int i = 0; i < 8; i++) {
    a.h[i] = A[m * 32 + 8 * kg + i];      // A row-major [m][k], 16 x 32
    b.h[i] = B[(8 * kg + i) * 16 + m];    // B row-major [k][n], 32 x 16, n = l % 16
  }
  f4 c = {0.f, 0.f, 0.f, 0.f};
  c = mfma32(a.get(), b.get(), c);
  for (int i = 0; i < 4; i++) D[(4 * kg + i) * 16 + m] = c[i];
}

// transposed fragments from LDS (the weights of the data gradient, both operands
// of the weight gradient)
typedef short s4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4 lds_s4;

// K = 32 fragment (8 bf16 per lane): rows k = 8 (lane / 16) .. + 7 of the lane's
// column lane % 16; p0, p1: this lane's 8-byte address among the first and the
// last four of its group's rows (row (lane % 16) / 4, channels 4 (lane % 4))
__device__ __forceinline__ bf8 ld_tr(const uint16_t *p0, const uint16_t *p1) {
  union {
    s4 h[2];
    bf8 v;
  } u;
  u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)p0);
  u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)p1);
  return u.v;
}

// vectors at their elements' alignment (one access where the address allows)
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t h4u __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ void st4(float *p, f4 v) { *(f4u *)p = v; }
__device__ __forceinline__ f4 ld4(const float *p) { return *(const f4u *)p; }

// The input of a layer: C0 channels from X, the rest from X2 (null when C0 is all).
// up = 1: X is at half the resolution and read upsampled (nearest): a decoder
// layer reads its two parents instead of a concatenated copy of them.
struct Input {
  const uint16_t *X, *X2;
  int C0, up;
};
__device__ __forceinline__ const uint16_t *input_at(const Input &in, int C, int b, int H, int W, int h, int w, int c) {
  if (c < in.C0) return in.X + (((int64_t)b * (H >> in.up) + (h >> in.up)) * (W >> in.up) + (w >> in.up)) * in.C0 + c;
  return in.X2 + (((int64_t)b * H + h) * W + w) * (C - in.C0) + c - in.C0;
}

// ---- convolution (implicit GEMM) ------------------------------------------------
// Y[p][co] = act(bias[co] + sum_{tap, ci} X[p + off(tap)][ci] * W[tap][co][ci])
// off(tap) = (ky - K/2, kx - K/2); X outside the image reads 0.  TR: the data
// gradient, whose weights are W[taps - 1 - tap][ci][co], read as they lie and
// transposed on the way out of LDS.
//
// Block: 4 WN wavefronts, a patch of 16 x 4R pixels and 16 NT WN output channels;
// a wavefront has R rows of 16 pixels and NT channel tiles.  The patch and its halo
// are staged in LDS with all their channels, as slabs of 32 ([slab][pixel][32]: a
// row's 16 pixels are one conflict-free 1 KB fragment); the weights follow in
// groups of taps, the next group's loads in flight while one is used.  Every
// output is summed tap by tap, within a tap by channel: the order is the same for
// every tile shape, so a network's activations do not depend on which one a size
// takes (a changed order flips bf16 roundings, and each layer multiplies them).
// The weights are the A operand, so a lane ends with four consecutive channels of
// one pixel.  The shapes are picked by conv_launch.
struct ConvArgs {
  Input in;
  const uint16_t *W;
  const float *bias;     // may be null
  const uint16_t *mask;  // the layer's own activations (a data gradient leaves through their ReLU), or null
  uint16_t *Y;        // bf16 output (or null)
  float *Yf;          // fp32 output (or null)
  int B, H, Wd, Cin, Cout, relu;
  int cout_real;  // channels >= cout_real are written as 0 (padding)
  int npx, npy;   // patches per image
  int slabs;      // of 32 input channels
  int group;      // taps whose weights are staged together
};

#define CONV_WPIECES 6  // 16-byte pieces of a weight group per thread

template <int K, int R, int NT, int WN, bool TR>
__global__ void __launch_bounds__(256 * WN) k_conv(ConvArgs a) {
  constexpr int H2 = K / 2, T = K * K, PW = 16 + 2 * H2, PH = 4 * R + 2 * H2, NP = PH * PW;
  constexpr int TH = 256 * WN, CO = 16 * NT * WN;
  extern __shared__ uint4 lds[];
  uint16_t *sx = (uint16_t *)lds, *sw = sx + a.slabs * NP * 32;
  const int tid = threadIdx.x, lane = tid & 63, wv = (tid >> 6) & 3, wn = tid >> 8;
  const int px = blockIdx.x % a.npx, py = (blockIdx.x / a.npx) % a.npy, b = blockIdx.x / (a.npx * a.npy);
  const int x0 = px * 16, y0 = py * 4 * R, c0 = blockIdx.y * CO;
  const int64_t img = (int64_t)b * a.H * a.Wd;
  uint4 rw[CONV_WPIECES];
  // weights of taps t0 .. t0 + group - 1, zeros past Cin and Cout:
  // [tap][slab][co][32 ci], TR: [tap][slab][32 k][co]
  auto load_w = [&](int t0) {
    const int n = min(a.group, T - t0) * a.slabs * CO * 4;
#pragma unroll
    for (int i = 0; i < CONV_WPIECES; i++) {
      const int q = tid + TH * i;
      rw[i] = make_uint4(0u, 0u, 0u, 0u);
      if (q >= n) continue;
      const int ts = q / (CO * 4), r = q - ts * (CO * 4);
      const int t = t0 + ts / a.slabs, k0 = (ts % a.slabs) * 32;
      if (!TR) {
        const int co = c0 + (r >> 2), ch = k0 + (r & 3) * 8;
        if (co < a.Cout && ch < a.Cin) rw[i] = *(const uint4 *)(a.W + ((int64_t)t * a.Cout + co) * a.Cin + ch);
      } else {
        const int k = k0 + r / (CO / 8), co = c0 + r % (CO / 8) * 8;
        if (co < a.Cout && k < a.Cin) rw[i] = *(const uint4 *)(a.W + ((int64_t)(T - 1 - t) * a.Cin + k) * a.Cout + co);
      }
    }
  };
  load_w(0);
  // the patch: 4 pieces a pixel and slab, SB slabs' loads in flight together
  constexpr int XC = (NP * 4 + TH - 1) / TH, SB = XC >= 12 ? 1 : 12 / XC;
#pragma unroll 1
  for (int s0 = 0; s0 < a.slabs; s0 += SB) {
    uint4 rx[SB][XC];
#pragma unroll
    for (int s = 0; s < SB; s++)
#pragma unroll
      for (int i = 0; i < XC; i++) {
        const int q = tid + TH * i, pix = q >> 2, c = (s0 + s) * 32 + (q & 3) * 8;
        const int hh = y0 + pix / PW - H2, ww = x0 + pix % PW - H2;
        const bool ok = q < NP * 4 && c < a.Cin && hh >= 0 && hh < a.H && ww >= 0 && ww < a.Wd;
        rx[s][i] = ok ? *(const uint4 *)input_at(a.in, a.Cin, b, a.H, a.Wd, hh, ww, c) : make_uint4(0u, 0u, 0u, 0u);
      }
#pragma unroll
    for (int s = 0; s < SB; s++)
#pragma unroll
      for (int i = 0; i < XC; i++)
        if (tid + TH * i < NP * 4 && s0 + s < a.slabs) *(uint4 *)&sx[(s0 + s) * NP * 32 + (tid + TH * i) * 8] = rx[s][i];
  }
  f4 acc[R][NT];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int n = 0; n < NT; n++) acc[r][n] = (f4){0.f, 0.f, 0.f, 0.f};
  const int li = lane & 15, g = lane >> 4;
#pragma unroll 1
  for (int t0 = 0; t0 < T; t0 += a.group) {
    const int tn = min(a.group, T - t0), n16 = tn * a.slabs * CO * 4;
    if (t0) __syncthreads();
#pragma unroll
    for (int i = 0; i < CONV_WPIECES; i++)
      if (tid + TH * i < n16) *(uint4 *)&sw[(tid + TH * i) * 8] = rw[i];
    __syncthreads();
    if (t0 + a.group < T) load_w(t0 + a.group);
    // (tap, slab) steps, the next step's fragments read while one is multiplied
    const uint16_t *wr = sw + (TR ? (8 * g + (li >> 2)) * CO + wn * 16 * NT + 4 * (li & 3) : (wn * 16 * NT + li) * 32 + 8 * g);
    int sl = 0, dy = t0 / K, dx = t0 - dy * K;
    bf8 fx[2][R], fw[2][NT];
    auto frag = [&](int f) {
      const uint16_t *xr = sx + sl * NP * 32 + (dy * PW + dx) * 32 + (R * wv * PW + li) * 32 + 8 * g;
#pragma unroll
      for (int n = 0; n < NT; n++)
        fw[f][n] = TR ? ld_tr(wr + 16 * n, wr + 16 * n + 4 * CO) : __builtin_bit_cast(bf8, *(const uint4 *)(wr + n * 16 * 32));
#pragma unroll
      for (int r = 0; r < R; r++) fx[f][r] = __builtin_bit_cast(bf8, *(const uint4 *)(xr + r * PW * 32));
      wr += CO * 32;
      if (++sl == a.slabs) {
        sl = 0;
        if (++dx == K) dx = 0, dy++;
      }
    };
    auto mul = [&](int f) {
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int r = 0; r < R; r++) acc[r][n] = mfma32(fw[f][n], fx[f][r], acc[r][n]);
    };
    const int steps = tn * a.slabs;
    frag(0);
    int it = 1;
#pragma unroll 1
    for (; it + 1 < steps; it += 2) {
      frag(1);
      mul(0);
      frag(0);
      mul(1);
    }
    if (it < steps) {
      frag(1);
      mul(0);
      mul(1);
    } else {
      mul(0);
    }
  }
  // D[m = 4 g + i][n = li]: channel 4 g + i of pixel li of the row
  const int ww = x0 + li;
#pragma unroll
  for (int n = 0; n < NT; n++) {
    const int co = c0 + 16 * (wn * NT + n) + 4 * g;
    if (co >= a.Cout) continue;  // Cout is a multiple of 16
    const f4 bv = a.bias ? ld4(a.bias + co) : (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int hh = y0 + R * wv + r;
      if (hh >= a.H || ww >= a.Wd) continue;
      f4 v = acc[r][n] + bv;
      h4u h;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (a.relu) v[i] = v[i] > 0.f ? v[i] : 0.f;
        if (co + i >= a.cout_real) v[i] = 0.f;
        h[i] = f2bf(v[i]);
      }
      const int64_t o = (img + (int64_t)hh * a.Wd + ww) * a.Cout + co;
      if (a.mask) {
        const h4u y = *(const h4u *)(a.mask + o);
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (!(bf2f(y[i]) > 0.f)) h[i] = 0;
      }
      if (a.Y) *(h4u *)(a.Y + o) = h;
      if (a.Yf) st4(a.Yf + o, v);
    }
  }
}

// The same sums with fragments straight from global memory, 2 x 2 tiles per
// wavefront, 64 pixels x 64 channels per block.  A pixel's addresses are formed once
// per tap.  conv_direct says which layers take it.  TR (1x1): the weights are read as
// they lie, 16 lanes a row; 1024 -> 1024, 4096 pixels: 55 us, 66 from turned weights.
template <int K, bool TR>
__global__ void __launch_bounds__(256) k_conv_direct(ConvArgs a) {
  constexpr int T = K * K;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
  const int64_t npix = (int64_t)a.B * a.H * a.Wd;
  const int64_t p0 = (int64_t)blockIdx.x * 64 + (wv & 1) * 32;
  const int c0 = blockIdx.y * 64 + (wv >> 1) * 32;
  const int C0 = a.in.C0, C1 = a.Cin - C0;
  int64_t pp[2];
  int pb[2], ph[2], pw[2];
#pragma unroll
  for (int r = 0; r < 2; r++) {
    const int64_t p = p0 + r * 16 + li, q = p < npix ? p : 0;
    pp[r] = p < npix ? q : -1;
    pw[r] = (int)(q % a.Wd);
    ph[r] = (int)((q / a.Wd) % a.H);
    pb[r] = (int)(q / ((int64_t)a.Wd * a.H));
  }
  const bf8 zero = __builtin_bit_cast(bf8, make_uint4(0u, 0u, 0u, 0u));
  auto weights = [&](const uint16_t *w, int k) {
    if (!TR) return __builtin_bit_cast(bf8, *(const uint4 *)(w + k));
    Bf8Builder e;
    for (int i = 0; i < 8; i++) e.h[i] = w[(int64_t)(k + i) * a.Cout];
    return e.get();
  };
  f4 acc[2][2] = {};
#pragma unroll 1
  for (int t = 0; t < T; t++) {
    const uint16_t *xa[2], *xb[2], *w[2];  // channels below C0, from C0 on; weights
    bool in[2], out[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const int h = ph[r] + t / K - K / 2, ww = pw[r] + t % K - K / 2;
      in[r] = pp[r] >= 0 && h >= 0 && h < a.H && ww >= 0 && ww < a.Wd;
      const int hi = in[r] ? h : 0, wi = in[r] ? ww : 0;
      xa[r] = a.in.X + (((int64_t)pb[r] * (a.H >> a.in.up) + (hi >> a.in.up)) * (a.Wd >> a.in.up) + (wi >> a.in.up)) * C0;
      xb[r] = C1 ? a.in.X2 + (((int64_t)pb[r] * a.H + hi) * a.Wd + wi) * C1 - C0 : xa[r];
    }
#pragma unroll
    for (int n = 0; n < 2; n++) {
      const int co = c0 + 16 * n + li;
      out[n] = co < a.Cout;
      w[n] = TR ? a.W + (int64_t)(T - 1 - t) * a.Cin * a.Cout + (out[n] ? co : 0)
                : a.W + ((int64_t)t * a.Cout + (out[n] ? co : 0)) * a.Cin;
    }
    for (int k0 = 0; k0 < a.Cin; k0 += 32) {
      const int k = k0 + 8 * g;
      const bool kin = k < a.Cin;
      bf8 fx[2], fw[2];
#pragma unroll
      for (int r = 0; r < 2; r++)
        fx[r] = in[r] && kin ? __builtin_bit_cast(bf8, *(const uint4 *)((k < C0 ? xa[r] : xb[r]) + k)) : zero;
#pragma unroll
      for (int n = 0; n < 2; n++) fw[n] = out[n] && kin ? weights(w[n], k) : zero;
#pragma unroll
      for (int n = 0; n < 2; n++)
#pragma unroll
        for (int r = 0; r < 2; r++) acc[r][n] = mfma32(fw[n], fx[r], acc[r][n]);
    }
  }
#pragma unroll
  for (int n = 0; n < 2; n++) {
    const int co = c0 + 16 * n + 4 * g;
    if (co >= a.Cout) continue;
    const f4 bv = a.bias ? ld4(a.bias + co) : (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 2; r++) {
      if (pp[r] < 0) continue;
      f4 v = acc[r][n] + bv;
      h4u h;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (a.relu) v[i] = v[i] > 0.f ? v[i] : 0.f;
        if (co + i >= a.cout_real) v[i] = 0.f;
        h[i] = f2bf(v[i]);
      }
      const int64_t o = pp[r] * a.Cout + co;
      if (a.mask) {
        const h4u y = *(const h4u *)(a.mask + o);
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (!(bf2f(y[i]) > 0.f)) h[i] = 0;
      }
      if (a.Y) *(h4u *)(a.Y + o) = h;
      if (a.Yf) st4(a.Yf + o, v);
    }
  }
}

// weights of the data gradient as a forward layer's: Wd[tap][ci][co] = W[T-1-tap][co][ci].
// 64 x 64 of a tap per block through LDS, so that both sides move 16 bytes a lane
// (1024 -> 1024, 3x3: 9 us; element by element 45)
__global__ void __launch_bounds__(256) k_flip_weights(const uint16_t *__restrict__ W, int T, int Cout, int Cin,
                                                      uint16_t *__restrict__ Wd) {
  __shared__ uint16_t sh[64][66];
  const int t = blockIdx.z, co0 = blockIdx.y * 64, ci0 = blockIdx.x * 64;
  const int64_t from = (int64_t)t * Cout * Cin, to = (int64_t)(T - 1 - t) * Cin * Cout;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int q = threadIdx.x + 256 * k, r = q >> 3, c = (q & 7) * 8;  // 8 of a row
    if (co0 + r >= Cout || ci0 + c >= Cin) continue;
    const uint4 v = *(const uint4 *)(W + from + (int64_t)(co0 + r) * Cin + ci0 + c);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) *(uint32_t *)&sh[r][c + 2 * i] = w[i];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int q = threadIdx.x + 256 * k, r = q >> 3, c = (q & 7) * 8;
    if (ci0 + r >= Cin || co0 + c >= Cout) continue;
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = (uint32_t)sh[c + 2 * i][r] | ((uint32_t)sh[c + 2 * i + 1][r] << 16);
    *(uint4 *)(Wd + to + (int64_t)(ci0 + r) * Cout + co0 + c) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// taps whose weights fit a stage's registers and 48 KB; 0: not one tap does
int conv_group(int T, int slabs, int CO, int threads) {
  const int per_tap = slabs * CO * 64;  // bytes
  int g = threads * CONV_WPIECES * 16 / per_tap;
  return g > T ? T : g;
}

template <int K, int R, int NT, int WN, bool TR>
bool conv_try(fvm_ctx *ctx, ConvArgs a, int64_t want, size_t most_lds) {
  constexpr int H2 = K / 2, NP = (4 * R + 2 * H2) * (16 + 2 * H2), CO = 16 * NT * WN;
  a.npx = (a.Wd + 15) / 16;
  a.npy = (a.H + 4 * R - 1) / (4 * R);
  a.slabs = (a.Cin + 31) / 32;
  a.group = conv_group(K * K, a.slabs, CO, 256 * WN);
  const int64_t nx = (int64_t)a.B * a.npx * a.npy, ny = (a.Cout + CO - 1) / CO;
  const size_t lds = (size_t)a.slabs * (NP + a.group * CO) * 64;
  if (a.group < 1 || nx * ny < want || lds > most_lds) return false;
  k_conv<K, R, NT, WN, TR><<<dim3((unsigned)nx, (unsigned)ny), 256 * WN, lds, ctx->stream>>>(a);
  return true;
}

// Layers for k_conv_direct.  The LDS kernel wins wherever two of its blocks fit a CU;
// a block with many slabs is alone on its CU, and what it then reaches is set by
// rounds, blocks over 256 CUs (tiled: of its smallest patch, with the channels a
// block is left with; direct: of 64 pixels x 64 channels).  Times in us, LDS / direct:
//   3x3, 19 or 20 slabs: 16 channels a block.  640 -> 128, 3 x 50 x 50 (5 rounds / 1):
//     106 / 86; 16384 pixels (8 / 2): 168 / 161; 640 -> 640, 2048 pixels (5 / 2): 104 /
//     157.  More than 20 slabs do not fit.  A data gradient turns its weights first
//     (640 -> 640, 2 x 20 x 20, 4 / 1: 87 / 92).
//   1x1, 13 slabs and more: 32 channels a block.  512 -> 1024, 2 x 20 x 20 (3 / 1): 17.9 /
//     11.8; 2048 pixels (4 / 2): 23.6 / 19.1; 512 -> 256, 2048 pixels (1 / 1): 7.2 / 11.7.
//   1x1, 11 or 12 slabs: 384 -> 384, 65536 pixels (24 / 24): 142 / 135; 3 x 50 x 50 (4 / 3):
//     24.4 / 21.9; 16384 (6 / 6): 35.8 / 38.0.
//   1x1 on large images is bound by reading its pixels, which the LDS kernel reads
//     once for every 32 (fewer than 64 outputs) or 64 channels; it loses where their
//     tile is padded most or filled from little LDS work.  131072 pixels: 80 -> 48
//     17.9 / 11.4, 32 -> 64 16.0 / 11.3, 32 -> 128 28.5 / 19.9; but 64 -> 32 9.9 / 11.4.
bool conv_direct(const ConvArgs &a, int K, bool tr) {
  const int slabs = (a.Cin + 31) / 32;
  const int64_t npix = (int64_t)a.B * a.H * a.Wd, patches = (int64_t)a.B * ((a.Wd + 15) / 16) * ((a.H + 3) / 4);
  auto rounds = [](int64_t blocks) { return (blocks + 255) / 256; };
  auto tiled = [&](int co) { return rounds(patches * ((a.Cout + co - 1) / co)); };
  const int64_t direct = rounds((npix + 63) / 64 * ((a.Cout + 63) / 64));
  if (K == 3) return slabs > 18 && (slabs > 20 || tiled(16) >= 4 * direct + (tr ? 1 : 0));
  if (slabs > 12) return 2 * tiled(32) >= 3 * direct + 2;
  if (slabs > 10) return tiled(64) > direct || tiled(64) >= 16;
  return npix >= 65536 && ((a.Cin < 64 && a.Cout >= 64) || (a.Cout > 32 && a.Cout < 64));
}

// The largest tile with blocks enough for the chip that leaves LDS for two of them on a
// CU (160 KB): 256 of 512 threads (64 channels side by side), 512 of 256 threads; then
// smaller tiles, 128 of the last but one, the smallest in any case.  A large tile reads
// its operands least often (R + NT fragments for R NT matrix instructions), but the
// deep levels have few pixels: 2048 at 16 x 16 and batch 8, 1024 when one 256 x 256
// state is predicted.  Over 980 layers (16 to 384 channels, 16 x 16 to 256 x 256 pixels,
// both directions) half these numbers of blocks cost 1 to 11 % by kind of layer, twice
// them 2 to 13 %, a quarter or four times 0 to 13 % and 3 to 11 %.
// flip: room for the weights (TR).
template <int K, bool TR>
void conv_launch(fvm_ctx *ctx, const ConvArgs &a, uint16_t *flip) {
  constexpr size_t HALF = 80 << 10, ALL = 160 << 10;
  if (!conv_direct(a, K, TR)) {
    if (a.Cout >= 64) {
      if (conv_try<K, 4, 2, 2, TR>(ctx, a, 256, HALF) || conv_try<K, 2, 2, 2, TR>(ctx, a, 256, HALF) ||
          conv_try<K, 1, 2, 2, TR>(ctx, a, 256, ALL))
        return;
    } else if (a.Cout >= 32) {
      if (conv_try<K, 4, 2, 1, TR>(ctx, a, 512, HALF) || conv_try<K, 2, 2, 1, TR>(ctx, a, 512, HALF)) return;
    } else if (conv_try<K, 4, 1, 1, TR>(ctx, a, 512, HALF)) {
      return;
    }
    if (a.Cout >= 32 && conv_try<K, 1, 1, 2, TR>(ctx, a, 128, ALL)) return;
    if (conv_try<K, 1, 1, 1, TR>(ctx, a, 0, ALL)) return;
  }
  ConvArgs d = a;
  if (TR && K == 3) {  // a layer with the channels exchanged
    k_flip_weights<<<dim3((a.Cout + 63) / 64, (a.Cin + 63) / 64, K * K), 256, 0, ctx->stream>>>(a.W, K * K, a.Cin, a.Cout,
                                                                                              flip);
    d.W = flip;
  }
  const int64_t npix = (int64_t)a.B * a.H * a.Wd;
  k_conv_direct<K, TR && K == 1>
      <<<dim3((unsigned)((npix + 63) / 64), (unsigned)((a.Cout + 63) / 64)), 256, 0, ctx->stream>>>(d);
}

// ---- weight gradient --------------------------------------------------------------
// dW[tap][co][ci] = sum_p dY[p][co] * X[p + off(tap)][ci]: a GEMM with M = Cout,
// N = Cin per tap and the pixels as K.  Both operands have K strided in memory
// (NHWC), so they are staged in LDS as they lie, [pixel][32 channels], and the
// fragments are read with the transposing LDS load (ds_read_b64_tr_b16: 16 lanes
// read four 32-byte rows, lane i gets column i of them); a tap is then only
// another row address.
//
// A wavefront has 32 co x 32 ci and all taps (36 accumulator tiles) and takes
// patches of 16 x 16 pixels in K steps of two rows, half its rows apart: the rows a
// tap needs, shifted by dy, are then another step's, and each is read once per dx.
// SPLIT (few channels): the block's 4 wavefronts share 32 co x 32 ci and split the
// patch's rows, their sums added in LDS at the end; otherwise they share a patch
// and have 64 co x 64 ci between them.  Blocks split the patches (`nchunk`) to fill
// the chip; their fp32 partials, and those of the bias, are added in chunk order
// by k_wgrad_reduce.  What bounds it is getting the patches in: all loads of a
// patch are issued together, and two blocks of a CU overlap.  Two blocks leave 256
// registers a lane, of which the sums of 64 x 64 channels (K = 3) take 144 and a patch on
// its way 76: that form spills 85 (320 bytes a lane), read and written once a patch.
// Before, every bf16 was gathered from global memory by itself and one thread
// summed a weight's partials over all chunks: one optimiser step's 15 gradients at
// batch 8, 128 x 128 took 3.29 ms; now 0.43.
#define KCH 256
#define WG_P 16              // patch edge
#define WG_HW (WG_P + 2)     // with the taps' halo
struct WgradArgs {
  Input in;
  const uint16_t *dY;
  float *part;  // [chunk][taps * Cout * Cin, then Cout (bias)]
  int B, H, Wd, Cin, Cout;
  int npx, npy, npatch, per_chunk;
  int want_bias;
  int aligned;  // the input and dY on 16-byte boundaries
};

__device__ __forceinline__ uint4 ld16(const uint16_t *p, int aligned) {
  if (aligned) return *(const uint4 *)p;
  uint32_t w[4];
  for (int i = 0; i < 4; i++) w[i] = (uint32_t)p[2 * i] | ((uint32_t)p[2 * i + 1] << 16);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// N 16-byte pieces per thread of a patch of PW x PH pixels at (x0, y0), slabs of 32
// channels from c0 (SL of them), into LDS as [slab][pixel][32]; zeros outside
template <int SL, int PW, int PH>
struct Patch {
  static constexpr int NP = PW * PH, N = (NP * 4 * SL + 255) / 256;
  uint4 r[N];
  __device__ __forceinline__ void load(const Input &in, int b, int H, int W, int C, int x0, int y0, int c0, int aligned) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int q = threadIdx.x + 256 * i, sl = q / (NP * 4), pix = (q - sl * NP * 4) >> 2, c = c0 + 32 * sl + (q & 3) * 8;
      const int hh = y0 + pix / PW, ww = x0 + pix % PW;
      const bool ok = q < NP * 4 * SL && hh >= 0 && hh < H && ww >= 0 && ww < W && c < C;
      r[i] = ok ? ld16(input_at(in, C, b, H, W, hh, ww, c), aligned) : make_uint4(0u, 0u, 0u, 0u);
    }
  }
  __device__ __forceinline__ void store(uint16_t *sh) const {
#pragma unroll
    for (int i = 0; i < N; i++)
      if (threadIdx.x + 256 * i < NP * 4 * SL) *(uint4 *)&sh[(threadIdx.x + 256 * i) * 8] = r[i];
  }
};

template <int K, bool SPLIT>
__global__ void __launch_bounds__(256, 2) k_wgrad(WgradArgs a) {
  constexpr int H2 = K / 2, HW = WG_P + 2 * H2, T = K * K, SL = SPLIT ? 1 : 2;
  constexpr int ROWS = SPLIT ? 4 : 16, STEPS = ROWS / 2;  // of a wavefront
  typedef Patch<SL, HW, HW> PX;
  typedef Patch<SL, WG_P, WG_P> PY;
  constexpr int TILES = SL * (HW * HW + WG_P * WG_P) * 64, RED = SPLIT ? 2 * T * 4 * 64 * 16 : 0;
  __shared__ uint4 lds[(TILES > RED ? TILES : RED) / 16];
  uint16_t *sx = (uint16_t *)lds, *sy = sx + SL * HW * HW * 32;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int co0 = blockIdx.y * 32 * SL, ci0 = blockIdx.z * 32 * SL;  // the block's
  const int row0 = SPLIT ? ROWS * wv : 0;
  const uint16_t *wx = SPLIT ? sx : sx + (wv & 1) * HW * HW * 32, *wy = SPLIT ? sy : sy + (wv >> 1) * WG_P * WG_P * 32;
  f4 acc[T][2][2];
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
      for (int n = 0; n < 2; n++) acc[t][m][n] = (f4){0.f, 0.f, 0.f, 0.f};
  float bsum[SL][8] = {};
  const bool bias = a.want_bias && blockIdx.z == 0;
  // fragment addresses: group g holds k = 8g.., i.e. row r + STEPS (g / 2), columns 8 (g % 2)..
  const int g = lane >> 4, li = lane & 15;
  const int frow = STEPS * (g >> 1), fcol = 8 * (g & 1) + (li >> 2), fch = 4 * (li & 3);
  const int p_end = min(a.npatch, ((int)blockIdx.x + 1) * a.per_chunk);
#pragma unroll 1
  for (int pt = blockIdx.x * a.per_chunk; pt < p_end; pt++) {
    const int px = pt % a.npx, py = (pt / a.npx) % a.npy, b = pt / (a.npx * a.npy);
    const int x0 = px * WG_P, y0 = py * WG_P;
    {
      PX tx;
      PY ty;
      tx.load(a.in, b, a.H, a.Wd, a.Cin, x0 - H2, y0 - H2, ci0, a.aligned);
      ty.load(Input{a.dY, nullptr, a.Cout, 0}, b, a.H, a.Wd, a.Cout, x0, y0, co0, a.aligned);
      __syncthreads();  // the tiles of the patch before are done with
      tx.store(sx);
      ty.store(sy);
      if (bias) {  // a thread's pieces of a slab are of the same 8 channels
#pragma unroll
        for (int i = 0; i < PY::N; i++) {
          const uint32_t w[4] = {ty.r[i].x, ty.r[i].y, ty.r[i].z, ty.r[i].w};
#pragma unroll
          for (int k = 0; k < 4; k++) {
            bsum[i / 4][2 * k] += __uint_as_float(w[k] << 16);
            bsum[i / 4][2 * k + 1] += __uint_as_float(w[k] & 0xffff0000u);
          }
        }
      }
    }
    __syncthreads();
    // row pairs (j, j + STEPS) of X meet the dY of steps j - dy
    bf8 fy[3][2];
#pragma unroll
    for (int j = -H2; j < STEPS + H2; j++) {
      const int ry = j + H2;  // the step that comes into reach
      if (ry < STEPS) {
#pragma unroll
        for (int m = 0; m < 2; m++) {
          const uint16_t *p = &wy[((row0 + ry + frow) * WG_P + fcol) * 32 + 16 * m + fch];
          fy[ry % 3][m] = ld_tr(p, p + 4 * 32);
        }
      }
#pragma unroll
      for (int dx = 0; dx < K; dx++) {
        bf8 fx[2];
#pragma unroll
        for (int n = 0; n < 2; n++) {
          const uint16_t *p = &wx[((row0 + j + H2 + frow) * HW + fcol + dx) * 32 + 16 * n + fch];
          fx[n] = ld_tr(p, p + 4 * 32);
        }
#pragma unroll
        for (int dy = 0; dy < K; dy++) {
          const int r = j - dy + H2;
          if (r < 0 || r >= STEPS) continue;
#pragma unroll
          for (int m = 0; m < 2; m++)
#pragma unroll
            for (int n = 0; n < 2; n++) acc[dy * K + dx][m][n] = mfma32(fy[r % 3][m], fx[n], acc[dy * K + dx][m][n]);
        }
      }
    }
  }
  const int64_t nw = (int64_t)T * a.Cout * a.Cin;
  float *out = a.part + (int64_t)blockIdx.x * (nw + a.Cout);
  if (SPLIT) {  // (w0 + w1) + (w2 + w3)
    f4 *red = (f4 *)lds;
    __syncthreads();
#pragma unroll
    for (int step = 0; step < 2; step++) {
      const bool give = step == 0 ? (wv & 1) : wv == 2, get = step == 0 ? !(wv & 1) : wv == 0;
      f4 *o = red + (step == 0 ? (wv >> 1) : 0) * T * 4 * 64 + lane;
      if (give) {
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
          for (int q = 0; q < 4; q++) o[(t * 4 + q) * 64] = acc[t][q >> 1][q & 1];
      }
      __syncthreads();
      if (get) {
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
          for (int q = 0; q < 4; q++) acc[t][q >> 1][q & 1] += o[(t * 4 + q) * 64];
      }
      __syncthreads();
    }
  }
  if (!SPLIT || wv == 0) {
    const int cb = co0 + (SPLIT ? 0 : 32 * (wv >> 1)), ib = ci0 + (SPLIT ? 0 : 32 * (wv & 1)) + li;
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
      for (int m = 0; m < 2; m++)
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int co = cb + 16 * m + 4 * g + i, ci = ib + 16 * n;
            if (co < a.Cout && ci < a.Cin) out[((int64_t)t * a.Cout + co) * a.Cin + ci] = acc[t][m][n][i];
          }
  }
  if (bias) {  // uniform over the block
    float *sb = (float *)lds;
    __syncthreads();
#pragma unroll
    for (int sl = 0; sl < SL; sl++)
#pragma unroll
      for (int i = 0; i < 8; i++) sb[(tid >> 2) * 33 * SL + 33 * sl + (tid & 3) * 8 + i] = bsum[sl][i];
    __syncthreads();
    if (tid < 32 * SL && co0 + tid < a.Cout) {
      float s = 0.f;
      for (int k = 0; k < 64; k++) s += sb[k * 33 * SL + 33 * (tid >> 5) + (tid & 31)];
      out[nw + co0 + tid] = s;
    }
  }
}

// dW and db from the chunks' partials: G groups of threads take every G-th chunk
// of 4 values, their sums are added in the groups' order
template <int G>
__global__ void __launch_bounds__(256) k_wgrad_reduce(const float *__restrict__ part, int nchunk, int64_t nw, int nb,
                                                      float *__restrict__ dW, float *__restrict__ db) {
  constexpr int Q = 256 / G;
  __shared__ f4 sh[256];
  const int64_t n = nw + nb;
  const int64_t q = ((int64_t)blockIdx.x * Q + threadIdx.x % Q) * 4;
  const int grp = threadIdx.x / Q;
  f4 s = {0.f, 0.f, 0.f, 0.f};
  if (q < n) {
#pragma unroll 4
    for (int c = grp; c < nchunk; c += G) s += ld4(&part[c * n + q]);
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  if (grp == 0 && q < n) {
#pragma unroll
    for (int k = 1; k < G; k++) s += sh[k * Q + threadIdx.x];
    if (q < nw) st4(&dW[q], s);
    else if (db) st4(&db[q - nw], s);
  }
}

// ---- elementwise layers ------------------------------------------------------------
__global__ void __launch_bounds__(256) k_relu_bwd(int64_t n, const uint16_t *__restrict__ y,
                                                  const uint16_t *__restrict__ dy, uint16_t *__restrict__ dz) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dz[i] = bf2f(y[i]) > 0.f ? dy[i] : (uint16_t)0;
}

// 2x2 average pooling (H, W even)
__global__ void __launch_bounds__(256) k_pool_fwd(const uint16_t *__restrict__ X, int B, int H, int W, int C,
                                                  uint16_t *__restrict__ Y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2;
  const int64_t n = (int64_t)B * Ho * Wo * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  const int64_t q = i / C;
  const int w = (int)(q % Wo), h = (int)((q / Wo) % Ho);
  const int64_t b = q / ((int64_t)Wo * Ho);
  const int64_t r0 = ((b * H + 2 * h) * W + 2 * w) * C + c, r1 = r0 + (int64_t)W * C;
  const float s = (bf2f(X[r0]) + bf2f(X[r0 + C])) + (bf2f(X[r1]) + bf2f(X[r1 + C]));
  Y[i] = f2bf(0.25f * s);
}

__global__ void __launch_bounds__(256) k_pool_bwd(const uint16_t *__restrict__ dY, int B, int H, int W, int C,
                                                  uint16_t *__restrict__ dX) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n = (int64_t)B * H * W * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  const int64_t q = i / C;
  const int w = (int)(q % W), h = (int)((q / W) % H);
  const int64_t b = q / ((int64_t)W * H);
  const int Ho = H / 2, Wo = W / 2;
  dX[i] = f2bf(0.25f * bf2f(dY[((b * Ho + h / 2) * Wo + w / 2) * C + c]));
}

// nearest-neighbour 2x upsampling written into channels [c0, c0+C) of a Ctot-channel tensor
__global__ void __launch_bounds__(256) k_up_fwd(const uint16_t *__restrict__ X, int B, int H, int W, int C,
                                                uint16_t *__restrict__ Y, int Ctot, int c0) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int H2 = 2 * H, W2 = 2 * W;
  const int64_t n = (int64_t)B * H2 * W2 * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  const int64_t q = i / C;
  const int w = (int)(q % W2), h = (int)((q / W2) % H2);
  const int64_t b = q / ((int64_t)W2 * H2);
  Y[q * Ctot + c0 + c] = X[((b * H + h / 2) * W + w / 2) * C + c];
}

__global__ void __launch_bounds__(256) k_up_bwd(const uint16_t *__restrict__ dY, int B, int H, int W, int C,
                                                int Ctot, int c0, uint16_t *__restrict__ dX) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n = (int64_t)B * H * W * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  const int64_t q = i / C;
  const int w = (int)(q % W), h = (int)((q / W) % H);
  const int64_t b = q / ((int64_t)W * H);
  const int W2 = 2 * W;
  const int64_t r0 = ((b * 2 * H + 2 * h) * W2 + 2 * w) * Ctot + c0 + c, r1 = r0 + (int64_t)W2 * Ctot;
  const float s = (bf2f(dY[r0]) + bf2f(dY[r0 + Ctot])) + (bf2f(dY[r1]) + bf2f(dY[r1 + Ctot]));
  dX[i] = f2bf(s);
}

// copy channels: Y[p][c0 + c] = X[p][c] (C channels of a Cx-channel X into a Ctot-channel Y)
__global__ void __launch_bounds__(256) k_copy_channels(const uint16_t *__restrict__ X, int64_t npix, int C, int Cx,
                                                       int xc0, uint16_t *__restrict__ Y, int Ctot, int c0) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npix * C) return;
  const int c = (int)(i % C);
  const int64_t p = i / C;
  Y[p * Ctot + c0 + c] = X[p * Cx + xc0 + c];
}

// add channels: Y[p][c] += X[p][xc0 + c]  (bf16 in, bf16 out, fp32 sum)
__global__ void __launch_bounds__(256) k_add_channels(const uint16_t *__restrict__ X, int64_t npix, int C, int Cx,
                                                      int xc0, uint16_t *__restrict__ Y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npix * C) return;
  const int c = (int)(i % C);
  const int64_t p = i / C;
  Y[i] = f2bf(bf2f(Y[i]) + bf2f(X[p * Cx + xc0 + c]));
}

// ---- the same layers eight channels a thread, as the whole passes use them ------------
struct H8 {
  uint16_t v[8];
};
__device__ __forceinline__ H8 ld_h8(const uint16_t *p) { return __builtin_bit_cast(H8, *(const uint4 *)p); }
__device__ __forceinline__ void st_h8(uint16_t *p, const H8 &h) { *(uint4 *)p = __builtin_bit_cast(uint4, h); }

__global__ void __launch_bounds__(256) k_copy8(int64_t n8, const uint16_t *__restrict__ X, uint16_t *__restrict__ Y) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n8) ((uint4 *)Y)[i] = ((const uint4 *)X)[i];
}

__global__ void __launch_bounds__(256) k_pool8(const uint16_t *__restrict__ X, int B, int H, int W, int C,
                                               uint16_t *__restrict__ Y) {
  const int C8 = C / 8, Ho = H / 2, Wo = W / 2;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)B * Ho * Wo * C8) return;
  const int c = (int)(i % C8) * 8;
  const int64_t q = i / C8;
  const int w = (int)(q % Wo), h = (int)((q / Wo) % Ho);
  const int64_t b = q / ((int64_t)Wo * Ho);
  const uint16_t *r0 = X + ((b * H + 2 * h) * W + 2 * w) * C + c, *r1 = r0 + (int64_t)W * C;
  const H8 a0 = ld_h8(r0), a1 = ld_h8(r0 + C), b0 = ld_h8(r1), b1 = ld_h8(r1 + C);
  H8 y;
#pragma unroll
  for (int k = 0; k < 8; k++) y.v[k] = f2bf(0.25f * ((bf2f(a0.v[k]) + bf2f(a1.v[k])) + (bf2f(b0.v[k]) + bf2f(b1.v[k]))));
  st_h8(Y + q * C + c, y);
}

// gradient of the upsampled part (channels [0, C) of dcat's Ctot), through the ReLU of
// the activations y it was upsampled from
__global__ void __launch_bounds__(256) k_up_bwd8(const uint16_t *__restrict__ dcat, int B, int H, int W, int C, int Ctot,
                                                 const uint16_t *__restrict__ y, uint16_t *__restrict__ dz) {
  const int C8 = C / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)B * H * W * C8) return;
  const int c = (int)(i % C8) * 8;
  const int64_t q = i / C8;
  const int w = (int)(q % W), h = (int)((q / W) % H);
  const int64_t b = q / ((int64_t)W * H);
  const uint16_t *r0 = dcat + ((b * 2 * H + 2 * h) * 2 * W + 2 * w) * Ctot + c, *r1 = r0 + (int64_t)2 * W * Ctot;
  const H8 a0 = ld_h8(r0), a1 = ld_h8(r0 + Ctot), b0 = ld_h8(r1), b1 = ld_h8(r1 + Ctot), m = ld_h8(y + q * C + c);
  H8 z;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const uint16_t s = f2bf((bf2f(a0.v[k]) + bf2f(a1.v[k])) + (bf2f(b0.v[k]) + bf2f(b1.v[k])));
    z.v[k] = bf2f(m.v[k]) > 0.f ? s : (uint16_t)0;
  }
  st_h8(dz + q * C + c, z);
}

// gradient of encoder activations y: the skip part (channels [c0, c0 + C) of dcat's
// Ctot) plus a quarter of the pooled gradient, through y's ReLU
__global__ void __launch_bounds__(256) k_skip_bwd8(const uint16_t *__restrict__ dcat, int Ctot, int c0,
                                                   const uint16_t *__restrict__ dpool, int B, int H, int W, int C,
                                                   const uint16_t *__restrict__ y, uint16_t *__restrict__ dz) {
  const int C8 = C / 8, Ho = H / 2, Wo = W / 2;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)B * H * W * C8) return;
  const int c = (int)(i % C8) * 8;
  const int64_t q = i / C8;
  const int w = (int)(q % W), h = (int)((q / W) % H);
  const int64_t b = q / ((int64_t)W * H);
  const H8 s = ld_h8(dcat + q * Ctot + c0 + c), p = ld_h8(dpool + ((b * Ho + h / 2) * Wo + w / 2) * C + c), m = ld_h8(y + q * C + c);
  H8 z;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const uint16_t v = f2bf(bf2f(s.v[k]) + bf2f(f2bf(0.25f * bf2f(p.v[k]))));
    z.v[k] = bf2f(m.v[k]) > 0.f ? v : (uint16_t)0;
  }
  st_h8(dz + q * C + c, z);
}

// masked mean squared error over the first Creal of C fp32 output channels:
// loss partials per block; dOut (bf16, C channels) = 2 (out - tgt) mask / count
#define MSE_PER 8  // values per thread, 256 apart: fewer partials for k_sum_f
__global__ void __launch_bounds__(256) k_mse(const float *__restrict__ out, const float *__restrict__ tgt,
                                             const float *__restrict__ mask, int64_t npix, int C, int Creal,
                                             float inv_count, uint16_t *__restrict__ dOut, float *__restrict__ part) {
  __shared__ float sh[256];
  float l = 0.f;
#pragma unroll
  for (int k = 0; k < MSE_PER; k++) {
    const int64_t i = ((int64_t)blockIdx.x * MSE_PER + k) * 256 + threadIdx.x;
    if (i >= npix * C) continue;
    const int c = (int)(i % C);
    const int64_t p = i / C;
    float g = 0.f;
    if (c < Creal) {
      const float m = mask ? mask[p * Creal + c] : 1.f;
      const float d = (out[i] - tgt[p * Creal + c]) * m;
      l += d * d * inv_count;
      g = 2.f * d * inv_count;
    }
    dOut[i] = f2bf(g);
  }
  sh[threadIdx.x] = l;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

__global__ void __launch_bounds__(256) k_sum_f(const float *__restrict__ part, int64_t n, float *__restrict__ out) {
  __shared__ float sh[256];
  float s = 0.f;
  for (int64_t i = threadIdx.x; i < n; i += 256) s += part[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = sh[0];
}

// Adam on fp32 master weights; the bf16 working copy is refreshed
struct AdamArgs {
  float *w;
  const float *g;
  float *m, *v;
  uint16_t *wb;  // or null
  int64_t n;
  float wd;
};
struct AdamRates {
  float lr, b1, b2, eps, c1, c2;
};
__device__ __forceinline__ void adam_at(const AdamArgs &a, const AdamRates &r, int64_t i) {
  const float gi = a.g[i] + a.wd * a.w[i];
  const float mi = r.b1 * a.m[i] + (1.f - r.b1) * gi;
  const float vi = r.b2 * a.v[i] + (1.f - r.b2) * gi * gi;
  a.m[i] = mi;
  a.v[i] = vi;
  const float wi = a.w[i] - r.lr * (mi / r.c1) / (sqrtf(vi / r.c2) + r.eps);
  a.w[i] = wi;
  if (a.wb) a.wb[i] = f2bf(wi);
}
__global__ void __launch_bounds__(256) k_adam(AdamArgs a, AdamRates r) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < a.n) adam_at(a, r, i);
}
// every tensor of a network in one launch (30 of them took 85 us one by one): block
// b works on the tensor k with first[k] <= b < first[k + 1]
#define ADAM_MAX 40
struct AdamAll {
  AdamArgs t[ADAM_MAX];
  int first[ADAM_MAX + 1];
  int n;
};
__global__ void __launch_bounds__(256) k_adam_all(AdamAll A, AdamRates r) {
  int k = 0;
  while (k + 1 < A.n && (int)blockIdx.x >= A.first[k + 1]) k++;
  const int64_t i = (int64_t)((int)blockIdx.x - A.first[k]) * 256 + threadIdx.x;
  if (i < A.t[k].n) adam_at(A.t[k], r, i);
}

__global__ void __launch_bounds__(256) k_f2bf(int64_t n, const float *__restrict__ x, uint16_t *__restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// ---- C ABI (sizes in elements; all pointers device) ---------------------------------
extern "C" int fvm_nn_mfma_selftest(fvm_ctx *ctx, const uint16_t *A, const uint16_t *B, float *D) {
  if (!ctx || !A || !B || !D) return FVM_ERR_ARG;
  k_mfma_selftest<<<1, 64, 0, ctx->stream>>>(A, B, D);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

static int conv_check(fvm_ctx *ctx, int B, int H, int W, int Cin, int Cout, int K) {
  if (B < 1 || H < 1 || W < 1 || Cin < 16 || Cin % 16 || Cout < 16 || Cout % 16 || (K != 1 && K != 3))
    return fvm_set_err(ctx, FVM_ERR_ARG, "conv: B,H,W >= 1, Cin and Cout multiples of 16, K in {1,3}");
  return FVM_OK;
}

// flip: K*K*Cin*Cout bf16 of workspace for a data gradient (tr), or null
static int conv_run(fvm_ctx *ctx, const ConvArgs &a, int K, bool tr, uint16_t *flip) {
  if ((int64_t)a.B * ((a.Wd + 15) / 16) * ((a.H + 3) / 4) > INT32_MAX)
    return fvm_set_err(ctx, FVM_ERR_ARG, "conv: too many pixels");
  if (K == 3) tr ? conv_launch<3, true>(ctx, a, flip) : conv_launch<3, false>(ctx, a, flip);
  else tr ? conv_launch<1, true>(ctx, a, flip) : conv_launch<1, false>(ctx, a, flip);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

extern "C" int fvm_nn_conv_fwd(fvm_ctx *ctx, const uint16_t *X, const uint16_t *W, const float *bias, int32_t B,
                               int32_t H, int32_t Wd, int32_t Cin, int32_t Cout, int32_t K, int32_t relu,
                               int32_t cout_real, uint16_t *Y, float *Yf) {
  if (!ctx || !X || !W || (!Y && !Yf)) return FVM_ERR_ARG;
  FVM_TRY(conv_check(ctx, B, H, Wd, Cin, Cout, K));
  ConvArgs a{Input{X, nullptr, Cin, 0}, W, bias, nullptr, Y, Yf, B, H, Wd, Cin, Cout, relu, cout_real > 0 ? cout_real : Cout};
  FVM_PHASE(ctx, FVM_PHASE_OTHER);
  return conv_run(ctx, a, K, false, nullptr);
}

// dX = conv(dY, flipped transposed W), the flip and the transposition made while
// the weights are read from LDS, or into Wd_scratch (K*K*Cout*Cin bf16) where they
// are read from memory
extern "C" int fvm_nn_conv_dgrad(fvm_ctx *ctx, const uint16_t *dY, const uint16_t *W, uint16_t *Wd_scratch, int32_t B,
                                 int32_t H, int32_t Wd, int32_t Cin, int32_t Cout, int32_t K, uint16_t *dX) {
  if (!ctx || !dY || !W || !Wd_scratch || !dX) return FVM_ERR_ARG;
  FVM_TRY(conv_check(ctx, B, H, Wd, Cin, Cout, K));
  ConvArgs a{Input{dY, nullptr, Cout, 0}, W, nullptr, nullptr, dX, nullptr, B, H, Wd, Cout, Cin, 0, Cin};
  FVM_PHASE(ctx, FVM_PHASE_OTHER);
  return conv_run(ctx, a, K, true, Wd_scratch);
}

// bytes of fp32 workspace fvm_nn_conv_wgrad needs
extern "C" size_t fvm_nn_wgrad_workspace(int32_t B, int32_t H, int32_t Wd, int32_t Cin, int32_t Cout, int32_t K) {
  const int64_t npix = (int64_t)B * H * Wd;
  const int64_t nchunk = (npix + KCH - 1) / KCH;
  return (size_t)nchunk * ((size_t)K * K * Cout * Cin + (size_t)Cout) * sizeof(float);
}

static int wgrad_run(fvm_ctx *ctx, const Input &in, const uint16_t *dY, int B, int H, int Wd, int Cin, int Cout, int K,
                     float *work, float *dW, float *db) {
  const int64_t npix = (int64_t)B * H * Wd;
  const int64_t nw = (int64_t)K * K * Cout * Cin;
  WgradArgs a{in, dY, work, B, H, Wd, Cin, Cout};
  a.npx = (Wd + WG_P - 1) / WG_P;
  a.npy = (H + WG_P - 1) / WG_P;
  if ((int64_t)B * a.npx * a.npy > INT32_MAX) return fvm_set_err(ctx, FVM_ERR_ARG, "conv: too many pixels");
  a.npatch = B * a.npx * a.npy;
  a.want_bias = db != nullptr;
  a.aligned = (((uintptr_t)in.X | (uintptr_t)in.X2 | (uintptr_t)dY) & 15) == 0;
  // wavefronts side by side in co and ci where both have 64 channels, else along
  // the pixels; two blocks a CU, within the workspace (one chunk per 256 pixels) and
  // with at least one patch each: more only grows the partials
  const bool split = Cout < 64 || Cin < 64;
  const int cw = split ? 32 : 64, tm = (Cout + cw - 1) / cw, tn = (Cin + cw - 1) / cw;
  int64_t nchunk = (512 + tm * tn - 1) / (tm * tn);
  const int64_t most = (npix + KCH - 1) / KCH;
  if (nchunk > most) nchunk = most;
  if (nchunk > a.npatch) nchunk = a.npatch;
  a.per_chunk = (int)((a.npatch + nchunk - 1) / nchunk);
  nchunk = (a.npatch + a.per_chunk - 1) / a.per_chunk;
  const dim3 grid((unsigned)nchunk, tm, tn);
  if (K == 3) split ? k_wgrad<3, true><<<grid, 256, 0, ctx->stream>>>(a) : k_wgrad<3, false><<<grid, 256, 0, ctx->stream>>>(a);
  else split ? k_wgrad<1, true><<<grid, 256, 0, ctx->stream>>>(a) : k_wgrad<1, false><<<grid, 256, 0, ctx->stream>>>(a);
  FVM_LAUNCH_CHECK(ctx);
  const int64_t quads = (nw + Cout) / 4;  // channel counts are multiples of 16
  if (nchunk >= 32)
    k_wgrad_reduce<16><<<(unsigned)((quads + 15) / 16), 256, 0, ctx->stream>>>(work, (int)nchunk, nw, Cout, dW, db);
  else
    k_wgrad_reduce<4><<<(unsigned)((quads + 63) / 64), 256, 0, ctx->stream>>>(work, (int)nchunk, nw, Cout, dW, db);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

// dW (fp32 [tap][Cout][Cin]) and db (fp32 [Cout], may be null)
extern "C" int fvm_nn_conv_wgrad(fvm_ctx *ctx, const uint16_t *X, const uint16_t *dY, int32_t B, int32_t H,
                                 int32_t Wd, int32_t Cin, int32_t Cout, int32_t K, float *work, float *dW, float *db) {
  if (!ctx || !X || !dY || !work || !dW) return FVM_ERR_ARG;
  FVM_TRY(conv_check(ctx, B, H, Wd, Cin, Cout, K));
  FVM_PHASE(ctx, FVM_PHASE_OTHER);
  return wgrad_run(ctx, Input{X, nullptr, Cin, 0}, dY, B, H, Wd, Cin, Cout, K, work, dW, db);
}

extern "C" int fvm_nn_relu_bwd(fvm_ctx *ctx, int64_t n, const uint16_t *y, const uint16_t *dy, uint16_t *dz) {
  if (!ctx || !y || !dy || !dz) return FVM_ERR_ARG;
  k_relu_bwd<<<nblk(n), 256, 0, ctx->stream>>>(n, y, dy, dz);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

extern "C" int fvm_nn_pool_fwd(fvm_ctx *ctx, const uint16_t *X, int32_t B, int32_t H, int32_t W, int32_t C,
                               uint16_t *Y) {
  if (!ctx || !X || !Y || H % 2 || W % 2) return FVM_ERR_ARG;
  k_pool_fwd<<<nblk((int64_t)B * (H / 2) * (W / 2) * C), 256, 0, ctx->stream>>>(X, B, H, W, C, Y);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

extern "C" int fvm_nn_pool_bwd(fvm_ctx *ctx, const uint16_t *dY, int32_t B, int32_t H, int32_t W, int32_t C,
                               uint16_t *dX) {
  if (!ctx || !dY || !dX || H % 2 || W % 2) return FVM_ERR_ARG;
  k_pool_bwd<<<nblk((int64_t)B * H * W * C), 256, 0, ctx->stream>>>(dY, B, H, W, C, dX);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

extern "C" int fvm_nn_up_fwd(fvm_ctx *ctx, const uint16_t *X, int32_t B, int32_t H, int32_t W, int32_t C, uint16_t *Y,
                             int32_t Ctot, int32_t c0) {
  if (!ctx || !X || !Y || c0 < 0 || c0 + C > Ctot) return FVM_ERR_ARG;
  k_up_fwd<<<nblk((int64_t)B * 4 * H * W * C), 256, 0, ctx->stream>>>(X, B, H, W, C, Y, Ctot, c0);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

extern "C" int fvm_nn_up_bwd(fvm_ctx *ctx, const uint16_t *dY, int32_t B, int32_t H, int32_t W, int32_t C,
                             int32_t Ctot, int32_t c0, uint16_t *dX) {
  if (!ctx || !dY || !dX || c0 < 0 || c0 + C > Ctot) return FVM_ERR_ARG;
  k_up_bwd<<<nblk((int64_t)B * H * W * C), 256, 0, ctx->stream>>>(dY, B, H, W, C, Ctot, c0, dX);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

extern "C" int fvm_nn_copy_channels(fvm_ctx *ctx, const uint16_t *X, int64_t npix, int32_t C, int32_t Cx, int32_t xc0,
                                    uint16_t *Y, int32_t Ctot, int32_t c0) {
  if (!ctx || !X || !Y || xc0 < 0 || xc0 + C > Cx || c0 < 0 || c0 + C > Ctot) return FVM_ERR_ARG;
  k_copy_channels<<<nblk(npix * C), 256, 0, ctx->stream>>>(X, npix, C, Cx, xc0, Y, Ctot, c0);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

extern "C" int fvm_nn_add_channels(fvm_ctx *ctx, const uint16_t *X, int64_t npix, int32_t C, int32_t Cx, int32_t xc0,
                                   uint16_t *Y) {
  if (!ctx || !X || !Y || xc0 < 0 || xc0 + C > Cx) return FVM_ERR_ARG;
  k_add_channels<<<nblk(npix * C), 256, 0, ctx->stream>>>(X, npix, C, Cx, xc0, Y);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

// loss (fp32 scalar, device) = sum over pixels and real channels of ((out - tgt) mask)^2 * inv_count
extern "C" int fvm_nn_mse(fvm_ctx *ctx, const float *out, const float *tgt, const float *mask, int64_t npix, int32_t C,
                          int32_t Creal, float inv_count, uint16_t *dOut, float *work, float *loss) {
  if (!ctx || !out || !tgt || !dOut || !work || !loss || Creal > C) return FVM_ERR_ARG;
  const int64_t n = npix * C;
  const unsigned nb = (unsigned)((n + 256 * MSE_PER - 1) / (256 * MSE_PER));
  k_mse<<<nb, 256, 0, ctx->stream>>>(out, tgt, mask, npix, C, Creal, inv_count, dOut, work);
  k_sum_f<<<1, 256, 0, ctx->stream>>>(work, nb, loss);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

extern "C" int fvm_nn_adam(fvm_ctx *ctx, int64_t n, float *w, const float *g, float *m, float *v, uint16_t *wb,
                           float lr, float b1, float b2, float eps, int32_t step, float wd) {
  if (!ctx || !w || !g || !m || !v || step < 1) return FVM_ERR_ARG;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  k_adam<<<nblk(n), 256, 0, ctx->stream>>>(AdamArgs{w, g, m, v, wb, n, wd}, AdamRates{lr, b1, b2, eps, c1, c2});
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

extern "C" int fvm_nn_f32_to_bf16(fvm_ctx *ctx, int64_t n, const float *x, uint16_t *y) {
  if (!ctx || !x || !y) return FVM_ERR_ARG;
  k_f2bf<<<nblk(n), 256, 0, ctx->stream>>>(n, x, y);
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

// ---- the whole network -----------------------------------------------------------------
// One call per pass, instead of one per layer: the host's part of a pass shrinks to its
// launches, and the layers' copies, concatenations and ReLU passes go into the
// kernels beside them.  Tensors are NHWC bf16 unless noted, level i at H >> i, W >> i.
#define NN_LEVELS 12  // the 13th, with 65536 channels at 16 on the first, fits no card
typedef struct {
  int32_t levels, B, H, W, cin, cout, cout_real;
  int32_t ch[NN_LEVELS];
  // layers e0_1, e0_2, e1_1, ..., d(L-2)_1, d(L-2)_2, ..., d0_2, out
  const uint16_t *wb[4 * NN_LEVELS];
  const float *b[4 * NN_LEVELS];
  float *gw[4 * NN_LEVELS], *gb[4 * NN_LEVELS];
  uint16_t *x[NN_LEVELS], *h[NN_LEVELS], *e[NN_LEVELS];  // encoder: input, first and second activations
  uint16_t *dh[NN_LEVELS], *d[NN_LEVELS];                // decoder: first and second activations
  float *out;                                            // fp32
  // backward: gradients of x, of the pre-activations of h, e (g1, g2), dh, d, of the
  // decoder's input (concatenated), of out (bf16)
  uint16_t *dx[NN_LEVELS], *g1[NN_LEVELS], *g2[NN_LEVELS], *gdh[NN_LEVELS], *gd[NN_LEVELS], *dcat[NN_LEVELS], *dout;
  float *work;  // fvm_nn_wgrad_workspace of the largest layer
} fvm_unet;

namespace {
struct Layer {
  int at, K, ci, co, lvl;
};
Layer enc(const fvm_unet &u, int i, int j) {
  return Layer{2 * i + j, 3, j ? u.ch[i] : (i ? u.ch[i - 1] : u.cin), u.ch[i], i};
}
Layer dec(const fvm_unet &u, int i, int j) {
  return Layer{2 * u.levels + 2 * (u.levels - 2 - i) + j, 3, j ? u.ch[i] : u.ch[i + 1] + u.ch[i], u.ch[i], i};
}
Layer last(const fvm_unet &u) { return Layer{4 * u.levels - 2, 1, u.ch[0], u.cout, 0}; }

int unet_check(fvm_ctx *ctx, const fvm_unet *u) {
  if (!ctx || !u || u->levels < 1 || u->levels > NN_LEVELS) return FVM_ERR_ARG;
  const int m = (1 << (u->levels - 1)) - 1;
  if (u->B < 1 || u->H < 1 || u->W < 1 || (u->H & m) || (u->W & m))
    return fvm_set_err(ctx, FVM_ERR_ARG, "unet: H and W must divide by 2^(levels-1)");
  for (int i = 0; i < u->levels; i++)
    if (u->ch[i] < 16 || u->ch[i] % 16) return fvm_set_err(ctx, FVM_ERR_ARG, "unet: channels must be multiples of 16");
  if (u->cin < 16 || u->cin % 16 || u->cout < 16 || u->cout % 16)
    return fvm_set_err(ctx, FVM_ERR_ARG, "unet: channels must be multiples of 16");
  return FVM_OK;
}
Input plain(const uint16_t *X, int C) { return Input{X, nullptr, C, 0}; }

int fwd(fvm_ctx *ctx, const fvm_unet &u, const Layer &l, const Input &in, uint16_t *Y, float *Yf) {
  ConvArgs a{in, u.wb[l.at], u.b[l.at], nullptr, Y, Yf, u.B, u.H >> l.lvl, u.W >> l.lvl, l.ci, l.co, Yf ? 0 : 1,
             Yf ? u.cout_real : l.co};
  return conv_run(ctx, a, l.K, false, nullptr);
}
// data gradient of layer l, through the ReLU of the activations it took (mask, or null);
// the weight gradients' workspace is free between them and has room for the weights
int dgrad(fvm_ctx *ctx, const fvm_unet &u, const Layer &l, const uint16_t *dY, const uint16_t *mask, uint16_t *dX) {
  ConvArgs a{plain(dY, l.co), u.wb[l.at], nullptr, mask, dX, nullptr, u.B, u.H >> l.lvl, u.W >> l.lvl, l.co, l.ci, 0, l.ci};
  return conv_run(ctx, a, l.K, true, (uint16_t *)u.work);
}
int wgrad(fvm_ctx *ctx, const fvm_unet &u, const Layer &l, const Input &in, const uint16_t *dY) {
  return wgrad_run(ctx, in, dY, u.B, u.H >> l.lvl, u.W >> l.lvl, l.ci, l.co, l.K, u.work, u.gw[l.at], u.gb[l.at]);
}
}  // namespace

extern "C" int fvm_nn_unet_forward(fvm_ctx *ctx, const fvm_unet *up, const uint16_t *X) {
  FVM_TRY(unet_check(ctx, up));
  const fvm_unet &u = *up;
  const int L = u.levels;
  FVM_PHASE(ctx, FVM_PHASE_OTHER);
  // the caller may refill X before the backward pass
  const int64_t npix = (int64_t)u.B * u.H * u.W, n8 = npix * u.cin / 8;
  if (!X) return FVM_ERR_ARG;
  if (((uintptr_t)X & 15) == 0) k_copy8<<<nblk(n8), 256, 0, ctx->stream>>>(n8, X, u.x[0]);
  else k_copy_channels<<<nblk(npix * u.cin), 256, 0, ctx->stream>>>(X, npix, u.cin, u.cin, 0, u.x[0], u.cin, 0);
  for (int i = 0; i < L; i++) {
    FVM_TRY(fwd(ctx, u, enc(u, i, 0), plain(u.x[i], enc(u, i, 0).ci), u.h[i], nullptr));
    FVM_TRY(fwd(ctx, u, enc(u, i, 1), plain(u.h[i], u.ch[i]), u.e[i], nullptr));
    if (i < L - 1) {
      const int h = u.H >> i, w = u.W >> i;
      k_pool8<<<nblk((int64_t)u.B * (h / 2) * (w / 2) * u.ch[i] / 8), 256, 0, ctx->stream>>>(u.e[i], u.B, h, w, u.ch[i],
                                                                                         u.x[i + 1]);
    }
  }
  const uint16_t *below = u.e[L - 1];
  for (int i = L - 2; i >= 0; i--) {
    FVM_TRY(fwd(ctx, u, dec(u, i, 0), Input{below, u.e[i], u.ch[i + 1], 1}, u.dh[i], nullptr));
    FVM_TRY(fwd(ctx, u, dec(u, i, 1), plain(u.dh[i], u.ch[i]), u.d[i], nullptr));
    below = u.d[i];
  }
  FVM_TRY(fwd(ctx, u, last(u), plain(below, u.ch[0]), nullptr, u.out));
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

// every gw, gb from dout
extern "C" int fvm_nn_unet_backward(fvm_ctx *ctx, const fvm_unet *up) {
  FVM_TRY(unet_check(ctx, up));
  const fvm_unet &u = *up;
  const int L = u.levels;
  FVM_PHASE(ctx, FVM_PHASE_OTHER);
  // top: the output layer, through the ReLU of the activations below it
  const uint16_t *act = L > 1 ? u.d[0] : u.e[0];
  uint16_t *g = L > 1 ? u.gd[0] : u.g2[0];
  FVM_TRY(wgrad(ctx, u, last(u), plain(act, u.ch[0]), u.dout));
  FVM_TRY(dgrad(ctx, u, last(u), u.dout, act, g));
  for (int i = 0; i < L - 1; i++) {
    const int h = u.H >> (i + 1), w = u.W >> (i + 1), cc = u.ch[i + 1] + u.ch[i];
    const uint16_t *below = i + 1 < L - 1 ? u.d[i + 1] : u.e[i + 1];
    FVM_TRY(wgrad(ctx, u, dec(u, i, 1), plain(u.dh[i], u.ch[i]), u.gd[i]));
    FVM_TRY(dgrad(ctx, u, dec(u, i, 1), u.gd[i], u.dh[i], u.gdh[i]));
    FVM_TRY(wgrad(ctx, u, dec(u, i, 0), Input{below, u.e[i], u.ch[i + 1], 1}, u.gdh[i]));
    FVM_TRY(dgrad(ctx, u, dec(u, i, 0), u.gdh[i], nullptr, u.dcat[i]));
    k_up_bwd8<<<nblk((int64_t)u.B * h * w * u.ch[i + 1] / 8), 256, 0, ctx->stream>>>(
        u.dcat[i], u.B, h, w, u.ch[i + 1], cc, below, i + 1 < L - 1 ? u.gd[i + 1] : u.g2[i + 1]);
  }
  for (int i = L - 1; i >= 0; i--) {
    const int h = u.H >> i, w = u.W >> i;
    if (i < L - 1)
      k_skip_bwd8<<<nblk((int64_t)u.B * h * w * u.ch[i] / 8), 256, 0, ctx->stream>>>(
          u.dcat[i], u.ch[i + 1] + u.ch[i], u.ch[i + 1], u.dx[i + 1], u.B, h, w, u.ch[i], u.e[i], u.g2[i]);
    FVM_TRY(wgrad(ctx, u, enc(u, i, 1), plain(u.h[i], u.ch[i]), u.g2[i]));
    FVM_TRY(dgrad(ctx, u, enc(u, i, 1), u.g2[i], u.h[i], u.g1[i]));
    FVM_TRY(wgrad(ctx, u, enc(u, i, 0), plain(u.x[i], enc(u, i, 0).ci), u.g1[i]));
    if (i > 0) FVM_TRY(dgrad(ctx, u, enc(u, i, 0), u.g1[i], nullptr, u.dx[i]));
  }
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}

// Adam on `nt` tensors (n[k] elements; wb[k] may be null), as fvm_nn_adam on each
extern "C" int fvm_nn_adam_all(fvm_ctx *ctx, int32_t nt, const int64_t *n, float *const *w, const float *const *g,
                               float *const *m, float *const *v, uint16_t *const *wb, const float *wd, float lr, float b1,
                               float b2, float eps, int32_t step) {
  if (!ctx || nt < 0 || !n || !w || !g || !m || !v || !wb || !wd || step < 1) return FVM_ERR_ARG;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  FVM_PHASE(ctx, FVM_PHASE_OTHER);
  for (int k0 = 0; k0 < nt; k0 += ADAM_MAX) {
    AdamAll A;
    A.n = nt - k0 < ADAM_MAX ? nt - k0 : ADAM_MAX;
    int64_t blocks = 0;
    for (int k = 0; k < A.n; k++) {
      const int q = k0 + k;
      if (!w[q] || !g[q] || !m[q] || !v[q] || n[q] < 0) return FVM_ERR_ARG;
      A.t[k] = AdamArgs{w[q], g[q], m[q], v[q], wb[q], n[q], wd[q]};
      A.first[k] = (int)blocks;
      blocks += nblk(n[q]);
      if (blocks > INT32_MAX) return FVM_ERR_ARG;
    }
    A.first[A.n] = (int)blocks;
    if (blocks) k_adam_all<<<(unsigned)blocks, 256, 0, ctx->stream>>>(A, AdamRates{lr, b1, b2, eps, c1, c2});
  }
  FVM_LAUNCH_CHECK(ctx);
  return FVM_OK;
}
