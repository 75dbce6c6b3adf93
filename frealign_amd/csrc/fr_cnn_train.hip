// fr_cnn_train.hip -- the mixed-precision training step of the orientation
// proposal for networks of 64 channels (every trained configuration; other
// channel counts take the general GEMMs of fr_cnn.hip).
//
// Same operands and arithmetic as the general step: FP32 activations and
// gradients in memory, each product's operands rounded to BF16 as they are
// read, FP32 accumulation on v_mfma_f32_16x16x32_bf16, bias, ReLU and bias
// gradients in FP32.  What differs is the layout and the split of the work.
//
// Layout: activations and gradients are [B][H][W][64], channels innermost, so
// that 8 consecutive K values of a fragment are 8 channels of one pixel (32
// contiguous bytes, two loads), the taps of a convolution are address offsets
// rather than an index division per element, and a pixel's 64 results are 256
// contiguous bytes.  Fragments go from global memory (L1 and L2: every pixel is
// read by at most 2.25 taps) straight to registers (a convolution's
// weights through LDS).
//
// What bounds it: at 256 images of 64^2 the layers are 65,536, 16,384 and
// 4,096 positions by 576 x 64, a few microseconds each on the matrix cores, and
// the first layer's activations are 64 MB: launches, load latency and that
// traffic, in this order.  So the input gradient is one launch for all four
// parity classes (each loads the four shifted gradients once and writes whole
// pixels; four launches of strided 4-byte stores before), the weight
// gradients' bias sums ride on the fragments they load anyway, all splits of
// all layers are added by one kernel at the end, and weights are put in
// fragment order once per step.
//
// Measured, forward and backward of that batch with 4 convolutions:
// 857 -> 251 us (convolution 1 forward 73 -> 27, its input gradient 161 -> 31,
// its weight gradient with its sums 142 -> 50).
#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fr_cnn.h"

namespace fr {

namespace {

constexpr int kT = 256;
constexpr int kC = 64;          // channels
constexpr int kW = 9 * kC * kC; // weights of a convolution after the first
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float fx4;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bfx8;

__device__ inline fx4 mfma(bfx8 a, bfx8 b, fx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ inline bfx8 round8(fx4 u, fx4 v) {
  bfx8 r;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    r[j] = (__bf16)u[j];
    r[4 + j] = (__bf16)v[j];
  }
  return r;
}

// 8 consecutive floats rounded to BF16
__device__ inline bfx8 frag8(const float* p) {
  return round8(*reinterpret_cast<const fx4*>(p), *reinterpret_cast<const fx4*>(p + 4));
}

// p's four floats where ok, else zeros.  The load is always made (p is a valid
// address either way): a branch around it would keep the compiler from having
// the next steps' loads in flight

__device__ inline fx4 load4_if(const float* p, bool ok) {
  const fx4 v = *reinterpret_cast<const fx4*>(p);
  return ok ? v : fx4{0.f, 0.f, 0.f, 0.f};
}

struct TrainShape {
  int S, L, K, Kp, F, P;  // Kp: classes rounded up to 32
  long long w_off[8], b_off[8], fw_off, fb_off;
};

// The step's weights in fragment order, BF16 (the values are BF16 already):
// per convolution l >= 1 the fragments (tap, half of K, block of 16 rows) as the
// 64 lanes hold them, 1 kB each: wf with rows co and K ci, wx with rows ci and K
// co; fully connected ff[k][p][c] and fx[p][c][Kp] (zero beyond K).
__global__ void __launch_bounds__(kT)
    k_train_weights(TrainShape t, const float* __restrict__ wq, __bf16* wf, __bf16* wx, __bf16* ff,
                    __bf16* fx) {
  const long long nconv = (long long)(t.L - 1) * kW, nff = (long long)t.K * t.F;
  long long i = blockIdx.x * (long long)kT + threadIdx.x;
  if (i < nconv) {
    const int l = 1 + (int)(i / kW), e = (int)(i % kW);
    const int j = e & 7, la = e >> 3 & 15, lg = e >> 7 & 3, m = e >> 9 & 3, h = e >> 11 & 1;
    const int tap = e >> 12, row = 16 * m + la, col = 32 * h + 8 * lg + j;
    const float* w = wq + t.w_off[l];
    wf[i] = (__bf16)w[(row * kC + col) * 9 + tap];
    wx[i] = (__bf16)w[(col * kC + row) * 9 + tap];
    return;
  }
  i -= nconv;
  if (i < nff) {
    const int c = (int)(i % kC), p = (int)(i / kC % t.P);
    const long long k = i / t.F;
    ff[i] = (__bf16)wq[t.fw_off + k * t.F + (long long)c * t.P + p];
    return;
  }
  i -= nff;
  if (i < (long long)t.F * t.Kp) {
    const int k = (int)(i % t.Kp);
    const long long f = i / t.Kp;
    const int c = (int)(f % kC), p = (int)(f / kC);
    fx[i] = (__bf16)(k < t.K ? wq[t.fw_off + (long long)k * t.F + (long long)c * t.P + p] : 0.f);
  }
}

// bias and ReLU of a 16-position column of accumulators; lane (la, lg) holds
// channels 16 m + 4 lg + r of position la
__device__ inline void store_relu(const fx4* acc, const float* __restrict__ bias, int lg,
                                  float* out) {
#pragma unroll
  for (int m = 0; m < 4; m++) {
    fx4 v;
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = fmaxf(acc[m][r] + bias[16 * m + 4 * lg + r], 0.f);
    *reinterpret_cast<fx4*>(out + 16 * m + 4 * lg) = v;
  }
}

// Convolution 0: 9 taps in one fragment (8 in the lanes of group 0, the ninth
// in group 1, zeros beyond).  A wave: 16 positions a time, four times.
__global__ void __launch_bounds__(kT)
    k_train_conv0(int B, int H, const float* __restrict__ img, const float* __restrict__ w,
                  const float* __restrict__ bias, float* out) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, la = lane & 15, lg = lane >> 4;
  const int Ho = H / 2, P = Ho * Ho, N = B * P;
  bfx8 a[4];
#pragma unroll
  for (int m = 0; m < 4; m++)
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int tap = 8 * lg + j;
      a[m][j] = (__bf16)(tap < 9 ? w[(16 * m + la) * 9 + tap] : 0.f);
    }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int n0 = blockIdx.x * 256 + wave * 64 + q * 16 + la, n = min(n0, N - 1);
    const int im = n / P, r = n - im * P, oy = r / Ho, ox = r - oy * Ho;
    const float* px = img + ((long long)im * H + 2 * oy) * H + 2 * ox;
    bfx8 b;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int tap = 8 * lg + j, ky = tap / 3, kx = tap - 3 * ky;
      const bool ok = tap < 9 && (ky > 0 || oy > 0) && (kx > 0 || ox > 0);
      const float v = px[ok ? (ky - 1) * H + kx - 1 : 0];
      b[j] = (__bf16)(ok ? v : 0.f);
    }
    fx4 acc[4];
#pragma unroll
    for (int m = 0; m < 4; m++) acc[m] = mfma(a[m], b, fx4{0.f, 0.f, 0.f, 0.f});
    if (n0 < N) store_relu(acc, bias, lg, out + (long long)n * kC);
  }
}

// A convolution's 72 weight fragments into LDS (all 256 threads), by loads that
// write LDS themselves: a wave's 64 x 16 bytes go to one address and the lanes
// after it.  train_weights_wait() before they are read.
constexpr int kFrags = 72;
constexpr size_t kWLds = (size_t)kW * sizeof(__bf16);

__device__ inline void train_weights_load(const __bf16* __restrict__ w, bfx8* wl) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < kFrags / 4; i++) {
    const int f = 4 * i + wave;
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void*)(w + ((size_t)f * 64 + lane) * 8),
        (__attribute__((address_space(3))) void*)(wl + f * 64), 16, 0, 0);
  }
}

__device__ inline void train_weights_wait() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// Convolution l >= 1: a wave computes the 64 channels of 16 positions over the
// 18 (tap, half of the channels) steps, all of its loads issued before the
// first product; the weights are in LDS, loaded once by a workgroup for all of
// its positions (read from L2 by every wave they were most of its time: 53 us
// for 65,536 positions, 15 us for 4,096; 27 and 8 us here).
__global__ void __launch_bounds__(kT, 2)
    k_train_conv(int B, int H, const float* __restrict__ in, const __bf16* __restrict__ wf,
                 const float* __restrict__ bias, float* out) {
  extern __shared__ bfx8 wl[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, la = lane & 15, lg = lane >> 4;
  const int Ho = H / 2, P = Ho * Ho, N = B * P;
  train_weights_load(wf, wl);
  for (int tile = blockIdx.x; tile * 64 < N; tile += gridDim.x) {
    const int n0 = tile * 64 + wave * 16 + la, n = min(n0, N - 1);
    const int im = n / P, r = n - im * P, oy = r / Ho, ox = r - oy * Ho;
    // the centre tap, inside for every position
    const float* px = in + (((long long)im * H + 2 * oy) * H + 2 * ox) * kC + 8 * lg;
    fx4 x[18][2];
#pragma unroll
    for (int s = 0; s < 18; s++) {
      const int ky = s / 6, kx = s / 2 % 3;
      // the padding: only row -1 and column -1 lie outside (H is even)
      const bool ok = (ky > 0 || oy > 0) && (kx > 0 || ox > 0);
      const float* p = px + (ok ? ((ky - 1) * H + kx - 1) * kC : 0) + 32 * (s & 1);
      x[s][0] = load4_if(p, ok);
      x[s][1] = load4_if(p + 4, ok);
    }
    if (tile == (int)blockIdx.x) train_weights_wait();
    fx4 acc[4];
#pragma unroll
    for (int m = 0; m < 4; m++) acc[m] = fx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 18; s++) {
      const bfx8 b = round8(x[s][0], x[s][1]);
#pragma unroll
      for (int m = 0; m < 4; m++) acc[m] = mfma(wl[(s * 4 + m) * 64 + lane], b, acc[m]);
    }
    if (n0 < N) store_relu(acc, bias, lg, out + (long long)n * kC);
  }
}

// sums the four waves' accumulators of one 16x16 block; wave 0 returns them
__device__ inline fx4 wave_sum(fx4 acc, fx4 (*red)[64], int wave, int lane) {
  red[wave][lane] = acc;
  __syncthreads();
  return (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

// logits[b][k] = sum_f Wfc[k][f] X[b][f] + bfc[k]: a workgroup 16 classes x 16
// images, its waves each a quarter of the 2 P steps over f = (p, c).
__global__ void __launch_bounds__(kT)
    k_train_fc(int K, int B, int F, const __bf16* __restrict__ ff, const float* __restrict__ bias,
               const float* __restrict__ X, float* logits) {
  __shared__ fx4 red[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, la = lane & 15, lg = lane >> 4;
  const int k = blockIdx.y * 16 + la, b = blockIdx.x * 16 + la;
  fx4 acc = fx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int f0 = 32 * wave; f0 < F; f0 += 128) {
    // rows and columns beyond the last are not stored
    const bfx8 av =
        *reinterpret_cast<const bfx8*>(ff + (long long)min(k, K - 1) * F + f0 + 8 * lg);
    const bfx8 bv = frag8(X + (long long)min(b, B - 1) * F + f0 + 8 * lg);
    acc = mfma(av, bv, acc);
  }
  const fx4 s = wave_sum(acc, red, wave, lane);
  if (wave || b >= B) return;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int kr = blockIdx.y * 16 + 4 * lg + r;
    if (kr < K) logits[(long long)b * K + kr] = s[r] + bias[kr];
  }
}

// gWfc[k][c P + p] = sum_b gL[b][k] X[b][(p, c)] and gbfc[k] = sum_b gL[b][k]:
// a wave 16 classes x 64 of f = (p, c), its four blocks interleaved (block i,
// column la: f0 + 4 la + i) so that a position's operands are one load.  The
// first wave of a class block adds the loss gradients it loads, in FP32.
__global__ void __launch_bounds__(kT)
    k_train_fc_wgrad(int K, int Kp, int B, int F, int P, const float* __restrict__ gL,
                     const float* __restrict__ X, float* gw, float* gb) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, la = lane & 15, lg = lane >> 4;
  const int k0 = blockIdx.y * 16, f0 = (blockIdx.x * 4 + wave) * 64;
  if (f0 >= F) return;
  fx4 acc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) acc[i] = fx4{0.f, 0.f, 0.f, 0.f};
  float sum = 0.f;
#pragma unroll 2
  for (int b0 = 0; b0 < B; b0 += 32) {
    bfx8 a, bv[4];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int b = b0 + 8 * lg + j;
      const bool on = b < B;
      const long long bc = on ? b : 0;
      const float gv = gL[bc * Kp + k0 + la], g = on ? gv : 0.f;
      const fx4 x = load4_if(X + bc * F + f0 + 4 * la, on);
      sum += g;
      a[j] = (__bf16)g;
#pragma unroll
      for (int i = 0; i < 4; i++) bv[i][j] = (__bf16)x[i];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = mfma(a, bv[i], acc[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int f = f0 + 4 * la + i, p = f / kC, c = f - p * kC;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int k = k0 + 4 * lg + r;
      if (k < K) gw[(long long)k * F + (long long)c * P + p] = acc[i][r];
    }
  }
  if (f0 == 0) {
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (lg == 0 && k0 + la < K) gb[k0 + la] = sum;
  }
}

// g[b][f] = (act[b][f] > 0) x sum_k Wfc[k][f] gL[b][k]: a wave 16 of f by 16
// images.
__global__ void __launch_bounds__(kT)
    k_train_fc_xgrad(int Kp, int B, int F, const __bf16* __restrict__ fx,
                     const float* __restrict__ gL, const float* __restrict__ act, float* g) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, la = lane & 15, lg = lane >> 4;
  const int f0 = (blockIdx.y * 4 + wave) * 16, b = blockIdx.x * 16 + la;
  fx4 acc = fx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k0 = 0; k0 < Kp; k0 += 32) {
    const bfx8 av =
        *reinterpret_cast<const bfx8*>(fx + (long long)(f0 + la) * Kp + k0 + 8 * lg);
    const bfx8 bv = frag8(gL + (long long)min(b, B - 1) * Kp + k0 + 8 * lg);
    acc = mfma(av, bv, acc);
  }
  if (b >= B) return;
  const long long at = (long long)b * F + f0 + 4 * lg;
  const fx4 m = *reinterpret_cast<const fx4*>(act + at);
#pragma unroll
  for (int r = 0; r < 4; r++) acc[r] = m[r] > 0.f ? acc[r] : 0.f;
  *reinterpret_cast<fx4*>(g + at) = acc;
}

// Input gradient of convolution l >= 1 through the ReLU below:
// gin[b][y][x][ci] = (act > 0) x sum over co, ky, kx of W[co][ci][ky][kx]
// g[b][oy][ox][co] with 2 oy + ky - 1 = y, 2 ox + kx - 1 = x.  For y = 2t + py
// the taps are ky = 1 (py = 0, oy = t) and ky = 0, 2 (py = 1, oy = t + 1, t),
// x alike: a wave takes 16 (t, u), loads the gradient at its four shifts and
// adds each of the 9 taps to its parity class's accumulators.
// Weights and loads as in the forward.
__global__ void __launch_bounds__(kT, 2)
    k_train_xgrad(int B, int H, const __bf16* __restrict__ wx, const float* __restrict__ g,
                  const float* __restrict__ act, float* gin) {
  extern __shared__ bfx8 wl[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, la = lane & 15, lg = lane >> 4;
  const int Ho = H / 2, P = Ho * Ho, N = B * P;
  train_weights_load(wx, wl);
  for (int tile = blockIdx.x; tile * 64 < N; tile += gridDim.x) {
    const int n0 = tile * 64 + wave * 16 + la, n = min(n0, N - 1);
    const int im = n / P, r = n - im * P, t = r / Ho, u = r - t * Ho;
    const float* gp = g + (long long)n * kC + 8 * lg;
    const long long at0 = (((long long)im * H + 2 * t) * H + 2 * u) * kC + 4 * lg;
    fx4 x[4][2][2], a[4][4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int dy = s >> 1, dx = s & 1;
      const bool ok = t + dy < Ho && u + dx < Ho;
      const float* p = gp + (ok ? (dy * Ho + dx) * kC : 0);
#pragma unroll
      for (int h = 0; h < 2; h++) {
        x[s][h][0] = load4_if(p + 32 * h, ok);
        x[s][h][1] = load4_if(p + 32 * h + 4, ok);
      }
    }
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int m = 0; m < 4; m++)
        a[c][m] = *reinterpret_cast<const fx4*>(act + at0 + ((c >> 1) * H + (c & 1)) * kC + 16 * m);
    if (tile == (int)blockIdx.x) train_weights_wait();
    bfx8 b[4][2];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int h = 0; h < 2; h++) b[s][h] = round8(x[s][h][0], x[s][h][1]);
#pragma unroll
    for (int c = 0; c < 4; c++) {
      fx4 acc[4];
#pragma unroll
      for (int m = 0; m < 4; m++) acc[m] = fx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int tap = 0; tap < 9; tap++) {
        const int ky = tap / 3, kx = tap - 3 * ky;
        if ((ky == 1 ? 0 : 2) + (kx == 1 ? 0 : 1) != c) continue;
        const int sh = (ky == 0 ? 2 : 0) + (kx == 0 ? 1 : 0);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int m = 0; m < 4; m++)
            acc[m] = mfma(wl[((tap * 2 + h) * 4 + m) * 64 + lane], b[sh][h], acc[m]);
      }
      if (n0 < N)
#pragma unroll
        for (int m = 0; m < 4; m++) {
          fx4 v;
#pragma unroll
          for (int q = 0; q < 4; q++) v[q] = a[c][m][q] > 0.f ? acc[m][q] : 0.f;
          *reinterpret_cast<fx4*>(gin + at0 + ((c >> 1) * H + (c & 1)) * kC + 16 * m) = v;
        }
    }
  }
}

// Weight gradient of convolution l >= 1 over one split of the positions:
// part[split][tap][co][ci] and, after the 9 taps, [co] of the bias.  A
// workgroup is one split and one ky, its three waves the kx: 64 x 64 results
// of one tap, 16 products of 32 positions from 16 loads.  Rows and columns of
// the four blocks are interleaved (block i, row m: channel 4 m + i), so that a
// position's four operands are one 16-byte load; the next 32 positions are
// loaded while these are multiplied.  39 us for 65,536 positions: the 144 kB
// that the nine taps load per 32 positions through L1.
__global__ void __launch_bounds__(192)
    k_train_wgrad(int B, int H, int chunk, const float* __restrict__ g,
                  const float* __restrict__ in, float* part) {
  const int lane = threadIdx.x & 63, kx = threadIdx.x >> 6, ky = blockIdx.y;
  const int la = lane & 15, lg = lane >> 4;
  const int Ho = H / 2, P = Ho * Ho, N = B * P;
  const int nbeg = blockIdx.x * chunk, nend = min(N, nbeg + chunk);
  fx4 acc[4][4], ga[8], xa[8], sum = fx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = fx4{0.f, 0.f, 0.f, 0.f};
  auto load = [&](int n0) {
    int n = n0 + 8 * lg;
    int im = n / P, r = n - im * P, oy = r / Ho, ox = r - oy * Ho;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      // at the padding and beyond the split: the tensors' first pixel, as zero
      const bool on = n < nend, ok = on && (ky > 0 || oy > 0) && (kx > 0 || ox > 0);
      ga[j] = load4_if(g + (on ? (long long)n * kC : 0) + 4 * la, on);
      xa[j] = load4_if(
          in + (ok ? (((long long)im * H + 2 * oy + ky - 1) * H + 2 * ox + kx - 1) * kC : 0) + 4 * la,
          ok);
      n++;
      if (++ox == Ho) {
        ox = 0;
        if (++oy == Ho) {
          oy = 0;
          im++;
        }
      }
    }
  };
  load(nbeg);
  for (int n0 = nbeg; n0 < nend; n0 += 32) {
    bfx8 a[4], b[4];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      sum += ga[j];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        a[i][j] = (__bf16)ga[j][i];
        b[i][j] = (__bf16)xa[j][i];
      }
    }
    if (n0 + 32 < nend) load(n0 + 32);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = mfma(a[i], b[j], acc[i][j]);
  }
  float* out = part + (long long)blockIdx.x * (kW + kC);
  float* ot = out + (ky * 3 + kx) * kC * kC;
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int co = 4 * (4 * lg + r) + i;
      const fx4 v{acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
      *reinterpret_cast<fx4*>(ot + co * kC + 4 * la) = v;
    }
  if (ky == 0 && kx == 0) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      sum[i] += __shfl_xor(sum[i], 16, 64);
      sum[i] += __shfl_xor(sum[i], 32, 64);
    }
    if (lg == 0) *reinterpret_cast<fx4*>(out + kW + 4 * la) = sum;
  }
}

// Weight gradient of convolution 0 over one split: part[split][tap][co], then
// [co] of the bias.  One block of columns holds the 9 taps; the waves take
// every fourth run of 32 positions.
__global__ void __launch_bounds__(kT)
    k_train_wgrad0(int B, int H, int chunk, const float* __restrict__ g,
                   const float* __restrict__ img, float* part) {
  __shared__ fx4 red[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, la = lane & 15, lg = lane >> 4;
  const int Ho = H / 2, P = Ho * Ho, N = B * P;
  const int nbeg = blockIdx.x * chunk, nend = min(N, nbeg + chunk);
  const int ky = la / 3, kx = la - 3 * ky;
  fx4 acc[4], sum = fx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; i++) acc[i] = fx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int n0 = nbeg + 32 * wave; n0 < nend; n0 += 128) {
    int n = n0 + 8 * lg;
    int im = n / P, r = n - im * P, oy = r / Ho, ox = r - oy * Ho;
    bfx8 a[4], b;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const bool on = n < nend, ok = on && la < 9 && (ky > 0 || oy > 0) && (kx > 0 || ox > 0);
      const fx4 gv = load4_if(g + (on ? (long long)n * kC : 0) + 4 * la, on);
      float xv = img[ok ? ((long long)im * H + 2 * oy + ky - 1) * H + 2 * ox + kx - 1 : 0];
      xv = ok ? xv : 0.f;
      sum += gv;
      b[j] = (__bf16)xv;
#pragma unroll
      for (int i = 0; i < 4; i++) a[i][j] = (__bf16)gv[i];
      n++;
      if (++ox == Ho) {
        ox = 0;
        if (++oy == Ho) {
          oy = 0;
          im++;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = mfma(a[i], b, acc[i]);
  }
  float* out = part + (long long)blockIdx.x * (10 * kC);
  // acc[i]: rows m = 4 lg + r are channels 4 m + i, column la the tap
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const fx4 s = wave_sum(acc[i], red, wave, lane);
    if (wave == 0 && la < 9)
#pragma unroll
      for (int r = 0; r < 4; r++) out[la * kC + 4 * (4 * lg + r) + i] = s[r];
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    sum[i] += __shfl_xor(sum[i], 16, 64);
    sum[i] += __shfl_xor(sum[i], 32, 64);
  }
  const fx4 s = wave_sum(sum, red, wave, lane);
  if (wave == 0 && lg == 0) *reinterpret_cast<fx4*>(out + 9 * kC + 4 * la) = s;
}

// The layers' splits added in a fixed order and put where the parameters lie.
// A block: 64 consecutive values of one layer's row (16 loads of 16 bytes) by
// 16 groups of splits.  One launch for the step, 577 blocks a layer; a serial
// loop over the splits per value took 54 us for one layer of 228 splits.
struct TrainSums {
  long long part[8], w_off[8], b_off[8];
  int nsplit[8], first[9];  // first block of each layer
};

__global__ void __launch_bounds__(kT)
    k_train_sums(TrainSums t, int L, const float* __restrict__ part, float* grad) {
  __shared__ fx4 red[16][16];
  int l = 0;
  while (l + 1 < L && (int)blockIdx.x >= t.first[l + 1]) l++;
  const int cin = l ? kC : 1, nw = 9 * kC * cin, row = nw + kC;
  const int col = threadIdx.x & 15, grp = threadIdx.x >> 4;
  const int e0 = ((int)blockIdx.x - t.first[l]) * 64 + 4 * col;
  const float* p = part + t.part[l] + e0;
  fx4 s = fx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int q = grp; q < t.nsplit[l]; q += 16)
    s += *reinterpret_cast<const fx4*>(p + (long long)q * row);
  red[grp][col] = s;
  __syncthreads();
  if (grp) return;
#pragma unroll
  for (int q = 1; q < 16; q++) s += red[q][col];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int e = e0 + i;
    if (e >= nw) {
      grad[t.b_off[l] + e - nw] = s[i];
    } else {
      // row [tap][co][ci]; parameters [co][ci][tap]
      const int tap = e / (kC * cin), r = e - tap * kC * cin;
      grad[t.w_off[l] + (long long)r * 9 + tap] = s[i];
    }
  }
}

inline unsigned nblk(long long n, long long per) { return (unsigned)((n + per - 1) / per); }

// splits of a layer's positions: at least 128 positions each, at most this
// many (partials of 148 kB a split are written and read back; 65,536 positions
// in 128 splits 39 us, in 205 46 us), and all layers' partials within
// kPartFloats
constexpr int kMaxSplit = 128, kMaxSplit0 = 512;
constexpr long long kPartFloats = 16ll << 20;

int split_count(const CnnLayout& lo, int l, long long N) {
  long long cap = kMaxSplit0;
  if (l > 0)
    cap = std::min<long long>(kMaxSplit, (kPartFloats - kMaxSplit0 * 10 * kC) /
                                             ((long long)(kW + kC) * (lo.L - 1)));
  return (int)std::max<long long>(1, std::min(cap, N / 128));
}

// workspace offsets (floats), each a multiple of 64
struct Ws {
  size_t act[8], logits, gL, gA, gB, part, wf, wx, ff, fx, total;
};

Ws ws_layout(const CnnLayout& lo, int B) {
  Ws w{};
  size_t o = 0;
  auto take = [&](size_t n) {
    const size_t at = o;
    o += (n + 63) / 64 * 64;
    return at;
  };
  const size_t Kp = (lo.K + 31) / 32 * 32;
  for (int l = 0; l < lo.L; l++) w.act[l] = take((size_t)kC * B * lo.hout(l) * lo.hout(l));
  w.logits = take((size_t)lo.K * B);
  w.gL = take(Kp * B);
  const size_t g0 = (size_t)kC * B * lo.hout(0) * lo.hout(0);
  w.gA = take(g0);
  w.gB = take(g0);
  w.part = take(kPartFloats);
  w.wf = take((size_t)(lo.L - 1) * kW / 2);
  w.wx = take((size_t)(lo.L - 1) * kW / 2);
  w.ff = take((size_t)lo.K * lo.F() / 2);
  w.fx = take((size_t)lo.F() * Kp / 2);
  w.total = o;
  return w;
}

}  // namespace

bool cnn_train_ok(const CnnLayout& lo) { return lo.C == kC; }

size_t cnn_train_workspace(const CnnLayout& lo, int B) { return ws_layout(lo, B).total; }

int cnn_train_backward(Ctx& c, const CnnLayout& lo, const float* wq, int B, const float* img,
                       const int* label, float* ws, float* loss, float* grad) {
  const int L = lo.L, K = lo.K, F = lo.F(), Kp = (K + 31) / 32 * 32;
  FR_CHECK((long long)B * lo.hout(0) * lo.hout(0) <= kCnnMaxPositions,
           "batch too large for the bias reduction");
  FR_CHECK(nblk(F, 64) < 65536u, "GEMM too tall");
  const Ws w = ws_layout(lo, B);
  TrainShape t{};
  t.S = lo.S;
  t.L = L;
  t.K = K;
  t.Kp = Kp;
  t.F = F;
  t.P = F / kC;
  for (int l = 0; l < L; l++) t.w_off[l] = lo.w_off[l];
  t.fw_off = lo.fw_off;
  __bf16* wf = reinterpret_cast<__bf16*>(ws + w.wf);
  __bf16* wx = reinterpret_cast<__bf16*>(ws + w.wx);
  __bf16* ff = reinterpret_cast<__bf16*>(ws + w.ff);
  __bf16* fx = reinterpret_cast<__bf16*>(ws + w.fx);
  const dim3 blk(kT);
  // two workgroups' weights fit a CU's LDS
  const unsigned kGrid = 512;
  FR_HIP(hipFuncSetAttribute((const void*)k_train_conv,
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)kWLds));
  FR_HIP(hipFuncSetAttribute((const void*)k_train_xgrad,
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)kWLds));
  hipLaunchKernelGGL(k_train_weights,
                     dim3(nblk((long long)(L - 1) * kW + (long long)K * F + (long long)F * Kp, kT)),
                     blk, 0, c.stream, t, wq, wf, wx, ff, fx);
  FR_HIP(hipGetLastError());
  // forward
  long long N[8];
  for (int l = 0; l < L; l++) N[l] = (long long)B * lo.hout(l) * lo.hout(l);
  hipLaunchKernelGGL(k_train_conv0, dim3(nblk(N[0], 256)), blk, 0, c.stream, B, lo.hin(0), img,
                     wq + lo.w_off[0], wq + lo.b_off[0], ws + w.act[0]);
  FR_HIP(hipGetLastError());
  for (int l = 1; l < L; l++) {
    hipLaunchKernelGGL(k_train_conv, dim3(std::min(kGrid, nblk(N[l], 64))), blk, kWLds, c.stream, B, lo.hin(l),
                       ws + w.act[l - 1], wf + (size_t)(l - 1) * kW, wq + lo.b_off[l],
                       ws + w.act[l]);
    FR_HIP(hipGetLastError());
  }
  const float* X = ws + w.act[L - 1];
  hipLaunchKernelGGL(k_train_fc, dim3(nblk(B, 16), nblk(K, 16)), blk, 0, c.stream, K, B, F, ff,
                     wq + lo.fb_off, X, ws + w.logits);
  FR_HIP(hipGetLastError());
  if (int r = cnn_softmax_xent(c, K, Kp, B, ws + w.logits, label, loss, ws + w.gL)) return r;
  // backward
  hipLaunchKernelGGL(k_train_fc_wgrad, dim3(nblk(F, 256), nblk(K, 16)), blk, 0, c.stream, K, Kp, B,
                     F, t.P, ws + w.gL, X, grad + lo.fw_off, grad + lo.fb_off);
  FR_HIP(hipGetLastError());
  float* gcur = ws + w.gA;
  float* gnext = ws + w.gB;
  hipLaunchKernelGGL(k_train_fc_xgrad, dim3(nblk(B, 16), nblk(F, 64)), blk, 0, c.stream, Kp, B, F,
                     fx, ws + w.gL, X, gcur);
  FR_HIP(hipGetLastError());
  TrainSums ts{};
  long long at = 0;
  for (int l = 0; l < L; l++) {
    ts.w_off[l] = lo.w_off[l];
    ts.b_off[l] = lo.b_off[l];
    ts.first[l + 1] = ts.first[l] + (l ? kW + kC : 10 * kC) / 64;
    ts.part[l] = at;
    const int split = split_count(lo, l, N[l]);
    // whole runs of 32 positions a split
    const long long chunk = ((N[l] + split - 1) / split + 31) / 32 * 32;
    ts.nsplit[l] = (int)((N[l] + chunk - 1) / chunk);
    at += (long long)ts.nsplit[l] * (l ? kW + kC : 10 * kC);
  }
  FR_CHECK(at <= kPartFloats, "weight-gradient split too large");
  for (int l = L - 1; l >= 0; l--) {
    const int chunk = (int)(((N[l] + split_count(lo, l, N[l]) - 1) / split_count(lo, l, N[l]) + 31) /
                            32 * 32);
    float* part = ws + w.part + ts.part[l];
    if (l == 0) {
      hipLaunchKernelGGL(k_train_wgrad0, dim3(ts.nsplit[0]), blk, 0, c.stream, B, lo.hin(0), chunk,
                         gcur, img, part);
      FR_HIP(hipGetLastError());
      break;
    }
    hipLaunchKernelGGL(k_train_wgrad, dim3(ts.nsplit[l], 3), dim3(192), 0, c.stream, B, lo.hin(l),
                       chunk, gcur, ws + w.act[l - 1], part);
    FR_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_train_xgrad, dim3(std::min(kGrid, nblk(N[l], 64))), blk, kWLds, c.stream, B, lo.hin(l),
                       wx + (size_t)(l - 1) * kW, gcur, ws + w.act[l - 1], gnext);
    FR_HIP(hipGetLastError());
    std::swap(gcur, gnext);
  }
  hipLaunchKernelGGL(k_train_sums, dim3(ts.first[L]), blk, 0, c.stream, ts, L, ws + w.part, grad);
  FR_HIP(hipGetLastError());
  return 0;
}

}  // namespace fr
