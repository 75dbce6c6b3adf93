// fr_search_f32.hip -- the exhaustive FP32 orientation x translation search with
// separable translations.
//
// With X'_p the particle's terms (CTF and c2r weights folded in, as in
// fr_search.hip) and Y = X'_p conj(T_o), the score map of ccp.f:194-252 is
//   cc(sx, sy) = Re sum_I e^{i I phi(sx)} Z(I, sy),
//   Z(I, sy)   = sum_J Y(I, J) e^{i J phi(sy)}
//              = sum_{J >= 0} [Y(I, J) + Y(I, -J)] cos J phi(sy)
//                         + i [Y(I, J) - Y(I, -J)] sin J phi(sy),
// phi(s) = 2 pi (s - 7) / NSAMR.  Both sums are FP32 matrix products: 32 I by 32
// J by 15 sy (the sums and differences halve the J), then 15 sx by 32 I by 15 sy,
// whose operand is what the first left in each lane's accumulators.  At
// MAXR2 = 32 a (particle, template) pair takes 76 16x16x4 products; the plain
// product of its 225 shift rows with the band took 1.5 MFLOP, ten times as much.
// All operands, sums and tables are FP32.
//
// A workgroup's four waves take four particles against the same templates.  The
// templates, bank rows over the annulus in order, go through LDS once for all
// four, to where the lane that consumes a point reads it (two buffers: the next
// template is written while this one is used); the particle's terms stay in
// registers.  Sum |c T|^2 for the normalisation accumulates beside the products.
//
// CCP takes the first maximum of the map's inner 13 x 13 and then a 3 x 3 box
// about it, so where two cells tie to a rounding the order of the sums decides, and
// the two boxes may differ by a percent.  A pair whose second cell lies within kTie
// of its first is therefore noted and its peak taken from the 225-row product
// (k_search_gemm_ties), by which list searches decide: the same pair has the same
// peak in both.  kTie: a cell is at most 2 x 1,640 products summed in FP32, each
// step rounded to 2^-24 of at most sqrt(sum |c T|^2 sum |X|^2); as a random walk
// sqrt(3280) 2^-24, times 4: 2^-16 of that root.  Two orders of the sums differ by
// up to 4.0e-6 of it over 50,400 pairs at MAXR2 = 32, a quarter; 0.3% of them tie.
//
// What bounds it: the matrix cores (76 x 32 cycles a pair) with about 430 vector
// instructions a pair beside them.  64 particles x 46,800 templates at MAXR2 = 32:
// 7.4 ms (0.3 of it the ties), 40.5 ms as the 225-row product with its separate norms.
#include <hip/hip_runtime.h>

#include "fr_common.h"
#include "fr_search.h"
#include "fr_search_dev.h"

namespace fr {

namespace {

constexpr int kThr = 256;
constexpr float kTie = 0x1p-16f;

template <int R>
struct Shape32 {
  static constexpr int kNT = (R + 15) / 16;  // row blocks of 16 I
  static constexpr int kKS = R / 4;          // steps of 4 |J|
  static constexpr int kPer = (R * (2 * R - 1) + kThr - 1) / kThr;  // bank values per thread
  // does the block hold a point with r < R
  static constexpr bool used(int t, int ks) { return 256 * t * t + 16 * ks * ks < R * R; }
};

template <int R>
__global__ void __launch_bounds__(kThr, 2)
    k_search_sep32(int np, int norient, int kc, int pitch, int nsamr, int ntile, int tile,
                   const int2* __restrict__ kidx, const float2* __restrict__ bank,
                   const float2* __restrict__ ap, const float* __restrict__ c2,
                   const float* __restrict__ sum2, float* __restrict__ score,
                   int* __restrict__ best_row, int* __restrict__ ntie, int* __restrict__ ties) {
  using S = Shape32<R>;
  constexpr int kNT = S::kNT, kKS = S::kKS, kPer = S::kPer, kF = kNT * kKS;
  // [buffer][block][lane]: (+J, -J) of the lane's point
  __shared__ float4 tpl[2][kF * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, g = lane >> 4;
  // blocks are dealt round-robin to the 8 XCDs; each XCD walks its own template
  // tiles with the particle quads innermost
  const int npq = (np + 3) / 4, xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int tl = (j / npq) * 8 + xcd;
  if (tl >= ntile) return;
  const int p0 = (j % npq) * 4, p = p0 + wave;
  const int lo = tl * tile, hi = min(norient, lo + tile);

  // where this thread's annulus points go in a buffer (in float2)
  int at[kPer];
#pragma unroll
  for (int r = 0; r < kPer; r++) {
    const int k = tid + r * kThr;
    at[r] = -1;
    if (k < kc) {
      const int2 ij = kidx[k];
      const int a = abs(ij.y);
      at[r] = (((ij.x >> 4) * kKS + (a >> 2)) * 64 + (a & 3) * 16 + (ij.x & 15)) * 2 + (ij.y < 0);
    }
  }
  for (int e = tid; e < 2 * kF * 64; e += kThr) (&tpl[0][0])[e] = make_float4(0.f, 0.f, 0.f, 0.f);
  // phase tables: J = 4 ks + g against sy = n, and sx = n against I = 16 t + 4 g + i
  float cy[kKS], sy[kKS], cx[kNT][4], sx[kNT][4];
#pragma unroll
  for (int ks = 0; ks < kKS; ks++) {
    cy[ks] = sy[ks] = 0.f;
    if (n < 15) phase((4 * ks + g) * (n - 7), nsamr, cy[ks], sy[ks]);
  }
#pragma unroll
  for (int t = 0; t < kNT; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      cx[t][i] = sx[t][i] = 0.f;
      if (n < 15) phase((16 * t + 4 * g + i) * (n - 7), nsamr, cx[t][i], sx[t][i]);
    }
  // the four particles' terms, through the first buffer into their waves' registers
  float4 x[kF];
  float2 cc[kF];
  for (int w = 0; w < 4; w++)
    for (int pass = 0; pass < 2; pass++) {
      __syncthreads();
      if (p0 + w < np) {
        const size_t row = (size_t)(p0 + w) * pitch;
#pragma unroll
        for (int r = 0; r < kPer; r++)
          if (at[r] >= 0)
            reinterpret_cast<float2*>(&tpl[0][0])[at[r]] =
                pass ? make_float2(c2[row + tid + r * kThr], 0.f) : ap[row + tid + r * kThr];
      }
      __syncthreads();
      if (wave == w) {
#pragma unroll
        for (int f = 0; f < kF; f++) {
          const float4 v = tpl[0][f * 64 + lane];
          if (pass) cc[f] = make_float2(v.x, v.z);
          else x[f] = v;
        }
      }
    }
  const float s2 = p < np ? sum2[p] : 0.f;
  float box_l = 0.f, norm_l = 0.f;  // lane k: pair k of the wave's last 64
  int row_l = 0;
  float2 pre[kPer];
  auto fetch = [&](int o) {
    const float2* row = bank + (size_t)o * pitch + tid;
#pragma unroll
    for (int r = 0; r < kPer; r++)
      if (at[r] >= 0) pre[r] = row[r * kThr];
  };
  auto put = [&](int b) {
#pragma unroll
    for (int r = 0; r < kPer; r++)
      if (at[r] >= 0) reinterpret_cast<float2*>(&tpl[b][0])[at[r]] = pre[r];
  };
  fetch(lo);
  __syncthreads();
  put(0);
  if (lo + 1 < hi) fetch(lo + 1);
  __syncthreads();
  for (int o = lo; o < hi; o++) {
    const int cur = (o - lo) & 1;
    if (o + 1 < hi) put(cur ^ 1);
    if (o + 2 < hi) fetch(o + 2);
    if (p < np) {
      floatx4 zr[kNT], zi[kNT];
#pragma unroll
      for (int t = 0; t < kNT; t++) zr[t] = zi[t] = floatx4{0.f, 0.f, 0.f, 0.f};
      float nacc = 0.f;
#pragma unroll
      for (int ks = 0; ks < kKS; ks++)
#pragma unroll
        for (int t = 0; t < kNT; t++) {
          if (!S::used(t, ks)) continue;
          const int f = t * kKS + ks;
          const float4 v = tpl[cur][f * 64 + lane];
          const float ur = x[f].x * v.x + x[f].y * v.y, ui = x[f].y * v.x - x[f].x * v.y;
          const float dr = x[f].z * v.z + x[f].w * v.w, di = x[f].w * v.z - x[f].z * v.w;
          nacc = fmaf(cc[f].x, v.x * v.x + v.y * v.y, nacc);
          nacc = fmaf(cc[f].y, v.z * v.z + v.w * v.w, nacc);
          zr[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ur + dr, cy[ks], zr[t], 0, 0, 0);
          zi[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ui + di, cy[ks], zi[t], 0, 0, 0);
          zr[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(di - ui, sy[ks], zr[t], 0, 0, 0);
          zi[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ur - dr, sy[ks], zi[t], 0, 0, 0);
        }
      nacc = wave_sum(nacc);
      floatx4 m[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int t = 0; t < kNT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          m[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(cx[t][i], zr[t][i], m[0], 0, 0, 0);
          m[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[t][i], zi[t][i], m[1], 0, 0, 0);
        }
      floatx4 map;
#pragma unroll
      for (int i = 0; i < 4; i++) map[i] = m[0][i] - m[1][i];
      float box, top;
      int row;
      ccp_peak(map, g, n, box, row, top);
      // cells at the top; none where the map has no ordered value
      const float tied = top - kTie * sqrtf(nacc * s2);
      int near = 0;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int sx = 4 * g + i;
        const bool in = sx >= 1 && sx <= 13 && n >= 1 && n <= 13;
        near += __popcll(__ballot(in && map[i] >= tied));
      }
      if (near != 1 && nacc > 0.f && s2 > 0.f && lane == 0)
        ties[(size_t)p * norient + atomicAdd(&ntie[p], 1)] = o;
      const int slot = (o - lo) & 63;
      if (lane == slot) {
        box_l = box;
        norm_l = nacc;
        row_l = row;
      }
      if (slot == 63 || o + 1 == hi) {
        if (lane <= slot) {
          const size_t e = (size_t)p * norient + o - slot + lane;
          score[e] = ccp_score(box_l, norm_l, s2);
          best_row[e] = row_l;
        }
      }
    }
    __syncthreads();
  }
}

__global__ void k_no_ties(int np, int* ntie) {
  const int p = blockIdx.x * kThr + threadIdx.x;
  if (p < np) ntie[p] = 0;
}

template <int R>
int launch_r(Ctx& c, int np, int norient, int kc, int pitch, int nsamr, const int* kidx,
             const void* bank, const float* ap, const float* c2, const float* sum2, float* score,
             int* best_row, int* ntie, int* ties) {
  if (c.cus <= 0) {
    hipDeviceProp_t prop;
    FR_HIP(hipGetDeviceProperties(&prop, c.device));
    c.cus = prop.multiProcessorCount;
  }
  // 256 templates per workgroup, which hides its set-up; fewer where that would
  // leave less than four workgroups per place on the device
  const int npq = (np + 3) / 4;
  int tile = 256;
  while (tile > 32 && (long long)((norient + tile - 1) / tile) * npq < 8ll * c.cus) tile /= 2;
  const int ntile = (norient + tile - 1) / tile;
  const size_t nblk = (size_t)((ntile + 7) / 8 * 8) * npq;
  FR_CHECK(nblk < (1u << 31), "search grid too large");
  hipLaunchKernelGGL(k_no_ties, dim3((np + kThr - 1) / kThr), dim3(kThr), 0, c.stream, np, ntie);
  FR_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_search_sep32<R>, dim3((unsigned)nblk), dim3(kThr), 0, c.stream, np, norient,
                     kc, pitch, nsamr, ntile, tile, reinterpret_cast<const int2*>(kidx),
                     reinterpret_cast<const float2*>(bank), reinterpret_cast<const float2*>(ap),
                     c2, sum2, score, best_row, ntie, ties);
  FR_HIP(hipGetLastError());
  return 0;
}

}  // namespace

int launch_search_sep32(Ctx& c, int np, int norient, int maxr2, int kc, int kpad, int nsamr,
                        const int* kidx, const void* bank, const float* ap, const float* c2,
                        const float* sum2, float* score, int* best_row, int* ntie, int* ties) {
  if (np <= 0 || norient <= 0) return 0;
  FR_CHECK(maxr2 <= kSepMaxR2, "the separable search holds MAXR2 <= %d (got %d)", kSepMaxR2, maxr2);
  auto go = [&](auto fn) {
    return fn(c, np, norient, kc, kpad / 2, nsamr, kidx, bank, ap, c2, sum2, score, best_row, ntie,
              ties);
  };
  if (maxr2 <= 16) return go(launch_r<16>);
  if (maxr2 <= 24) return go(launch_r<24>);
  return go(launch_r<32>);
}

}  // namespace fr
