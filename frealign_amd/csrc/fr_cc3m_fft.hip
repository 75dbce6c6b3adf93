// fr_cc3m_fft.hip -- CC3M (cc3m.f:8-169) and PRESB (presb.f:8-160) on the
// particle's grid, for any box, band and AMAG.
//
// The section lives on the columns I < MAXR2 of the half-plane only, before and
// after the mask, so only those are held (a band of CB columns, a multiple of 8)
// and each step goes over them once:
//   k_band_cols   gathers 8 columns of an item's section times the CTF straight
//                 into LDS and runs their backward column FFT
//   k_band_mean   MASKCOS2's ring mean per item.  The ring sum is linear in the
//                 section: sum of w_I Re X(I, J) Rhat(I, J), Rhat the transform of
//                 the ring's pixels, formed in k_band_cols (AMAG = 1); an item of
//                 another AMAG takes its rows to real space here
//   k_band_rows   row c2r, (x - mean) w, row r2c, in LDS.  The mean's own term is
//                 the DC point, which no shell counts
//   k_band_sums   forward column FFT of 8 columns and their part of the shell sums:
//                 shell s is s^2-s+1 <= r^2 <= s^2+s, a run of J per column, so a
//                 thread takes a shell's points of one sign of J in order
//   k_band_score  the shells of an item, the columns' parts in order
// Sums run in a fixed order: a rerun gives the same bits.
//
// What bounds it: the band goes through memory as write, read, write, read (512
// items of a 320 box at MAXR2 = 80: 105 MB each time), the gather and the FFTs'
// exchanges through LDS; before, whole half-planes went through it twelve times.
// That call: 1,122 us as whole planes, now 304 (columns 94, rows 133, sums 57).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "fr_common.h"
#include "fr_extract.h"
#include "fr_fft_dev.h"
#include "fr_kernels.h"

namespace fr {

namespace bandfft {

struct Band {
  int nsam, nitem, cb, jmax, maxr12, maxr22, nsh;
  float ri2, ri3, rih, halfw;
  int flip;
  int skip;  // items with AMAG = 1 are the band grid's (fr_cc3m.hip): left alone
  __device__ bool left(float amag) const { return skip && amag == 1.0f; }
};

struct BandWork {
  float2* band;
  float4* psum;
  float *part, *mean;
};

struct BandCall {
  const float *a3df, *spec, *ctff;
  const int* pidx;
  const float *dm, *shift, *amag;
};

}  // namespace bandfft

namespace {

using namespace fftdev;
using bandfft::Band;
using bandfft::BandCall;
using bandfft::BandWork;
constexpr int kThr = kFftThreads;
constexpr int kCw = 8;  // columns per workgroup
constexpr float kPi = 3.1415926535897f;

constexpr int rows_nseq(int n) { return n >= 1024 ? 2 : 2048 / n; }

// N > 0: the length is known at compile time; N = 0: passes of a length known at
// run time between two buffers of sequences of pitch n + 1
template <int N>
using Cols = Fft<N ? N : 64, kCw, true>;
template <int N>
using Rows = Fft<N ? N : 64, rows_nseq(N ? N : 64), false>;
template <int N>
using RowsBack = Fft<N ? N : 64, rows_nseq(N ? N : 64), false, true>;

template <int N>
__global__ void __launch_bounds__(kThr)
    k_band_cols(Band b, Plan pl, const float2* __restrict__ a3df, const float* __restrict__ dm,
                const int* __restrict__ pidx, const float2* __restrict__ ctff,
                const float* __restrict__ rhat, const float* __restrict__ amag,
                float2* __restrict__ work, float* __restrict__ part,
                const float2* __restrict__ tw) {
  extern __shared__ float2 smem[];
  __shared__ float red[kThr / 64];
  const int n = N ? N : pl.n, ld = n + 1, jc = n / 2 + 1;
  const size_t ic = (size_t)n * jc;
  using F = Cols<N>;
  auto at = [&](int q, int y) { return N ? F::at(q, y) : q * ld + y; };
  float2* buf = smem;
  // an item's column blocks in XCD-contiguous order: they share lines
  const int nblk = b.cb / kCw, lb = xcd_block(blockIdx.x, gridDim.x);
  const int it = lb / nblk, x0 = (lb - it * nblk) * kCw;
  if (it >= b.nitem || b.left(amag[it])) return;
  for (int e = threadIdx.x; e < kCw * (N ? F::LD : ld); e += kThr) buf[e] = make_float2(0.f, 0.f);
  __syncthreads();
  const float* d = dm + 9 * (size_t)it;
  const float2* cp = ctff + (size_t)pidx[it] * 2 * ic;
  const float scal = 1.0f / (float)n / (float)n;
  const bool inner = ainterpo_inner(jc, d, b.jmax + 1);
  float rsum = 0.f;
#pragma unroll 2
  for (int e = threadIdx.x; e < kCw * (2 * b.jmax + 1); e += kThr) {
    const int i = x0 + (e & (kCw - 1)), j = e / kCw - b.jmax, r2 = i * i + j * j;
    if (r2 < b.maxr12 || r2 >= b.maxr22) continue;
    const size_t id = (size_t)i + (size_t)jc * wrapn(j, n);
    const float2 cr = cp[id], cl = cp[id + ic];
    cf a = inner ? ainterpo_inner_dev(n, jc, a3df, d, i, j) : ainterpo_dev(n, a3df, d, i, j);
    if (b.flip) {  // cc3.f:86-89
      if (cr.x + cl.x < 0.0f) a = cf{-a.re, -a.im};
    } else {
      a = cmul(a, cf{cr.x + cl.x, cr.y - cl.y});
    }
    a = cscale(a, scal);
    buf[at(e & (kCw - 1), wrapn(j, n))] = make_float2(a.re, a.im);
    rsum += (i ? 2.0f : 1.0f) * a.re * rhat[(size_t)abs(j) * b.cb + i];
  }
  for (int off = 32; off > 0; off >>= 1) rsum += __shfl_xor(rsum, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = rsum;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int q = 0; q < kThr / 64; q++) s += red[q];
    part[lb] = s;
  }
  float2* out = work + (size_t)it * n * b.cb + x0;
  if constexpr (N > 0) {
    float2 u[F::IF][F::RF], z[F::IL][F::RL];
    F::template each<F::RF>([&](int k, int q, int y) {
#pragma unroll
      for (int r = 0; r < F::RF; r++) u[k][r] = buf[F::at(q, y + r * F::TF)];
    });
    F::template run<+1, true>(u, z, buf, tw);
    F::template each<F::RL>([&](int k, int q, int y) {
#pragma unroll
      for (int r = 0; r < F::RL; r++) out[(size_t)(y + r * F::TL) * b.cb + q] = z[k][r];
    });
  } else {
    const float2* res = lds_fft(buf, smem + kCw * ld, pl, ld, kCw, +1, tw);
    for (int e = threadIdx.x; e < n * kCw; e += kThr)
      out[(size_t)(e / kCw) * b.cb + (e & (kCw - 1))] = res[(e & (kCw - 1)) * ld + e / kCw];
  }
}

// point k of the sequence of rows 2q and 2q+1 (ra: their CB columns each)
__device__ inline float2 band_pair(const float2* ra, int n, int cb, int k) {
  const int m = 2 * k <= n ? k : n - k;
  float2 a = make_float2(0.f, 0.f), c = a;
  if (m < cb) {
    a = ra[m];
    c = ra[cb + m];
  }
  return pair_point(a, c, k, n);
}

// the row pairs pair0 .. of `work` (npairs in all; beyond: the last again)
// through the c2r: f(q, x, (pixel x of row 2q, of row 2q + 1))
template <int N, typename F>
__device__ inline void band_c2r(float2* smem, const Plan& pl, const float2* work, int pair0,
                                int npairs, int cb, const float2* __restrict__ tw, F f) {
  const int n = N ? N : pl.n, ld = n + 1, nseq = rows_nseq(n);
  if constexpr (N > 0) {
    using T = Rows<N>;
    float2 u[T::IF][T::RF], z[T::IL][T::RL];
    T::template each<T::RF>([&](int k, int q, int x) {
      const float2* ra = work + (size_t)min(pair0 + q, npairs - 1) * 2 * cb;
#pragma unroll
      for (int r = 0; r < T::RF; r++) u[k][r] = band_pair(ra, N, cb, x + r * T::TF);
    });
    T::template run<+1, true>(u, z, smem, tw);
    T::template each<T::RL>([&](int k, int q, int x) {
#pragma unroll
      for (int r = 0; r < T::RL; r++) f(q, x + r * T::TL, z[k][r]);
    });
  } else {
    for (int e = threadIdx.x; e < nseq * n; e += kThr) {
      const int q = e / n, k = e - q * n;
      smem[q * ld + k] = band_pair(work + (size_t)min(pair0 + q, npairs - 1) * 2 * cb, n, cb, k);
    }
    __syncthreads();
    const float2* res = lds_fft(smem, smem + nseq * ld, pl, ld, nseq, +1, tw);
    for (int e = threadIdx.x; e < nseq * n; e += kThr) {
      const int q = e / n, x = e - q * n;
      f(q, x, res[q * ld + x]);
    }
    __syncthreads();
  }
}

// squared wrapped distances of MASKCOS2 (origin 1)
__device__ inline float wrap2(int v, int n) {
  const int d = v < n / 2 ? v : v - n;
  return (float)(d * d);
}

template <int N>
__global__ void __launch_bounds__(kThr)
    k_band_mean(Band b, Plan pl, const float2* __restrict__ work, const float* __restrict__ part,
                int ring_cnt, const float* __restrict__ amag, float* __restrict__ mean,
                const float2* __restrict__ tw) {
  extern __shared__ float2 smem[];
  __shared__ float red[kThr / 64];
  __shared__ int redc[kThr / 64];
  const int n = N ? N : pl.n, it = blockIdx.x, nblk = b.cb / kCw;
  const float am = amag[it];
  if (am == 1.0f) {
    if (threadIdx.x == 0 && !b.skip) {
      float s = 0.f;
      for (int q = 0; q < nblk; q++) s += part[(size_t)it * nblk + q];
      mean[it] = ring_cnt ? s / (float)ring_cnt : s;
    }
    return;
  }
  const float ri2p = b.ri2 / am / am, ri3p = b.ri3 / am / am;
  const int nseq = rows_nseq(n), end = (it + 1) * (n / 2);
  float s = 0.f;
  int cnt = 0;
  for (int p0 = it * (n / 2); p0 < end; p0 += nseq)
    band_c2r<N>(smem, pl, work, p0, end, b.cb, tw, [&](int q, int x, float2 z) {
      if (p0 + q >= end) return;
      const int row = 2 * (p0 + q - it * (n / 2));
      const float ra = wrap2(x, n) + wrap2(row, n), rc = wrap2(x, n) + wrap2(row + 1, n);
      if (ra > ri2p && ra <= ri3p) s += z.x, cnt++;
      if (rc > ri2p && rc <= ri3p) s += z.y, cnt++;
    });
  for (int off = 32; off > 0; off >>= 1) {
    s += __shfl_xor(s, off, 64);
    cnt += __shfl_xor(cnt, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = s;
    redc[threadIdx.x >> 6] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    s = 0.f;
    cnt = 0;
    for (int q = 0; q < kThr / 64; q++) s += red[q], cnt += redc[q];
    mean[it] = cnt ? s / (float)cnt : s;
  }
}

template <int N>
__global__ void __launch_bounds__(kThr)
    k_band_rows(Band b, Plan pl, float2* __restrict__ work, const float* __restrict__ amag,
                const float* __restrict__ mean, const float2* __restrict__ tw) {
  extern __shared__ float2 smem[];
  const int n = N ? N : pl.n, ld = n + 1, nh = n / 2, nseq = rows_nseq(n);
  const int pair0 = blockIdx.x * nseq, npairs = b.nitem * nh;
  if (b.skip) {  // rows of items that are left alone only
    const int last = min(pair0 + nseq, npairs) - 1;
    bool any = false;
    for (int it = pair0 / nh; it <= last / nh; it++) any |= !b.left(amag[it]);
    if (!any) return;
  }
  // (z - mean) weight of pixel x of both rows of pair pr
  auto masked = [&](int pr, int x, float2 z) {
    const int it = pr / nh, row = 2 * (pr - it * nh);
    const float am = amag[it], mu = mean[it];
    const float ri2p = b.ri2 / am / am, ri3p = b.ri3 / am / am, rihp = b.rih / am;
    auto weight = [&](float r2) {
      if (r2 > ri3p) return 0.0f;
      if (r2 > ri2p) return (1.0f + cosf(kPi * (sqrtf(r2) - rihp) / b.halfw)) / 2.0f;
      return 1.0f;
    };
    const float dx = wrap2(x, n);
    return make_float2((z.x - mu) * weight(dx + wrap2(row, n)),
                       (z.y - mu) * weight(dx + wrap2(row + 1, n)));
  };
  const float2* out;
  if constexpr (N > 0) {
    // a thread masks the pixels its last pass leaves it and starts the transform
    // back with them
    using F = Rows<N>;
    using G = RowsBack<N>;
    static_assert(G::RF == F::RL && G::IF == F::IL, "the passes do not meet");
    float2 u[F::IF][F::RF], z[F::IL][F::RL], o[G::IL][G::RL];
    F::template each<F::RF>([&](int k, int q, int x) {
      const float2* ra = work + (size_t)min(pair0 + q, npairs - 1) * 2 * b.cb;
#pragma unroll
      for (int r = 0; r < F::RF; r++) u[k][r] = band_pair(ra, N, b.cb, x + r * F::TF);
    });
    F::template run<+1, false>(u, z, smem, tw);
    F::template each<F::RL>([&](int k, int q, int x) {
      const int pr = min(pair0 + q, npairs - 1);
#pragma unroll
      for (int r = 0; r < F::RL; r++) z[k][r] = masked(pr, x + r * F::TL, z[k][r]);
    });
    G::template run<-1, true>(z, o, smem, tw);
    __syncthreads();
    G::template each<G::RL>([&](int k, int q, int x) {
#pragma unroll
      for (int r = 0; r < G::RL; r++) {
        const int y = x + r * G::TL;
        if (y < b.cb || N - y < b.cb) smem[G::at(q, y)] = o[k][r];
      }
    });
    __syncthreads();
    out = smem;
  } else {
    float2* tmp = smem + nseq * ld;
    for (int e = threadIdx.x; e < nseq * n; e += kThr) {
      const int q = e / n, k = e - q * n;
      smem[q * ld + k] = band_pair(work + (size_t)min(pair0 + q, npairs - 1) * 2 * b.cb, n, b.cb, k);
    }
    __syncthreads();
    float2* res = lds_fft(smem, tmp, pl, ld, nseq, +1, tw);
    for (int e = threadIdx.x; e < nseq * n; e += kThr) {
      const int q = e / n, x = e - q * n;
      res[q * ld + x] = masked(min(pair0 + q, npairs - 1), x, res[q * ld + x]);
    }
    __syncthreads();
    out = lds_fft(res, res == smem ? tmp : smem, pl, ld, nseq, -1, tw);
  }
  for (int e = threadIdx.x; e < nseq * b.cb; e += kThr) {
    const int q = e / b.cb, k = e - q * b.cb;
    if (pair0 + q >= npairs) continue;
    auto at = [&](int x) { return N ? RowsBack<N>::at(q, x) : q * ld + x; };
    float2* ra = work + (size_t)(pair0 + q) * 2 * b.cb + k;
    split_pair(out[at(k)], out[at(k ? n - k : 0)], ra[0], ra[b.cb]);
  }
}

template <int N>
__global__ void __launch_bounds__(kThr)
    k_band_sums(Band b, Plan pl, const float2* __restrict__ work, const float2* __restrict__ spec,
                const int* __restrict__ pidx, const float* __restrict__ shift,
                const float* __restrict__ amag, float4* __restrict__ psum,
                const float2* __restrict__ tw) {
  extern __shared__ float2 smem[];
  using F = Cols<N>;
  const int n = N ? N : pl.n, ld = n + 1, jc = n / 2 + 1;
  // the transform's buffers, then per point of the band the masked section and
  // (REAL(SAMP CONJG(AINPO)), |SAMP|^2): after it (N > 0) or in it
  const int ldj = 2 * b.jmax + 1;
  float2* ey = smem + (N ? max(kCw * F::LD, 2 * kCw * ldj) : 2 * kCw * ld);  // e^{i SHY J}
  __shared__ float2 ex[kCw];
  const int nblk = b.cb / kCw, lb = xcd_block(blockIdx.x, gridDim.x);
  const int it = lb / nblk, x0 = (lb - it * nblk) * kCw;
  if (it >= b.nitem || b.left(amag[it])) return;
  const float2* in = work + (size_t)it * n * b.cb + x0;
  const float shx = shift[2 * it], shy = shift[2 * it + 1];
  for (int j = threadIdx.x; j <= b.jmax; j += kThr) {
    float sn, cs;
    sincosf(shy * (float)j, &sn, &cs);
    ey[j] = make_float2(cs, sn);
  }
  if (threadIdx.x < kCw) {
    float sn, cs;
    sincosf(shx * (float)(x0 + (int)threadIdx.x), &sn, &cs);
    ex[threadIdx.x] = make_float2(cs, sn);
  }
  const float2* sp = spec + (size_t)pidx[it] * n * jc;
  auto point = [&](int c, int j, float2 a) {
    const int i = x0 + c, r2 = i * i + j * j;
    if (r2 < b.maxr12 || r2 >= b.maxr22) return make_float2(0.f, 0.f);
    const float2 s = sp[(size_t)i + (size_t)jc * wrapn(j, n)];
    const float2 u = ex[c], v = ey[abs(j)];
    const float vs = j < 0 ? -v.y : v.y;
    const float cs = u.x * v.x - u.y * vs, sn = u.x * vs + u.y * v.x;
    const float re = s.x * a.x + s.y * a.y, im = s.y * a.x - s.x * a.y;
    return make_float2(re * cs - im * sn, s.x * s.x + s.y * s.y);
  };
  float2 *res, *pt;
  auto pos = [&](int c, int j) { return N ? c * ldj + j + b.jmax : c * ld + (j < 0 ? n + j : j); };
  if constexpr (N > 0) {
    float2 u[F::IF][F::RF], z[F::IL][F::RL];
    F::template each<F::RF>([&](int k, int c, int y) {
#pragma unroll
      for (int r = 0; r < F::RF; r++) u[k][r] = in[(size_t)(y + r * F::TF) * b.cb + c];
    });
    F::template run<-1, false>(u, z, smem, tw);
    __syncthreads();
    res = smem;
    pt = smem + kCw * ldj;
    F::template each<F::RL>([&](int k, int c, int y) {
#pragma unroll
      for (int r = 0; r < F::RL; r++) {
        const int row = y + r * F::TL, j = 2 * row <= N ? row : row - N;
        if (abs(j) > b.jmax) continue;
        res[pos(c, j)] = z[k][r];
        pt[pos(c, j)] = point(c, j, z[k][r]);
      }
    });
  } else {
    for (int e = threadIdx.x; e < n * kCw; e += kThr)
      smem[(e & (kCw - 1)) * ld + e / kCw] = in[(size_t)(e / kCw) * b.cb + (e & (kCw - 1))];
    __syncthreads();
    res = lds_fft(smem, smem + kCw * ld, pl, ld, kCw, -1, tw);
    pt = res == smem ? smem + kCw * ld : smem;
    for (int e = threadIdx.x; e < kCw * ldj; e += kThr) {
      const int c = e & (kCw - 1), j = e / kCw - b.jmax;
      pt[pos(c, j)] = point(c, j, res[pos(c, j)]);
    }
  }
  __syncthreads();
  for (int base = 0; base < 2 * b.nsh; base += kThr) {
    const int e = base + threadIdx.x, s = e >> 1, neg = e & 1;
    float q = 0.f, s2 = 0.f, a2 = 0.f, cnt = 0.f;
    if (s < b.nsh) {
      for (int c = 0; c < kCw; c++) {
        const int i = x0 + c;
        const int hi = min(s * s + s, b.maxr22 - 1) - i * i;
        if (hi < 0) break;
        const int lo = max(s ? s * s - s + 1 : 0, b.maxr12) - i * i;
        const int j1 = isqrt(hi);
        int j0 = lo > 0 ? isqrt(lo - 1) + 1 : 0;
        if (neg) j0 = max(j0, 1);
        for (int j = j0; j <= j1; j++) {
          const int at = pos(c, neg ? -j : j);
          const float2 p = pt[at], a = res[at];
          q += p.x;
          s2 += p.y;
          a2 += a.x * a.x + a.y * a.y;
          cnt += 1.0f;
        }
      }
    }
    q += __shfl_xor(q, 1, 64);
    s2 += __shfl_xor(s2, 1, 64);
    a2 += __shfl_xor(a2, 1, 64);
    cnt += __shfl_xor(cnt, 1, 64);
    if (s < b.nsh && !neg) psum[(size_t)lb * b.nsh + s] = make_float4(q, s2, a2, cnt);
  }
}

#ifndef FR_LEN
__device__ inline float4 shell(const float4* psum, const Band& b, int it, int s) {
  const int nblk = b.cb / kCw;
  float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = 0; k < nblk; k++) {
    const float4 p = psum[((size_t)it * nblk + k) * b.nsh + s];
    t.x += p.x;
    t.y += p.y;
    t.z += p.z;
    t.w += p.w;
  }
  return t;
}

// cc3m.f:139-167 over shells 1 .. NSAM/2-1: one wave per item, FP64 sums reduced
// by a fixed butterfly
__global__ void __launch_bounds__(64)
    k_band_score(Band b, float rbfact, const float4* __restrict__ psum,
                 const float* __restrict__ fsct, const float* __restrict__ amag,
                 float* __restrict__ score) {
  const int it = blockIdx.x, lane = threadIdx.x;
  if (b.left(amag[it])) return;
  double s1 = 0.0, s2 = 0.0, s3 = 0.0;
  for (int s = 1 + lane; s < min(b.nsam / 2, b.nsh); s += 64) {
    const float4 t = shell(psum, b, it, s);
    if (t.w == 0.0f) continue;
    float r = t.x / sqrtf(t.z);
    if (!b.flip && fsct[s] < 0.95f) r = fabsf(r);
    const float wgt = expf(-rbfact * (float)(s * s));
    s3 += (double)(r * wgt);
    s2 += (double)(wgt * wgt * t.y);
    s1 += 1.0;
  }
  for (int off = 32; off > 0; off >>= 1) {
    s1 += __shfl_xor(s1, off, 64);
    s2 += __shfl_xor(s2, off, 64);
    s3 += __shfl_xor(s3, off, 64);
  }
  if (lane == 0) {
    if (s1 * s2 != 0.0) s3 = s3 / sqrt(s1 * s2);
    score[it] = (float)s3;
  }
}

// presb.f:95-123: per-shell correlation; shells with no point leave RBIN untouched
__global__ void __launch_bounds__(64)
    k_band_presb(Band b, const float4* __restrict__ psum, float* __restrict__ rbin) {
  const int it = blockIdx.x;
  float* rb = rbin + (size_t)it * b.nsam;
  for (int s = threadIdx.x; s < min(b.nsam / 2, b.nsh); s += 64) {
    const float4 t = shell(psum, b, it, s);
    if (t.w == 0.0f) continue;
    rb[2 * s] = t.x / sqrtf(t.y * t.z);
    rb[2 * s + 1] = 1.0f;
  }
}

// The ring's sums on the device: on the host they were 2 ms of the first PRESB of a
// 256 box
__device__ inline double ring_mult(int v, int n) { return v == 0 || 2 * v == n ? 1.0 : 2.0; }

__global__ void __launch_bounds__(kThr)
    k_ring_rows(int n, int cb, float ri2, float ri3, double* __restrict__ row) {
  const int y = blockIdx.x;
  for (int i = threadIdx.x; i < cb; i += kThr) {
    double s = 0.0;
    for (int x = 0; 2 * x <= n; x++) {
      const float r2 = (float)(x * x + y * y);
      if (r2 > ri2 && r2 <= ri3) s += ring_mult(x, n) * cospi(2.0 * (i * x % n) / n);
    }
    row[(size_t)y * cb + i] = ring_mult(y, n) * s;
  }
}

__global__ void __launch_bounds__(kThr)
    k_ring_hat(int n, int cb, const double* __restrict__ row, float* __restrict__ out) {
  __shared__ double co[kCc3mMaxBox / 2 + 1];
  const int j = blockIdx.x;
  for (int y = threadIdx.x; 2 * y <= n; y += kThr) co[y] = cospi(2.0 * (j * y % n) / n);
  __syncthreads();
  for (int i = threadIdx.x; i < cb; i += kThr) {
    double s = 0.0;
    for (int y = 0; 2 * y <= n; y++) s += co[y] * row[(size_t)y * cb + i];
    out[(size_t)j * cb + i] = (float)s;
  }
}

int band_cb(int maxr2) { return (maxr2 + kCw - 1) / kCw * kCw; }
int band_nsh(int maxr2) { return maxr2 + 1; }

size_t align16(size_t b) { return (b + 15) & ~(size_t)15; }

BandWork band_work(void* base, int nsam, int maxr2, size_t n, size_t* bytes) {
  const size_t cb = band_cb(maxr2), nblk = cb / kCw;
  char* p = static_cast<char*>(base);
  size_t o = 0;
  BandWork w;
  auto take = [&](auto*& q, size_t k) {
    q = reinterpret_cast<std::remove_reference_t<decltype(q)>>(p + o);
    o += align16(sizeof(*q) * k);
  };
  take(w.band, n * nsam * cb);
  take(w.psum, n * nblk * band_nsh(maxr2));
  take(w.part, n * nblk);
  take(w.mean, n);
  *bytes = o;
  return w;
}
#endif  // FR_LEN

}  // namespace

template <int N>
int launch_band_n(Ctx& c, const Band& b, const BandCall& p, const Cc3mRing& ring,
                  const BandWork& w) {
  Plan pl;
  FR_CHECK(make_plan(b.nsam, &pl), "FFT length %d not supported", b.nsam);
  const float2* tw = c.twiddles(b.nsam);
  FR_CHECK(tw != nullptr, "twiddle table allocation failed");
  const int n = b.nsam, nseq = rows_nseq(n);
  const int cols = round8(b.nitem * (b.cb / kCw)), npairs = b.nitem * (n / 2);
  const size_t lc = N ? Cols<N>::kLds : sizeof(float2) * 2 * kCw * (n + 1);
  const size_t lr = N ? Rows<N>::kLds : sizeof(float2) * 2 * nseq * (n + 1);
  const size_t ls = sizeof(float2) * (b.jmax + 1) +
                    (N ? std::max(lc, sizeof(float2) * 2 * kCw * (2 * b.jmax + 1)) : lc);
  auto big = [](const void* fn, size_t lds) {
    return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  };
  FR_HIP(big((const void*)k_band_cols<N>, lc));
  FR_HIP(big((const void*)k_band_mean<N>, lr));
  FR_HIP(big((const void*)k_band_rows<N>, lr));
  FR_HIP(big((const void*)k_band_sums<N>, ls));
  hipLaunchKernelGGL(k_band_cols<N>, dim3(cols), dim3(kThr), lc, c.stream, b, pl,
                     reinterpret_cast<const float2*>(p.a3df), p.dm, p.pidx,
                     reinterpret_cast<const float2*>(p.ctff), ring.rhat, p.amag, w.band, w.part,
                     tw);
  FR_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_band_mean<N>, dim3(b.nitem), dim3(kThr), lr, c.stream, b, pl, w.band,
                     w.part, ring.cnt, p.amag, w.mean, tw);
  FR_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_band_rows<N>, dim3((npairs + nseq - 1) / nseq), dim3(kThr), lr, c.stream, b,
                     pl, w.band, p.amag, w.mean, tw);
  FR_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_band_sums<N>, dim3(cols), dim3(kThr), ls, c.stream, b, pl, w.band,
                     reinterpret_cast<const float2*>(p.spec), p.pidx, p.shift, p.amag, w.psum,
                     tw);
  FR_HIP(hipGetLastError());
  return 0;
}

#ifdef FR_LEN
template int launch_band_n<FR_LEN>(Ctx&, const Band&, const BandCall&, const Cc3mRing&,
                                   const BandWork&);
#else
#define FR_EXTERN(N)                                                                        \
  extern template int launch_band_n<N>(Ctx&, const Band&, const BandCall&, const Cc3mRing&, \
                                       const BandWork&);
FR_LENGTHS(FR_EXTERN)

namespace {

int launch_band(Ctx& c, const Band& b, const BandCall& p, const Cc3mRing& ring, const BandWork& w) {
  return with_length(b.nsam, [&](auto len) { return launch_band_n<len()>(c, b, p, ring, w); });
}

Band make_band(int nsam, int n, int maxr12, int maxr2, float ri2, float ri3, float rih,
               float halfw, int flip, int skip) {
  int jmax = maxr2 - 1;
  return Band{nsam, n,   band_cb(maxr2), jmax, maxr12, maxr2 * maxr2, band_nsh(maxr2),
              ri2,  ri3, rih,            halfw, flip,   skip};
}

}  // namespace

size_t cc3m_fft_bytes(int nsam, int maxr2, size_t n) {
  size_t bytes = 0;
  (void)band_work(nullptr, nsam, maxr2, n, &bytes);
  return bytes;
}

// Pixels of the MASKCOS2 ring at AMAG = 1, as the kernels test them.
int cc3m_ring_count(int nsam, float ri2, float ri3) {
  const int h = nsam / 2;
  auto mult = [&](int v) { return v == 0 || v == h ? 1 : 2; };
  int cnt = 0;
  for (int y = 0; y <= h; y++)
    for (int x = 0; x <= h; x++) {
      const float r2 = (float)(x * x + y * y);
      if (r2 > ri2 && r2 <= ri3) cnt += mult(x) * mult(y);
    }
  return cnt;
}

size_t cc3m_ring_bytes(int nsam, int maxr2) {
  return band_cb(maxr2) * (sizeof(double) * (nsam / 2 + 1) + sizeof(float) * (size_t)maxr2);
}

// Rhat[J][I] = sum over the ring's pixels (x, y) of cos(2 pi I x/N) cos(2 pi J y/N),
// J < MAXR2, I < CB, in 64 bits; in front of it, for the launch alone, the rows' sums
// over x.
int launch_ring_hat(Ctx& c, int nsam, float ri2, float ri3, int maxr2, void* buf,
                    const float** rhat) {
  const int h = nsam / 2, cb = band_cb(maxr2);
  double* row = static_cast<double*>(buf);
  float* out = reinterpret_cast<float*>(row + (size_t)(h + 1) * cb);
  hipLaunchKernelGGL(k_ring_rows, dim3(h + 1), dim3(kThr), 0, c.stream, nsam, cb, ri2, ri3, row);
  FR_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_ring_hat, dim3(maxr2), dim3(kThr), 0, c.stream, nsam, cb, row, out);
  FR_HIP(hipGetLastError());
  *rhat = out;
  return 0;
}

int launch_cc3m(Ctx& c, const Cc3mArgs& a, const float* a3df, const float* spec, const float* ctff,
                const int* pidx, const float* dm, const float* shift, const float* amag,
                const float* fsct, const Cc3mRing& ring, void* work, float* score,
                bool skip_unit) {
  if (a.n <= 0) return 0;
  FR_CHECK(a.nsam <= kCc3mMaxBox, "box too large for CC3M bins");
  FR_CHECK(a.maxr2 < a.nsam / 2, "CC3M needs MAXR2 < NSAM/2 (got %d)", a.maxr2);
  FR_CHECK(ring.rhat && work, "CC3M tables missing");
  const Band b = make_band(a.nsam, a.n, a.maxr1 * a.maxr1, a.maxr2, a.ri2, a.ri3, a.rih, a.halfw,
                           a.cc3, skip_unit);
  size_t bytes;
  const BandWork w = band_work(work, a.nsam, a.maxr2, a.n, &bytes);
  if (int r = launch_band(c, b, BandCall{a3df, spec, ctff, pidx, dm, shift, amag}, ring, w))
    return r;
  hipLaunchKernelGGL(k_band_score, dim3(a.n), dim3(64), 0, c.stream, b, a.rbfact, w.psum, fsct,
                     amag, score);
  FR_HIP(hipGetLastError());
  return 0;
}

// PRESB for a batch: the CC3M steps over 1 <= r^2 < (NSAM/2)^2
int launch_presb(Ctx& c, int nsam, int n, const float* a3df, const float* spec, const float* ctff,
                 const int* pidx, const float* dm, const float* shift, const float* amag,
                 float ri2, float ri3, float rih, float halfw, const Cc3mRing& ring, void* work,
                 float* rbin) {
  if (n <= 0) return 0;
  FR_CHECK(nsam <= kCc3mMaxBox, "box too large for PRESB bins");
  FR_CHECK(ring.rhat && work, "PRESB tables missing");
  const Band b = make_band(nsam, n, 1, nsam / 2, ri2, ri3, rih, halfw, 0, 0);
  size_t bytes;
  const BandWork w = band_work(work, nsam, nsam / 2, n, &bytes);
  if (int r = launch_band(c, b, BandCall{a3df, spec, ctff, pidx, dm, shift, amag}, ring, w))
    return r;
  hipLaunchKernelGGL(k_band_presb, dim3(n), dim3(64), 0, c.stream, b, w.psum, rbin);
  FR_HIP(hipGetLastError());
  return 0;
}

#endif  // FR_LEN

}  // namespace fr
