// fr_fft.hip -- batched 2D real FFTs for the particle and projection planes.
//
// Replaces the FFTW 3.3 plans of fftw_plans.f:12-13 (fftwf_plan_dft_r2c_2d /
// fftwf_plan_dft_c2r_2d, in place, unnormalised) for the box sizes the hot
// path uses: N = 2^a 3^b 5^c, N <= 1024 (64, 96, 128, 160, 256 and the 4x
// padded 1024 of pad.f).
//
// Structure: row pass (two real rows packed into one complex sequence),
// column pass over the JC half-plane columns, both as Stockham autosort FFTs
// with an accurate twiddle table (W_N^k computed on the host in FP64): in
// registers with exchanges through LDS where the length is compiled in, with
// radix-4/2/3/5 butterflies in LDS where it is not.
#include <hip/hip_runtime.h>

#include <vector>

#include "fr_common.h"
#include "fr_fft_dev.h"

namespace fr {

namespace {

using namespace fftdev;
constexpr int kThreads = kFftThreads;
#ifndef FR_LEN
// ---- row pass, forward: rows (2q, 2q+1) -> z = a + i b -> FFT -> unpack to half spectra
__global__ void __launch_bounds__(kThreads) k_rows_r2c(float* data, Plan pl, int nrows_per_img,
                                                       size_t img_stride, int npairs, int nseq,
                                                       const float2* __restrict__ tw) {
  extern __shared__ float2 smem[];
  const int n = pl.n, ld = n + 1;
  float2* buf = smem;
  float2* tmp = smem + nseq * ld;
  const int pair0 = blockIdx.x * nseq;
  const int pitch = n + 2;
  for (int e = threadIdx.x; e < nseq * n; e += blockDim.x) {
    int s = e / n, x = e - s * n;
    int pr = pair0 + s;
    float2 v = f2(0.f, 0.f);
    if (pr < npairs) {
      int img = (2 * pr) / nrows_per_img, row = (2 * pr) % nrows_per_img;
      const float* ra = data + img * img_stride + (size_t)row * pitch;
      v = f2(ra[x], ra[x + pitch]);
    }
    buf[s * ld + x] = v;
  }
  __syncthreads();
  float2* res = lds_fft(buf, tmp, pl, ld, nseq, -1, tw);
  const int jc = n / 2 + 1;
  for (int e = threadIdx.x; e < nseq * jc; e += blockDim.x) {
    int s = e / jc, k = e - s * jc;
    int pr = pair0 + s;
    if (pr >= npairs) continue;
    float2 zk = res[s * ld + k];
    float2 zm = res[s * ld + ((n - k) % n)];
    // Xa = (Z_k + conj Z_-k)/2 ; Xb = (Z_k - conj Z_-k)/(2i)
    float2 xa = f2(0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y));
    float2 xb = f2(0.5f * (zk.y + zm.y), -0.5f * (zk.x - zm.x));
    int img = (2 * pr) / nrows_per_img, row = (2 * pr) % nrows_per_img;
    float* ra = data + img * img_stride + (size_t)row * pitch;
    ra[2 * k] = xa.x;
    ra[2 * k + 1] = xa.y;
    ra[pitch + 2 * k] = xb.x;
    ra[pitch + 2 * k + 1] = xb.y;
  }
}

// ---- row pass, backward: half spectra of rows (2q, 2q+1) -> real rows
__global__ void __launch_bounds__(kThreads) k_rows_c2r(float* data, Plan pl, int nrows_per_img,
                                                       size_t img_stride, int npairs, int nseq,
                                                       const float2* __restrict__ tw) {
  extern __shared__ float2 smem[];
  const int n = pl.n, ld = n + 1, jc = n / 2 + 1, pitch = n + 2;
  float2* buf = smem;
  float2* tmp = smem + nseq * ld;
  const int pair0 = blockIdx.x * nseq;
  for (int e = threadIdx.x; e < nseq * jc; e += blockDim.x) {
    int s = e / jc, k = e - s * jc;
    int pr = pair0 + s;
    float2 a = f2(0.f, 0.f), b = f2(0.f, 0.f);
    if (pr < npairs) {
      int img = (2 * pr) / nrows_per_img, row = (2 * pr) % nrows_per_img;
      const float* ra = data + img * img_stride + (size_t)row * pitch;
      a = f2(ra[2 * k], ra[2 * k + 1]);
      b = f2(ra[pitch + 2 * k], ra[pitch + 2 * k + 1]);
    }
    if (k == 0 || 2 * k == n) { a.y = 0.f; b.y = 0.f; }
    // Z_k = A_k + i B_k ; Z_{n-k} = conj(A_k) + i conj(B_k)
    buf[s * ld + k] = f2(a.x - b.y, a.y + b.x);
    if (k > 0 && 2 * k < n) buf[s * ld + (n - k)] = f2(a.x + b.y, -a.y + b.x);
  }
  __syncthreads();
  float2* res = lds_fft(buf, tmp, pl, ld, nseq, +1, tw);
  for (int e = threadIdx.x; e < nseq * pitch; e += blockDim.x) {
    int s = e / pitch, x = e - s * pitch;
    int pr = pair0 + s;
    if (pr >= npairs) continue;
    int img = (2 * pr) / nrows_per_img, row = (2 * pr) % nrows_per_img;
    float* ra = data + img * img_stride + (size_t)row * pitch;
    float2 z = x < n ? res[s * ld + x] : f2(0.f, 0.f);
    ra[x] = z.x;
    ra[pitch + x] = z.y;
  }
}

// ---- column pass over the half-plane: JC columns of length n (complex, stride JC)
__global__ void __launch_bounds__(kThreads) k_cols(float* data, Plan pl, size_t img_stride, int cw,
                                                   int nimg, int sign,
                                                   const float2* __restrict__ tw) {
  extern __shared__ float2 smem[];
  const int n = pl.n, ld = n + 1, jc = n / 2 + 1;
  float2* buf = smem;
  float2* tmp = smem + cw * ld;
  // column blocks of one image in XCD-contiguous order
  const int jb = (jc + cw - 1) / cw;
  const int lb = xcd_block(blockIdx.x, gridDim.x);
  const int img = lb / jb;
  if (img >= nimg) return;
  const int x0 = (lb - img * jb) * cw;
  const int ncol = min(cw, jc - x0);
  float2* base = reinterpret_cast<float2*>(data + img * img_stride);
  for (int e = threadIdx.x; e < n * cw; e += blockDim.x) {
    int y = e / cw, c = e - y * cw;
    float2 v = f2(0.f, 0.f);
    if (c < ncol) v = base[(size_t)y * jc + x0 + c];
    buf[c * ld + y] = v;
  }
  __syncthreads();
  float2* res = lds_fft(buf, tmp, pl, ld, cw, sign, tw);
  for (int e = threadIdx.x; e < n * cw; e += blockDim.x) {
    int y = e / cw, c = e - y * cw;
    if (c < ncol) base[(size_t)y * jc + x0 + c] = res[c * ld + y];
  }
}

// the third axis of a 3D transform: ncols columns of length n, element y of
// column q at complex index y * rs + q (rs = JC*NSAM for a padded volume)
__global__ void __launch_bounds__(kThreads) k_cols_z(float* data, Plan pl, int ncols, size_t rs,
                                                     int cw, int sign,
                                                     const float2* __restrict__ tw) {
  extern __shared__ float2 smem[];
  const int n = pl.n, ld = n + 1;
  float2* buf = smem;
  float2* tmp = smem + cw * ld;
  const int lb = xcd_block(blockIdx.x, gridDim.x);
  const int x0 = lb * cw;
  if (x0 >= ncols) return;
  const int ncol = min(cw, ncols - x0);
  float2* base = reinterpret_cast<float2*>(data);
  for (int e = threadIdx.x; e < n * cw; e += blockDim.x) {
    int y = e / cw, c = e - y * cw;
    float2 v = f2(0.f, 0.f);
    if (c < ncol) v = base[(size_t)y * rs + x0 + c];
    buf[c * ld + y] = v;
  }
  __syncthreads();
  float2* res = lds_fft(buf, tmp, pl, ld, cw, sign, tw);
  for (int e = threadIdx.x; e < n * cw; e += blockDim.x) {
    int y = e / cw, c = e - y * cw;
    if (c < ncol) base[(size_t)y * rs + x0 + c] = res[c * ld + y];
  }
}

int row_seqs(int n) {
  int s = 2048 / n;
  return s < 1 ? 1 : s;
}
#endif

// ---- the same three kernels with the length known at compile time
template <int N>
using RowFft = Fft<N, 2048 / N, false>;
template <int N>
using ColFft = Fft<N, cols_cw(N), true>;

template <int N>
__global__ void __launch_bounds__(kThreads) k_rows_r2c_t(float* data, size_t img_stride,
                                                         int npairs, const float2* __restrict__ tw) {
  using F = RowFft<N>;
  constexpr int NSEQ = 2048 / N, JC = N / 2 + 1, PITCH = N + 2;
  extern __shared__ float2 smem[];
  const int pair0 = blockIdx.x * NSEQ;
  // rows of pair pr, as an image's start and the pair's in it
  auto row = [&](int pr) {
    return data + (2 * pr / N) * img_stride + (size_t)(2 * pr % N) * PITCH;
  };
  float2 a[F::IF][F::RF], z[F::IL][F::RL];
  F::template each<F::RF>([&](int it, int s, int i) {
    const float* ra = row(min(pair0 + s, npairs - 1)) + i;
#pragma unroll
    for (int r = 0; r < F::RF; r++) a[it][r] = f2(ra[r * F::TF], ra[r * F::TF + PITCH]);
  });
  F::template run<-1, false>(a, z, smem, tw);
  __syncthreads();
  F::template each<F::RL>([&](int it, int s, int i) {
#pragma unroll
    for (int q = 0; q < F::RL; q++) smem[F::at(s, i + q * F::TL)] = z[it][q];
  });
  __syncthreads();
  for (int e = threadIdx.x; e < NSEQ * JC; e += kThreads) {
    const int s = e / JC, k = e - s * JC;
    if (pair0 + s >= npairs) continue;
    float2* ra = reinterpret_cast<float2*>(row(pair0 + s)) + k;
    split_pair(smem[F::at(s, k)], smem[F::at(s, k ? N - k : 0)], ra[0], ra[JC]);
  }
}

template <int N>
__global__ void __launch_bounds__(kThreads) k_rows_c2r_t(float* data, size_t img_stride,
                                                         int npairs, const float2* __restrict__ tw) {
  using F = RowFft<N>;
  constexpr int NSEQ = 2048 / N, JC = N / 2 + 1, PITCH = N + 2;
  extern __shared__ float2 smem[];
  const int pair0 = blockIdx.x * NSEQ;
  auto row = [&](int pr) {
    return data + (2 * pr / N) * img_stride + (size_t)(2 * pr % N) * PITCH;
  };
  float2 a[F::IF][F::RF], z[F::IL][F::RL];
  F::template each<F::RF>([&](int it, int s, int i) {
    const float2* ra = reinterpret_cast<const float2*>(row(min(pair0 + s, npairs - 1)));
#pragma unroll
    for (int r = 0; r < F::RF; r++) {
      const int k = i + r * F::TF, m = 2 * k <= N ? k : N - k;
      a[it][r] = pair_point(ra[m], ra[m + JC], k, N);
    }
  });
  // every load is in registers once the first exchange's barriers are passed:
  // the rows may be written in place
  F::template run<+1, false>(a, z, smem, tw);
  F::template each<F::RL>([&](int it, int s, int i) {
    if (pair0 + s >= npairs) return;
    float* ra = row(pair0 + s);
#pragma unroll
    for (int q = 0; q < F::RL; q++) {
      ra[i + q * F::TL] = z[it][q].x;
      ra[i + q * F::TL + PITCH] = z[it][q].y;
    }
    if (i < 2) ra[N + i] = ra[N + i + PITCH] = 0.f;
  });
}


template <int N, int SIGN>
__global__ void __launch_bounds__(kThreads) k_cols_t(float* data, size_t img_stride, int nimg,
                                                     const float2* __restrict__ tw) {
  using F = ColFft<N>;
  constexpr int JC = N / 2 + 1;
  constexpr int CW = cols_cw(N);
  constexpr int JB = (JC + CW - 1) / CW;
  extern __shared__ float2 smem[];
  // column blocks of one image in XCD-contiguous order
  const int lb = xcd_block(blockIdx.x, gridDim.x);
  const int img = lb / JB;
  if (img >= nimg) return;
  const int x0 = (lb - img * JB) * CW;
  const int ncol = min(CW, JC - x0);
  float2* base = reinterpret_cast<float2*>(data + img * img_stride) + x0;
  float2 a[F::IF][F::RF], z[F::IL][F::RL];
  F::template each<F::RF>([&](int it, int c, int i) {
    const float2* col = base + min(c, ncol - 1) + (size_t)i * JC;
#pragma unroll
    for (int r = 0; r < F::RF; r++) a[it][r] = col[(size_t)r * F::TF * JC];
  });
  F::template run<SIGN, false>(a, z, smem, tw);
  F::template each<F::RL>([&](int it, int c, int i) {
    if (c >= ncol) return;
    float2* col = base + c + (size_t)i * JC;
#pragma unroll
    for (int q = 0; q < F::RL; q++) col[(size_t)q * F::TL * JC] = z[it][q];
  });
}

}  // namespace

template <int N>
int rows_pass_t(Ctx& c, int nimg, float* data, size_t img_stride, bool fwd, const float2* tw) {
  constexpr int NSEQ = 2048 / N;
  const int npairs = nimg * (N / 2);
  const size_t lds = RowFft<N>::kLds;
  dim3 grid((npairs + NSEQ - 1) / NSEQ);
  if (fwd)
    hipLaunchKernelGGL(k_rows_r2c_t<N>, grid, dim3(kThreads), lds, c.stream, data, img_stride,
                       npairs, tw);
  else
    hipLaunchKernelGGL(k_rows_c2r_t<N>, grid, dim3(kThreads), lds, c.stream, data, img_stride,
                       npairs, tw);
  FR_HIP(hipGetLastError());
  return 0;
}

template <int N>
int cols_pass_t(Ctx& c, int nimg, float* data, size_t img_stride, int sign, const float2* tw) {
  constexpr int JC = N / 2 + 1;
  constexpr int CW = cols_cw(N);
  const size_t lds = ColFft<N>::kLds;
  const long long nblk = (long long)((JC + CW - 1) / CW) * nimg;
  FR_CHECK(nblk <= (1ll << 30), "too many images in one FFT batch (%d)", nimg);
  dim3 grid(round8((int)nblk));
  if (sign < 0)
    hipLaunchKernelGGL((k_cols_t<N, -1>), grid, dim3(kThreads), lds, c.stream, data, img_stride,
                       nimg, tw);
  else
    hipLaunchKernelGGL((k_cols_t<N, +1>), grid, dim3(kThreads), lds, c.stream, data, img_stride,
                       nimg, tw);
  FR_HIP(hipGetLastError());
  return 0;
}

#ifdef FR_LEN
template int rows_pass_t<FR_LEN>(Ctx&, int, float*, size_t, bool, const float2*);
template int cols_pass_t<FR_LEN>(Ctx&, int, float*, size_t, int, const float2*);
#else
#define FR_EXTERN(N)                                                                  \
  extern template int rows_pass_t<N>(Ctx&, int, float*, size_t, bool, const float2*); \
  extern template int cols_pass_t<N>(Ctx&, int, float*, size_t, int, const float2*);
FR_LENGTHS(FR_EXTERN)

bool fft_supported(int nsam) {
  Plan p;
  return (nsam % 2 == 0) && make_plan(nsam, &p);
}

static int rows_pass_any(Ctx&, const Plan&, int, float*, size_t, bool, const float2*);
static int cols_pass_any(Ctx&, const Plan&, int, float*, size_t, int, const float2*);

static int rows_pass(Ctx& c, int nsam, int nimg, float* data, size_t img_stride, bool fwd) {
  Plan pl;
  FR_CHECK(make_plan(nsam, &pl) && nsam % 2 == 0, "FFT length %d not supported", nsam);
  const float2* tw = c.twiddles(nsam);
  FR_CHECK(tw != nullptr, "twiddle table allocation failed");
  return with_length(nsam, [&](auto len) {
    if constexpr (len() > 0)
      return rows_pass_t<len()>(c, nimg, data, img_stride, fwd, tw);
    else
      return rows_pass_any(c, pl, nimg, data, img_stride, fwd, tw);
  });
}

static int rows_pass_any(Ctx& c, const Plan& pl, int nimg, float* data, size_t img_stride, bool fwd,
                         const float2* tw) {
  const int nsam = pl.n;
  int npairs = nimg * (nsam / 2);
  int nseq = row_seqs(nsam);
  size_t lds = sizeof(float2) * 2 * nseq * (nsam + 1);
  dim3 grid((npairs + nseq - 1) / nseq);
  if (fwd)
    hipLaunchKernelGGL(k_rows_r2c, grid, dim3(kThreads), lds, c.stream, data, pl, nsam, img_stride,
                       npairs, nseq, tw);
  else
    hipLaunchKernelGGL(k_rows_c2r, grid, dim3(kThreads), lds, c.stream, data, pl, nsam, img_stride,
                       npairs, nseq, tw);
  FR_HIP(hipGetLastError());
  return 0;
}

static int cols_pass(Ctx& c, int nsam, int nimg, float* data, size_t img_stride, int sign) {
  Plan pl;
  FR_CHECK(make_plan(nsam, &pl), "FFT length %d not supported", nsam);
  const float2* tw = c.twiddles(nsam);
  FR_CHECK(tw != nullptr, "twiddle table allocation failed");
  FR_CHECK(nimg <= 65535, "too many images in one FFT batch (%d)", nimg);
  return with_length(nsam, [&](auto len) {
    if constexpr (len() > 0)
      return cols_pass_t<len()>(c, nimg, data, img_stride, sign, tw);
    else
      return cols_pass_any(c, pl, nimg, data, img_stride, sign, tw);
  });
}

static int cols_pass_any(Ctx& c, const Plan& pl, int nimg, float* data, size_t img_stride, int sign,
                         const float2* tw) {
  const int nsam = pl.n;
  int jc = nsam / 2 + 1;
  int cw = 2048 / nsam;
  if (cw < 1) cw = 1;
  if (cw > jc) cw = jc;
  size_t lds = sizeof(float2) * 2 * cw * (nsam + 1);
  const long long nblk = (long long)((jc + cw - 1) / cw) * nimg;
  FR_CHECK(nblk <= (1ll << 30), "too many images in one FFT batch (%d)", nimg);
  dim3 grid(round8((int)nblk));
  hipLaunchKernelGGL(k_cols, grid, dim3(kThreads), lds, c.stream, data, pl, img_stride, cw, nimg,
                     sign, tw);
  FR_HIP(hipGetLastError());
  return 0;
}

int fft_rows_2d(Ctx& c, int nsam, int nimg, float* data, size_t img_stride, bool fwd) {
  if (nimg <= 0) return 0;
  return rows_pass(c, nsam, nimg, data, img_stride, fwd);
}

int fft_r2c_2d(Ctx& c, int nsam, int nimg, float* data, size_t img_stride) {
  if (nimg <= 0) return 0;
  if (int r = rows_pass(c, nsam, nimg, data, img_stride, true)) return r;
  return cols_pass(c, nsam, nimg, data, img_stride, -1);
}

int fft_c2r_2d(Ctx& c, int nsam, int nimg, float* data, size_t img_stride) {
  if (nimg <= 0) return 0;
  if (int r = cols_pass(c, nsam, nimg, data, img_stride, +1)) return r;
  return rows_pass(c, nsam, nimg, data, img_stride, false);
}

static int z_pass(Ctx& c, int nsam, float* data, int sign) {
  Plan pl;
  FR_CHECK(make_plan(nsam, &pl), "FFT length %d not supported", nsam);
  const float2* tw = c.twiddles(nsam);
  FR_CHECK(tw != nullptr, "twiddle table allocation failed");
  const int jc = nsam / 2 + 1;
  const int ncols = jc * nsam;
  int cw = 2048 / nsam;
  if (cw < 1) cw = 1;
  const size_t lds = sizeof(float2) * 2 * cw * (nsam + 1);
  dim3 grid(round8((ncols + cw - 1) / cw));
  hipLaunchKernelGGL(k_cols_z, grid, dim3(kThreads), lds, c.stream, data, pl, ncols,
                     (size_t)ncols, cw, sign, tw);
  FR_HIP(hipGetLastError());
  return 0;
}

// 3D transforms of a padded volume (NSAM+2 row pitch, NSAM^2 rows): the 2D
// transform of every z-slice, then the z axis
int fft_r2c_3d(Ctx& c, int nsam, float* data) {
  const size_t img = (size_t)nsam * (nsam + 2);
  if (int r = fft_r2c_2d(c, nsam, nsam, data, img)) return r;
  return z_pass(c, nsam, data, -1);
}

int fft_c2r_3d(Ctx& c, int nsam, float* data) {
  const size_t img = (size_t)nsam * (nsam + 2);
  if (int r = z_pass(c, nsam, data, +1)) return r;
  return fft_c2r_2d(c, nsam, nsam, data, img);
}

#endif  // FR_LEN

}  // namespace fr
