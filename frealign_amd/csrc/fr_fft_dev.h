// fr_fft_dev.h -- device building blocks of the batched FFTs: complex
// helpers, the butterflies and the Stockham autosort passes, with the length
// known at compile time or at run time.  Used by the FFT kernels and by
// kernels that run a transform between other work on the same tile.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace fr {
namespace fftdev {

constexpr int kFftThreads = 256;  // threads of every workgroup that runs these passes

// XCD-aware block order.  The hardware deals a launch's workgroups to the 8
// XCDs round robin (workgroup p to XCD p mod 8); with a grid of g8 blocks (a
// multiple of 8), logical block (p mod 8) (g8 / 8) + p / 8 gives each XCD a
// contiguous range of logical blocks, so neighbouring blocks whose data share
// cache lines (the 8-column blocks of one half-plane row) share one L2.
__device__ inline int xcd_block(int p, int g8) { return (p & 7) * (g8 >> 3) + (p >> 3); }
inline int round8(int g) { return (g + 7) & ~7; }

// No contraction is left to the compiler in these: it would choose by what
// surrounds a transform, and the same transform in two kernels would differ in
// its last bits.
__device__ inline float2 f2(float a, float b) { return make_float2(a, b); }
__device__ inline float2 add2(float2 a, float2 b) {
#pragma clang fp contract(off)
  return f2(a.x + b.x, a.y + b.y);
}
__device__ inline float2 sub2(float2 a, float2 b) {
#pragma clang fp contract(off)
  return f2(a.x - b.x, a.y - b.y);
}
__device__ inline float2 mul2(float2 a, float2 b) {
#pragma clang fp contract(off)
  return f2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x));
}
__device__ inline float2 scl2(float2 a, float s) {
#pragma clang fp contract(off)
  return f2(a.x * s, a.y * s);
}
// multiply by i*sign
__device__ inline float2 muli(float2 a, int sign) { return sign > 0 ? f2(-a.y, a.x) : f2(a.y, -a.x); }

template <int R>
__device__ inline void butterfly(float2* u, int sign) {
  if constexpr (R == 2) {
    float2 a = u[0], b = u[1];
    u[0] = add2(a, b);
    u[1] = sub2(a, b);
  } else if constexpr (R == 4) {
    float2 a0 = add2(u[0], u[2]), a1 = sub2(u[0], u[2]);
    float2 b0 = add2(u[1], u[3]), jt = muli(sub2(u[1], u[3]), sign);
    u[0] = add2(a0, b0);
    u[2] = sub2(a0, b0);
    u[1] = add2(a1, jt);
    u[3] = sub2(a1, jt);
  } else if constexpr (R == 8) {
    const float h = 0.70710678118654752440f;
    float2 e[4] = {u[0], u[2], u[4], u[6]}, o[4] = {u[1], u[3], u[5], u[7]};
    butterfly<4>(e, sign);
    butterfly<4>(o, sign);
    // o[k] times e^{sign i pi k / 4}
    const float2 j1 = muli(o[1], sign), j3 = muli(o[3], sign);
    o[1] = scl2(add2(o[1], j1), h);
    o[2] = muli(o[2], sign);
    o[3] = scl2(sub2(j3, o[3]), h);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      u[k] = add2(e[k], o[k]);
      u[k + 4] = sub2(e[k], o[k]);
    }
  } else if constexpr (R == 3) {
    const float h = 0.86602540378443864676f;
    float2 s = add2(u[1], u[2]), d = sub2(u[1], u[2]);
    float2 v0 = add2(u[0], s);
    float2 m = sub2(u[0], scl2(s, 0.5f));
    float2 nn = scl2(muli(d, sign), h);
    u[0] = v0;
    u[1] = add2(m, nn);
    u[2] = sub2(m, nn);
  } else if constexpr (R == 5) {
    const float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
    const float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;
    float2 a1 = add2(u[1], u[4]), b1 = sub2(u[1], u[4]);
    float2 a2 = add2(u[2], u[3]), b2 = sub2(u[2], u[3]);
    float2 v0 = add2(add2(u[0], a1), a2);
    float2 p1 = add2(u[0], add2(scl2(a1, c1), scl2(a2, c2)));
    float2 q1 = muli(add2(scl2(b1, s1), scl2(b2, s2)), sign);
    float2 p2 = add2(u[0], add2(scl2(a1, c2), scl2(a2, c1)));
    float2 q2 = muli(sub2(scl2(b1, s2), scl2(b2, s1)), sign);
    u[0] = v0;
    u[1] = add2(p1, q1);
    u[4] = sub2(p1, q1);
    u[2] = add2(p2, q2);
    u[3] = sub2(p2, q2);
  }
}

// largest j >= 0 with j*j <= v (v >= 0, below 2^20)
__device__ inline int isqrt(int v) {
  int j = (int)sqrtf((float)v);
  if (j * j > v) j--;
  if ((j + 1) * (j + 1) <= v) j++;
  return j;
}

// ---- transforms whose length is known at compile time
//
// A Stockham pass of radix R takes butterfly i (of N / R) of a sequence from the
// points i + r N / R and leaves it at points N / R apart once it is the last
// one.  So the first pass takes its points from wherever they are (global
// memory, a computation) and the last leaves them in registers: LDS only
// carries the exchanges between passes, two for 8 x 8 x 4 at 256 points, in one
// buffer (18.5 kB for 2,048 points, so that the waves, not LDS, fill a CU).
// Radix-4 passes from LDS to LDS, with the tile put there before and read back
// after, took eight passages through two buffers; the r2c of 256 images of 256^2
// 74 -> 49 us.

// radix of pass i of a length n: eights first, then fours, threes, fives
constexpr int fft_radix(int n, int i) {
  int t = 0, m = n;
  while (m % 2 == 0) { m /= 2; t++; }
  int n8 = t / 3, n4 = 0, n2 = 0;
  if (t % 3 == 2) n4 = 1;
  else if (t % 3 == 1 && n8) { n8--; n4 = 2; }
  else if (t % 3 == 1) n2 = 1;
  if (i < n8) return 8;
  if (i < n8 + n4) return 4;
  if (i < n8 + n4 + n2) return 2;
  i -= n8 + n4 + n2;
  while (m % 3 == 0) { if (i-- == 0) return 3; m /= 3; }
  while (m % 5 == 0) { if (i-- == 0) return 5; m /= 5; }
  return 0;
}

constexpr int fft_npass(int n) {
  int k = 0;
  while (fft_radix(n, k)) k++;
  return k;
}

// NSEQ sequences of N points by kFftThreads threads.  kCols: neighbouring
// threads take the same butterfly of neighbouring sequences (columns of an
// image), else neighbouring butterflies of one sequence.  kRev: the passes in
// the opposite order; its first pass takes the points where the other order's
// last pass left them, so that a transform, a step on its points and the
// transform back need no exchange between them.
template <int N, int NSEQ, bool kCols, bool kRev = false>
struct Fft {
  static constexpr int NP = fft_npass(N);
  static constexpr int radix(int i) { return fft_radix(N, kRev ? NP - 1 - i : i); }
  static constexpr int iters(int r) { return (NSEQ * (N / r) + kFftThreads - 1) / kFftThreads; }
  static constexpr int RF = radix(0), TF = N / RF, IF = iters(RF);            // first pass
  static constexpr int RL = radix(NP - 1), TL = N / RL, IL = iters(RL);       // last pass
  // a word after every 8 points and sequences 8 points apart modulo 32: the
  // strided writes of a pass then fall on different banks, along a sequence
  // and across columns
  static constexpr int LP = N + N / 8, LD = LP + (40 - LP % 32) % 32;
  static constexpr size_t kLds = sizeof(float2) * NSEQ * LD;
  static __device__ inline int at(int s, int x) { return s * LD + x + (x >> 3); }

  // f(it, s, i) for this thread's butterflies of a pass of radix R
  template <int R, typename F>
  static __device__ inline void each(F f) {
    constexpr int T = N / R;
#pragma unroll
    for (int it = 0; it < iters(R); it++) {
      const int b = (int)threadIdx.x + it * kFftThreads;
      if (NSEQ * T % kFftThreads && b >= NSEQ * T) continue;
      if constexpr (kCols) f(it, b % NSEQ, b / NSEQ);
      else f(it, b / T, b % T);
    }
  }

  // the passes after pass I's points are in u
  template <int SIGN, bool kBusy, int I, int P, int IT, int R>
  static __device__ inline void pass(float2 (&u)[IT][R], float2 (&z)[IL][RL], float2* buf,
                                     const float2* __restrict__ tw) {
    each<R>([&](int it, int, int i) {
      if constexpr (P > 1) {
        const int k = i % P;
#pragma unroll
        for (int r = 1; r < R; r++) {
          float2 w = tw[r * k * (N / (P * R))];
          if (SIGN > 0) w.y = -w.y;
          u[it][r] = mul2(u[it][r], w);
        }
      }
      butterfly<R>(u[it], SIGN);
    });
    if constexpr (I == NP - 1) {
#pragma unroll
      for (int it = 0; it < IT; it++)
#pragma unroll
        for (int r = 0; r < R; r++) z[it][r] = u[it][r];
    } else {
      if (kBusy || I > 0) __syncthreads();
      each<R>([&](int it, int s, int i) {
        const int k = i % P, base = (i - k) * R + k;
#pragma unroll
        for (int q = 0; q < R; q++) buf[at(s, base + q * P)] = u[it][q];
      });
      __syncthreads();
      constexpr int R2 = radix(I + 1), T2 = N / R2;
      float2 v[iters(R2)][R2];
      each<R2>([&](int it, int s, int i) {
#pragma unroll
        for (int r = 0; r < R2; r++) v[it][r] = buf[at(s, i + r * T2)];
      });
      pass<SIGN, kBusy, I + 1, P * R>(v, z, buf, tw);
    }
  }

  // a[it][r]: point i + r TF of butterfly (it, s, i) of each<RF>; z[it][q]: point
  // i + q TL of each<RL>.  kBusy: other threads may still read buf.  They read it
  // after the return too: a barrier before it is written again.
  template <int SIGN, bool kBusy>
  static __device__ inline void run(float2 (&a)[IF][RF], float2 (&z)[IL][RL], float2* buf,
                                    const float2* __restrict__ tw) {
    pass<SIGN, kBusy, 0, 1>(a, z, buf, tw);
  }
};

// The point k of the sequence that carries two half spectra a and b (of N real
// values each) as Z = A + i B, from the half planes' points (k or N - k): the
// imaginary parts at k = 0 and N/2 are ignored, as the c2r does.
__device__ inline float2 pair_point(float2 a, float2 b, int k, int n) {
#pragma clang fp contract(off)
  if (k == 0 || 2 * k == n) a.y = b.y = 0.f;
  return 2 * k <= n ? make_float2(a.x - b.y, a.y + b.x) : make_float2(a.x + b.y, -a.y + b.x);
}

// The two half spectra's points k from Z_k and Z_{N-k}.
__device__ inline void split_pair(float2 zk, float2 zm, float2& a, float2& b) {
#pragma clang fp contract(off)
  a = make_float2(0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y));
  b = make_float2(0.5f * (zk.y + zm.y), -0.5f * (zk.x - zm.x));
}

// ---- radix-2/3/4/5 passes from LDS to LDS with the length known at run time
constexpr int kMaxPass = 12;

struct Plan {
  int n;
  int npass;
  int radix[kMaxPass];
};

inline bool make_plan(int n, Plan* p) {
  if (n < 2 || n > 1024) return false;
  p->n = n;
  p->npass = 0;
  int m = n;
  while (m % 4 == 0 && p->npass < kMaxPass) { p->radix[p->npass++] = 4; m /= 4; }
  while (m % 2 == 0 && p->npass < kMaxPass) { p->radix[p->npass++] = 2; m /= 2; }
  while (m % 3 == 0 && p->npass < kMaxPass) { p->radix[p->npass++] = 3; m /= 3; }
  while (m % 5 == 0 && p->npass < kMaxPass) { p->radix[p->npass++] = 5; m /= 5; }
  return m == 1;
}

template <int R>
__device__ inline void stockham_pass(const float2* in, float2* out, int n, int ld, int nseq, int p,
                                     int sign, const float2* __restrict__ tw) {
  const int T = n / R;
  const int stride = n / (p * R);
  for (int b = threadIdx.x; b < nseq * T; b += blockDim.x) {
    int s = b / T, i = b - s * T;
    int k = i % p;
    const float2* x = in + s * ld;
    float2 u[R];
#pragma unroll
    for (int r = 0; r < R; r++) u[r] = x[i + r * T];
#pragma unroll
    for (int r = 1; r < R; r++) {
      int e = (r * k * stride) % n;
      float2 w = tw[e];
      if (sign > 0) w.y = -w.y;
      u[r] = mul2(u[r], w);
    }
    butterfly<R>(u, sign);
    float2* y = out + s * ld;
    int base = (i - k) * R + k;
#pragma unroll
    for (int q = 0; q < R; q++) y[base + q * p] = u[q];
  }
}

// In-LDS FFT of nseq sequences (stride ld); returns the buffer holding the result.
__device__ inline float2* lds_fft(float2* buf, float2* tmp, const Plan& pl, int ld, int nseq, int sign,
                           const float2* __restrict__ tw) {
  int p = 1;
  for (int ps = 0; ps < pl.npass; ps++) {
    int R = pl.radix[ps];
    switch (R) {
      case 4: stockham_pass<4>(buf, tmp, pl.n, ld, nseq, p, sign, tw); break;
      case 2: stockham_pass<2>(buf, tmp, pl.n, ld, nseq, p, sign, tw); break;
      case 3: stockham_pass<3>(buf, tmp, pl.n, ld, nseq, p, sign, tw); break;
      default: stockham_pass<5>(buf, tmp, pl.n, ld, nseq, p, sign, tw); break;
    }
    __syncthreads();
    float2* t = buf;
    buf = tmp;
    tmp = t;
    p *= R;
  }
  return buf;
}

// The lengths that are compiled in: the even ones from 64 to 512 (an index division
// or modulus by a run-time length costs more than its butterfly: preparing 300
// images of 160^2 takes 173 us, 357 with passes of a run-time length).  A source with
// kernels of a length is compiled once per length as well, with FR_LEN defined, and
// then holds that length's alone: the device code is loaded where a program first
// uses it, and all lengths of the preparation's kernels together were 11 ms of its
// first call.
#define FR_LENGTHS(X) \
  X(64) X(72) X(80) X(90) X(96) X(100) X(108) X(120) X(128) \
  X(144) X(150) X(160) X(162) X(180) X(192) X(200) X(216) X(240) \
  X(250) X(256) X(270) X(288) X(300) X(320) X(324) X(360) X(384) \
  X(400) X(432) X(450) X(480) X(486) X(500) X(512)

// f(integral_constant<N>), or N = 0, the passes of a run-time length, for any other
template <typename F>
inline int with_length(int n, F f) {
#define FR_CASE(N) \
  case N: return f(std::integral_constant<int, N>{});
  switch (n) {
    FR_LENGTHS(FR_CASE)
    default: return f(std::integral_constant<int, 0>{});
  }
#undef FR_CASE
}

// columns per workgroup of a column pass: 64 bytes or more of a row, and 2,048
// points where the columns are short (16 at 256 measured no faster)
constexpr int cols_cw(int n) { return n <= 64 ? 32 : n <= 128 ? 16 : 8; }

// row pairs per workgroup of a row pass that stays in one image: the largest
// divisor of the image's pairs within 2,048 points
constexpr int rows_in_image(int n) {
  int k = 2048 / n;
  while (n / 2 % k) k--;
  return k;
}

}  // namespace fftdev
}  // namespace fr
