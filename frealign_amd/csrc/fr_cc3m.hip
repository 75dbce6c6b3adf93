// fr_cc3m.hip -- CC3M (cc3m.f:8-169) on the band's own grid.
//
// CC3M extracts a section on the annulus MAXR1 <= r < MAXR2, goes to real
// space on the NSAM x NSAM grid, applies MASKCOS2 and comes back, and reads
// only the annulus again.  With R = MAXR2 - 1 the largest frequency on either
// side, the masked band is
//   out[k] = sum_j W[k - j] X[j],   |k|, |j| <= R,
// W the transform of the mask's weights: only its frequencies up to 2 R
// matter.  So the same numbers come from any M x M grid with M >= 4 R + 1
// that carries the mask with W cut at M/2 - 1 (what aliases falls outside the
// band), whatever NSAM is: 64, 96 or 128 points for MAXR2 <= 16, 24, 32.
// The mean that MASKCOS2 takes over its ring is linear in the band (the table
// Q, formed on the NSAM grid).  This needs the weights of one AMAG; the kernel
// takes the items with AMAG = 1 and leaves the others to the NSAM-grid form.
//
// One workgroup per item, persistent over a contiguous run of items (the
// candidates of one particle reuse its CTF and spectrum, held in registers).
// Every pass is a product with T[m][2i] = cos(2 pi i m/M), T[m][2i+1] =
// -sin(2 pi i m/M) on the FP32 matrix cores:
//   column c2c  Y[m][c]   = sum_J T[m][.] B[c][.]   B: the +-J pairs
//   row c2r     x[r][m]   = sum_I T[r][.] w_I Y[m][.]
//   mask        y = (x - mean) w, the same w at r and M - r
//   row r2c     Z[m][k]   = sum_r T[r][k] y[r][m]  (+ M mean at k = 0)
//   column r2c  out[j][k] = sum_m T[m][j] Z[m][k]
// folded over the table's symmetries: rows m and M - m differ by the sign of the
// sines, rows m and M/2 - m by that of the odd cosines and the even sines.  So
// the cosine and sine parts of even and odd frequencies, each a product over
// m < M/4, give all four rows, and the transforms back take the four rows' sums
// and differences (row M/4 is its own partner, in plain sums).  At MAXR2 <= 16,
// where 8 frequencies of one parity would not fill a tile, only over M - m.
// Then the shell sums of cc3m.f:117-150, each thread its own (I, +-J) pairs,
// reduced by shell in a fixed order.
//
// What bounds it: at MAXR2 = 32 an item takes 768 16x16x4 FP32 MFMA (2.5 us of
// one CU's matrix cores; 1,536 folded once, 4,896 on a 256 grid), 3,200 gathered
// points and the barriers between the passes.  LDS is 71 KB (149 KB on the 256
// grid), so two workgroups share a CU and one's gathers and sums run under the
// other's products.  8,192 items of a 256 box: 291 us (1,370 on the 256 grid,
// 393 folded once).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "fr_common.h"
#include "fr_extract.h"
#include "fr_kernels.h"

namespace fr {

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float fx4;

__device__ inline fx4 mfma4(float a, float b, fx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// sum over the 16 lanes of a row, in every lane, on the vector ALU
template <int kCtrl>
__device__ inline float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf,
                                                        false));
}
__device__ inline float row16_sum(float v) {
  v = dpp_add<0xB1>(v);   // quad_perm 1,0,3,2
  v = dpp_add<0x4E>(v);   // quad_perm 2,3,0,1
  v = dpp_add<0x141>(v);  // row_half_mirror
  return dpp_add<0x140>(v);  // row_mirror
}

template <int RB, int M>
struct BandShape {
  static constexpr int kThreads = RB == 32 ? 512 : 256;
  static constexpr int kWaves = kThreads / 64;
  // the products folded over quarters of the grid, a wave's tile 16 frequencies
  // of one parity: 16 of RB = 32 fill it, 8 of RB = 16 would not
  static constexpr bool kQuarter = RB == 32;
  static constexpr int kK = 2 * RB;      // reals per row: RB frequencies
  static constexpr int kP = kK + 4;      // LDS row pitch (floats): conflict-free operand reads
  static constexpr int kPairs = RB * RB / kThreads;  // (I, |J|) pairs per thread
  static constexpr int kT = (M / 2 + 1) * kP, kY = M * kP, kB = kK * kP;
  // T, Y/Z (then the pairs' sums), B/out, the shells' terms
  static constexpr int kLds = kT + kY + kB;
  static_assert(3 * RB * RB <= kY, "the pairs' sums use the Y buffer");
  static_assert(M / 16 <= kWaves, "one row block per wave");
};

// kWin: instead of the score, each item's cross-spectrum sums and differences
// over +-J for every pair, and its shells' |AINPO|^2 and norm, for k_cc3m_window
template <int RB, int M, bool kWin>
__global__ void __launch_bounds__((BandShape<RB, M>::kThreads), 4)
    k_cc3m_band(int nsam, int nitem, float rbfact,
                const float2* __restrict__ a3df, const float* __restrict__ dm,
                const int* __restrict__ pidx, const float2* __restrict__ ctff,
                const float2* __restrict__ spec, const float* __restrict__ shift,
                const float* __restrict__ amag_arr, const float* __restrict__ fsct,
                const float* __restrict__ tab, const int* __restrict__ pairs,
                const float* __restrict__ ring_tab, int ring_cnt,
                const float* __restrict__ wmap, float* __restrict__ score, int flip, int mixed,
                Cc3mWinBuf wb) {
  using S = BandShape<RB, M>;
  constexpr int kThr = S::kThreads, kK = S::kK, kP = S::kP, kPr = S::kPairs, H = M / 2;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* Ts = lds;          // [M/2 + 1][kP]
  float* Ys = Ts + S::kT;   // [M][kP]
  float* Bs = Ys + S::kY;   // [kK][kP]
  __shared__ float red_s[S::kWaves];
  __shared__ float2 phx[RB], phy[RB];  // e^{i SHX I}, e^{i SHY J}
  __shared__ double term[RB][2];       // per shell: R_k WGT and WGT^2 sum |SAMP|^2

  const int tid0 = threadIdx.x;
  const int jc = nsam / 2 + 1;
  const size_t ic = (size_t)nsam * jc;
  auto ld2 = [](const float* p) { return *reinterpret_cast<const float2*>(p); };
  auto ld4 = [](const float* p) { return *reinterpret_cast<const fx4*>(p); };

  const int per = (nitem + (int)gridDim.x - 1) / (int)gridDim.x;
  const int it0 = blockIdx.x * per, it1 = min(nitem, it0 + per);

  if (mixed) {  // no item of this form: nothing to set up
    bool any = false;
    for (int it = it0 + tid0; it < it1; it += kThr) any |= amag_arr[it] == 1.0f;
    if (!__syncthreads_or(any)) return;
  }
  // ---- what does not depend on the item
  for (int e = tid0; e < (H + 1) * (kK / 4); e += kThr) {
    const int r = e / (kK / 4), q = e % (kK / 4);
    *reinterpret_cast<float4*>(Ts + r * kP + 4 * q) =
        *reinterpret_cast<const float4*>(tab + (size_t)r * kK + 4 * q);
  }
  // this thread's pairs (I, +-J): the place of the pair's sums in shell order
  // (below 0: off the band)
  int pos[kPr];
#pragma unroll
  for (int u = 0; u < kPr; u++) pos[u] = pairs[kCc3mPairHdr + tid0 + u * kThr];
  // this 16-lane row's shell: its pairs, point count, weight and sign rule
  const int sh = 1 + (tid0 >> 4);
  const int sb0 = pairs[sh], sb1 = pairs[sh + 1];
  const int top = min(nsam / 2, kCc3mShells);
  const bool used = sh < top && sb1 > sb0;
  const float wgt = expf(-rbfact * (float)(sh * sh));
  const bool absr = used && !flip && fsct[sh] < 0.95f;
  // shells with points (SUM1 of cc3m.f:139-167)
  double nshell = 0.0;
  for (int s = 1; s < top && s <= RB; s++)
    if (pairs[s + 1] > pairs[s]) nshell += 1.0;
  float2 cpos[kPr], cneg[kPr];
  int pprev = -1;

  for (int it = it0; it < it1; it++) {
    if (amag_arr[it] != 1.0f) continue;  // the NSAM-grid form's item
    // Opaque copies, made anew for each item: addresses formed from them and
    // values loaded through them are not kept across items, which would cost
    // more registers (as spills, read back through L2) than forming them again.
    int tid = tid0;
    const float *wtab = wmap, *qtab = ring_tab;
    asm volatile("" : "+v"(tid), "+s"(wtab), "+s"(qtab));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int la = lane & 15, lg = lane >> 4;
    const int m0 = wave * 16, m = m0 + la;
    const bool rows = m0 < M;
    const int p = pidx[it];
    if (p != pprev) {
      pprev = p;
      const float2* cp = ctff + (size_t)p * 2 * ic;
#pragma unroll
      for (int u = 0; u < kPr; u++) {
        cpos[u] = cneg[u] = make_float2(0.f, 0.f);
        if (pos[u] >= 0) {
          const int e = tid + u * kThr, i = e / RB, jj = e % RB;
          const size_t ip = (size_t)i + (size_t)jc * jj;
          const size_t in = (size_t)i + (size_t)jc * wrapn(-jj, nsam);
          float2 cr = cp[ip], cl = cp[ip + ic];
          cpos[u] = make_float2(cr.x + cl.x, cr.y - cl.y);
          cr = cp[in], cl = cp[in + ic];
          cneg[u] = make_float2(cr.x + cl.x, cr.y - cl.y);
        }
      }
    }
    if (tid < 2 * RB) {
      float sn, cs;
      sincosf(shift[2 * it + (tid < RB ? 0 : 1)] * (float)(tid % RB), &sn, &cs);
      (tid < RB ? phx : phy)[tid % RB] = make_float2(cs, sn);
    }
    // ---- B[c][k], c = (I, re|im), k = (J, cos|sin), from the CTF-multiplied
    // section (cc3m.f:74-112); the ring sum on the way
    float rsum = 0.f;
    {
      const float* d = dm + 9 * (size_t)it;
      const bool inner = ainterpo_inner(jc, d, RB);
      const float scal = 1.0f / (float)nsam / (float)nsam;
#pragma unroll
      for (int u = 0; u < kPr; u++) {
        // one pair's gathers in flight at a time: two pairs' do not fit the registers
        if (u) __builtin_amdgcn_sched_barrier(0);
        const int e = tid + u * kThr, i = e / RB, jj = e % RB;
        cf ap = {0.f, 0.f}, an = ap;
        if (pos[u] >= 0) {
          if (inner) {
            ap = ainterpo_inner_dev(nsam, jc, a3df, d, i, jj);
            an = ainterpo_inner_dev(nsam, jc, a3df, d, i, -jj);
          } else {
            ap = ainterpo_dev(nsam, a3df, d, i, jj);
            an = ainterpo_dev(nsam, a3df, d, i, -jj);
          }
        }
        if (flip) {  // cc3.f:86-89
          if (cpos[u].x < 0.0f) ap = cf{-ap.re, -ap.im};
          if (cneg[u].x < 0.0f) an = cf{-an.re, -an.im};
        } else {
          ap = cmul(ap, cf{cpos[u].x, cpos[u].y});
          an = cmul(an, cf{cneg[u].x, cneg[u].y});
        }
        const cf xp = cscale(ap, scal), xn = jj ? cscale(an, scal) : cf{0.f, 0.f};
        const cf P = cadd(xp, xn);
        const cf Q = jj ? csub(xp, xn) : cf{0.f, 0.f};
        // Y_re = P_re T_re + Q_im T_im, Y_im = P_im T_re - Q_re T_im
        *reinterpret_cast<float2*>(Bs + (2 * i) * kP + 2 * jj) = make_float2(P.re, Q.im);
        *reinterpret_cast<float2*>(Bs + (2 * i + 1) * kP + 2 * jj) = make_float2(P.im, -Q.re);
        const float2 qa = ld2(qtab + (2 * i) * kCc3mRingPitch + 2 * jj);
        const float2 qb = ld2(qtab + (2 * i + 1) * kCc3mRingPitch + 2 * jj);
        rsum += qa.x * P.re + qa.y * Q.im + qb.x * P.im - qb.y * Q.re;
      }
    }
    for (int off = 32; off > 0; off >>= 1) rsum += __shfl_xor(rsum, off, 64);
    if (lane == 0) red_s[wave] = rsum;
    __syncthreads();

    // ---- column c2c, times the c2r weight
    if constexpr (S::kQuarter) {
      // m < M/4 and the frequencies' parity: Ee, Eo, Oe, Oo give Y at m, M - m,
      // M/2 - m and M/2 + m
      const int y0 = (wave / (kK / 16)) * 16, c0 = (wave % (kK / 16)) * 16;
      fx4 ee = {0.f, 0.f, 0.f, 0.f}, eo = ee, oe = ee, oo = ee;
#pragma unroll
      for (int s = 0; s < RB / 8; s++) {
        const fx4 tv = ld4(Ts + (y0 + la) * kP + 16 * s + 4 * lg);
        const fx4 bv = ld4(Bs + (c0 + la) * kP + 16 * s + 4 * lg);
        ee = mfma4(tv[0], bv[0], ee);
        oe = mfma4(tv[1], bv[1], oe);
        eo = mfma4(tv[2], bv[2], eo);
        oo = mfma4(tv[3], bv[3], oo);
      }
      const float wc = (c0 + la) < 2 ? 1.0f : 2.0f;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int y = y0 + 4 * lg + i;
        if (M % 128 && y >= M / 4) continue;
        float* yp = Ys + c0 + la;
        const float ep = ee[i] + eo[i], em = ee[i] - eo[i];
        const float op = oe[i] + oo[i], om = oe[i] - oo[i];
        yp[y * kP] = (ep + op) * wc;
        yp[(H - y) * kP] = (em - om) * wc;
        if (y) {
          yp[(M - y) * kP] = (ep - op) * wc;
          yp[(H + y) * kP] = (em + om) * wc;
        }
      }
      // rows M/4 and 3M/4, eight threads per column: even J by the cosines, odd J
      // by the sines
      const int c = tid >> 3, q = tid & 7;
      float v = 0.f;
#pragma unroll
      for (int j = 0; j < RB; j += 8) v += Bs[c * kP + 2 * (j + q) + (q & 1)];
      if ((q ^ (q >> 1)) & 1) v = -v;
      v += __shfl_xor(v, 2, 64);
      v += __shfl_xor(v, 4, 64);
      const float o = __shfl_xor(v, 1, 64);
      if (q == 0) {
        Ys[(M / 4) * kP + c] = (v + o) * (c < 2 ? 1.0f : 2.0f);
        Ys[(3 * M / 4) * kP + c] = (v - o) * (c < 2 ? 1.0f : 2.0f);
      }
    } else {
      // m < M/2: E against the cosine rows of B and O against its sine rows give
      // Y[m] = E + O, Y[M-m] = E - O
      constexpr int kTiles = (H / 16) * (kK / 16);
#pragma unroll
      for (int t0 = 0; t0 < kTiles; t0 += S::kWaves) {
        const int t = t0 + wave;
        if (kTiles % S::kWaves && t >= kTiles) break;
        const int y0 = (t / (kK / 16)) * 16, c0 = (t % (kK / 16)) * 16;
        fx4 e = {0.f, 0.f, 0.f, 0.f}, o = e;
#pragma unroll
        for (int ks = 0; ks < RB / 4; ks++) {
          const float2 tv = ld2(Ts + (y0 + la) * kP + 8 * ks + 2 * lg);
          const float2 bv = ld2(Bs + (c0 + la) * kP + 8 * ks + 2 * lg);
          e = mfma4(tv.x, bv.x, e);
          o = mfma4(tv.y, bv.y, o);
        }
        const float wc = (c0 + la) < 2 ? 1.0f : 2.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int y = y0 + 4 * lg + i;
          Ys[y * kP + c0 + la] = (e[i] + o[i]) * wc;
          if (y) Ys[(M - y) * kP + c0 + la] = (e[i] - o[i]) * wc;
        }
      }
      // row M/2: Y[c] = sum_J (-1)^J B[c][cos J], eight threads per column
      const int c = tid >> 3, q = tid & 7;
      float y = 0.f;
#pragma unroll
      for (int j = 0; j < RB; j += 8) y += Bs[c * kP + 2 * (j + q)];
      if (q & 1) y = -y;
      y += __shfl_xor(y, 1, 64);
      y += __shfl_xor(y, 2, 64);
      y += __shfl_xor(y, 4, 64);
      if (q == 0) Ys[H * kP + c] = y * (c < 2 ? 1.0f : 2.0f);
    }
    __syncthreads();

    // ---- rows of this wave's block: x = c2r of Y, y = (x - mean) w, Z = r2c of y
    float tot = 0.f;
#pragma unroll
    for (int k = 0; k < S::kWaves; k++) tot += red_s[k];
    const float mean = ring_cnt ? tot / (float)ring_cnt : tot;
    if constexpr (S::kQuarter) {
      // r < M/4 by parity as above: w is the same at r and M - r, and at M/2 - r
      // and M/2 + r.  Z at even and odd k takes the sums and differences of the
      // four y over the halves
      if (rows) {
        constexpr int kQt = (M / 4 + 15) / 16;
        fx4 w[kQt], wm[kQt];
#pragma unroll
        for (int t = 0; t < kQt; t++) {
          w[t] = ld4(wtab + (size_t)m * M + 16 * t + 4 * lg);
#pragma unroll
          for (int i = 0; i < 4; i++) wm[t][i] = wtab[(size_t)m * M + H - (16 * t + 4 * lg + i)];
        }
        const float wq = wtab[(size_t)m * M + M / 4];
        fx4 yv[RB / 8];
#pragma unroll
        for (int s = 0; s < RB / 8; s++) yv[s] = ld4(Ys + m * kP + 16 * s + 4 * lg);
        fx4 zce = {0.f, 0.f, 0.f, 0.f}, zse = zce, zco = zce, zso = zce;
#pragma unroll
        for (int t = 0; t < kQt; t++) {
          __builtin_amdgcn_sched_barrier(0);  // one tile's operands at a time
          fx4 ee = {0.f, 0.f, 0.f, 0.f}, eo = ee, oe = ee, oo = ee, ce, se, co, so;
#pragma unroll
          for (int s = 0; s < RB / 8; s++) {
            const fx4 tv = ld4(Ts + (16 * t + la) * kP + 16 * s + 4 * lg);
            ee = mfma4(tv[0], yv[s][0], ee);
            oe = mfma4(tv[1], yv[s][1], oe);
            eo = mfma4(tv[2], yv[s][2], eo);
            oo = mfma4(tv[3], yv[s][3], oo);
          }
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float ep = ee[i] + eo[i] - mean, em = ee[i] - eo[i] - mean;
            const float op = oe[i] + oo[i], om = oe[i] - oo[i];
            float ya = (ep + op) * w[t][i], yb = (ep - op) * w[t][i];
            float yc = (em - om) * wm[t][i], yd = (em + om) * wm[t][i];
            if (t == 0 && i == 0 && lg == 0) yb = yd = 0.f;  // r = 0 and M/2: their own partners
            if (M % 64 && 16 * t + 4 * lg + i >= M / 4) ya = yb = yc = yd = 0.f;
            const float p = ya + yb, q = yc + yd, u = ya - yb, v = yc - yd;
            ce[i] = p + q;
            co[i] = p - q;
            se[i] = u - v;
            so[i] = u + v;
          }
          // k-step i takes r = 16t + 4 lg + i: the C layout of the sums is the B layout
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const fx4 tv = ld4(Ts + (16 * t + 4 * lg + i) * kP + 4 * la);
            zce = mfma4(tv[0], ce[i], zce);
            zse = mfma4(tv[1], se[i], zse);
            zco = mfma4(tv[2], co[i], zco);
            zso = mfma4(tv[3], so[i], zso);
          }
        }
        // rows M/4 and 3M/4: x = P + Q and P - Q, P of the even I (8 s + 2 lg), Q of the odd
        float xp = 0.f, xq = 0.f;
#pragma unroll
        for (int s = 0; s < RB / 8; s++) {
          xp += yv[s][0];
          xq -= yv[s][3];
        }
        if (lg & 1) xp = -xp, xq = -xq;
        xp += __shfl_xor(xp, 16, 64);
        xq += __shfl_xor(xq, 16, 64);
        xp += __shfl_xor(xp, 32, 64);
        xq += __shfl_xor(xq, 32, 64);
        const float ya = (xp + xq - mean) * wq, yb = (xp - xq - mean) * wq;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          zce[i] += (i & 1) ? -(ya + yb) : ya + yb;
          zso[i] += (i & 1) ? ya - yb : yb - ya;
        }
        if (lg == 0) zce[0] += mean * (float)M;  // k = 0, the mean's own term
        // this wave alone read rows m0 .. m0 + 15 of Ys
#pragma unroll
        for (int i = 0; i < 4; i++)
          *reinterpret_cast<fx4*>(Ys + m * kP + 4 * (4 * lg + i)) =
              fx4{zce[i], zse[i], zco[i], zso[i]};
      }
    } else {
      // E and O of a tile of T rows r < M/2 give x[r] = E + O and x[M-r] = E - O
      // (the same w at both); Z's cosine part takes y[r] + y[M-r], its sine part
      // y[r] - y[M-r]
      fx4 w[M / 32];
      float wh = 0.f;
      if (rows) {
#pragma unroll
        for (int t = 0; t < M / 32; t++)
          w[t] = *reinterpret_cast<const fx4*>(wtab + (size_t)m * M + 16 * t + 4 * lg);
        wh = wtab[(size_t)m * M + H];
      }
      if (rows) {
        float2 yv[RB / 4];
#pragma unroll
        for (int ks = 0; ks < RB / 4; ks++) yv[ks] = ld2(Ys + m * kP + 8 * ks + 2 * lg);
        fx4 zc[RB / 16], zs[RB / 16];
#pragma unroll
        for (int kt = 0; kt < RB / 16; kt++) zc[kt] = zs[kt] = fx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < M / 32; t++) {
          __builtin_amdgcn_sched_barrier(0);  // one tile's operands at a time
          fx4 e = {0.f, 0.f, 0.f, 0.f}, o = e, sp, sm;
#pragma unroll
          for (int ks = 0; ks < RB / 4; ks++) {
            const float2 tv = ld2(Ts + (16 * t + la) * kP + 8 * ks + 2 * lg);
            e = mfma4(tv.x, yv[ks].x, e);
            o = mfma4(tv.y, yv[ks].y, o);
          }
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float ya = (e[i] + o[i] - mean) * w[t][i];
            float yb = (e[i] - o[i] - mean) * w[t][i];
            if (t == 0 && i == 0 && lg == 0) yb = 0.f;  // r = 0: its own partner
            sp[i] = ya + yb;
            sm[i] = ya - yb;
          }
          // k-step i takes r = 16t + 4 lg + i: the C layout of E, O is the B layout
#pragma unroll
          for (int i = 0; i < 4; i++)
#pragma unroll
            for (int kt = 0; kt < RB / 16; kt++) {
              const float2 tv = ld2(Ts + (16 * t + 4 * lg + i) * kP + 2 * (16 * kt + la));
              zc[kt] = mfma4(tv.x, sp[i], zc[kt]);
              zs[kt] = mfma4(tv.y, sm[i], zs[kt]);
            }
        }
        // row M/2: x = sum_I (-1)^I wYre[m][I], I = 4 ks + lg
        float xs = 0.f;
#pragma unroll
        for (int ks = 0; ks < RB / 4; ks++) xs += yv[ks].x;
        xs = (lg & 1) ? -xs : xs;
        xs += __shfl_xor(xs, 16, 64);
        xs += __shfl_xor(xs, 32, 64);
        const float yh = (xs - mean) * wh;
#pragma unroll
        for (int kt = 0; kt < RB / 16; kt++)
#pragma unroll
          for (int i = 0; i < 4; i++) zc[kt][i] += (i & 1) ? -yh : yh;
        if (lg == 0) zc[0][0] += mean * (float)M;  // k = 0, the mean's own term
        // this wave alone read rows m0 .. m0 + 15 of Ys
#pragma unroll
        for (int kt = 0; kt < RB / 16; kt++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            *reinterpret_cast<float2*>(Ys + m * kP + 2 * (16 * kt + 4 * lg + i)) =
                make_float2(zc[kt][i], zs[kt][i]);
      }
    }
    __syncthreads();

    // the pairs' spectrum, in flight under the column r2c
    float2 spos[kPr], sneg[kPr];
#pragma unroll
    for (int u = 0; u < kPr; u++) {
      const int e = tid + u * kThr, i = e / RB, jj = e % RB;
      spos[u] = sneg[u] = make_float2(0.f, 0.f);
      if (pos[u] >= 0) {
        const float2* sp = spec + (size_t)p * ic + i;
        spos[u] = sp[(size_t)jc * jj];
        sneg[u] = sp[(size_t)jc * wrapn(-jj, nsam)];
      }
    }
    // ---- column r2c, folded over m
    if constexpr (S::kQuarter) {
      // a wave's 16 j of one parity: cosine rows take (Z[m] + Z[M-m]) +- (Z[M/2-m] +
      // Z[M/2+m]), sine rows (Z[m] - Z[M-m]) -+ (Z[M/2-m] - Z[M/2+m])
      const int par = wave / (kK / 16), c0 = (wave % (kK / 16)) * 16;
      const float sg = par ? -1.0f : 1.0f;
      fx4 ac = {0.f, 0.f, 0.f, 0.f}, as = ac;
      const float* zp = Ys + c0 + la;
      const float* tp = Ts + lg * kP + 4 * la + 2 * par;
#pragma unroll
      for (int s = 0; s < M / 16; s++) {
        const int mm = 4 * s + lg;
        // m = 0 and M/2 have no partner (row M does not exist)
        const bool alone = s == 0 && lg == 0;
        const float za = zp[mm * kP], zc = zp[(H - mm) * kP], zd = zp[(H + mm) * kP];
        const float zb = zp[(alone ? 0 : M - mm) * kP];
        const float2 tv = ld2(tp + 4 * s * kP);
        ac = mfma4(tv.x, alone ? za + sg * zc : (za + zb) + sg * (zc + zd), ac);
        as = mfma4(tv.y, alone ? 0.f : (za - zb) - sg * (zc - zd), as);
      }
      // m = M/4 and 3M/4: the cosines of even j and the sines of odd j are +-1
      const float z1 = zp[(M / 4) * kP], z3 = zp[(3 * M / 4) * kP];
      const float ec = par ? 0.f : z1 + z3, es = par ? z3 - z1 : 0.f;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int j = 2 * (4 * lg + i) + par;
        Bs[j * kP + c0 + la] = ac[i] + ((i & 1) ? -ec : ec);
        Bs[(RB + j) * kP + c0 + la] = as[i] + ((i & 1) ? -es : es);
      }
    } else {
      // cosine rows take Z[m] + Z[M-m], sine rows Z[m] - Z[M-m] (m = 0 and M/2 are
      // their own partners)
      constexpr int kTiles = (RB / 16) * (kK / 16);
      if (wave < kTiles) {
        const int j0 = (wave / (kK / 16)) * 16, c0 = (wave % (kK / 16)) * 16;
        fx4 ac = {0.f, 0.f, 0.f, 0.f}, as = ac;
        // rows m = 4 s + lg upward and their partners M - m downward, each from
        // one base and a constant offset per step
        constexpr int kSteps = M / 8;
        const float* zp = Ys + lg * kP + c0 + la;
        const float* zq = Ys + (M - 4 * (kSteps - 1) - lg) * kP + c0 + la;
        const float* tp = Ts + lg * kP + 2 * (j0 + la);
#pragma unroll
        for (int s = 0; s < kSteps; s++) {
          const float za = zp[4 * s * kP];
          // m = 0 has no partner (its row M does not exist)
          const float zb = s ? zq[4 * (kSteps - 1 - s) * kP]
                             : Ys[(lg ? M - lg : 0) * kP + c0 + la];
          const float2 tv = ld2(tp + 4 * s * kP);
          const bool alone = s == 0 && lg == 0;
          ac = mfma4(tv.x, alone ? za : za + zb, ac);
          as = mfma4(tv.y, alone ? 0.f : za - zb, as);
        }
        // m = M/2: T = (-1)^j, no sine
        const float zh = Ys[H * kP + c0 + la];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float c = ac[i] + ((i & 1) ? -zh : zh);
          Bs[(j0 + 4 * lg + i) * kP + c0 + la] = c;
          Bs[(RB + j0 + 4 * lg + i) * kP + c0 + la] = as[i];
        }
      }
    }
    __syncthreads();

    // ---- cc3m.f:117-150: shifted particle x conj(masked projection) of this
    // thread's pairs, to the pair's place in shell order
#pragma unroll
    for (int u = 0; u < kPr; u++) {
      if (pos[u] < 0) continue;
      const int e = tid + u * kThr, i = e / RB, jj = e % RB;
      const float2 c = ld2(Bs + jj * kP + 2 * i), s = ld2(Bs + (RB + jj) * kP + 2 * i);
      const float2 ex = phx[i], ey = phy[jj];
      const float2 apv = make_float2(c.x - s.y, c.y + s.x);
      if constexpr (kWin) {
        // C = SPEC CONJG(AINPO) e^{i (SHX I + SHY J)} at the window's centre
        auto cross = [&](float2 v, float2 a, float cs, float sn) {
          const float re = v.x * a.x + v.y * a.y, im = v.y * a.x - v.x * a.y;
          return make_float2(re * cs - im * sn, re * sn + im * cs);
        };
        const float2 cp =
            cross(spos[u], apv, ex.x * ey.x - ex.y * ey.y, ex.x * ey.y + ex.y * ey.x);
        float2 cn = make_float2(0.f, 0.f);
        float s2 = spos[u].x * spos[u].x + spos[u].y * spos[u].y;
        float a2 = apv.x * apv.x + apv.y * apv.y;
        if (jj) {
          const float2 anv = make_float2(c.x + s.y, c.y - s.x);
          cn = cross(sneg[u], anv, ex.x * ey.x + ex.y * ey.y, ex.y * ey.x - ex.x * ey.y);
          s2 += sneg[u].x * sneg[u].x + sneg[u].y * sneg[u].y;
          a2 += anv.x * anv.x + anv.y * anv.y;
        }
        wb.cross[(size_t)it * wb.npair + pos[u]] =
            make_float4(cp.x + cn.x, cp.y + cn.y, cp.x - cn.x, cp.y - cn.y);
        Ys[RB * RB + pos[u]] = s2;
        Ys[2 * RB * RB + pos[u]] = a2;
        continue;
      }
      // REAL(SAMP CONJG(AINPO)) with SAMP = SPEC e^{i (SHX I + SHY J)}
      auto corr = [&](float2 v, float2 a, float cs, float sn) {
        const float re = v.x * a.x + v.y * a.y, im = v.y * a.x - v.x * a.y;
        return re * cs - im * sn;
      };
      float q = corr(spos[u], apv, ex.x * ey.x - ex.y * ey.y, ex.x * ey.y + ex.y * ey.x);
      float s2 = spos[u].x * spos[u].x + spos[u].y * spos[u].y;
      float a2 = apv.x * apv.x + apv.y * apv.y;
      if (jj) {
        const float2 anv = make_float2(c.x + s.y, c.y - s.x);
        q += corr(sneg[u], anv, ex.x * ey.x + ex.y * ey.y, ex.y * ey.x - ex.x * ey.y);
        s2 += sneg[u].x * sneg[u].x + sneg[u].y * sneg[u].y;
        a2 += anv.x * anv.x + anv.y * anv.y;
      }
      Ys[pos[u]] = q;
      Ys[RB * RB + pos[u]] = s2;
      Ys[2 * RB * RB + pos[u]] = a2;
    }
    __syncthreads();
    // one 16-lane row per shell, a fixed order; cc3m.f:139-167
    {
      float q = 0.f, s2 = 0.f, a2 = 0.f;
      for (int e = sb0 + la; e < sb1; e += 16) {
        if (!kWin) q += Ys[e];
        s2 += Ys[RB * RB + e];
        a2 += Ys[2 * RB * RB + e];
      }
      q = row16_sum(q);
      s2 = row16_sum(s2);
      a2 = row16_sum(a2);
      if (kWin && la == 0) {
        wb.a2[(size_t)it * kCc3mWinShells + sh - 1] = a2;
        term[sh - 1][1] = used ? (double)(wgt * wgt * s2) : 0.0;
      }
      if (!kWin && la == 0) {
        float r = q / sqrtf(a2);
        if (absr) r = fabsf(r);
        term[sh - 1][0] = used ? (double)(r * wgt) : 0.0;
        term[sh - 1][1] = used ? (double)(wgt * wgt * s2) : 0.0;
      }
    }
    __syncthreads();
    if (wave == 0) {
      double s3 = !kWin && lane < RB ? term[lane][0] : 0.0, s2 = lane < RB ? term[lane][1] : 0.0;
      for (int off = RB / 2; off > 0; off >>= 1) {
        s3 += __shfl_xor(s3, off, 64);
        s2 += __shfl_xor(s2, off, 64);
      }
      if (lane == 0) {
        if (kWin) {
          wb.norm[it] = nshell * s2 != 0.0 ? sqrt(nshell * s2) : 1.0;
        } else {
          if (nshell * s2 != 0.0) s3 = s3 / sqrt(nshell * s2);
          score[it] = (float)s3;
        }
      }
    }
  }
}

// ---- CC3M at every shift of a window (cc3m.f:117-167): with C the item's
// cross spectrum at the window's centre, S and D its sums and differences over
// +-J, and a, b the shift's offsets, the shell sums are
//   Re sum C e^{i (a I + b J)} = T1 - T2 - T3 - T4,
//   T1 = sum Re S cos aI cos bJ,   T2 = sum Im D cos aI sin bJ,
//   T3 = sum Im S sin aI cos bJ,   T4 = sum Re D sin aI sin bJ,
// and -a or -b only change signs: four products over a quarter of the window.
// Per shell each is a matrix product of 16 items by the shell's pairs with the
// pairs by the quarter's shifts, on the FP32 matrix cores; the phase factors are
// formed from two small tables.  A workgroup takes 16 items at a time, its eight
// waves the shells in zig-zag; a shell's terms join the wave's FP64 sums per shift,
// and these add up in LDS in wave order: the same sums whatever the launch holds.
// On the vector units, one item a workgroup and one shift a lane, the sums were
// most of the window's time: 52,728 items of a 128 box x 81 shifts took 10.6 ms,
// and take 2.05 ms.  With all of an item's shells in one wave and four such waves of
// 16 items a workgroup, this kernel took 107 us for 27 items and 111 for 500; 30 and 31 now.
constexpr int kWinWaves = 8, kWinItems = 16;
constexpr int kWinHalf = kCc3mWinMax / 2 + 1;  // offsets 0 .. 5 per axis

template <int NT>
__global__ void __launch_bounds__(64 * kWinWaves)
    k_cc3m_window(int nitem, int rb, int top, float rbfact, const int* __restrict__ pairs,
                  const float* __restrict__ fsct, const float* __restrict__ amag_arr, int flip,
                  Cc3mWindow win, Cc3mWinBuf wb, float* __restrict__ score,
                  int* __restrict__ code) {
  constexpr int kN = 16 * NT + 4;  // pitch: conflict-free
  __shared__ float2 tx[32][kWinHalf], ty[32][kWinHalf];  // (cos, sin) of a dsx I, b dsy J
  __shared__ unsigned short ij[32 * 32];                 // the pairs in shell order
  __shared__ double sums[4][kWinItems][kN];              // [signs][item][quarter shift]
  const int tid = threadIdx.x, lane = tid & 63, la = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int e = tid; e < 32 * kWinHalf; e += 64 * kWinWaves) {
    const int i = e / kWinHalf, a = e % kWinHalf;
    float sn, cs;
    sincosf((float)a * win.dsx * (float)i, &sn, &cs);
    tx[i][a] = make_float2(cs, sn);
    sincosf((float)a * win.dsy * (float)i, &sn, &cs);
    ty[i][a] = make_float2(cs, sn);
  }
  for (int e = tid; e < rb * rb; e += 64 * kWinWaves) {
    const int p = pairs[kCc3mPairHdr + e];
    if (p >= 0) ij[p] = (unsigned short)((e / rb) | ((e % rb) << 8));
  }
  __syncthreads();
  const int hx = win.nsx / 2, hy = win.nsy / 2, nq = (hx + 1) * (hy + 1);
  int qa[NT], qb[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int n = min(16 * t + la, nq - 1);
    qa[t] = n / (hy + 1);
    qb[t] = n % (hy + 1);
  }
  for (int base = blockIdx.x * kWinItems; base < nitem; base += gridDim.x * kWinItems) {
    const float4* row = wb.cross + (size_t)min(base + la, nitem - 1) * wb.npair;
    double acc[NT][4][4];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) acc[t][i][k] = 0.0;
    for (int sh = 1; sh < top && sh <= rb; sh++) {
      const int z = sh & (2 * kWinWaves - 1);
      if ((z < kWinWaves ? z : 2 * kWinWaves - 1 - z) != wave) continue;
      const int b0 = pairs[sh], b1 = pairs[sh + 1];
      if (b0 == b1) continue;
      fx4 T[NT][4];
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int k = 0; k < 4; k++) T[t][k] = fx4{0.f, 0.f, 0.f, 0.f};
      for (int e0 = b0; e0 < b1; e0 += 4) {
        const int e = e0 + lg;
        float4 v = row[min(e, b1 - 1)];
        if (e >= b1) v = make_float4(0.f, 0.f, 0.f, 0.f);
        const int pk = ij[min(e, b1 - 1)], i = pk & 0xff, j = pk >> 8;
#pragma unroll
        for (int t = 0; t < NT; t++) {
          const float2 x = tx[i][qa[t]], y = ty[j][qb[t]];
          T[t][0] = mfma4(v.x, x.x * y.x, T[t][0]);
          T[t][1] = mfma4(v.w, x.x * y.y, T[t][1]);
          T[t][2] = mfma4(v.y, x.y * y.x, T[t][2]);
          T[t][3] = mfma4(v.z, x.y * y.y, T[t][3]);
        }
      }
      const float wgt = expf(-rbfact * (float)(sh * sh));
      const bool absr = !flip && fsct[sh] < 0.95f;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int it = min(base + 4 * lg + i, nitem - 1);
        const float ra = sqrtf(wb.a2[(size_t)it * kCc3mWinShells + sh - 1]);
#pragma unroll
        for (int t = 0; t < NT; t++) {
          const float u = T[t][0][i], w = T[t][1][i], x = T[t][2][i], y = T[t][3][i];
          float r[4] = {(u - w) - (x + y), (u + w) - (x - y), (u - w) + (x + y),
                        (u + w) + (x - y)};
#pragma unroll
          for (int k = 0; k < 4; k++) {
            r[k] = r[k] / ra;
            if (absr) r[k] = fabsf(r[k]);
            acc[t][i][k] += (double)(r[k] * wgt);
          }
        }
      }
    }
    for (int w = 0; w < kWinWaves; w++) {
      if (wave == w)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
          for (int i = 0; i < 4; i++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
              double& s = sums[k][4 * lg + i][16 * t + la];
              s = w ? s + acc[t][i][k] : acc[t][i][k];
            }
      __syncthreads();
    }
    // the first maximum of each item in window order (IX outer, IY inner)
    for (int m = wave; m < kWinItems; m += kWinWaves) {
      const int it = base + m;
      if (it >= nitem) break;
      const double norm = wb.norm[it];
      float bv = -3.0e38f;
      int bs = 0x7fffffff;
      for (int e = lane; e < 4 * nq; e += 64) {
        const int n = e >> 2, k = e & 3, a = n / (hy + 1), b = n % (hy + 1);
        const float v = (float)(sums[k][m][n] / norm);
        const int s = (hx + (k & 2 ? -a : a)) * win.nsy + hy + (k & 1 ? -b : b);
        if (v > bv || (v == bv && s < bs)) {
          bv = v;
          bs = s;
        }
      }
      for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(bv, off, 64);
        const int os = __shfl_xor(bs, off, 64);
        if (ov > bv || (ov == bv && os < bs)) {
          bv = ov;
          bs = os;
        }
      }
      if (lane == 0 && amag_arr[it] == 1.0f) {
        score[it] = bv;
        code[it] = bs < win.nsx * win.nsy ? bs : 0;
      }
    }
    __syncthreads();  // the sums are written again
  }
}

}  // namespace

// Every band that the kernel's registers hold, at the boxes of the NSAM-grid form
// and, below NSAM/2, at the boxes of the particle's grid: an item with AMAG = 1
// comes here at any of them (8,192 items of a 250 box at MAXR2 32: 274 us, on the
// particle's grid 1,928)
bool cc3m_band_ok(int nsam, int maxr2) {
  return maxr2 >= 1 && maxr2 <= 32 &&
         (cc3m_fused_ok(nsam, maxr2) || (maxr2 < nsam / 2 && nsam <= kCc3mMaxBox));
}

int cc3m_band_grid(int nsam, int maxr2) {
  if (maxr2 > 32 || maxr2 < 1) return 0;
  const int need = maxr2 <= 16 ? 64 : maxr2 <= 24 ? 96 : 128;
  // the particle's own grid where it is one of the sizes and no larger
  return (nsam == 64 || nsam == 96 || nsam == 128) && nsam < need ? nsam : need;
}

int cc3m_band_rb(int maxr2) { return maxr2 <= 16 ? 16 : 32; }

// T[m][2i] = cos(2 pi i m/M), T[m][2i+1] = -sin(2 pi i m/M), m = 0 .. M/2
void cc3m_band_dft(int M, int rb, std::vector<float>& tab) {
  tab.assign((size_t)(M / 2 + 1) * 2 * rb, 0.f);
  for (int m = 0; m <= M / 2; m++)
    for (int i = 0; i < rb; i++) {
      const double ph = 2.0 * M_PI * (double)((i * m) % M) / (double)M;
      tab[(size_t)m * 2 * rb + 2 * i] = (float)std::cos(ph);
      tab[(size_t)m * 2 * rb + 2 * i + 1] = (float)-std::sin(ph);
    }
}

// Offsets of the shells INT(SQRT(FLOAT(I*I+J*J))+0.5) in the list of the pairs
// (I, |J|) of the band sorted by shell, then each pair's place in it
void cc3m_band_pairs(int maxr12, int maxr22, int rb, std::vector<int>& out) {
  std::vector<std::vector<int>> by(kCc3mShells + 1);
  for (int i = 0; i < rb; i++)
    for (int j = 0; j < rb; j++) {
      const int r2 = i * i + j * j;
      if (r2 >= maxr12 && r2 < maxr22) by[(int)(sqrtf((float)r2) + 0.5f)].push_back(i * rb + j);
    }
  out.assign((size_t)kCc3mPairHdr + rb * rb, -1);
  int n = 0;
  for (int s = 0; s < kCc3mPairHdr; s++) {
    out[s] = n;
    if (s <= kCc3mShells)
      for (int e : by[s]) out[kCc3mPairHdr + e] = n++;
  }
}

// The mask on the M grid, [m][n]: the NSAM-grid weights of cc3m_fused_wmap
// with their transform cut at M/2 - 1 (M = NSAM: the weights themselves).
// They are even in both axes, so cosines do.
void cc3m_band_wmap(int nsam, int M, const std::vector<float>& full, std::vector<float>& w) {
  if (M == nsam) {
    w = full;
    return;
  }
  // Every step runs along rows, so that the compiler vectorises it, and over a
  // quarter of the result: on a 256 box 1.1 ms, 11.0 as sums
  // per element.
  const int h = nsam / 2, Q = M / 2;  // frequencies 0 .. Q - 1
  auto table = [&](int rows, int cols, int n) {  // [r][c] = cos(2 pi r c/n)
    std::vector<double> co(n), t((size_t)rows * cols);
    for (int k = 0; k < n; k++) co[k] = std::cos(2.0 * M_PI * k / n);
    for (int r = 0; r < rows; r++)
      for (int c = 0, at = 0; c < cols; c++) {
        t[(size_t)r * cols + c] = co[at];
        at = (at + r) % n;
      }
    return t;
  };
  // y += v x
  auto add = [](int n, double v, const double* x, double* y) {
    for (int k = 0; k < n; k++) y[k] += v * x[k];
  };
  auto mult = [&](int n) { return n == 0 || n == h ? 1.0 : 2.0; };
  const std::vector<double> cn = table(h + 1, Q, nsam), cm = table(Q, Q + 1, M);
  // a[m][q] = sum_n w[m][n] cos(2 pi q n/N), then f[p][q] over m
  std::vector<double> a((size_t)(h + 1) * Q, 0.0), f((size_t)Q * Q, 0.0);
  for (int m = 0; m <= h; m++) {
    double* am = &a[(size_t)m * Q];
    for (int n = 0; n <= h; n++)
      if (const float v = full[(size_t)m * nsam + n])
        add(Q, mult(n) * (double)v, &cn[(size_t)n * Q], am);
    for (int p = 0; p < Q; p++) add(Q, mult(m) * cn[(size_t)m * Q + p], am, &f[(size_t)p * Q]);
  }
  for (int p = 0; p < Q; p++)
    for (int q = 0; q < Q; q++)
      f[(size_t)p * Q + q] *= (p ? 2.0 : 1.0) * (q ? 2.0 : 1.0) / ((double)nsam * nsam);
  // b[p][n] = sum_q f[p][q] cos(2 pi q n/M), n <= M/2, then the rows
  std::vector<double> b((size_t)Q * (Q + 1), 0.0), row(Q + 1);
  for (int p = 0; p < Q; p++)
    for (int q = 0; q < Q; q++)
      add(Q + 1, f[(size_t)p * Q + q], &cm[(size_t)q * (Q + 1)], &b[(size_t)p * (Q + 1)]);
  w.assign((size_t)M * M, 0.f);
  for (int m = 0; m <= Q; m++) {
    std::fill(row.begin(), row.end(), 0.0);
    for (int p = 0; p < Q; p++)
      add(Q + 1, cm[(size_t)p * (Q + 1) + m], &b[(size_t)p * (Q + 1)], row.data());
    for (int n = 0; n <= Q; n++) {
      const float v = (float)row[n];
      for (int y : {m, (M - m) % M})
        for (int x : {n, (M - n) % M}) w[(size_t)y * M + x] = v;
    }
  }
}

int cc3m_band_npair(int maxr12, int maxr22, int rb) {
  int n = 0;
  for (int i = 0; i < rb; i++)
    for (int j = 0; j < rb; j++) n += i * i + j * j >= maxr12 && i * i + j * j < maxr22;
  return n;
}

size_t cc3m_window_bytes(int npair) {
  return sizeof(float4) * (size_t)npair + sizeof(float) * kCc3mWinShells + sizeof(double);
}

Cc3mWinBuf cc3m_window_buf(void* base, int npair, size_t n) {
  Cc3mWinBuf b;
  b.npair = npair;
  b.cross = static_cast<float4*>(base);
  b.norm = reinterpret_cast<double*>(b.cross + (size_t)npair * n);
  b.a2 = reinterpret_cast<float*>(b.norm + n);
  return b;
}

namespace {
struct BandCall {
  const float *a3df, *spec, *ctff;
  const int* pidx;
  const float *dm, *shift, *amag, *fsct;
};

template <int RB, int M, bool kWin>
int launch_band(Ctx& c, const Cc3mArgs& a, const BandCall& p, const Cc3mBandTables& t,
                float* score, int blocks, const Cc3mWinBuf& wb) {
  using S = BandShape<RB, M>;
  auto fn = k_cc3m_band<RB, M, kWin>;
  const size_t lds = sizeof(float) * S::kLds;
  FR_HIP(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)lds));
  int grid = 0;
  if (int r = cc3m_grid(c, (const void*)fn, S::kThreads, lds, a.n, blocks, &grid)) return r;
  hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(S::kThreads), lds, c.stream, a.nsam, a.n,
                     a.rbfact, reinterpret_cast<const float2*>(p.a3df), p.dm, p.pidx,
                     reinterpret_cast<const float2*>(p.ctff),
                     reinterpret_cast<const float2*>(p.spec), p.shift, p.amag, p.fsct, t.dft,
                     t.pairs, t.ring, t.ring_cnt, t.wmap, score, a.cc3, a.mixed, wb);
  FR_HIP(hipGetLastError());
  return 0;
}

template <bool kWin>
int launch_any(Ctx& c, const Cc3mArgs& a, const BandCall& p, const Cc3mBandTables& t,
               float* score, int blocks, const Cc3mWinBuf& wb) {
  FR_CHECK(t.dft && t.pairs && t.ring && t.wmap, "band CC3M tables missing");
  const int M = cc3m_band_grid(a.nsam, a.maxr2), rb = cc3m_band_rb(a.maxr2);
  if (rb == 16 && M == 64) return launch_band<16, 64, kWin>(c, a, p, t, score, blocks, wb);
  if (rb == 32 && M == 64) return launch_band<32, 64, kWin>(c, a, p, t, score, blocks, wb);
  if (rb == 32 && M == 96) return launch_band<32, 96, kWin>(c, a, p, t, score, blocks, wb);
  if (rb == 32 && M == 128) return launch_band<32, 128, kWin>(c, a, p, t, score, blocks, wb);
  return fail("band CC3M: no grid for MAXR2 %d", a.maxr2);
}

template <int NT>
int launch_window(Ctx& c, const Cc3mArgs& a, const float* fsct, const float* amag,
                  const Cc3mBandTables& t, const Cc3mWindow& win, const Cc3mWinBuf& wb,
                  float* score, int* code) {
  const int top = a.nsam / 2 < kCc3mShells ? a.nsam / 2 : kCc3mShells;
  int grid = 0;
  if (int r = cc3m_grid(c, (const void*)k_cc3m_window<NT>, 64 * kWinWaves, 0,
                        (a.n + kWinItems - 1) / kWinItems, -1, &grid))
    return r;
  hipLaunchKernelGGL(k_cc3m_window<NT>, dim3((unsigned)grid), dim3(64 * kWinWaves), 0, c.stream,
                     a.n, cc3m_band_rb(a.maxr2), top, a.rbfact, t.pairs, fsct, amag, a.cc3, win,
                     wb, score, code);
  FR_HIP(hipGetLastError());
  return 0;
}
}  // namespace

int launch_cc3m_band(Ctx& c, const Cc3mArgs& a, const float* a3df, const float* spec,
                     const float* ctff, const int* pidx, const float* dm, const float* shift,
                     const float* amag, const float* fsct, const Cc3mBandTables& t, float* score,
                     int blocks) {
  if (a.n <= 0) return 0;
  return launch_any<false>(c, a, BandCall{a3df, spec, ctff, pidx, dm, shift, amag, fsct}, t, score,
                           blocks, Cc3mWinBuf{});
}

int launch_cc3m_band_window(Ctx& c, const Cc3mArgs& a, const float* a3df, const float* spec,
                            const float* ctff, const int* pidx, const float* dm,
                            const float* shift, const float* amag, const float* fsct,
                            const Cc3mBandTables& t, const Cc3mWindow& win, void* buf,
                            float* score, int* code, int blocks) {
  if (a.n <= 0) return 0;
  FR_CHECK(buf && code, "window buffers missing");
  FR_CHECK(win.nsx >= 1 && win.nsy >= 1 && win.nsx <= kCc3mWinMax && win.nsy <= kCc3mWinMax &&
               win.nsx % 2 == 1 && win.nsy % 2 == 1,
           "shift window %d x %d: odd sizes up to %d", win.nsx, win.nsy, kCc3mWinMax);
  const int npair =
      cc3m_band_npair(a.maxr1 * a.maxr1, a.maxr2 * a.maxr2, cc3m_band_rb(a.maxr2));
  const Cc3mWinBuf wb = cc3m_window_buf(buf, npair, a.n);
  if (int r = launch_any<true>(c, a, BandCall{a3df, spec, ctff, pidx, dm, shift, amag, fsct}, t,
                               score, blocks, wb))
    return r;
  const int nq = (win.nsx / 2 + 1) * (win.nsy / 2 + 1);
  if (nq <= 16) return launch_window<1>(c, a, fsct, amag, t, win, wb, score, code);
  if (nq <= 32) return launch_window<2>(c, a, fsct, amag, t, win, wb, score, code);
  return launch_window<3>(c, a, fsct, amag, t, win, wb, score, code);
}

}  // namespace fr
