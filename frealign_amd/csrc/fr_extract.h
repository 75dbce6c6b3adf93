// fr_extract.h -- device-side trilinear gather from the Hermitian half-volume.
#pragma once
#include "fr_common.h"

namespace fr {

// two neighbouring points of the half-volume, 8-byte aligned
typedef float PointPair __attribute__((ext_vector_type(4), aligned(8)));

// AINTERPO3DS (ainterpo3ds.f:22-98, IPAD=1) evaluated at X3 = DM*(I,J): the
// plane coordinates are formed in the reference's FP32 operation order
// (X3 = DM(1)*I + DM(4)*J, no FMA), and the eight corners use the same
// integer rules, so the voxels read are bit-identical to the reference.
__device__ inline cf ainterpo_dev(int nsam, const float2* __restrict__ a3df, const float* d, int i,
                                  int j) {
  const int jc = nsam / 2 + 1;
  float x, y, z;
  int ls, lt, ms, mt, ns, nt;
  bool neg;
  {
#pragma clang fp contract(off)
    float fi = (float)i, fj = (float)j;
    float xx = d[0] * fi + d[3] * fj;
    float yy = d[1] * fi + d[4] * fj;
    float zz = d[2] * fi + d[5] * fj;
    neg = xx < 0.0f;
    x = neg ? -xx : xx;
    y = neg ? -yy : yy;
    z = neg ? -zz : zz;
  }
  ls = (int)x;
  lt = ls + 1;
  if (lt >= jc) lt = jc - 1;
  ms = (int)y;
  mt = ms + 1;
  if (y < 0.0f) { ms--; mt--; }
  if (ms <= -jc) ms = -jc + 1;
  if (mt >= jc) mt = jc - 1;
  ns = (int)z;
  nt = ns + 1;
  if (z < 0.0f) { ns--; nt--; }
  if (ns <= -jc) ns = -jc + 1;
  if (nt >= jc) nt = jc - 1;
  // Guards beyond the reference's clamps: they only act where the reference
  // itself would index outside the half-volume (|coordinate| >= JC, possible
  // for |AMAG| < 1 or non-finite input), so in-range results are unchanged.
  ls = min(max(ls, 0), jc - 1);
  lt = min(max(lt, 0), jc - 1);
  ms = min(max(ms, -jc + 1), jc - 1);
  mt = min(max(mt, -jc + 1), jc - 1);
  ns = min(max(ns, -jc + 1), jc - 1);
  nt = min(max(nt, -jc + 1), jc - 1);
  const float ax0 = 1.0f - fabsf(x - (float)ls), ax1 = 1.0f - fabsf(x - (float)lt);
  const float ay0 = 1.0f - fabsf(y - (float)ms), ay1 = 1.0f - fabsf(y - (float)mt);
  const float az0 = 1.0f - fabsf(z - (float)ns), az1 = 1.0f - fabsf(z - (float)nt);
  const size_t my0 = (size_t)jc * wrapn(ms, nsam), my1 = (size_t)jc * wrapn(mt, nsam);
  const size_t nz0 = (size_t)jc * nsam * wrapn(ns, nsam), nz1 = (size_t)jc * nsam * wrapn(nt, nsam);
  // LS and LT are neighbours (or the same point at JC-1): one 16-byte load
  // takes both from the pair that starts at min(LS, JC-2)
  const int lb = min(ls, jc - 2);
  const bool sl = ls != lb, tl = lt != lb;
  auto pair = [&](size_t row, float2& s0, float2& t0) {
    const PointPair v = *reinterpret_cast<const PointPair*>(a3df + row + lb);
    s0 = sl ? make_float2(v[2], v[3]) : make_float2(v[0], v[1]);
    t0 = tl ? make_float2(v[2], v[3]) : make_float2(v[0], v[1]);
  };
  float2 c000, c100, c010, c110, c001, c101, c011, c111;
  pair(my0 + nz0, c000, c100);
  pair(my1 + nz0, c010, c110);
  pair(my0 + nz1, c001, c101);
  pair(my1 + nz1, c011, c111);
  float w000 = ax0 * ay0 * az0, w100 = ax1 * ay0 * az0, w010 = ax0 * ay1 * az0, w110 = ax1 * ay1 * az0;
  float w001 = ax0 * ay0 * az1, w101 = ax1 * ay0 * az1, w011 = ax0 * ay1 * az1, w111 = ax1 * ay1 * az1;
  float re = c000.x * w000 + c100.x * w100 + c010.x * w010 + c110.x * w110 + c001.x * w001 +
             c101.x * w101 + c011.x * w011 + c111.x * w111;
  float im = c000.y * w000 + c100.y * w100 + c010.y * w010 + c110.y * w110 + c001.y * w001 +
             c101.y * w101 + c011.y * w011 + c111.y * w111;
  return neg ? cf{re, -im} : cf{re, im};
}

// ainterpo_dev where every coordinate of the plane's points keeps below JC - 1
// in size, so that no clamp acts: the same voxels and the same sums with 24-bit
// index products (JC NSAM < 2^24) and no selects.
__device__ inline cf ainterpo_inner_dev(int nsam, int jc, const float2* __restrict__ a3df,
                                        const float* d, int i, int j) {
  float x, y, z;
  bool neg;
  {
#pragma clang fp contract(off)
    float fi = (float)i, fj = (float)j;
    float xx = d[0] * fi + d[3] * fj;
    float yy = d[1] * fi + d[4] * fj;
    float zz = d[2] * fi + d[5] * fj;
    neg = xx < 0.0f;
    x = neg ? -xx : xx;
    y = neg ? -yy : yy;
    z = neg ? -zz : zz;
  }
  const int ls = (int)x;
  int ms = (int)y, ns = (int)z;
  if (y < 0.0f) ms--;
  if (z < 0.0f) ns--;
  const float fl = (float)ls, fm = (float)ms, fn = (float)ns;
  const float ax0 = 1.0f - fabsf(x - fl), ax1 = 1.0f - fabsf(x - (fl + 1.0f));
  const float ay0 = 1.0f - fabsf(y - fm), ay1 = 1.0f - fabsf(y - (fm + 1.0f));
  const float az0 = 1.0f - fabsf(z - fn), az1 = 1.0f - fabsf(z - (fn + 1.0f));
  const unsigned my0 = __umul24(jc, wrapn(ms, nsam)), my1 = __umul24(jc, wrapn(ms + 1, nsam));
  const unsigned plane = __umul24(jc, nsam);
  const unsigned nz0 = __umul24(plane, wrapn(ns, nsam)) + ls,
                 nz1 = __umul24(plane, wrapn(ns + 1, nsam)) + ls;
  const PointPair c00 = *reinterpret_cast<const PointPair*>(a3df + (my0 + nz0));
  const PointPair c10 = *reinterpret_cast<const PointPair*>(a3df + (my1 + nz0));
  const PointPair c01 = *reinterpret_cast<const PointPair*>(a3df + (my0 + nz1));
  const PointPair c11 = *reinterpret_cast<const PointPair*>(a3df + (my1 + nz1));
  float w000 = ax0 * ay0 * az0, w100 = ax1 * ay0 * az0, w010 = ax0 * ay1 * az0, w110 = ax1 * ay1 * az0;
  float w001 = ax0 * ay0 * az1, w101 = ax1 * ay0 * az1, w011 = ax0 * ay1 * az1, w111 = ax1 * ay1 * az1;
  float re = c00[0] * w000 + c00[2] * w100 + c10[0] * w010 + c10[2] * w110 + c01[0] * w001 +
             c01[2] * w101 + c11[0] * w011 + c11[2] * w111;
  float im = c00[1] * w000 + c00[3] * w100 + c10[1] * w010 + c10[3] * w110 + c01[1] * w001 +
             c01[3] * w101 + c11[1] * w011 + c11[3] * w111;
  return neg ? cf{re, -im} : cf{re, im};
}

// Whether ainterpo_inner_dev serves the points (I, J), I*I + J*J <= R*R, of the
// plane d: |coordinate| <= R sqrt(d_k^2 + d_{3+k}^2) on axis k.
__device__ inline bool ainterpo_inner(int jc, const float* d, int r) {
  const float lim = (float)(jc - 2) / (float)r, l2 = lim > 0.f ? lim * lim * 0.9999f : -1.f;
  return d[0] * d[0] + d[3] * d[3] < l2 && d[1] * d[1] + d[4] * d[4] < l2 &&
         d[2] * d[2] + d[5] * d[5] < l2;
}

}  // namespace fr
