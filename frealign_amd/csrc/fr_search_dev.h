// fr_search_dev.h -- device code shared by the searches with separable shifts.
#pragma once
#include <hip/hip_runtime.h>

namespace fr {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

// Wave-wide maximum and sum through DPP row operations (fixed order), the
// result read from lane 63: a uniform value.
template <int kCtrl, int kRowMask>
__device__ inline float dpp_f(float old, float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), kCtrl,
                                                    kRowMask, 0xF, false));
}

__device__ inline float wave_max(float v) {
  const float lo = -3.4e38f;
  v = fmaxf(v, dpp_f<0xB1, 0xF>(lo, v));   // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp_f<0x4E, 0xF>(lo, v));   // quad_perm [2,3,0,1]
  v = fmaxf(v, dpp_f<0x141, 0xF>(lo, v));  // row_half_mirror
  v = fmaxf(v, dpp_f<0x140, 0xF>(lo, v));  // row_mirror
  v = fmaxf(v, dpp_f<0x142, 0xA>(lo, v));  // row_bcast15
  v = fmaxf(v, dpp_f<0x143, 0xC>(lo, v));  // row_bcast31
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ inline float wave_sum(float v) {
  v += dpp_f<0xB1, 0xF>(0.f, v);
  v += dpp_f<0x4E, 0xF>(0.f, v);
  v += dpp_f<0x141, 0xF>(0.f, v);
  v += dpp_f<0x140, 0xF>(0.f, v);
  v += dpp_f<0x142, 0xA>(0.f, v);
  v += dpp_f<0x143, 0xC>(0.f, v);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// cos and sin of 2 pi (a mod n) / n: the argument reduced exactly first
__device__ inline void phase(int a, int n, float& c, float& s) {
  int r = a % n;
  if (r < 0) r += n;
  sincosf(6.283185307179586f * (float)r / (float)n, &s, &c);
}

// The peak of one (particle, template) pair's map (ccp.f:229-251): lane (g, n)
// holds map[sx = 4 g + i][sy = n].  The argmax over the inner 13 x 13, x outer,
// first maximum: the maximum value across the wave, then the first (sx, sy)
// holding it from the lanes' ballots (of the lanes of one i, the lowest has the
// smallest sx and then the smallest sy); the 3 x 3 box sum around it by lane
// reads.  Uniform results; m is the maximum.
__device__ __forceinline__ void ccp_peak(const floatx4& map, int g, int n, float& box, int& row,
                                         float& m) {
  bool ok[4];
  m = -3.4e38f;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int sx = 4 * g + i;
    ok[i] = sx >= 1 && sx <= 13 && n >= 1 && n <= 13;
    if (ok[i]) m = fmaxf(m, map[i]);
  }
  m = wave_max(m);
  int key = 15 * 16;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const unsigned long long hit = __ballot(ok[i] && map[i] == m);
    const int b = __builtin_ctzll(hit | 1ull << 63);
    const int k = (4 * (b >> 4) + i) * 16 + (b & 15);
    if (hit && k < key) key = k;
  }
  if (key == 15 * 16) key = 7 * 16 + 7;  // no ordered value (NaN map): the centre
  const int bx = key >> 4, by = key & 15;
  box = 0.f;
#pragma unroll
  for (int dx = -1; dx <= 1; dx++) {
    const int sxn = bx + dx, ii = sxn & 3;
    const float v = ii == 0 ? map[0] : ii == 1 ? map[1] : ii == 2 ? map[2] : map[3];
#pragma unroll
    for (int dy = -1; dy <= 1; dy++)
      box += __int_as_float(
          __builtin_amdgcn_readlane(__float_as_int(v), (sxn >> 2) * 16 + by + dy));
  }
  row = bx * 15 + by;
}

// ccp.f:252 with nacc = sum |c T|^2, s2 = sum |X|^2.  A wave takes its pairs'
// scores 64 at a time, a lane each: the square root and the divisions cost more
// instructions than the search of the peak (with the lane reads above, the BF16
// search of 128 particles x 46,800 templates: 6.20 -> 5.55 ms).
__device__ __forceinline__ float ccp_score(float box, float nacc, float s2) {
  return (nacc > 0.f && s2 > 0.f) ? box / sqrtf(nacc) / sqrtf(s2) / 9.0f : -3.0e38f;
}

}  // namespace fr
