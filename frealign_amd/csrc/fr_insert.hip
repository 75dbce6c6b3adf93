// fr_insert.hip -- CTF-weighted trilinear Fourier insertion, scattered per voxel
// tile in LDS.
//
// Replaces PINSERT_TRILIN (pinsert_trilin.f:8-244) as driven by PINSERT
// (pinsert.f:8-195) for a buffer of particles, the A3D3/A3D3_S flush
// (a3d3.f:107-143).  A task is (particle, symmetry copy); its plane points
// are the (I,J) of the full central plane with I^2+J^2 <= IRREC^2, at
// X3 = DM*(I,J), each adding to the voxels L in [max(0,FLOOR(X3)),
// min(NSAM/2,FLOOR(X3+1))] (and likewise M, N within +-NSAM/2) with the
// trilinear weight (1-|X3-L|)(1-|Y3-M|)(1-|Z3-N|).
//
// A workgroup owns one 8x8x8 tile of one half-map.  It lists, in task order,
// the half's tasks whose plane passes within reach of the tile; its four waves
// take a contiguous quarter of the list each.  A wave takes two tasks at a
// time, 32 lanes each: the lanes bound the J of 32 rows I against the tile
// grown by the trilinear reach (a form linear in I), a prefix sum packs the
// rows, and the points go through 32 at a time, a lane a point: its FP32
// coordinates and voxel range in the reference's operation order (no FMA
// contraction), eight corners added to sums in LDS.  A point near a tile's face
// is visited by the neighbouring tiles too; corners outside the tile are
// left out.
//
// The sums are plain reads and writes: LDS float atomics take about 100 cycles
// a wave here (measured: 4.4 of 5.1 ms).  No two lanes may then meet in a voxel
// in one instruction.  Each 32 lanes have sums of their own, and take the
// plane's points by classes (I mod q, J mod q): q steps of the plane's axes are
// longer than a cell's diagonal sqrt(3) (q = 2 unless AMAG > 1.15), so the
// points of a class lie in different cells, and a wave's LDS accesses complete
// in program order.  The eight sums of a voxel are added in a fixed order at the
// end: reruns give the same bits, NKSUM and TTD likewise.  No global atomics.
// Tiles near the origin, which every plane crosses, are dispatched first so
// that they do not trail the launch.  The per-point terms (sample x phase ramp
// x CTF x weight, and CTF^2 x weight) depend only on the particle, so they are
// formed once per particle, J innermost.
//
// What bounds it: the vector units (about 300 instructions per 64 lanes' points,
// near half of them filled) and the latency of a point's eight dependent LDS
// updates; the sums' 48 KB let three workgroups share a CU.  The gather that this
// replaces gave each voxel a thread, which tested every point that could reach it,
// most of them in vain: 64 particles x 14 copies at 256^3 3,790 us, now 1,456;
// 300 particles in C1 at 150^3 1,150 us, now 310.
//
// The _SE variant (PINSERT_TRILIN_SE with NNSTAT = 1,
// pinsert_trilin_se.f:186-194) also sums, per voxel, the count, |term|^2,
// |term| and the phase difference to the reference transform of the terms it
// receives, over both halves: a second launch of the same form, whose sums are
// these and whose lists hold both halves' tasks.  A point's eight terms are its
// sample times real weights, so their size and phase are formed once, and the
// reference's phases once per tile.  In one launch with the sums, both took
// 112 KB, one workgroup a CU: 4 particles at 256^3 450 us, 64 particles 1,458,
// 300 at 150^3 1,296; now 224, 711 and 650 (as the gather 237, 711 and 1,534).
#include <hip/hip_runtime.h>

#include <math.h>

#include <type_traits>

#include "fr_common.h"
#include "fr_kernels.h"

namespace fr {

namespace {

constexpr int kThreads = 256;
constexpr int kTile = 8;  // voxels per tile edge
constexpr int kVox = kTile * kTile * kTile;
constexpr int kWaves = 4;        // per tile
constexpr int kSets = 2;         // tasks a wave takes at a time, each with sums of its own
constexpr int kLanes = 64 / kSets;
constexpr int kSplit = 8;        // shorter task lists are split by classes
constexpr int kList = kThreads;  // tasks tested per pass
constexpr int kReduceThreads = 1024;
static_assert(kThreads == 64 * kWaves && kSets == 2, "32 lanes per set of sums");

// Per task, in the order half 0 then half 1 (task order within a half):
//   [0] d0 d1 d2 d3   [1] d4 d5 IRREC^2 part
//   [2] h1 (I = h1 . P for P on the plane), ilo | ihi << 16
//   [3] h2 (J = h2 . P), bit k: |b_k| too small for 1/b_k (axis k bounds no J)
//   [4] 1/b per axis, classes per axis   [5] a_k / b_k per axis (0 where b_k ~ 0)
constexpr int kRec = 6;

__host__ __device__ inline size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

struct Scratch {
  int* first;        // [nb] first task of each particle (or -1)
  int* ord;          // [ntask] tasks by half
  int* n0;           // tasks of half 0
  float4* hit;       // [ntask] plane normal, squared reach (below 0: no plane)
  float4* rec;       // [ntask][kRec]
  float4* pts;       // [nb][w*w] (samp.re, samp.im, ctfv2, 0), J innermost
  unsigned long long* pcount;  // [ntiles][2]
  double* pttd;      // [ntiles][2]
  size_t bytes;
};

Scratch scratch_layout(void* base, int nsam, int nb, int ntask, int ntiles) {
  const int jc = nsam / 2 + 1, w = 2 * jc - 1;
  char* p = static_cast<char*>(base);
  Scratch s;
  size_t o = 0;
  auto take = [&](auto*& q, size_t n) {
    q = reinterpret_cast<std::remove_reference_t<decltype(q)>>(p + o);
    o += align256(sizeof(*q) * n);
  };
  take(s.first, (size_t)nb);
  take(s.ord, (size_t)ntask);
  take(s.n0, 1);
  take(s.hit, (size_t)ntask);
  take(s.rec, (size_t)ntask * kRec);
  take(s.pts, (size_t)nb * w * w);
  take(s.pcount, 2 * (size_t)ntiles);
  take(s.pttd, 2 * (size_t)ntiles);
  s.bytes = o;
  return s;
}

void tile_counts(int nsam, int* tx, int* ty, int* tz) {
  const int jc = nsam / 2 + 1;
  *tx = (jc + kTile - 1) / kTile;
  *ty = (nsam + kTile - 1) / kTile;
  *tz = (nsam + kTile - 1) / kTile;
}

// One workgroup: the tasks of half 0 and then those of half 1, each in task
// order, and the first task of each run of tasks of one particle (tasks come
// grouped by particle; a particle's copies share its shift, weight and radius)
__global__ void __launch_bounds__(1024)
    k_insert_order(int ntask, int nb, const InsertTask* __restrict__ tasks, int* first, int* ord,
                   int* n0) {
  __shared__ int tot[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int p = tid; p < nb; p += 1024) first[p] = -1;
  int mine = 0;
  for (int k = tid; k < ntask; k += 1024) mine += tasks[k].half ? 0 : 1;
  for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off, 64);
  if (lane == 0) tot[wave] = mine;
  __syncthreads();
  int zeros = 0;
  for (int q = 0; q < 16; q++) zeros += tot[q];
  if (tid == 0) *n0 = zeros;
  int seen0 = 0;  // tasks of half 0 before this pass
  for (int base = 0; base < ntask; base += 1024) {
    const int k = base + tid;
    const bool in = k < ntask;
    const bool h0 = in && !tasks[k].half;
    if (in) {
      const int part = tasks[k].part;
      if (part >= 0 && part < nb && (k == 0 || tasks[k - 1].part != part)) first[part] = k;
    }
    const unsigned long long bal = __ballot(h0);
    __syncthreads();
    if (lane == 0) tot[wave] = __popcll(bal);
    __syncthreads();
    int before = seen0 + __popcll(bal & ((1ull << lane) - 1ull));
    for (int q = 0; q < 16; q++) {
      if (q < wave) before += tot[q];
      seen0 += tot[q];
    }
    if (in) ord[h0 ? before : zeros + k - before] = k;
  }
}

// pinsert_trilin.f:60-87: the weighted sample and CTF^2 of every plane point
// of a particle, exactly as the reference's scatter forms them; a workgroup
// takes 16 x 16 points, read with I innermost and written with J innermost
__global__ void __launch_bounds__(kThreads)
    k_insert_points(int nsam, const int* __restrict__ first,
                    const InsertTask* __restrict__ tasks, const float2* __restrict__ datc,
                    const float2* __restrict__ ctff, float4* pts) {
  __shared__ float4 turn[16][17];
  const int b = blockIdx.y;
  const int k = first[b];
  if (k < 0) return;
  const InsertTask t = tasks[k];
  const int jc = nsam / 2 + 1, w = 2 * jc - 1, nt = (w + 15) / 16;
  const size_t ic = (size_t)nsam * jc;
  const int bi = (blockIdx.x % nt) * 16, bj = (blockIdx.x / nt) * 16;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int i = bi + tx - (jc - 1);
  const int j = bj + ty - (jc - 1);
  float4 out = make_float4(0.f, 0.f, 0.f, 0.f);
  float g2;
  bool inside;
  {
#pragma clang fp contract(off)
    g2 = (float)(i * i + j * j);
    inside = g2 <= (float)t.irrec2 && i < jc && j < jc;
  }
  if (inside) {
    const float2* sp = datc + (size_t)t.part * ic;
    const float2* cp = ctff + (size_t)t.part * 2 * ic;
    size_t id;
    bool mate = i < 0;
    if (!mate) id = (size_t)i + (size_t)jc * wrapn(j, nsam);
    else id = (size_t)(-i) + (size_t)jc * wrapn(-j, nsam);
    float2 s = sp[id];
    if (mate) s.y = -s.y;
    float2 cr = cp[id], cl = cp[id + ic];
    cf ctfs = cf{cr.x + cl.x, cr.y - cl.y};  // CTFR + CONJG(CTFL)
    float phase = t.shx * (float)i + t.shy * (float)j;
    float sn, cs;
    sincosf(phase, &sn, &cs);
    float wgt = expf(t.tmp * g2) * t.occ;
    cf samp = cmul(cmul(cf{s.x, s.y}, cf{cs, sn}), ctfs);
    float ctfv2 = 0.25f * (ctfs.re * ctfs.re + ctfs.im * ctfs.im) * wgt;
    samp = cscale(samp, wgt);
    out = make_float4(samp.re, samp.im, ctfv2, 0.f);
  }
  turn[tx][ty] = out;
  __syncthreads();
  const int oi = bi + ty, oj = bj + tx;
  if (oi < w && oj < w) pts[(size_t)b * w * w + (size_t)oi * w + oj] = turn[ty][tx];
}

// per-task plane geometry for the candidate search (double, then rounded; the
// margins of the search cover the rounding)
__global__ void __launch_bounds__(kThreads)
    k_insert_geo(int ntask, int nb, int nsam, const InsertTask* __restrict__ tasks,
                 const int* __restrict__ ord, float4* hit, float4* rec) {
  const int q = blockIdx.x * kThreads + threadIdx.x;
  if (q >= ntask) return;
  const InsertTask t = tasks[ord[q]];
  const double ax = t.dm[0], ay = t.dm[1], az = t.dm[2];
  const double bx = t.dm[3], by = t.dm[4], bz = t.dm[5];
  const double nx = ay * bz - az * by, ny = az * bx - ax * bz, nz = ax * by - ay * bx;
  const double aa = ax * ax + ay * ay + az * az, bb = bx * bx + by * by + bz * bz;
  const double ab = ax * bx + ay * by + az * bz;
  const double det = aa * bb - ab * ab;
  const bool valid = t.irrec2 >= 0 && det > 1e-12 && t.part >= 0 && t.part < nb;
  const double id = valid ? 1.0 / det : 0.0;
  // points reach |P| <= sqrt(IRREC^2 * lambda_max(G)) within the square
  // |I|,|J| <= NSAM/2; a voxel they touch lies within sqrt(3) more
  const double lmax = 0.5 * (aa + bb + sqrt((aa - bb) * (aa - bb) + 4.0 * ab * ab));
  const double jcm = (double)(nsam / 2);
  const double r2pts = t.irrec2 < 2.0 * jcm * jcm ? (double)t.irrec2 : 2.0 * jcm * jcm;
  const double reach = sqrt(r2pts * lmax) + 1.7320508 + 0.01;
  // classes of points: q steps of the plane's lattice span more than a cell's
  // diagonal (distances are at least the square root of G's smaller eigenvalue)
  const double lmin = fmax(aa + bb - lmax, 0.0);
  const int q2 = valid ? (int)fmin(fmax(ceil(1.7322 / sqrt(lmin)), 2.0), 2.0 * jcm + 1.0) : 2;
  hit[q] = make_float4((float)nx, (float)ny, (float)nz, valid ? (float)(reach * reach) : -1.f);
  const bool zx = !(fabs(bx) > 1e-6), zy = !(fabs(by) > 1e-6), zz = !(fabs(bz) > 1e-6);
  float4* r = rec + (size_t)q * kRec;
  r[0] = make_float4(t.dm[0], t.dm[1], t.dm[2], t.dm[3]);
  r[1] = make_float4(t.dm[4], t.dm[5], __int_as_float(t.irrec2), __int_as_float(t.part));
  r[2] = make_float4((float)((bb * ax - ab * bx) * id), (float)((bb * ay - ab * by) * id),
                     (float)((bb * az - ab * bz) * id),
                     __int_as_float((int)(unsigned short)t.ilo | (int)t.ihi << 16));
  r[3] = make_float4((float)((aa * bx - ab * ax) * id), (float)((aa * by - ab * ay) * id),
                     (float)((aa * bz - ab * az) * id),
                     __int_as_float((zx ? 1 : 0) | (zy ? 2 : 0) | (zz ? 4 : 0)));
  r[4] = make_float4(zx ? 0.f : (float)(1.0 / bx), zy ? 0.f : (float)(1.0 / by),
                     zz ? 0.f : (float)(1.0 / bz), __int_as_float(q2));
  r[5] = make_float4(zx ? 0.f : (float)(ax / bx), zy ? 0.f : (float)(ay / by),
                     zz ? 0.f : (float)(az / bz), 0.f);
}

// logical intervals covered by the storage range [s0, s1] of a wrapped axis
__device__ inline int logical_ranges(int s0, int s1, int nsam, int* lo, int* hi) {
  const int h = nsam / 2;
  int n = 0;
  if (s0 <= h) {  // the non-negative part s0 .. min(s1, h)
    lo[n] = s0;
    hi[n] = s1 < h ? s1 : h;
    n++;
  }
  if (s1 >= h) {  // the negative part max(s0, h) - nsam .. s1 - nsam
    lo[n] = (s0 > h ? s0 : h) - nsam;
    hi[n] = s1 - nsam;
    n++;
  }
  return n;
}

// does the plane through the origin with normal g.xyz reach the box [lo, hi]
// grown by one voxel (the trilinear reach), within the plane's disc?
__device__ inline bool plane_reaches(const float4& g, float xl, float xh, float yl, float yh,
                                     float zl, float zh) {
  xl -= 1.01f; yl -= 1.01f; zl -= 1.01f;
  xh += 1.01f; yh += 1.01f; zh += 1.01f;
  const float mn = (g.x > 0.f ? g.x * xl : g.x * xh) + (g.y > 0.f ? g.y * yl : g.y * yh) +
                   (g.z > 0.f ? g.z * zl : g.z * zh);
  const float mx = (g.x > 0.f ? g.x * xh : g.x * xl) + (g.y > 0.f ? g.y * yh : g.y * yl) +
                   (g.z > 0.f ? g.z * zh : g.z * zl);
  const float slack = 1e-3f * (fabsf(g.x) + fabsf(g.y) + fabsf(g.z)) + 1e-3f;
  if (mn > slack || mx < -slack) return false;
  // nearest point of the box to the origin
  const float cx = xl > 0.f ? xl : (xh < 0.f ? xh : 0.f);
  const float cy = yl > 0.f ? yl : (yh < 0.f ? yh : 0.f);
  const float cz = zl > 0.f ? zl : (zh < 0.f ? zh : 0.f);
  return cx * cx + cy * cy + cz * cz <= g.w;
}

// Phases as whole turns times 2^32, whose differences wrap by themselves: exact
// octants and the arctangent of a ratio up to 1, scaled in 64 bits.  Against 64
// bits a difference is 4.0e-8 radians off (rms of 2e7, most 2.1e-7), as the
// arctangent of the product formed in FP32 is (4.0e-8, 2.9e-7).
__device__ inline unsigned turns(float x, float y) {
  const float ax = fabsf(x), ay = fabsf(y), mx = fmaxf(ax, ay);
  const double a = atanf(mx > 0.f ? fminf(ax, ay) / mx : 0.f);
  unsigned u = (unsigned)(a * 683565275.57643158 + 0.5);  // 2^32 / 2 pi
  if (ay > ax) u = (1u << 30) - u;
  if (x < 0.f) u = (1u << 31) - u;
  return y < 0.f ? 0u - u : u;
}

// A voxel's reference phase, odd; kNoPhase where the value is zero (pdiff.f:8-24:
// no difference), kBadPhase where it is no number
constexpr unsigned kNoPhase = 0u, kBadPhase = 2u;
__device__ inline unsigned ref_phase(float2 r) {
  if (!(fabsf(r.x) <= 3.4e38f && fabsf(r.y) <= 3.4e38f)) return kBadPhase;
  return r.x == 0.f && r.y == 0.f ? kNoPhase : turns(r.x, r.y) | 1u;
}

// pdiff.f:8-24: |phase of b conj(r)| of a term of size ab and phase p
__device__ inline float pdiff_dev(float ab, unsigned p, unsigned ref) {
  if (ref == kBadPhase) return __int_as_float(0x7fc00000);
  const int d = (int)(p - ref);
  const unsigned m = d < 0 ? 0u - (unsigned)d : (unsigned)d;
  const float v = (float)((double)m * 1.4629180792671596e-9);  // 2 pi / 2^32
  return ab == 0.f || ref == kNoPhase ? 0.f : v + (ab - ab);
}

// inclusive prefix sum over each 32 lanes, on the vector ALU
template <int kCtrl, int kRows>
__device__ inline int dpp_acc(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, kCtrl, kRows, 0xf, false);
}
__device__ inline int half_scan(int v) {
  v = dpp_acc<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8 within 16 lanes
  v = dpp_acc<0x112, 0xf>(v);
  v = dpp_acc<0x114, 0xf>(v);
  v = dpp_acc<0x118, 0xf>(v);
  return dpp_acc<0x142, 0xa>(v);  // row_bcast 15 into the odd rows
}

// LDS written by some lanes of a wave and read by others: the wave's own
// accesses complete in order, so only the compiler has to be held
__device__ inline void wave_lds() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

struct Sum {
  float re, im, c2;  // numerator, CTF^2
  __device__ void add(const Sum& o) {
    re += o.re;
    im += o.im;
    c2 += o.c2;
  }
};
constexpr int kOut = 1 << 20;             // byte offset of a corner outside the tile

// pinsert_trilin.f:88-111 on one axis: the voxels S..T of a point (S = INT(A1),
// minus 1 for A1 < 0, with A1 = (X + 0.5) - 0.5; T likewise with A2 = X + 1);
// those outside the tile's [lo, hi], which lies within the reference's clamps,
// are left out.  T - S is 0, 1 or (at negative integers) 2.
struct Axis {
  int s, t;
  __device__ Axis(float x) {
#pragma clang fp contract(off)
    const float a1 = (x + 0.5f) - 0.5f, a2 = x + 1.0f;
    s = (int)a1;
    if (a1 < 0.0f) s--;
    t = (int)a2;
    if (a2 < 0.0f) t--;
  }
  // byte offset of voxel s + k of an axis whose tile holds lo .. lo + n from
  // offset `at` on, or kOut
  __device__ int off(int k, int lo, int n, int at, int mul) const {
    const int v = s + k - lo;
    return (unsigned)v <= (unsigned)n && (k == 0 || s + k <= t) ? v * mul + at : kOut;
  }
};

// the _SE statistics of a voxel
struct StatSum {
  float v, a, p;  // |term|^2, |term|, phase difference
  int n;
  __device__ void add(const StatSum& o) {
    v += o.v;
    a += o.a;
    p += o.p;
    n += o.n;
  }
};

template <bool kStats>
struct TileSums {
  using Acc = std::conditional_t<kStats, StatSum, Sum>;
  Acc sum[kWaves][kSets * kVox];
  unsigned ref[kStats ? kVox : 1];     // the reference transform's phases in the tile
  int list[kList];
  int tot[kWaves];
  int2 row[kWaves][kSets][kLanes];     // I | first J << 16, start
  unsigned flag[kWaves][kSets][8];     // a bit where a row starts
  unsigned live[kWaves];
  unsigned long long rc[kWaves];
  double rt[kWaves];
};

// kStats: the statistics of the terms, both halves' together, instead of their sums
template <bool kStats>
__global__ void __launch_bounds__(kThreads)
    k_insert_scatter(int nsam, int ntask, int tx, int ty, int tz, const int* __restrict__ n0p,
                     const float4* __restrict__ hit, const float4* __restrict__ rec,
                     const float4* __restrict__ pts, float2* num0, float* ctf2_0, float2* num1,
                     float* ctf2_1, unsigned long long* pcount, double* pttd, InsertStats st) {
  extern __shared__ __attribute__((aligned(16))) char lds_raw[];
  using Acc = typename TileSums<kStats>::Acc;
  TileSums<kStats>& S = *reinterpret_cast<TileSums<kStats>*>(lds_raw);
  const int jc = nsam / 2 + 1, h = nsam / 2, w = 2 * jc - 1;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // a tile's two halves are neighbouring workgroups (one workgroup for statistics)
  const int b = kStats ? blockIdx.x : blockIdx.x >> 1;
  const int half = kStats ? 0 : blockIdx.x & 1;
  // no term in the tile: the sums' launch has counted them
  if (kStats && (pcount[2 * (size_t)b] | pcount[2 * (size_t)b + 1]) == 0) return;
  // tiles go out slab by slab in order of |logical n|, rows in order of
  // |logical m| (storage rows 0, last, 1, last - 1, ...): the tiles near the
  // origin, which every plane crosses, start first instead of last
  const int tmf = (b / tx) % ty, tnf = b / (tx * ty);
  const int l0 = (b % tx) * kTile;
  const int m0 = ((tmf & 1) ? ty - 1 - (tmf >> 1) : (tmf >> 1)) * kTile;
  const int n0 = ((tnf & 1) ? tz - 1 - (tnf >> 1) : (tnf >> 1)) * kTile;
  const int l1 = min(l0 + kTile - 1, jc - 1);
  // the tile's logical boxes (a wrapped axis may split in two)
  int mlo[2], mhi[2], nlo[2], nhi[2];
  const int nmr = logical_ranges(m0, min(m0 + kTile - 1, nsam - 1), nsam, mlo, mhi);
  const int nnr = logical_ranges(n0, min(n0 + kTile - 1, nsam - 1), nsam, nlo, nhi);
  unsigned live = 0u;  // this wave's sets that are set up, a bit each
  bool any = false;    // a plane reaches the tile
  const int rl = lane & (kLanes - 1), slot = lane / kLanes;
  const unsigned long long lt = (1ull << lane) - 1ull;
  char* const set = reinterpret_cast<char*>(&S.sum[wave][slot * kVox]);

  {
    const int k0 = half ? *n0p : 0, k1 = half || kStats ? ntask : *n0p;
    unsigned cnt = 0u;
    unsigned long long cnt64 = 0ull;
    double ttd = 0.0;
    for (int box = 0; box < nmr * nnr; box++) {
      const int ml = mlo[box % nmr], mh = mhi[box % nmr];
      const int nl = nlo[box / nmr], nh = nhi[box / nmr];
      // where the box starts in the tile's sums, in bytes
      constexpr int kB = sizeof(Acc), kM = kTile * kB, kN = kTile * kM;
      const int ms = ((ml < 0 ? nsam : 0) - m0 + ml) * kM, ns = ((nl < 0 ? nsam : 0) - n0 + nl) * kN;
      const float cx = 0.5f * (float)(l0 + l1), hx = 0.5f * (float)(l1 - l0) + 1.02f;
      const float cy = 0.5f * (float)(ml + mh), hy = 0.5f * (float)(mh - ml) + 1.02f;
      const float cz = 0.5f * (float)(nl + nh), hz = 0.5f * (float)(nh - nl) + 1.02f;
      for (int base = k0; base < k1; base += kList) {
        // list the tasks reaching this box, in task order (ballot compaction)
        const int k = base + tid;
        bool on = false;
        if (k < k1) {
          const float4 g = hit[k];
          on = g.w >= 0.f && plane_reaches(g, (float)l0, (float)l1, (float)ml, (float)mh,
                                           (float)nl, (float)nh);
        }
        const unsigned long long bal = __ballot(on);
        __syncthreads();  // the previous list is no longer read
        if (lane == 0) S.tot[wave] = __popcll(bal);
        __syncthreads();
        int nlist = 0, before = 0;
        for (int q = 0; q < kWaves; q++) {
          if (q == wave) before = nlist;
          nlist += S.tot[q];
        }
        if (on) S.list[before + __popcll(bal & lt)] = k;
        __syncthreads();
        // This wave's quarter of the tasks, two at a time.  A short list is split by
        // the classes of its points instead, a class (of each four) to a wave: one
        // wave at work would leave a CU, which holds three tiles, nearly idle.
        const bool split = nlist < kSplit;
        const int q0 = split ? 0 : nlist * wave / kWaves;
        const int q1 = split ? nlist : nlist * (wave + 1) / kWaves;
        if constexpr (kStats)
          if (nlist && !any) {  // read per term they were most of a pass: 600 cycles each of eight
            for (int v = tid; v < kVox; v += kThreads) {
              const int l = l0 + (v & 7), m = m0 + (v >> 3 & 7), n = n0 + (v >> 6);
              if (l < jc && m < nsam && n < nsam)
                S.ref[v] = ref_phase(reinterpret_cast<const float2*>(
                    st.ref)[(size_t)l + (size_t)jc * ((size_t)m + (size_t)nsam * n)]);
            }
            __syncthreads();
          }
        any |= nlist != 0;
        if (!live && q0 < q1 && rl < 8) S.flag[wave][slot][rl] = 0u;
        for (int k = 0; k < min(q1 - q0, kSets); k++)
          if (!(live >> k & 1)) {
            live |= 1u << k;
            for (int e = lane; e < kVox; e += 64) S.sum[wave][k * kVox + e] = Acc{};
          }
        wave_lds();
        for (int qb = q0; qb < q1; qb += kSets) {
          const int q = qb + slot;
          const float4* R = rec + (size_t)S.list[min(q, q1 - 1)] * kRec;
          const float4 r0 = R[0], r1 = R[1], r2 = R[2], r3 = R[3], r4 = R[4], r5 = R[5];
          const float4* tp = pts + (size_t)__float_as_int(r1.w) * w * w;
          const int za = __float_as_int(r3.w), ir2 = __float_as_int(r1.z);
          // classes per axis: the most that either needs
          int nc = __float_as_int(r4.w);
          nc = __builtin_amdgcn_readfirstlane(max(nc, __shfl_xor(nc, 32, 64)));
          const float ci = r2.x * cx + r2.y * cy + r2.z * cz;
          const float cj = r3.x * cx + r3.y * cy + r3.z * cz;
          const float ri = fabsf(r2.x) * hx + fabsf(r2.y) * hy + fabsf(r2.z) * hz + 0.02f;
          const float rj = fabsf(r3.x) * hx + fabsf(r3.y) * hy + fabsf(r3.z) * hz + 0.02f;
          const float lim = (float)h;
          const int ilo = max((int)fminf(fmaxf(ceilf(ci - ri), -lim), lim + 1.f),
                              (int)(short)__float_as_int(r2.w));
          const int ihi = min((int)fminf(fmaxf(floorf(ci + ri), -lim - 1.f), lim),
                              __float_as_int(r2.w) >> 16);
          const float jlo = fmaxf(ceilf(cj - rj), -lim), jhi = fminf(floorf(cj + rj), lim);
          // per axis, J in (c_k - I a_k) / b_k -+ h_k / |b_k|
          const float ex = cx * r4.x, ey = cy * r4.y, ez = cz * r4.z;
          const float ox = za & 1 ? 3.0e38f : hx * fabsf(r4.x);
          const float oy = za & 2 ? 3.0e38f : hy * fabsf(r4.y);
          const float oz = za & 4 ? 3.0e38f : hz * fabsf(r4.z);
          const int nrow = q < q1 ? ihi - ilo + 1 : 0;
          for (int rb = 0; __any(rb < nrow); rb += kLanes) {
            const int i = ilo + rb + rl;
            const float fi = (float)i;
            int j0 = 0, j1 = -1;
            if (q < q1 && i <= ihi) {
              const float jx = ex - fi * r5.x, jy = ey - fi * r5.y, jz = ez - fi * r5.z;
              const float jl = fmaxf(fmaxf(jlo, jx - ox), fmaxf(jy - oy, jz - oz));
              const float jh = fminf(fminf(jhi, jx + ox), fminf(jy + oy, jz + oz));
              bool on = jl <= jh + 0.02f;
              if (za) {  // an axis with b_k ~ 0: the row is in reach or not
                const float slack = 1e-3f * (float)jc;
                if ((za & 1) && fabsf(cx - fi * r0.x) > hx + slack * fabsf(r0.w)) on = false;
                if ((za & 2) && fabsf(cy - fi * r0.y) > hy + slack * fabsf(r1.x)) on = false;
                if ((za & 4) && fabsf(cz - fi * r0.z) > hz + slack * fabsf(r1.y)) on = false;
              }
              if (on) {
                j0 = (int)fmaxf(ceilf(jl - 0.01f), jlo);
                j1 = (int)fminf(floorf(jh + 0.01f), jhi);
              }
            }
            const int imod = nc == 2 ? i & 1 : (i + nc * 1024) % nc;
            const int jmod = nc == 2 ? j0 & 1 : (j0 + nc * 1024) % nc;
            for (int cls = split ? wave : 0; cls < nc * nc; cls += split ? kWaves : 1) {
              const int ca = nc == 2 ? cls & 1 : cls % nc, cb = nc == 2 ? cls >> 1 : cls / nc;
              const int f0 = j0 + (cb >= jmod ? cb - jmod : cb - jmod + nc);
              int c = 0;
              if (imod == ca && f0 <= j1) c = nc == 2 ? ((j1 - f0) >> 1) + 1 : (j1 - f0) / nc + 1;
              // a class holds at most 16 of 32 rows: with 16 points of a row at a
              // time a pass holds at most 256
              for (int jb = 0; __any(jb < c); jb += 16) {
                const int cc = min(max(c - jb, 0), 16);
                const unsigned some = (unsigned)(__ballot(cc > 0) >> (slot * kLanes));
                const int end = half_scan(cc), start = end - cc;
                const int total = __shfl(end, slot * kLanes + kLanes - 1, 64);
                if (cc > 0) {
                  S.row[wave][slot][__popc(some & ((1u << rl) - 1u))] =
                      make_int2((i & 0xffff) | (f0 + jb * nc) << 16, start);
                  atomicOr(&S.flag[wave][slot][start >> 5], 1u << (start & 31));
                }
                wave_lds();
                int before = -1;  // rows started before these 32 points, less one
                for (int p0 = 0; __any(p0 < total); p0 += kLanes) {
                  const unsigned mask = S.flag[wave][slot][p0 / kLanes];
                  const int p = p0 + rl;
                  const int at = before + (int)__popc(mask & (~0u >> (31 - rl)));
                  const int2 rw = S.row[wave][slot][max(at, 0)];
                  before += (int)__popc(mask);
                  const bool on = p < total;
                  const int pi = on ? (short)rw.x : 0;
                  const int pj = on ? (rw.x >> 16) + (p - rw.y) * nc : 0;
                  const float4 pv = tp[__mul24(pi + h, w) + pj + h];
                  float x3, y3, z3;
                  {
#pragma clang fp contract(off)
                    const float fpi = (float)pi, fpj = (float)pj;
                    x3 = r0.x * fpi + r0.w * fpj;
                    y3 = r0.y * fpi + r1.x * fpj;
                    z3 = r0.z * fpi + r1.y * fpj;
                  }
                  const Axis X(x3), Y(y3), Z(z3);
                  const bool inside = on && pi * pi + pj * pj <= ir2;
                  // a point's terms are its sample times real weights: one size and
                  // one phase for the eight
                  float pab = 0.f;
                  unsigned pph = 0u;
                  if constexpr (kStats) {
                    pab = hypotf(pv.x, pv.y);
                    pph = turns(pv.x, pv.y);
                  }
                  // corner (kx, ky, kz) of every lane's point: pinsert_trilin.f:113-131,
                  // the weights' product in its order
                  auto corner = [&](int off, float bxy, float bz) {
                    const float box = bxy * bz;
                    if (off < kOut) {
                      Acc& t = *reinterpret_cast<Acc*>(set + off);
                      Acc u = t;
                      if constexpr (kStats) {
                        const float ab = pab * fabsf(box);  // a weight may round to -1e-7
                        u.v += ab * ab;
                        u.a += ab;
                        u.p += pdiff_dev(ab, pph + (__float_as_uint(box) & 1u << 31),
                                         S.ref[off / kB]);
                        u.n++;
                      } else {
                        u.re += pv.x * box;
                        u.im += pv.y * box;
                        u.c2 += pv.z * box;
                      }
                      t = u;
                    }
                    wave_lds();  // another lane's next corner may be this voxel
                  };
                  if (!__any(X.t - X.s > 1 || Y.t - Y.s > 1 || Z.t - Z.s > 1)) {
                    int ax[2], ay[2], az[2];
                    float wx[2], wy[2], wz[2];
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                      ax[k] = inside ? X.off(k, l0, l1 - l0, 0, kB) : kOut;
                      ay[k] = Y.off(k, ml, mh - ml, ms, kM);
                      az[k] = Z.off(k, nl, nh - nl, ns, kN);
                      wx[k] = 1.0f - fabsf(x3 - (float)(X.s + k));
                      wy[k] = 1.0f - fabsf(y3 - (float)(Y.s + k));
                      wz[k] = 1.0f - fabsf(z3 - (float)(Z.s + k));
                    }
                    // NKSUM; TTD's terms over the tile's corners, their weights
                    // added per axis in 64 bits
                    auto n2 = [](const int(&o)[2]) { return (o[0] < kOut) + (o[1] < kOut); };
                    auto w2 = [](const int(&o)[2], const float(&f)[2]) {
                      return (double)(o[0] < kOut ? f[0] : 0.f) +
                             (double)(o[1] < kOut ? f[1] : 0.f);
                    };
                    const int nv = n2(ax) * n2(ay) * n2(az);
                    cnt += nv;
                    if (nv) ttd += (double)pv.z * w2(ax, wx) * w2(ay, wy) * w2(az, wz);
#pragma unroll
                    for (int kz = 0; kz < 2; kz++)
#pragma unroll
                      for (int ky = 0; ky < 2; ky++)
#pragma unroll
                        for (int kx = 0; kx < 2; kx++)
                          corner(ax[kx] + ay[ky] + az[kz], wx[kx] * wy[ky], wz[kz]);
                  } else {  // negative integers: three voxels on an axis
                    for (int kz = 0; kz < 3; kz++)
                      for (int ky = 0; ky < 3; ky++)
                        for (int kx = 0; kx < 3; kx++) {
                          const int off = (inside ? X.off(kx, l0, l1 - l0, 0, kB) : kOut) +
                                          Y.off(ky, ml, mh - ml, ms, kM) +
                                          Z.off(kz, nl, nh - nl, ns, kN);
                          const float bx = 1.0f - fabsf(x3 - (float)(X.s + kx));
                          const float by = 1.0f - fabsf(y3 - (float)(Y.s + ky));
                          const float bz = 1.0f - fabsf(z3 - (float)(Z.s + kz));
                          if (off < kOut) {
                            cnt++;
                            ttd += (double)pv.z * (double)bx * (double)by * (double)bz;
                          }
                          corner(off, bx * by, bz);
                        }
                  }
                }
                wave_lds();
                if (rl < 8) S.flag[wave][slot][rl] = 0u;
                wave_lds();
              }
            }
          }
          cnt64 += cnt;
          cnt = 0u;
        }
      }
    }
    if (!any) {
      if (!kStats && tid == 0) {
        pcount[2 * (size_t)b + half] = 0;
        pttd[2 * (size_t)b + half] = 0.0;
      }
      return;
    }
    // the waves' sums in wave order, into the half-map or the statistics: every
    // set's value is read, those in use added, so that eight loads are in flight
    // instead of one after the other
    if (lane == 0) S.live[wave] = live;
    __syncthreads();
    unsigned use[kWaves];
#pragma unroll
    for (int q = 0; q < kWaves; q++) use[q] = S.live[q];
    for (int v = tid; v < kVox; v += kThreads) {
      const int l = l0 + (v & 7), m = m0 + (v >> 3 & 7), n = n0 + (v >> 6);
      const size_t at = (size_t)l + (size_t)jc * ((size_t)m + (size_t)nsam * n);
      Acc t{};
#pragma unroll
      for (int q = 0; q < kWaves; q++)
#pragma unroll
        for (int k = 0; k < kSets; k++) {
          const Acc u = S.sum[q][k * kVox + v];
          if (use[q] >> k & 1) t.add(u);
        }
      if (l >= jc || m >= nsam || n >= nsam) continue;
      if constexpr (kStats) {
        if (!t.n) continue;
        st.ksum[at] += t.n;
        st.vsum[at] += t.v;
        st.psum[at] += t.p;
        st.asum[at] += t.a;
      } else if (t.re != 0.f || t.im != 0.f || t.c2 != 0.f) {
        float2* num = half ? num1 : num0;
        float* ctf2 = half ? ctf2_1 : ctf2_0;
        const float2 o = num[at];
        num[at] = make_float2(o.x + t.re, o.y + t.im);
        ctf2[at] += t.c2;
      }
    }
    if (kStats) return;
    // the tile's NKSUM and TTD: a fixed reduction order
    for (int off = 32; off > 0; off >>= 1) {
      cnt64 += __shfl_xor(cnt64, off, 64);
      ttd += __shfl_xor(ttd, off, 64);
    }
    if (lane == 0) {
      S.rc[wave] = cnt64;
      S.rt[wave] = ttd;
    }
    __syncthreads();
    if (tid == 0) {
      unsigned long long uc = 0;
      double ut = 0.0;
      for (int q = 0; q < kWaves; q++) {
        uc += S.rc[q];
        ut += S.rt[q];
      }
      pcount[2 * (size_t)b + half] = uc;
      pttd[2 * (size_t)b + half] = ut;
    }
  }
}

// NKSUM and TTD of the launch: tiles summed in a fixed order
__global__ void __launch_bounds__(kReduceThreads)
    k_insert_reduce(int ntiles, const unsigned long long* __restrict__ pcount,
                    const double* __restrict__ pttd, unsigned long long* nksum, double* ttd) {
  __shared__ unsigned long long rc[kReduceThreads / 64][2];
  __shared__ double rt[kReduceThreads / 64][2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  unsigned long long u0 = 0, u1 = 0;
  double t0 = 0.0, t1 = 0.0;
  for (int b = tid; b < ntiles; b += kReduceThreads) {
    u0 += pcount[2 * (size_t)b];
    u1 += pcount[2 * (size_t)b + 1];
    t0 += pttd[2 * (size_t)b];
    t1 += pttd[2 * (size_t)b + 1];
  }
  for (int off = 32; off > 0; off >>= 1) {
    u0 += __shfl_xor(u0, off, 64);
    u1 += __shfl_xor(u1, off, 64);
    t0 += __shfl_xor(t0, off, 64);
    t1 += __shfl_xor(t1, off, 64);
  }
  if (lane == 0) {
    rc[wave][0] = u0;
    rc[wave][1] = u1;
    rt[wave][0] = t0;
    rt[wave][1] = t1;
  }
  __syncthreads();
  if (tid < 2) {
    unsigned long long cc = 0;
    double tt = 0.0;
    for (int q = 0; q < kReduceThreads / 64; q++) {
      cc += rc[q][tid];
      tt += rt[q][tid];
    }
    if (cc) {
      nksum[tid] += cc;
      ttd[tid] += tt;
    }
  }
}

}  // namespace

size_t insert_scratch_bytes(int nsam, int nb, int ntask) {
  int tx, ty, tz;
  tile_counts(nsam, &tx, &ty, &tz);
  return scratch_layout(nullptr, nsam, nb, ntask, tx * ty * tz).bytes;
}

int launch_insert(Ctx& c, int nsam, int nb, int ntask, const InsertTask* d_tasks,
                  const float* d_datc, const float* d_ctff, float* num0, float* ctf2_0,
                  float* num1, float* ctf2_1, unsigned long long* d_nksum, double* d_ttd,
                  void* scratch, const InsertStats* stats) {
  if (ntask <= 0 || nb <= 0) return 0;
  FR_CHECK(scratch != nullptr, "insertion scratch missing");
  FR_CHECK(nb <= 65535, "too many particles in one insertion (%d)", nb);
  FR_CHECK(!stats || (stats->ref && stats->ksum && stats->vsum && stats->psum && stats->asum),
           "insertion statistics arrays missing");
  const int jc = nsam / 2 + 1, w = 2 * jc - 1;
  int tx, ty, tz;
  tile_counts(nsam, &tx, &ty, &tz);
  const int ntiles = tx * ty * tz;
  Scratch s = scratch_layout(scratch, nsam, nb, ntask, ntiles);
  hipLaunchKernelGGL(k_insert_order, dim3(1), dim3(1024), 0, c.stream, ntask, nb, d_tasks, s.first,
                     s.ord, s.n0);
  FR_HIP(hipGetLastError());
  const int nt = (w + 15) / 16;
  hipLaunchKernelGGL(k_insert_points, dim3(nt * nt, nb), dim3(kThreads), 0, c.stream, nsam,
                     s.first, d_tasks, reinterpret_cast<const float2*>(d_datc),
                     reinterpret_cast<const float2*>(d_ctff), s.pts);
  FR_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_insert_geo, dim3((ntask + kThreads - 1) / kThreads), dim3(kThreads), 0,
                     c.stream, ntask, nb, nsam, d_tasks, s.ord, s.hit, s.rec);
  FR_HIP(hipGetLastError());
  const size_t lds = sizeof(TileSums<false>);
  hipLaunchKernelGGL(k_insert_scatter<false>, dim3(2 * ntiles), dim3(kThreads), lds, c.stream,
                     nsam, ntask, tx, ty, tz, s.n0, s.hit, s.rec, s.pts,
                     reinterpret_cast<float2*>(num0), ctf2_0, reinterpret_cast<float2*>(num1),
                     ctf2_1, s.pcount, s.pttd, InsertStats{});
  if (stats) {
    FR_HIP(hipGetLastError());
    const size_t lds_st = sizeof(TileSums<true>);
    FR_HIP(hipFuncSetAttribute((const void*)k_insert_scatter<true>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_st));
    hipLaunchKernelGGL(k_insert_scatter<true>, dim3(ntiles), dim3(kThreads), lds_st, c.stream, nsam,
                       ntask, tx, ty, tz, s.n0, s.hit, s.rec, s.pts, reinterpret_cast<float2*>(num0),
                       ctf2_0, reinterpret_cast<float2*>(num1), ctf2_1, s.pcount, s.pttd, *stats);
  }
  FR_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_insert_reduce, dim3(1), dim3(kReduceThreads), 0, c.stream, ntiles,
                     s.pcount, s.pttd, d_nksum, d_ttd);
  FR_HIP(hipGetLastError());
  return 0;
}

}  // namespace fr
