// mw3_step.h -- the radial kinetic correction and the fused update of one
// Chebyshev step (device templates; instantiated per operator precision in
// mw3_step_f32.hip and mw3_step_f64.hip).
//
// The radial term is T psi = c psi - S (c - E)_+ divi S psi on the low modes
// k1 < k1lo, k2 < k2lo (mw3_setup.cpp).  In FP64 the products over r come first
// and last, so that both ride in the update, which has every r row of its columns
// in hand:
//   update of the step before:  G[k1][R]  = sum_r S(r, k1) psi(r, R)
//   k_rad_rr:                   G2[k1][R] = sum_k2 S(R, k2) (c - E(k1, k2))_+ divi
//                                           sum_R' S(R', k2) G[k1][R']
//   update:                     corr[r][R] = sum_k1 S(r, k1) G2[k1][R]
// psi is then read once for the radial term (as the update's own psi), and
// neither the transformed rows nor the correction pass through a dense slab:
// G and G2 hold k1lo rows instead of n1 (38 of 256 at 256 x 512 x 120).  Mixed
// precision forms the correction before the update, with the products over R
// first (the order of its FP32 sums is part of its results), and its update reads
// it.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "mw3_internal.h"

namespace mw3 {
namespace step {

template <typename T>
struct Mma;
template <>
struct Mma<double> {
  typedef double V __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ V mma(double a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // row of D held in register r by lane group g (lane / 16)
  static __host__ __device__ constexpr int row(int g, int r) { return 4 * r + g; }
};
template <>
struct Mma<float> {  // (no r products: the rows alone)
  typedef float V __attribute__((ext_vector_type(4)));
  static __host__ __device__ constexpr int row(int g, int r) { return 4 * g + r; }
};

// ---------------------------------------------------------------------------
// buffer access: a descriptor of num_records bytes at a wave-uniform base.  A
// lane whose offset lies past the end reads zero and stores nothing, without
// a memory access and without a branch, so lanes that hold no kept point cost
// no traffic and every load of a tile is issued before any is waited for.
// ---------------------------------------------------------------------------
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr uint32_t kOff = 0x80000000u;  // past the end of every descriptor

static __device__ __forceinline__ Rsrc rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
}

typedef uint32_t U2 __attribute__((ext_vector_type(2)));
typedef uint32_t U4 __attribute__((ext_vector_type(4)));

// N consecutive values of type T at byte offset off
template <typename T, int N>
static __device__ __forceinline__ void bld(Rsrc r, uint32_t off, T (&v)[N]) {
  constexpr int B = sizeof(T) * N;
  static_assert(B == 4 || B == 8 || B == 16, "");
  if constexpr (B == 4) {
    const uint32_t x = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
    __builtin_memcpy(&v[0], &x, 4);
  } else if constexpr (B == 8) {
    const U2 x = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
    __builtin_memcpy(&v[0], &x, 8);
  } else {
    const U4 x = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    __builtin_memcpy(&v[0], &x, 16);
  }
}

template <typename T, int N>
static __device__ __forceinline__ void bst(Rsrc r, uint32_t off, const T (&v)[N]) {
  constexpr int B = sizeof(T) * N;
  if constexpr (B == 4) {
    uint32_t x;
    __builtin_memcpy(&x, &v[0], 4);
    __builtin_amdgcn_raw_buffer_store_b32(x, r, off, 0, 0);
  } else if constexpr (B == 8) {
    U2 x;
    __builtin_memcpy(&x, &v[0], 8);
    __builtin_amdgcn_raw_buffer_store_b64(x, r, off, 0, 0);
  } else {
    U4 x;
    __builtin_memcpy(&x, &v[0], 16);
    __builtin_amdgcn_raw_buffer_store_b128(x, r, off, 0, 0);
  }
}

// the lane index as a value the compiler cannot trace: what is computed from it
// inside a loop stays there, instead of being kept in registers across it
static __device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// LDS values that a wave's lanes leave for each other: what was written before is
// seen by the reads after, and what was read before is not overwritten by the
// writes after (a wave's LDS operations execute in order, so this costs no
// instruction; it keeps the compiler to that order)
static __device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// four consecutive values
template <typename T>
static __device__ __forceinline__ void ldv4(const T* p, T (&v)[4]) {
  typedef T T4 __attribute__((ext_vector_type(4)));
  const T4 x = *(const T4*)p;
#pragma unroll
  for (int q = 0; q < 4; q++) v[q] = x[q];
}

template <typename T, int N>
static __device__ __forceinline__ void ldvn(const T* p, T (&v)[N]) {
  if constexpr (N == 1) {
    v[0] = p[0];
  } else {
    typedef T TN __attribute__((ext_vector_type(N)));
    const TN x = *(const TN*)p;
#pragma unroll
    for (int q = 0; q < N; q++) v[q] = x[q];
  }
}

template <typename T, int N>
static __device__ __forceinline__ void stvn(T* p, const T (&v)[N]) {
  if constexpr (N == 1) {
    p[0] = v[0];
  } else {
    typedef T TN __attribute__((ext_vector_type(N)));
    TN x;
#pragma unroll
    for (int q = 0; q < N; q++) x[q] = v[q];
    *(TN*)p = x;
  }
}

// ---------------------------------------------------------------------------
// k_update: V psi, compressed-grid projection, damped update
// (SRC/mod_Hphi_01y2.f:838-853, SRC/main_madwave3.f:245-248, 332-339), the
// per-step projections of the new psi (SRC/mod_flux_01y2.f:598-628, 672-702;
// SRC/mod_coortrans01_02.f:694-740) and the two r products of the radial term.
//
// A tile is 16 r rows of a strip, 16 NT consecutive R of one (channel, angle);
// only tiles with a kept point are listed, strip by strip.  Each wave takes a
// run of the list; the part of a strip in one block's runs is a segment, whose
// sums over r (G, the flux line, the product weights) are added up in the block
// (the waves after the segment's first leave theirs in LDS) and go to the
// segment's place; their readers add a strip's segments, in order.  Lane (g, i) holds R = 16 NT strip + NT i + t (t < NT) of the rows
// that register q of an MFMA result holds, so the back product's result, the
// element-wise work and the forward product's right operand share one layout
// and nothing moves between lanes.  FP32 takes two R per lane (whole 128-byte
// lines per row), FP64 one.
//
// Bound by memory: at 256 x 512 x 120 (5.55 M kept points) a step moves 40
// bytes per point in mixed precision (psi32 4, psi_{k-1} 8, angular and radial
// slabs and V 12, product weights 4, stores 12), 43 us at the rate of a large copy
// (5.2 TB/s), 45 measured (with the angular kernel beside it 51); the row-item
// form before it, one wave per 64 R, took 54 and a second stream's sums.  In FP64
// it moves 48 (51 us), and the two r products are 2 x 0.66 GFLOP of matrix work
// under the loads (18 us at the rate of a large product): 75 us, in place of 76 us
// plus an R-first radial term of 98 us (R passes 72, r passes 26).  Equal runs:
// a block per strip left the last blocks alone at 74 (mixed) and 104 us.
// ---------------------------------------------------------------------------
constexpr int kUpWaves = 4;  // waves per block

struct UpSeg {
  int32_t cia, c, ia, strip;  // cia = c na + ia
  int32_t nn, taboff;         // r DST size, element offset of its table
  int32_t rflux;              // flux row ir1flux - 1
  int32_t seg;                // its index
};

struct UpWave {
  UpSeg s;       // first segment
  int32_t nt;    // tiles
  int32_t cont;  // the first segment began in a wave before, in the same block
  int32_t nadd;  // waves after this one, in the same block, in the last segment
  int32_t pad[5];
};

struct UpArgs {
  const UpWave* waves;    // [nwaves]
  const UpSeg* segs;      // [nseg]
  const uint32_t* tiles;  // [nwaves][tmax][64]: new segment << 31 | row tile << 8 |
                          // keep bits q NT + t
  int nwaves, nseg, tmax;
  const double* absfr2;
  const double* rowtab;  // [n1][4]: absfr1, Re and Im zAR1flux, 0
  // tables are stored in the order the lanes read them (one contiguous load
  // per wave: rows at a stride of a power of two meet on the same cache sets)
  const double* tab;     // S(r, k1) [size][row tile][NK1][lane (g, i)][4]: row i,
                         // k1 = 16 j + 4 g + q
  const double* g2;      // [nc na][strip][kst][16]
  double* g1;            // [nseg][kst][16]
  int ns, kst;           // strips of a row, rows of G2
  const double* psi;     // psi_k
  const void* psi32;     // its FP32 copy (mixed precision)
  double* out;           // hout (mode 0) or psi_{k-1} -> psi_{k+1}
  float* out32;          // FP32 copy of the new psi (mixed precision)
  const void* tkin;      // correction slab (NK1 = 0)
  const void* ang;
  const void* v;
  const double* psi0;    // autocorrelation reference or null
  const void* tprod;     // product weights or null
  int64_t tp_cstride;
  const int32_t* ch_elec;
  const int32_t* ch_omega;
  const int32_t* ch_cpl;
  int nc, ne, na, n1, n2;
  double emindlt, rdelta2, radcut, rsah2;
  int mode;              // 0: out = H psi; 1: undamped first step; 2: damped step
  // ring slot: *dslot when set (captured steps), else slot; the next captured
  // step reads *dslot_next
  const int32_t* dslot;
  int32_t* dslot_next;
  int slot;
  // what the step leaves for the ring's sums, at place slot mod its depth (a power
  // of two)
  double* part;          // [kRing][nwaves][2] (norm, autocorrelation)
  double* upart;         // [seg_ring][nseg][3 or 4][16 NT]: sum_r of Re and Im zAR1flux
                         // psi, psi at the flux row, with product weights those
                         // times psi; or null
  double* slice;         // [slice_ring][nc na][n1] or null
  int seg_ring, slice_ring;
  int ir2abs;
};

// what a launch needs of psi, by template: CPL 0 one electronic state, 1 up to
// 4 channels per Omega (listed), 2 any; AUX bit 0 product weights, bit 1
// autocorrelation; MODE 2 the step, 1 the general form (a.mode 0 or 1), 3 only
// G of psi
template <typename T, int NK1, int NT, int CPL, int AUX, int MODE>
__global__ __launch_bounds__(64 * kUpWaves, 2) void k_update(UpArgs a) {
  typedef typename Mma<T>::V V;
  constexpr bool M32 = sizeof(T) == 4;
  static_assert(NK1 == 0 ? MODE != 3 : !M32, "the r products are FP64's");
  constexpr bool P32 = M32 && MODE == 2;  // psi_k from its FP32 copy
  constexpr int SW = 16 * NT, KP = 16 * NK1, NKA = NK1 > 0 ? NK1 : 1;
  constexpr bool FWD = NK1 > 0 && MODE >= 2, BACK = NK1 > 0 && MODE != 3;
  constexpr bool PRODP = (AUX & 1) && MODE == 2, AUTO = (AUX & 2) && MODE != 3;
  constexpr int NCPL = CPL == 1 ? 3 : 1;
  constexpr uint32_t ES = sizeof(T);
  // LDS, per wave: G2 of the strip and a tile's table rows (padded so that the
  // lane groups of a read fall on different banks); for all: the r rows'
  // absorption factors and flux weights
  constexpr int LG = SW, LS = KP + (NK1 % 4 ? 0 : 4);
  constexpr int NG = BACK ? KP * LG : 0, NSTG = FWD ? 16 * LS : 0;
  __shared__ __align__(16) T lds[kUpWaves * (NG + NSTG) > 0 ? kUpWaves * (NG + NSTG) : 4];
  // sums of a first segment that belongs to a wave before
  constexpr int NH = FWD ? NKA * 4 * NT * 64 : 1;
  __shared__ __align__(16) T hacc[kUpWaves - 1][NH];
  __shared__ __align__(16) double hsum[kUpWaves - 1][MODE == 2 ? 4 : 1][SW];
  extern __shared__ double rowl[];  // [n1][3]
  const int lane0 = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int w = blockIdx.x * kUpWaves + wave;
  const int wc = w < a.nwaves ? w : a.nwaves - 1;
  const uint32_t* const tiles = a.tiles + (int64_t)wc * a.tmax * 64;
  uint32_t tn = tiles[lane0], tnn = a.tmax > 1 ? tiles[64 + lane0] : 0u;
  const UpWave* const wr = a.waves + wc;
  UpSeg sg = wr->s;
  const int nt = w < a.nwaves ? wr->nt : 0;
  bool head = wr->cont != 0;  // in a first segment that belongs to a wave before
  const int nadd = wr->nadd;
  const int n1 = a.n1, n2 = a.n2;
  const int64_t plane = (int64_t)n1 * n2, slab = (int64_t)a.na * plane;
  const uint32_t rb = (uint32_t)n2 * 16u;  // values of a row tile
  T* const gl = lds + wave * (NG + NSTG);
  T* const stg = gl + NG;
  const int slot = a.dslot ? *a.dslot : a.slot;
  if (a.dslot_next && blockIdx.x == 0 && threadIdx.x == 0) *a.dslot_next = slot + 1;
  if constexpr (MODE != 3)
    for (int k = threadIdx.x; k < 3 * n1; k += 64 * kUpWaves) {
      const int r = k / 3;
      rowl[k] = a.rowtab[4 * r + (k - 3 * r)];
    }

  // per segment: absorption of its columns, the other channels of its Omega
  // (CPL 1; -1: none, read through a descriptor of no bytes), G2 in LDS (rows
  // past kst repeat the last one, against zero columns of the table)
  double f2[NT];
  int cs2[NCPL];
  int cself = 0;  // partners listed before the channel itself
  auto begin_seg = [&](const UpSeg& s) {
    const int lane = opaque(lane0), i = lane & 15;
    if constexpr (MODE != 3) {
      const int R0 = s.strip * SW + NT * i;
#pragma unroll
      for (int t = 0; t < NT; t++) f2[t] = a.absfr2[R0 + t < n2 ? R0 + t : n2 - 1];
    }
    if constexpr (CPL == 1) {
      int n = 0;
#pragma unroll
      for (int k = 0; k < NCPL; k++) cs2[k] = -1;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int s2 = a.ch_cpl[4 * s.c + k];
        if (s2 >= 0 && s2 != s.c) {
#pragma unroll
          for (int m = 0; m < NCPL; m++)
            if (m == n) cs2[m] = s2;
          n++;
        } else if (s2 == s.c) {
          cself = n;
        }
      }
    }
    if constexpr (BACK) {
      const T* g2 = a.g2 + ((int64_t)s.cia * a.ns + s.strip) * a.kst * SW;
      constexpr int NV = KP * SW / 256;  // 4-value vectors per lane
      T y[NV][4];
#pragma unroll
      for (int l = 0; l < NV; l++) {
        const int v = lane + 64 * l;
        const int k1 = v / (SW / 4), x = 4 * (v - k1 * (SW / 4));
        ldv4(g2 + (k1 < a.kst ? k1 : a.kst - 1) * SW + x, y[l]);
      }
      wave_lds_sync();  // the last segment's reads
#pragma unroll
      for (int l = 0; l < NV; l++) {
        const int v = lane + 64 * l;
        const int k1 = v / (SW / 4), x = 4 * (v - k1 * (SW / 4));
        stvn<T, 4>(&gl[k1 * LG + x], y[l]);
      }
      wave_lds_sync();
    }
  };

  V acc[NKA][NT];
  double s_norm = 0.0, s_auto = 0.0, zre[NT], zim[NT], zval[NT], spr[NT];
  auto clear_seg = [&]() {
#pragma unroll
    for (int m = 0; m < NKA; m++)
#pragma unroll
      for (int t = 0; t < NT; t++) acc[m][t] = (V){0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < NT; t++) zre[t] = zim[t] = zval[t] = spr[t] = 0.0;
  };
  clear_seg();

  // a tile's operands
  float pf[4][NT];   // psi_k (FP32 copy)
  double pd[4][NT];  // psi_k
  double ob[4][NT], p0[4][NT];
  T an[4][NT], vv[4][NT], tk[4][NT], tp[4][NT];
  T av[NKA][4];  // left operands of the back product
  uint32_t eo[4];
  auto load = [&](uint32_t tw, const UpSeg& s) {
    const int lane = opaque(lane0), g = lane >> 4, i = lane & 15;
    const int rt = __builtin_amdgcn_readfirstlane((int)((tw >> 8) & 0x7fffffu));
    const int64_t ro = (int64_t)rt * rb;
    const int64_t vb = (int64_t)s.ia * plane + ro, base = (int64_t)s.c * slab + vb;
    const int R0 = s.strip * SW + NT * i;
    if constexpr (NK1 > 0) {
      const T* tr = a.tab + s.taboff + (int64_t)rt * (16 * KP) + 4 * lane;
#pragma unroll
      for (int j = 0; j < NK1; j++) ldv4(tr + 256 * j, av[j]);
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
      eo[q] = ((tw >> (q * NT)) & ((1u << NT) - 1u))
                  ? (uint32_t)(Mma<T>::row(g, q) * n2 + R0) * 4u
                  : kOff;
    auto o8 = [&](int q) { return eo[q] == kOff ? kOff : eo[q] * 2u; };
    auto oT = [&](int q) { return ES == 4 ? eo[q] : o8(q); };
    if constexpr (P32) {
      const Rsrc r = rsrc((const float*)a.psi32 + base, rb * 4u);
#pragma unroll
      for (int q = 0; q < 4; q++) bld<float, NT>(r, eo[q], pf[q]);
    } else {
      const Rsrc r = rsrc(a.psi + base, rb * 8u);
#pragma unroll
      for (int q = 0; q < 4; q++) bld<double, NT>(r, o8(q), pd[q]);
    }
    if constexpr (MODE == 3) return;
    if constexpr (MODE == 2) {
      const Rsrc r = rsrc(a.out + base, rb * 8u);
#pragma unroll
      for (int q = 0; q < 4; q++) bld<double, NT>(r, o8(q), ob[q]);
    }
    {
      const Rsrc r = rsrc((const T*)a.ang + base, rb * ES);
#pragma unroll
      for (int q = 0; q < 4; q++) bld<T, NT>(r, oT(q), an[q]);
    }
    if constexpr (NK1 == 0) {
      const Rsrc r = rsrc((const T*)a.tkin + base, rb * ES);
#pragma unroll
      for (int q = 0; q < 4; q++) bld<T, NT>(r, oT(q), tk[q]);
    }
    if constexpr (CPL <= 1) {
      const int et = CPL == 0 ? 0 : a.ch_elec[s.c];
      const Rsrc r = rsrc((const T*)a.v + ((int64_t)et * a.ne + et) * slab + vb, rb * ES);
#pragma unroll
      for (int q = 0; q < 4; q++) bld<T, NT>(r, oT(q), vv[q]);
    }
    if constexpr (PRODP) {
      const Rsrc r = rsrc((const T*)a.tprod + (int64_t)s.c * a.tp_cstride + vb, rb * ES);
#pragma unroll
      for (int q = 0; q < 4; q++) bld<T, NT>(r, oT(q), tp[q]);
    }
    if constexpr (AUTO) {
      const Rsrc r = rsrc(a.psi0 + base, a.psi0 ? rb * 8u : 0u);
#pragma unroll
      for (int q = 0; q < 4; q++) bld<double, NT>(r, o8(q), p0[q]);
    }
  };
  // sum over the lane groups of the segment's FP64 sums
  auto gsum = [&](int k, double (&x)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      x[t] = k == 0 ? zre[t] : k == 1 ? zim[t] : k == 2 ? zval[t] : spr[t];
      x[t] += __shfl_xor(x[t], 16);
      x[t] += __shfl_xor(x[t], 32);
    }
  };
  // a first segment's sums, for the wave before
  auto save_seg = [&]() {
    const int lane = opaque(lane0), g = lane >> 4, i = lane & 15;
    if constexpr (FWD) {
#pragma unroll
      for (int m = 0; m < NK1; m++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int t = 0; t < NT; t++)
            hacc[wave - 1][(m * 4 * NT + r * NT + t) * 64 + lane] = acc[m][t][r];
    }
    if constexpr (MODE == 2) {
#pragma unroll
      for (int k = 0; k < (PRODP ? 4 : 3); k++) {
        double x[NT];
        gsum(k, x);
        if (g == 0) stvn<double, NT>(&hsum[wave - 1][k][NT * i], x);
      }
    }
  };
  // the segment's sums, with those of the na waves after this one, to their
  // places
  auto end_seg = [&](const UpSeg& s, int na) {
    const int lane = opaque(lane0), g = lane >> 4, i = lane & 15;
    if constexpr (FWD) {
      for (int k = 0; k < na; k++)
#pragma unroll
        for (int m = 0; m < NK1; m++)
#pragma unroll
          for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < NT; t++)
              acc[m][t][r] += hacc[wave + k][(m * 4 * NT + r * NT + t) * 64 + lane];
      T* g1 = a.g1 + (int64_t)s.seg * a.kst * SW + NT * i;
#pragma unroll
      for (int m = 0; m < NK1; m++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int k1 = 16 * m + Mma<T>::row(g, r);
          T x[NT];
#pragma unroll
          for (int t = 0; t < NT; t++) x[t] = acc[m][t][r];
          if (k1 < a.kst) stvn<T, NT>(g1 + k1 * SW, x);
        }
    }
    if constexpr (MODE == 2) {
      if (a.upart) {
        const int64_t at = (int64_t)(slot & (a.seg_ring - 1)) * a.nseg + s.seg;
        double* up = a.upart + at * ((PRODP ? 4 : 3) * SW) + NT * i;
#pragma unroll
        for (int k = 0; k < (PRODP ? 4 : 3); k++) {
          double x[NT];
          gsum(k, x);
          for (int q = 0; q < na; q++)
#pragma unroll
            for (int t = 0; t < NT; t++) x[t] += hsum[wave + q][k][NT * i + t];
          if (g == 0) stvn<double, NT>(up + k * SW, x);
        }
      }
    }
  };

  // Vector memory operations end in order: a tile's loads are issued before
  // the stores of the tile before it (a wait for them does not wait for those
  // stores), its table rows before its data (the back product starts while the
  // data are in flight), and its list word a tile earlier.
  if (nt > 0) {
    load(tn, sg);
    begin_seg(sg);
  }
  if constexpr (MODE != 3) __syncthreads();  // rowl
  uint32_t tl = tn;
  tn = tnn;
  // (a wave's segments are consecutive)
  int seg_next = sg.seg + 1 < a.nseg ? sg.seg + 1 : a.nseg - 1;
  UpSeg sn = a.segs[seg_next];
  for (int t0 = 0; t0 < nt;) {
    const int lane = opaque(lane0), g = lane >> 4, i = lane & 15;
    const int rt = __builtin_amdgcn_readfirstlane((int)((tl >> 8) & 0x7fffffu));
    const uint32_t keep = tl;
    const int64_t ro = (int64_t)rt * rb;
    const int64_t vb = (int64_t)sg.ia * plane + ro, base = (int64_t)sg.c * slab + vb;
    uint32_t so4[4];
#pragma unroll
    for (int q = 0; q < 4; q++) so4[q] = eo[q];
    auto so8 = [&](int q) { return so4[q] == kOff ? kOff : so4[q] * 2u; };
    auto soT = [&](int q) { return ES == 4 ? so4[q] : so8(q); };
    double o[4][NT];
    T bv[4][NT];  // the new psi (MODE 3: psi) in operator precision, zero off the grid
    if constexpr (FWD) {  // the tile's table rows, for the forward product
      wave_lds_sync();  // the last tile's reads
#pragma unroll
      for (int j = 0; j < NK1; j++) stvn<T, 4>(stg + i * LS + 16 * j + 4 * g, av[j]);
      wave_lds_sync();
    }
    if constexpr (MODE == 3) {
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int t = 0; t < NT; t++) bv[q][t] = ((keep >> (q * NT + t)) & 1u) ? (T)pd[q][t] : (T)0;
    } else {
      // the coupled channels' V and psi, in flight during the back product
      T cv[NCPL][4][NT];
      double cd[NCPL][4][NT];
      float cf[NCPL][4][NT];
      auto load_cpl = [&](int k, int s2, uint32_t nby) {
        const int et = a.ch_elec[sg.c];
        const Rsrc rv = rsrc((const T*)a.v + ((int64_t)et * a.ne + a.ch_elec[s2]) * slab + vb,
                             nby * ES);
#pragma unroll
        for (int q = 0; q < 4; q++) bld<T, NT>(rv, soT(q), cv[k][q]);
        if constexpr (P32) {
          const Rsrc rp = rsrc((const float*)a.psi32 + (int64_t)s2 * slab + vb, nby * 4u);
#pragma unroll
          for (int q = 0; q < 4; q++) bld<float, NT>(rp, so4[q], cf[k][q]);
        } else {
          const Rsrc rp = rsrc(a.psi + (int64_t)s2 * slab + vb, nby * 8u);
#pragma unroll
          for (int q = 0; q < 4; q++) bld<double, NT>(rp, so8(q), cd[k][q]);
        }
      };
      if constexpr (CPL == 1) {
#pragma unroll
        for (int k = 0; k < NCPL; k++) load_cpl(k, cs2[k] >= 0 ? cs2[k] : sg.c, cs2[k] >= 0 ? rb : 0u);
      }
      // correction of the tile: corr[row][R] = sum_k1 S(row, k1) G2[k1][R]
      V co[NT];
#pragma unroll
      for (int t = 0; t < NT; t++) co[t] = (V){0, 0, 0, 0};
      if constexpr (NK1 > 0) {
#pragma unroll
        for (int j = 0; j < NK1; j++)
#pragma unroll
          for (int q = 0; q < 4; q++) {
            T gb[NT];
            ldvn<T, NT>(&gl[(16 * j + 4 * g + q) * LG + NT * i], gb);
#pragma unroll
            for (int t = 0; t < NT; t++) co[t] = Mma<T>::mma(av[j][q], gb[t], co[t]);
          }
      }
      __builtin_amdgcn_sched_barrier(0);
      double h[4][NT], p[4][NT];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int r = 16 * rt + Mma<T>::row(g, q);
#pragma unroll
        for (int t = 0; t < NT; t++) {
          p[q][t] = P32 ? (double)pf[q][t] : pd[q][t];
          const double k = NK1 > 0 ? (double)co[t][q] : (double)tk[q][t];
          // T psi = radcut psi - low-mode correction on r < nn1; psi beyond
          // (the reference's tail identity)
          h[q][t] = (r < sg.nn ? a.radcut * p[q][t] - k : p[q][t]) + (double)an[q][t];
          if constexpr (CPL == 0) h[q][t] += p[q][t] * (double)vv[q][t];
        }
      }
      auto add_cpl = [&](int k) {
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
          for (int t = 0; t < NT; t++)
            h[q][t] += (P32 ? (double)cf[k][q][t] : cd[k][q][t]) * (double)cv[k][q][t];
      };
      if constexpr (CPL == 1) {  // in the order of the list
#pragma unroll
        for (int k = 0; k <= NCPL; k++) {
          if (k == cself) {
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
              for (int t = 0; t < NT; t++) h[q][t] += p[q][t] * (double)vv[q][t];
          }
          if (k < NCPL) add_cpl(k < NCPL ? k : 0);
        }
      } else if constexpr (CPL == 2) {
        for (int s2 = 0; s2 < a.nc; s2++) {
          if (a.ch_omega[s2] != a.ch_omega[sg.c]) continue;
          load_cpl(0, s2, rb);
          add_cpl(0);
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int r = 16 * rt + Mma<T>::row(g, q);
        const double* rw = rowl + 3 * (r < n1 ? r : n1 - 1);
        const double f1 = rw[0], za = rw[1], zb = rw[2];
#pragma unroll
        for (int t = 0; t < NT; t++) {
          const double hn = (h[q][t] - a.emindlt * p[q][t]) * a.rdelta2;
          double x;
          if constexpr (MODE == 2) {
            const double f = f1 * f2[t];
            x = (2.0 * hn - f * ob[q][t]) * f;
          } else {
            x = a.mode == 1 ? hn : h[q][t];
          }
          o[q][t] = ((keep >> (q * NT + t)) & 1u) ? x : 0.0;
          bv[q][t] = (T)o[q][t];
          s_norm += o[q][t] * o[q][t];
          if constexpr (AUTO) s_auto += p0[q][t] * o[q][t];
          if constexpr (PRODP) spr[t] += (double)tp[q][t] * o[q][t];
          if constexpr (MODE == 2) {
            zre[t] += za * o[q][t];
            zim[t] += zb * o[q][t];
            zval[t] = r == sg.rflux ? o[q][t] : zval[t];
          }
        }
      }
    }
    // scheduling barriers between the phases: without them the LDS reads and
    // the next tile's loads are moved up across the element-wise work, and the
    // registers they hold no longer fit two waves per SIMD
    __builtin_amdgcn_sched_barrier(0);
    t0++;
    const bool more = t0 < nt;
    const bool chg = more && (__builtin_amdgcn_readfirstlane((int)tn) < 0);
    tl = tn;
    if (more) {
      const UpSeg s2 = chg ? sn : sg;
      load(tn, s2);
      tn = t0 + 1 < nt ? tiles[(t0 + 1) * 64 + lane0] : 0u;
    }
    if constexpr (MODE != 3) {
      const Rsrc ro8 = rsrc(a.out + base, rb * 8u);
      const Rsrc ro4 = rsrc(a.out32 + base, M32 && a.out32 ? rb * 4u : 0u);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        bst<double, NT>(ro8, so8(q), o[q]);
        if constexpr (M32) {
          float o32[NT];
#pragma unroll
          for (int t = 0; t < NT; t++) o32[t] = (float)o[q][t];
          bst<float, NT>(ro4, so4[q], o32);
        }
        if (MODE == 2 && a.slice && (a.ir2abs - 1) / SW == sg.strip) {
          double* sl =
              a.slice + ((int64_t)(slot & (a.slice_ring - 1)) * a.nc * a.na + sg.cia) * n1;
#pragma unroll
          for (int t = 0; t < NT; t++)
            if (sg.strip * SW + NT * i + t == a.ir2abs - 1 && ((keep >> (q * NT + t)) & 1u))
              sl[16 * rt + Mma<T>::row(g, q)] = o[q][t] * a.rsah2;
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FWD) {
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int m = 0; m < NK1; m++) {
          const T fa = stg[Mma<T>::row(g, q) * LS + 16 * m + i];
#pragma unroll
          for (int t = 0; t < NT; t++) acc[m][t] = Mma<T>::mma(fa, bv[q][t], acc[m][t]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if ((FWD || MODE == 2) && (chg || (!more && head))) {
      if (head) save_seg();
      else end_seg(sg, 0);
      if (chg) clear_seg();
    }
    if (chg) {
      head = false;
      sg = sn;
      begin_seg(sg);
      seg_next = seg_next + 1 < a.nseg ? seg_next + 1 : a.nseg - 1;
      sn = a.segs[seg_next];
    }
  }
  if constexpr (FWD || MODE == 2) {
    __syncthreads();
    if (nt > 0 && !head) end_seg(sg, nadd);
  }
  if constexpr (MODE != 3) {
    for (int of = 32; of > 0; of >>= 1) {
      s_norm += __shfl_xor(s_norm, of);
      if constexpr (AUTO) s_auto += __shfl_xor(s_auto, of);
    }
    if (lane0 == 0 && a.part && w < a.nwaves) {
      double* p = a.part + 2 * ((int64_t)slot * a.nwaves + w);
      p[0] = s_norm;
      p[1] = s_auto;
    }
  }
}

// ---------------------------------------------------------------------------
// k_rad_rr (FP64): G -> G2 of one (channel, angle) and 16 modes k1: fold over R,
// sum over R to the low k2 modes of both parities, weights, and back to R.
// S(n2-1-R, k2) = (-1)^k2 S(R, k2), so with u = G[R] + G[n2-1-R] and
// v = G[R] - G[n2-1-R] the even modes see u and the odd ones v, and back
// G2[R] = E + O, G2[n2-1-R] = E - O: half the products of the plain sums.
// G is the sum of the strips' segments, in segment order.  Eight waves: in the
// first product each takes one parity and a quarter of the R pairs (LDS adds
// the quarters' partial tiles), in the second an eighth of the R tiles.  The
// first product's result layout is the second one's right operand as it
// stands.  A wave runs each loop only a few times, so the time is that of a
// chain of memory latencies: the next block's G is in flight behind the products.
// The tables are read where they are used; their registers would push the
// block's second copy off the CU.  29 us at 256 x 512 x 120 (38 k1 by 77 k2 modes
// of 120 angles).
// ---------------------------------------------------------------------------
struct RrArgs {
  const double* g1;
  double* g2;
  const double* tf;  // [nb][parity][NP][lane (g, i)][4]: S(j, 2 k + parity), k = 16 t + i,
                     // j = 16 jb + 4 g + e
  const double* tb;  // [nb][parity][NP][lane][4]: the back product's, in MFMA order
  const double* wt;  // weights (c - E(k1, k2))_+ divi [na][k1 tile][parity][NP][lane][4] of
                     // the first product's results
  int na, n1, n2, nk1, kst, nb;
  const int32_t* sfirst;  // [nc na ns + 1] first segment of each strip
  // strips per row, log2 of their width (4; with a constant the compiler forms more
  // addresses ahead and spills at NP = 3), most segments of one
  int ns, swl, segmax;
};

template <int NP, bool VEC>
__global__ __launch_bounds__(512, 4) void k_rad_rr(RrArgs a) {
  typedef double T;
  typedef Mma<T> M;
  typedef M::V V;
  constexpr uint32_t ES = sizeof(T);
  __shared__ V red[4][2][NP][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int par = wave & 1, jw = wave >> 1;
  const int g = lane >> 4, i = lane & 15;
  const int cia = blockIdx.x / a.nk1, mt = blockIdx.x - cia * a.nk1;
  const int ia = cia % a.na;
  const int n2 = a.n2, nb = a.nb, h = n2 / 2, ke = n2 - h, kst = a.kst, swl = a.swl, sw = 1 << swl;
  const int k1 = 16 * mt + i, k1c = k1 < kst ? k1 : kst - 1;
  if (mt * 16 >= kst) return;  // no row of this tile is kept
  const T* tf = a.tf + par * NP * 256 + 4 * lane;
  const T* tb = a.tb;
  const int32_t* sf = a.sfirst + (int64_t)cia * a.ns;
  const int64_t segw = (int64_t)kst * sw;  // values of a segment
  // segments 0 and 1 of the strip that holds the 16-column block b, 4 columns
  // from c on (b is wave-uniform); a second segment the strip does not have
  // reads zero, without a memory access
  auto gload = [&](int b, int c, T (&y)[2][4]) {
    const int s = (16 * b) >> swl, s0 = sf[s], n = sf[s + 1] - s0;
    const Rsrc r = rsrc(a.g1 + s0 * segw, (uint32_t)((n < 2 ? n : 2) * segw) * ES);
    const uint32_t o = (uint32_t)(k1c * sw + 16 * b - s * sw + c) * ES;
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const uint32_t oq = o + q * (uint32_t)segw * ES;
      T z0[2], z1[2];
      bld<T, 2>(r, oq, z0);
      bld<T, 2>(r, oq + 16u, z1);
      y[q][0] = z0[0], y[q][1] = z0[1], y[q][2] = z1[0], y[q][3] = z1[1];
    }
  };
  // the same columns of the segments from k on
  auto gmore = [&](int o, int k, T (&y)[4]) {
    const int s = o >> swl, s1 = sf[s + 1];
    for (int q = sf[s] + k; q < s1; q++) {
      const T* G = a.g1 + q * segw + k1c * sw + (o - s * sw);
#pragma unroll
      for (int e = 0; e < 4; e++) y[e] += G[e];
    }
  };
  T xn[2][4], mn[2][4];
  auto prefetch = [&](int jb) {
    if constexpr (VEC) {
      gload(jb, 4 * g, xn);
      gload(n2 / 16 - 1 - jb, 12 - 4 * g, mn);
    }
  };
  V acc[NP];
#pragma unroll
  for (int t = 0; t < NP; t++) acc[t] = (V){0, 0, 0, 0};
  if (jw < nb) prefetch(jw);
#pragma unroll 1
  for (int jb = jw; jb < nb; jb += 4) {
    T at[NP][4], xs[4] = {0, 0, 0, 0}, ms[4] = {0, 0, 0, 0}, u[4];
    const int j0 = 16 * jb + 4 * g;
#pragma unroll
    for (int t = 0; t < NP; t++) ldv4(tf + (int64_t)(jb * 2 * NP + t) * 256, at[t]);
    if constexpr (VEC) {
      T mm[4] = {0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        xs[e] = xn[0][e] + xn[1][e];
        mm[e] = mn[0][e] + mn[1][e];
      }
      if (a.segmax > 2) {
        gmore(j0, 2, xs);
        gmore(n2 - 4 - j0, 2, mm);
      }
#pragma unroll
      for (int e = 0; e < 4; e++) ms[e] = mm[3 - e];  // mirrored columns come in reverse order
    } else {
      gmore(j0, 0, xs);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int o1 = n2 - 1 - j0 - e, o = o1 > 0 ? o1 : 0, s = o >> swl;
        for (int q = sf[s]; q < sf[s + 1]; q++)
          ms[e] += a.g1[q * segw + k1c * sw + (o - s * sw)];
      }
    }
    if (jb + 4 < nb) prefetch(jb + 4);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int j = j0 + e;
      // the middle of an odd n2 counts once, in the even modes; rows past it
      // meet zero columns
      u[e] = j < h ? (par ? xs[e] - ms[e] : xs[e] + ms[e]) : (j < ke && !par ? xs[e] : (T)0);
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int t = 0; t < NP; t++) acc[t] = M::mma(at[t][e], u[e], acc[t]);
  }
#pragma unroll
  for (int t = 0; t < NP; t++) red[jw][par][t][lane] = acc[t];
  T wt[2][NP][4];
  {
    const T* w = a.wt + (int64_t)(ia * a.nk1 + mt) * (2 * NP * 256) + 4 * lane;
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int t = 0; t < NP; t++) ldv4(w + (p * NP + t) * 256, wt[p][t]);
  }
  __syncthreads();
  V hw[2][NP];
#pragma unroll
  for (int p = 0; p < 2; p++)
#pragma unroll
    for (int t = 0; t < NP; t++) {
      const V s = (red[0][p][t][lane] + red[1][p][t][lane]) +
                  (red[2][p][t][lane] + red[3][p][t][lane]);
#pragma unroll
      for (int r = 0; r < 4; r++) hw[p][t][r] = s[r] * wt[p][t][r];
    }
  T* out = a.g2 + (int64_t)cia * a.ns * segw + k1 * sw;
  auto at2 = [&](int R) { return out + (R >> swl) * segw + (R & (sw - 1)); };  // column R of row k1
#pragma unroll 1
  for (int rt = wave; rt < nb; rt += 8) {
    V e = {0, 0, 0, 0}, o = {0, 0, 0, 0};
    T ae[NP][4], ao[NP][4];
#pragma unroll
    for (int t = 0; t < NP; t++) {
      ldv4(tb + (int64_t)(rt * 2 * NP + t) * 256 + 4 * lane, ae[t]);
      ldv4(tb + (int64_t)(rt * 2 * NP + NP + t) * 256 + 4 * lane, ao[t]);
    }
#pragma unroll
    for (int t = 0; t < NP; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        e = M::mma(ae[t][r], hw[0][t][r], e);
        o = M::mma(ao[t][r], hw[1][t][r], o);
      }
    const int R = 16 * rt + 4 * g;  // registers r: R + r
    if (k1 >= kst) continue;
    if constexpr (VEC) {
      if (R < h) {
        T lo[4], hi[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          lo[r] = e[r] + o[r];
          hi[3 - r] = e[r] - o[r];
        }
        stvn<T, 4>(at2(R), lo);
        stvn<T, 4>(at2(n2 - 4 - R), hi);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        if (R + r < ke) *at2(R + r) = e[r] + o[r];
        if (R + r < h) *at2(n2 - 1 - R - r) = e[r] - o[r];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <typename U>
static hipError_t upload_v(U** dst, const std::vector<U>& v) {
  hipError_t e = hipMalloc((void**)dst, sizeof(U) * std::max<size_t>(v.size(), 1));
  if (e != hipSuccess || v.empty()) return e;
  return hipMemcpy(*dst, v.data(), sizeof(U) * v.size(), hipMemcpyHostToDevice);
}

static hipError_t zalloc(void** p, size_t n) {
  hipError_t e = hipMalloc(p, std::max<size_t>(n, 16));
  return e == hipSuccess ? hipMemset(*p, 0, std::max<size_t>(n, 16)) : e;
}

// blocks of the step's update that a CU holds, of the two that its registers
// allow: 160 KB of LDS over what the kernel takes (its sums and tables, and 24
// bytes per r row)
template <typename T, int NK1, int NT>
static hipError_t resident(int n1, int* blocks) {
  hipFuncAttributes f{};
  const hipError_t e = hipFuncGetAttributes(&f, (const void*)k_update<T, NK1, NT, 0, 0, 2>);
  *blocks = f.sharedSizeBytes + sizeof(double) * 3 * (size_t)n1 > 80 * 1024 ? 1 : 2;
  return e;
}

template <typename T>
static hipError_t resident(const Ctx* c, int* blocks) {
  const int n1 = c->t.n1;
  if constexpr (sizeof(T) == 4) {
    return c->up_nt == 2 ? resident<T, 0, 2>(n1, blocks) : resident<T, 0, 1>(n1, blocks);
  } else {
    switch (c->up_nk1) {
      case 1: return resident<T, 1, 1>(n1, blocks);
      case 3: return resident<T, 3, 1>(n1, blocks);
      case 4: return resident<T, 4, 1>(n1, blocks);
      default: return resident<T, 0, 1>(n1, blocks);
    }
  }
}

// FP64: the tables of k_rad_rr (S(R, k2) by parity for the R products, and the
// weights), G and G2
static hipError_t build_rr(Ctx* c, int k1max, int k2max) {
  typedef Mma<double> M;
  const HostTables& t = c->t;
  const int n1 = t.n1, n2 = t.n2, na = t.na;
  const int h = n2 / 2, ke = n2 - h, nb = (ke + 15) / 16, NP = c->rr_np;
  c->up_kst = k1max;
  c->rr_nb = nb;
  int q2 = 0;
  while (t.dst_sizes[q2] != n2) q2++;
  auto S = [&](int j, int k) {
    return j < ke && k < k2max ? t.dst_tables[(size_t)t.low_off[q2] + (size_t)k * t.low_ld[q2] + j]
                               : 0.0;
  };
  std::vector<double> tf((size_t)nb * 2 * NP * 256), tb(tf.size());
  size_t o = 0;
  // back: row i of a table tile gives D's row i, which is to be R offset
  // 4 g + r where i = row(g, r); its columns are the modes that result
  // register r of lane group g holds
  int inv[16];
  for (int g = 0; g < 4; g++)
    for (int r = 0; r < 4; r++) inv[M::row(g, r)] = 4 * g + r;
  for (int b = 0; b < nb; b++)
    for (int p = 0; p < 2; p++)
      for (int u = 0; u < NP; u++)
        for (int l = 0; l < 256; l++, o++) {
          const int lg = l >> 6, li = (l >> 2) % 16, x = l % 4;
          tf[o] = S(16 * b + 4 * lg + x, 2 * (16 * u + li) + p);
          tb[o] = S(16 * b + inv[li], 2 * (16 * u + M::row(lg, x)) + p);
        }
  std::vector<double> wt((size_t)na * c->up_nk1 * 2 * NP * 256);
  o = 0;
  for (int ia = 0; ia < na; ia++)
    for (int mt = 0; mt < c->up_nk1; mt++)
      for (int p = 0; p < 2; p++)
        for (int u = 0; u < NP; u++)
          for (int l = 0; l < 256; l++, o++) {
            const int k1 = 16 * mt + (l >> 2) % 16;
            const int k2 = 2 * (16 * u + M::row(l >> 6, l % 4)) + p;
            double w = 0.0;
            if (k1 < t.k1lo[ia] && k2 < t.k2lo[ia])
              w = t.radcut - (t.p2r1[(size_t)ia * n1 + k1] + t.p2r2[k2]);
            wt[o] = w > 0.0 ? w * t.divi[ia] : 0.0;
          }
  hipError_t e;
  const size_t row = sizeof(double) * (size_t)k1max * 16;
  if ((e = upload_v(&c->d_rr_w, wt)) != hipSuccess) return e;
  if ((e = upload_v(&c->d_rr_f, tf)) != hipSuccess) return e;
  if ((e = upload_v(&c->d_rr_b, tb)) != hipSuccess) return e;
  if ((e = zalloc((void**)&c->d_g1, row * (size_t)c->up_nseg)) != hipSuccess) return e;
  return zalloc((void**)&c->d_g2, row * (size_t)t.nc * na * c->up_ns);
}

// strips and tiles of the update, and in FP64, where the low modes fit the
// kernels, tables of the radial products
template <typename T>
static hipError_t build(Ctx* c) {
  const HostTables& t = c->t;
  hipError_t e;
  const int n1 = t.n1, n2 = t.n2, na = t.na;
  // low modes: 16-mode tiles of k1, of k2 per parity
  int k1max = 0, k2max = 0;
  for (int ia = 0; ia < na; ia++) {
    k1max = std::max(k1max, t.k1lo[ia]);
    k2max = std::max(k2max, t.k2lo[ia]);
  }
  const int nk = (k1max + 15) / 16, np = ((k2max + 1) / 2 + 15) / 16;
  // (mixed precision keeps the R products first: the order of the FP32 sums,
  // and with it their rounding, is part of its results)
  c->up_nk1 = sizeof(T) == 4 ? 0 : nk < 1 ? 0 : nk <= 1 ? 1 : nk <= 3 ? 3 : nk <= 4 ? 4 : 0;
  c->rr_np = np <= 4 ? np : 0;
  // (four mode tiles take 94 KB of LDS beside 24 bytes per r row)
  if (!c->rr_np || n1 > 2048) c->up_nk1 = 0;
  if (!c->up_nk1) c->rr_np = 0;
  // FP32: two R per lane where rows are 8-byte aligned
  c->up_nt = sizeof(T) == 4 && n2 % 2 == 0 ? 2 : 1;
  const int NT = c->up_nt, SW = 16 * NT, ns = (n2 + SW - 1) / SW;
  const int nrt = (n1 + 15) / 16;
  std::vector<uint32_t> tiles;
  tiles.reserve((size_t)na * ns * nrt * 16);
  std::vector<int32_t> first((size_t)na * ns), cnt((size_t)na * ns);
  // bit x: kept point R + x of a row (x < 16 NT), eight mask bytes (0 or 1) to a
  // product whose top byte gathers them
  auto row_bits = [&](const uint8_t* row, int R) {
    uint32_t b = 0;
    for (int x = 0; x < SW && R + x < n2; x += 8) {
      uint64_t v = 0;
      if (R + x + 8 <= n2) std::memcpy(&v, row + R + x, 8);
      else std::memcpy(&v, row + R + x, (size_t)(n2 - R - x));
      b |= (uint32_t)((v * 0x0102040810204080ull) >> 56) << x;
    }
    return b;
  };
  for (int ia = 0; ia < na; ia++)
    for (int s = 0; s < ns; s++) {
      const size_t q0 = (size_t)ia * ns + s;
      first[q0] = (int32_t)(tiles.size() / 64);
      for (int rt = 0; rt < nrt; rt++) {
        uint32_t b[16], any = 0;
        for (int i = 0; i < 16; i++) {
          const int r = 16 * rt + i;
          b[i] = r < n1 ? row_bits(&t.mask[(size_t)ia * t.nplane + (size_t)r * n2], s * SW) : 0u;
          any |= b[i];
        }
        if (!any) continue;
        for (int lane = 0; lane < 64; lane++) {
          uint32_t w = (uint32_t)rt << 8;
          for (int q = 0; q < 4; q++)
            w |= ((b[Mma<T>::row(lane >> 4, q)] >> (NT * (lane & 15))) & ((1u << NT) - 1u))
                 << (q * NT);
          tiles.push_back(w);
        }
      }
      cnt[q0] = (int32_t)(tiles.size() / 64) - first[q0];
    }
  // S(r, k1) per r size, zero at r >= nn1 and past the size's low modes
  const int kp = 16 * c->up_nk1;
  std::vector<double> tab;
  std::vector<int> off((size_t)na, 0), qoff(t.dst_sizes.size(), -1);
  for (int ia = 0; ia < na && kp; ia++) {
    int q = 0;
    while (t.dst_sizes[q] != t.nn1[ia]) q++;
    if (qoff[q] < 0) {
      qoff[q] = (int)tab.size();
      int kcap = 0;
      for (int ja = 0; ja < na; ja++)
        if (t.nn1[ja] == t.nn1[ia]) kcap = std::max(kcap, t.k1lo[ja]);
      for (int rt = 0; rt < nrt; rt++)
        for (int j = 0; j < c->up_nk1; j++)
          for (int l = 0; l < 256; l++) {
            const int r = 16 * rt + (l >> 2) % 16, k = 16 * j + 4 * (l >> 6) + l % 4;
            tab.push_back(r < t.nn1[ia] && k < kcap
                              ? t.dst_tables[(size_t)t.low_off[q] + (size_t)k * t.low_ld[q] + r]
                              : 0.0);
          }
    }
    off[ia] = qoff[q];
  }
  if (kp && (e = upload_v(&c->d_up_tab, tab)) != hipSuccess) return e;
  // Waves.  Few strips (every strip's block resident at once): a block per
  // strip, its waves an equal part each, so that a strip is one segment.  Else
  // runs of equal length over all channels' tiles, for as many waves as are
  // resident at once, so that the one resident set ends together.  Runs too
  // where a strip's quarter is more than twice their length, which leaves most
  // of the chip idle: few strips of many rows (us a step, a block per strip ->
  // runs: 64 x 64 x 8 FP64 18.4 either way, 256 x 64 x 8 26.7 -> 20.8, mixed
  // 1500 x 64 x 16 98 -> 71, 3000 x 64 x 16 170 -> 117).  Runs for two blocks per
  // CU where one fits took longer than those for one (4096 x 64 x 16 mixed 165
  // against 150, FP64 210 against 195, four mode tiles at 160 x 256 x 60 53
  // against 47).
  int64_t total = 0, nstrip = 0;
  for (int x : cnt) {
    total += x;
    nstrip += x > 0;
  }
  total *= t.nc;
  nstrip *= t.nc;
  int dev = 0, ncu = 0;
  if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
  if ((e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess)
    return e;
  int res = 0;
  if ((e = resident<T>(c, &res)) != hipSuccess) return e;
  const int nw = res * kUpWaves * ncu;  // resident waves
  int tmax = (int)std::max<int64_t>(1, (total + nw - 1) / nw);
  int per = 1;  // tiles of a wave, a block to each strip
  for (int x : cnt) per = std::max(per, (x + kUpWaves - 1) / kUpWaves);
  const bool aligned = nstrip <= res * ncu && per <= 2 * tmax;
  if (aligned) tmax = per;
  std::vector<UpWave> waves;
  std::vector<UpSeg> segs;
  std::vector<uint32_t> lists;
  std::vector<int32_t> sfirst;
  lists.reserve((size_t)(aligned ? kUpWaves * nstrip : (total + tmax - 1) / tmax) * tmax * 64);
  int segmax = 1;
  for (int ch = 0; ch < t.nc; ch++)
    for (int ia = 0; ia < na; ia++)
      for (int s = 0; s < ns; s++) {
        const size_t q0 = (size_t)ia * ns + s;
        const int rf = t.ir1flux.empty() ? -1 : t.ir1flux[ia] - 1;
        sfirst.push_back((int32_t)segs.size());
        const int run = aligned ? (cnt[q0] + kUpWaves - 1) / kUpWaves : tmax;
        for (int k = 0; k < cnt[q0]; k++) {
          const bool neww = waves.empty() || (aligned ? k % run == 0 : waves.back().nt == run);
          const bool newb = neww && waves.size() % kUpWaves == 0;
          if (k == 0 || newb)
            segs.push_back(UpSeg{ch * na + ia, ch, ia, s, t.nn1[ia], off[ia], rf,
                                 (int32_t)segs.size()});
          if (neww) {
            const bool cont = k > 0 && !newb;
            if (cont) {  // counted by the segment's first wave of the block
              size_t o = waves.size() - 1;
              while (waves[o].cont && waves[o].s.seg == segs.back().seg) o--;
              waves[o].nadd++;
            }
            waves.push_back(UpWave{segs.back(), 0, cont ? 1 : 0, 0, {0, 0, 0, 0, 0}});
            lists.resize(lists.size() + (size_t)tmax * 64, 0u);
          }
          uint32_t* w = &lists[((waves.size() - 1) * tmax + waves.back().nt) * 64];
          for (int lane = 0; lane < 64; lane++)
            w[lane] = tiles[((size_t)first[q0] + k) * 64 + lane] |
                      (k == 0 && waves.back().nt > 0 ? 0x80000000u : 0u);
          waves.back().nt++;
        }
        if (aligned && cnt[q0])
          while (waves.size() % kUpWaves) {  // a whole block per strip
            waves.push_back(UpWave{segs.back(), 0, 1, 0, {0, 0, 0, 0, 0}});
            lists.resize(lists.size() + (size_t)tmax * 64, 0u);
          }
        segmax = std::max(segmax, (int)segs.size() - sfirst.back());
      }
  sfirst.push_back((int32_t)segs.size());
  c->up_nwaves = (int)waves.size();
  c->up_nseg = (int)segs.size();
  c->up_tmax = tmax;
  c->up_ns = ns;
  c->up_segmax = segmax;
  if ((e = upload_v((UpWave**)&c->d_up_wave, waves)) != hipSuccess) return e;
  if ((e = upload_v((UpSeg**)&c->d_up_seg, segs)) != hipSuccess) return e;
  if ((e = upload_v(&c->d_up_tile, lists)) != hipSuccess) return e;
  if ((e = upload_v(&c->d_up_sfirst, sfirst)) != hipSuccess) return e;
  return c->up_nk1 ? build_rr(c, k1max, k2max) : hipSuccess;
}

template <typename T, int NK1, int NT, int CPL, int AUX, int MODE>
static void launch_k(Ctx* c, const UpArgs& a) {
  hipLaunchKernelGGL((k_update<T, NK1, NT, CPL, AUX, MODE>), dim3((unsigned)((c->up_nwaves + kUpWaves - 1) / kUpWaves)),
                     dim3(64 * kUpWaves), MODE != 3 ? sizeof(double) * 3 * (size_t)a.n1 : 0, c->stream, a);
}

// aux: bit 0 product weights, bit 1 autocorrelation
template <typename T, int NK1, int NT>
static void launch_nk(Ctx* c, const UpArgs& a, int cpl, int aux, int mode) {
  if (mode == 3) {
    if constexpr (NK1 > 0) launch_k<T, NK1, NT, 0, 0, 3>(c, a);
  } else if (mode == 2 && cpl == 0) {
    if (aux == 0) launch_k<T, NK1, NT, 0, 0, 2>(c, a);
    else if (aux == 1) launch_k<T, NK1, NT, 0, 1, 2>(c, a);
    else if (aux == 2) launch_k<T, NK1, NT, 0, 2, 2>(c, a);
    else launch_k<T, NK1, NT, 0, 3, 2>(c, a);
  } else if (mode == 2 && cpl == 1) {
    if (aux == 0) launch_k<T, NK1, NT, 1, 0, 2>(c, a);
    else if (aux == 2) launch_k<T, NK1, NT, 1, 2, 2>(c, a);
    else launch_k<T, NK1, NT, 1, 3, 2>(c, a);
  } else if (mode == 2) {
    if (aux & 1) launch_k<T, NK1, NT, 2, 3, 2>(c, a);
    else launch_k<T, NK1, NT, 2, 2, 2>(c, a);
  } else if (cpl == 0) {
    launch_k<T, NK1, NT, 0, 0, 1>(c, a);
  } else {
    launch_k<T, NK1, NT, 2, 0, 1>(c, a);
  }
}

template <typename T>
static hipError_t update(Ctx* c, const UpArgs& a, int nk1, int cpl, int aux, int mode) {
  if (c->up_nwaves == 0) return hipSuccess;
  if constexpr (sizeof(T) == 4) {
    if (c->up_nt == 2) launch_nk<T, 0, 2>(c, a, cpl, aux, mode);
    else launch_nk<T, 0, 1>(c, a, cpl, aux, mode);
  } else {
    switch (nk1) {
      case 0: launch_nk<T, 0, 1>(c, a, cpl, aux, mode); break;
      case 1: launch_nk<T, 1, 1>(c, a, cpl, aux, mode); break;
      case 3: launch_nk<T, 3, 1>(c, a, cpl, aux, mode); break;
      case 4: launch_nk<T, 4, 1>(c, a, cpl, aux, mode); break;
      default: return hipErrorInvalidValue;
    }
  }
  return hipGetLastError();
}

template <int NP>
static void launch_rr(Ctx* c, const RrArgs& a) {
  const unsigned nb = (unsigned)(c->t.nc * c->t.na * c->up_nk1);
  if (c->t.n2 % 16 == 0)
    hipLaunchKernelGGL((k_rad_rr<NP, true>), dim3(nb), dim3(512), 0, c->stream, a);
  else
    hipLaunchKernelGGL((k_rad_rr<NP, false>), dim3(nb), dim3(512), 0, c->stream, a);
}

}  // namespace step
}  // namespace mw3
