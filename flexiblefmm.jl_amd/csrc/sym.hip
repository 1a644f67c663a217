// The translations of the cube and the harmonic methods in the reflection symmetry of the cube.
//
// The surfaces of a box are lattices that the three reflections x -> -x, y -> -y, z -> -z
// map onto themselves, and the Laplace kernel is invariant under them.  With an even
// number of points per edge no point lies on a reflection plane, so the points form orbits
// of exactly 8: point (r, h) is orbit r's representative (the octant of smallest
// coordinates) with the coordinates of h's set bits reflected; the 8 children of a box are
// one orbit too.  In the basis of the orbits' Walsh-Hadamard transforms,
//   x^chi_r = sum_h (-1)^popcount(chi & h) x_(r, h),   chi = 0 .. 7,
// every operator that commutes with the reflections splits into 8 blocks, one per chi, an
// eighth of its size on each side: the pseudo-inverses (296 x 1352 at p = 8: 8 blocks of
// 37 x 169), M2M and L2L (296 x 2368: 8 blocks of 37 x 296, an input orbit being
// x_(c = d ^ h, r, h) over the children c).  So the products cost an eighth of the dense
// forms' (src/operators/ki_common.jl:52-68, 176-199), the butterflies 24 additions per 8
// values.  The blocks of the pseudo-inverses are factored by their own SVDs (U_chi, S_chi,
// V_chi); together these are a singular value decomposition of the whole check matrix, so
// P = V S^-1 U^T is applied factor by factor as before, with no folded pseudo-inverse.
//
// Small- and large-surface points are kept in orbit order (8 r + h) in device memory, so an
// orbit is 64 contiguous bytes.  Every kernel here is one workgroup of 8 waves per 16
// columns (nodes or sibling groups): wave chi multiplies block chi on the matrix cores
// (v_mfma_f64_16x16x4, the 16 columns being the tile's), the operands
// passing through LDS rows of 17 entries (stride 17: a lane per row writes, and a row of
// 16 columns reads, without bank conflicts).  Two workgroups share a CU, so that one's
// loads, potentials and butterflies run beside the other's products.
#include "ffmm_internal.h"

#include <algorithm>
#include <cmath>
#include <numeric>

namespace ffmm {

constexpr double C4PI = 0.07957747154594767;   // 1 / (4 pi)
constexpr int SY_TB = 512;                     // 8 waves: wave chi multiplies block chi
constexpr int SY_N = 16;                       // columns per workgroup
constexpr int SY_K = 64;                       // orbits per chunk
constexpr int SY_S = SY_N + 1;                 // LDS row stride

typedef double sy_f64x4 __attribute__((ext_vector_type(4)));
static __device__ __forceinline__ sy_f64x4 mma(double a, double b, sy_f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);   // lane (lk, li): rows lk + 4 e of column li
}

// v[chi] <- sum_h (-1)^popcount(chi & h) v[h]
__device__ __forceinline__ void wht8(double v[8]) {
#pragma unroll
  for (int b = 1; b < 8; b <<= 1)
#pragma unroll
    for (int i = 0; i < 8; i++)
      if (!(i & b)) {
        const double x = v[i], y = v[i | b];
        v[i] = x + y;
        v[i | b] = x - y;
      }
}

// lane d of 8 takes register h of lane d ^ h: v_(c, h) -> v_(d = c ^ h, h) and back
__device__ __forceinline__ void skew8(double v[8]) {
#pragma unroll
  for (int h = 1; h < 8; h++) v[h] = __shfl_xor(v[h], h, 64);
}

__device__ __forceinline__ void load8(const double *__restrict__ p, double v[8]) {
#pragma unroll
  for (int h = 0; h < 8; h += 2) {
    const double2 x = *reinterpret_cast<const double2 *>(p + h);
    v[h] = x.x;
    v[h + 1] = x.y;
  }
}
__device__ __forceinline__ void store8(double *__restrict__ p, const double v[8]) {
#pragma unroll
  for (int h = 0; h < 8; h += 2) *reinterpret_cast<double2 *>(p + h) = make_double2(v[h], v[h + 1]);
}

// acc += A[.., k] X[k, ..] over ng groups of 4 k-steps: A (k-major, row stride R) at this
// lane's (lk, li), X in LDS at this wave's block.  The next group's operator rows are
// loaded before this group's products (12 MFMAs of 64 cycles at p = 8: longer than an L2
// round trip); the operator copies are padded by a group, so the last prefetch stays inside.
template <int RT>
__device__ __forceinline__ void mma_chunk(sy_f64x4 acc[RT], const double *__restrict__ A, const double *X, int ng, int lk,
                                          int li) {
  constexpr int R = 16 * RT;
  double a[4][RT], an[4][RT];
#pragma unroll
  for (int s = 0; s < 4; s++)
#pragma unroll
    for (int i = 0; i < RT; i++) a[s][i] = A[(size_t)4 * s * R + 16 * i];
  for (int g = 0; g < ng; g++) {
    A += (size_t)16 * R;
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int i = 0; i < RT; i++) an[s][i] = A[(size_t)4 * s * R + 16 * i];
    double b[4];
#pragma unroll
    for (int s = 0; s < 4; s++) b[s] = X[(16 * g + 4 * s + lk) * SY_S + li];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int i = 0; i < RT; i++) acc[i] = mma(a[s][i], b[s], acc[i]);
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int i = 0; i < RT; i++) a[s][i] = an[s][i];
  }
}

// this wave's rows of a product (RT tiles) into its LDS block
template <int RT>
__device__ __forceinline__ void put_rows(double *X, const sy_f64x4 acc[RT], int lk, int li) {
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int e = 0; e < 4; e++) X[(16 * i + lk + 4 * e) * SY_S + li] = acc[i][e];
}

// LDS accesses of one wave are in order; this keeps the compiler from moving them
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------
// S2M: the check potentials at the 8 points of an orbit (representative a, reflections
// -a), transformed.  The squared differences of a coordinate are shared by the 4 points
// with that sign, so an orbit takes 20 FP32 operations and 8 rsq where 8 separate points
// take 48 and 8.  The mixed form: FP32 terms over at most 256 sources folded into FP64
// (positions relative to the node centre, differences formed in FP64 and rounded once).
// ---------------------------------------------------------------------------
template <bool F32> struct SySrc;
template <> struct SySrc<true> {
  using T = float4;
  using S = float;
  static constexpr int CAP = 640;
};
template <> struct SySrc<false> {
  using T = double4;
  using S = double;
  static constexpr int CAP = 320;
};
constexpr int SY_FOLD = 256;   // FP32 terms per fold

template <bool F32, class Fetch>
__device__ __forceinline__ void orbit_potentials(double a0, double a1, double a2, int32_t j0, int32_t j1, int32_t step,
                                                 Fetch &&src, double v[8]) {
  using S = typename SySrc<F32>::S;
  const S x0 = (S)a0, y0 = (S)a1, z0 = (S)a2;
#pragma unroll
  for (int h = 0; h < 8; h++) v[h] = 0.0;
  auto add = [&](const typename SySrc<F32>::T &s, S part[8]) {
    const S xm = x0 - s.x, xp = -x0 - s.x, ym = y0 - s.y, yp = -y0 - s.y, zm = z0 - s.z, zp = -z0 - s.z;
    const S qx[2] = {xm * xm, xp * xp};
    S qxy[4];
#pragma unroll
    for (int h = 0; h < 4; h++) qxy[h] = fma(h & 2 ? yp : ym, h & 2 ? yp : ym, qx[h & 1]);
#pragma unroll
    for (int h = 0; h < 8; h++) {
      const S r2 = fma(h & 4 ? zp : zm, h & 4 ? zp : zm, qxy[h & 3]);
      if constexpr (F32) part[h] = fmaf(__builtin_amdgcn_rsqf(r2), s.w, part[h]);
      else part[h] = fma(rsqrt_f64(r2), s.w, part[h]);
    }
  };
  if constexpr (F32) {
    for (int32_t jb = j0; jb < j1; jb += SY_FOLD * step) {
      const int32_t je = min(j1, jb + SY_FOLD * step);
      float part[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int32_t j = jb; j < je; j += step) add(src(j), part);
#pragma unroll
      for (int h = 0; h < 8; h++) v[h] += (double)part[h];
    }
  } else {
    for (int32_t j = j0; j < j1; j += step) add(src(j), v);
  }
#pragma unroll
  for (int h = 0; h < 8; h++) v[h] *= C4PI;
}

struct SyNodes {               // the childless sourced nodes and the sorted points
  const int32_t *nodes;
  int64_t nq, nn;
  const double *centers, *lam;
  const int32_t *level, *plo, *phi;
  const double *sx, *sy, *sz, *tau;
  const double *rep;           // 3 x nk: the orbits' representatives at the reference width
  int nk;
};

// The transformed check potentials of a few nodes, pMh[(q 8 + chi) KP + k] (0 for
// nk <= k < KP): one workgroup per (node, 64 orbits), its 4 waves splitting the sources.
// Used where 16 nodes per workgroup of the fused kernel would leave CUs idle.
template <bool F32>
__global__ void __launch_bounds__(256) k_sym_s2m(SyNodes a, int KP, double *__restrict__ pMh) {
  __shared__ double red[3][8][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t q = blockIdx.x;
  const int k = blockIdx.y * SY_K + lane;
  const int node = a.nodes[q];
  const double c0 = a.centers[node], c1 = a.centers[a.nn + node], c2 = a.centers[2 * a.nn + node];
  const double sc = a.lam[a.level[node]];
  const int kk = min(k, a.nk - 1);
  double v[8];
  orbit_potentials<F32>(a.rep[kk] * sc, a.rep[a.nk + kk] * sc, a.rep[2 * a.nk + kk] * sc, a.plo[node] + w,
                        a.phi[node] + 1, 4,
                        [&](int32_t j) -> typename SySrc<F32>::T {
                          using S = typename SySrc<F32>::S;
                          return {(S)(a.sx[j] - c0), (S)(a.sy[j] - c1), (S)(a.sz[j] - c2), (S)a.tau[j]};
                        },
                        v);
  if (w > 0)
#pragma unroll
    for (int h = 0; h < 8; h++) red[w - 1][h][lane] = v[h];
  __syncthreads();
  if (w > 0) return;
#pragma unroll
  for (int h = 0; h < 8; h++) v[h] = k < a.nk ? ((v[h] + red[0][h][lane]) + red[1][h][lane]) + red[2][h][lane] : 0.0;
  wht8(v);
#pragma unroll
  for (int h = 0; h < 8; h++) pMh[(q * 8 + h) * KP + k] = v[h];
}

// UC2E: M = lam V_chi S_chi^-1 (U_chi^T p_chi) (src/device_passes.jl:496-502), with S2M
// inside (MODE 0: FP64, 1: mixed) or from pMh (MODE 2).  Per chunk of 64 orbits the waves
// form the transformed potentials of their nodes (a lane per orbit, a node per wave: every
// source read is an LDS broadcast), then each wave multiplies its block.
template <int MODE, int NR>
__global__ void __launch_bounds__(SY_TB, 4) k_sym_uc2e(SyNodes a, const double *__restrict__ A1,
                                                       const double *__restrict__ A2, int KP,
                                                       const double *__restrict__ pMh, double *__restrict__ Mp) {
  constexpr int RT = (NR + 15) / 16, R = 16 * RT, KG = (NR + 15) / 16;   // k groups of 16 of the second factor
  constexpr bool F32 = MODE == 1;
  using ST = typename SySrc<F32>::T;
  using S = typename SySrc<F32>::S;
  constexpr int CAP = MODE == 2 ? 1 : SySrc<F32>::CAP;
  __shared__ double P[8][SY_K * SY_S];
  __shared__ __attribute__((aligned(16))) ST src[CAP];
  __shared__ int32_t off[SY_N + 1], first[SY_N], nid[SY_N];
  __shared__ double scl[SY_N], ctr[3][SY_N];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int64_t q0 = (int64_t)blockIdx.x * SY_N;
  if (t < 64) {
    const int64_t q = q0 + t;
    int32_t cnt = 0;
    if (t < SY_N) {
      int32_t p = 0;
      double s = 0.0, c[3] = {0.0, 0.0, 0.0};
      int node = -1;
      if (q < a.nq) {
        node = a.nodes[q];
        s = a.lam[a.level[node]];
        if (MODE != 2) {
          p = a.plo[node];
          cnt = a.phi[node] - p + 1;
          for (int d = 0; d < 3; d++) c[d] = a.centers[d * a.nn + node];
        }
      }
      nid[t] = node;
      scl[t] = s;
      first[t] = p;
      for (int d = 0; d < 3; d++) ctr[d][t] = c[d];
    }
    int32_t v = cnt;
#pragma unroll
    for (int o = 1; o < SY_N; o <<= 1) {
      const int32_t u = __shfl_up(v, o, 64);
      if (lane >= o) v += u;
    }
    if (t < SY_N) off[t + 1] = v;
    if (t == 0) off[0] = 0;
  }
  __syncthreads();
  const int32_t total = MODE == 2 ? 0 : off[SY_N];
  const bool staged = total <= CAP;
  if (MODE != 2 && staged) {
    for (int32_t i = t; i < total; i += SY_TB) {
      int n = 0;
#pragma unroll
      for (int m = SY_N / 2; m > 0; m >>= 1)
        if (off[n + m] <= i) n += m;
      const int32_t j = first[n] + (i - off[n]);
      src[i] = ST{(S)(a.sx[j] - ctr[0][n]), (S)(a.sy[j] - ctr[1][n]), (S)(a.sz[j] - ctr[2][n]), (S)a.tau[j]};
    }
    __syncthreads();
  }
  sy_f64x4 acc[RT];
#pragma unroll
  for (int i = 0; i < RT; i++) acc[i] = sy_f64x4{0.0, 0.0, 0.0, 0.0};
  const double *A = A1 + ((size_t)w * KP + lk) * R + li;
  for (int k0 = 0; k0 < a.nk; k0 += SY_K) {
    const int k = k0 + lane;
    const int kk = min(k, a.nk - 1);
    double r0 = 0.0, r1 = 0.0, r2 = 0.0;
    if (MODE != 2) {
      r0 = a.rep[kk];
      r1 = a.rep[a.nk + kk];
      r2 = a.rep[2 * a.nk + kk];
    }
    if (k0 > 0) lds_barrier();   // the previous chunk's products have read P
#pragma unroll
    for (int m = 0; m < SY_N / 8; m++) {
      const int n = w + 8 * m;
      double v[8];
      if constexpr (MODE == 2) {
        const double *__restrict__ p = pMh + (q0 + n) * 8 * (int64_t)KP + k;
#pragma unroll
        for (int h = 0; h < 8; h++) v[h] = q0 + n < a.nq ? p[(int64_t)h * KP] : 0.0;
      } else {
        const double sc = scl[n];
        const int32_t j0 = off[n], j1 = off[n + 1];
        if (staged) {
          orbit_potentials<F32>(r0 * sc, r1 * sc, r2 * sc, j0, j1, 1, [&](int32_t j) -> ST { return src[j]; }, v);
        } else {
          const int32_t f = first[n] - j0;
          const double c0 = ctr[0][n], c1 = ctr[1][n], c2 = ctr[2][n];
          orbit_potentials<F32>(r0 * sc, r1 * sc, r2 * sc, j0, j1, 1,
                                [&](int32_t j) -> ST {
                                  const int32_t g = f + j;
                                  return ST{(S)(a.sx[g] - c0), (S)(a.sy[g] - c1), (S)(a.sz[g] - c2), (S)a.tau[g]};
                                },
                                v);
        }
        if (k >= a.nk)
#pragma unroll
          for (int h = 0; h < 8; h++) v[h] = 0.0;
        wht8(v);
      }
#pragma unroll
      for (int h = 0; h < 8; h++) P[h][lane * SY_S + n] = v[h];
    }
    lds_barrier();
    mma_chunk<RT>(acc, A + (size_t)k0 * R, P[w], (min(SY_K, a.nk - k0) + 15) / 16, lk, li);
  }
  // the second factor, through this wave's own block of P (only it reads and writes there)
  wave_lds_fence();
  put_rows<RT>(P[w], acc, lk, li);
  wave_lds_fence();
  sy_f64x4 out[RT];
#pragma unroll
  for (int i = 0; i < RT; i++) out[i] = sy_f64x4{0.0, 0.0, 0.0, 0.0};
  mma_chunk<RT>(out, A2 + ((size_t)w * (R + 16) + lk) * R + li, P[w], KG, lk, li);
  wave_lds_fence();
  put_rows<RT>(P[w], out, lk, li);
  lds_barrier();
  // back to the points (the transform's 1/8 is in A2), scaled by the level's power of two
  for (int i = t; i < SY_N * NR; i += SY_TB) {
    const int n = i / NR, r = i % NR;
    if (nid[n] < 0) continue;
    double v[8];
#pragma unroll
    for (int h = 0; h < 8; h++) v[h] = P[h][r * SY_S + n];
    wht8(v);
#pragma unroll
    for (int h = 0; h < 8; h++) v[h] *= scl[n];
    store8(Mp + ((int64_t)nid[n] * NR + r) * 8, v);
  }
}

// M2M of a level's sibling groups: the parents' multipoles from their 8 children's, in FP64
// in both forms (the FP64 multipoles are what it reads: bound by memory, FP32 products
// would not be faster).  Chunks of 8 orbits of the 8 children: lane (r, c) loads its child's
// orbit, the lanes exchange so that lane (r, d) holds x_(d ^ h, r, h), and transforms it.
template <int NR>
__global__ void __launch_bounds__(SY_TB, 4) k_sym_m2m(const double *__restrict__ B, int KP,
                                                      const int32_t *__restrict__ parent,
                                                      const uint8_t *__restrict__ has_source, int64_t first, int64_t ng,
                                                      double *__restrict__ Mp) {
  constexpr int RT = (NR + 15) / 16, R = 16 * RT;
  __shared__ double P[8][SY_K * SY_S];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int64_t g0 = (int64_t)blockIdx.x * SY_N;
  const int rl = lane >> 3, c = lane & 7;
  sy_f64x4 acc[RT];
#pragma unroll
  for (int i = 0; i < RT; i++) acc[i] = sy_f64x4{0.0, 0.0, 0.0, 0.0};
  bool live[SY_N / 8];
#pragma unroll
  for (int m = 0; m < SY_N / 8; m++) {
    const int64_t g = g0 + w + 8 * m;
    live[m] = g < ng && has_source[first + NCHILD * g + c];
  }
  const double *A = B + ((size_t)w * KP + lk) * R + li;
  for (int r0 = 0; r0 < NR; r0 += 8) {
    double v[SY_N / 8][8];
#pragma unroll
    for (int m = 0; m < SY_N / 8; m++) {
#pragma unroll
      for (int h = 0; h < 8; h++) v[m][h] = 0.0;
      if (live[m] && r0 + rl < NR) load8(Mp + ((first + NCHILD * (g0 + w + 8 * m) + c) * NR + r0 + rl) * 8, v[m]);
      skew8(v[m]);
      wht8(v[m]);
    }
    if (r0 > 0) lds_barrier();
#pragma unroll
    for (int m = 0; m < SY_N / 8; m++)
#pragma unroll
      for (int h = 0; h < 8; h++) P[h][lane * SY_S + w + 8 * m] = v[m][h];
    lds_barrier();
    mma_chunk<RT>(acc, A + (size_t)r0 * 8 * R, P[w], (min(8, NR - r0) * 8 + 15) / 16, lk, li);
  }
  wave_lds_fence();
  put_rows<RT>(P[w], acc, lk, li);
  lds_barrier();
  for (int i = t; i < SY_N * NR; i += SY_TB) {
    const int n = i / NR, r = i % NR;
    if (g0 + n >= ng) continue;
    double v[8];
#pragma unroll
    for (int h = 0; h < 8; h++) v[h] = P[h][r * SY_S + n];
    wht8(v);
    store8(Mp + ((int64_t)parent[first + NCHILD * (g0 + n)] * NR + r) * 8, v);
  }
}

// The downward operators: input columns of NR orbits, transformed into LDS; wave chi keeps
// its operand (NR rows, 16 columns) in registers; the output rows in chunks of 64.
//   MODE 0, L2L: the children's partial locals of a sibling group from the parent's
//     (output row 8 r + d of block chi: orbit r of the children c = d ^ h);
//   MODE 1, DC2E: U_chi S_chi^-1 (V_chi^T lam l_chi) of a leaf (src/device_passes.jl:583-593),
//     output row k: orbit k of the large surface.
struct SyDown {
  const double *A1;            // MODE 1: V_chi^T
  const double *A2;            // k-major, row stride RP
  int RP, nrow;                // padded and actual output rows
  const int32_t *col;          // MODE 0: the parents (of sibling group g: col[first + 8 g]); MODE 1: the leaves
  int64_t first, n;
  const int32_t *level;
  const double *lam;
  const double *in;
  double *out;
};
template <int MODE, int NR>
__global__ void __launch_bounds__(SY_TB, 4) k_sym_down(SyDown a) {
  constexpr int RT = (NR + 15) / 16, R = 16 * RT, KS = (NR + 3) / 4;
  constexpr int ROWS = R > SY_K ? R : SY_K;
  __shared__ double P[8][ROWS * SY_S];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int64_t q0 = (int64_t)blockIdx.x * SY_N;
  for (int i = t; i < SY_N * R; i += SY_TB) {
    const int n = i / R, r = i % R;
    const int64_t q = q0 + n;
    double v[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (q < a.n && r < NR) {
      const int32_t c = MODE == 0 ? a.col[a.first + NCHILD * q] : a.col[q];
      load8(a.in + ((int64_t)c * NR + r) * 8, v);
      if (MODE == 1) {
        const double s = a.lam[a.level[c]];
#pragma unroll
        for (int h = 0; h < 8; h++) v[h] *= s;
      }
      wht8(v);
    }
#pragma unroll
    for (int h = 0; h < 8; h++) P[h][r * SY_S + n] = v[h];
  }
  lds_barrier();
  if (MODE == 1) {
    sy_f64x4 acc[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) acc[i] = sy_f64x4{0.0, 0.0, 0.0, 0.0};
    mma_chunk<RT>(acc, a.A1 + ((size_t)w * (R + 16) + lk) * R + li, P[w], RT, lk, li);
    wave_lds_fence();
    put_rows<RT>(P[w], acc, lk, li);
    wave_lds_fence();
  }
  double b[KS];
#pragma unroll
  for (int s = 0; s < KS; s++) b[s] = P[w][(4 * s + lk) * SY_S + li];
  wave_lds_fence();
  const double *A = a.A2 + ((size_t)w * 4 * KS + lk) * a.RP + li;
  for (int k0 = 0; k0 < a.nrow; k0 += SY_K) {
    sy_f64x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = sy_f64x4{0.0, 0.0, 0.0, 0.0};
    const int nt = (min(SY_K, a.nrow - k0) + 15) / 16;
    if (nt == 4) {
#pragma unroll
      for (int s = 0; s < KS; s++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = mma(A[(size_t)4 * s * a.RP + k0 + 16 * i], b[s], acc[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 3; i++)
        if (i < nt)
#pragma unroll
          for (int s = 0; s < KS; s++) acc[i] = mma(A[(size_t)4 * s * a.RP + k0 + 16 * i], b[s], acc[i]);
    }
    if (k0 > 0) lds_barrier();   // the previous chunk's rows are read
    put_rows<4>(P[w], acc, lk, li);
    lds_barrier();
#pragma unroll
    for (int m = 0; m < SY_N / 8; m++) {
      const int n = w + 8 * m, row = k0 + lane;
      const int64_t q = q0 + n;
      double v[8];
#pragma unroll
      for (int h = 0; h < 8; h++) v[h] = P[h][lane * SY_S + n];
      wht8(v);                     // the transform's 1/8 is in A2
      if (MODE == 0) skew8(v);     // lane (r, d) holds the children d ^ h: back to lane (r, c)
      if (q < a.n && row < a.nrow) {
        if (MODE == 0) store8(a.out + ((a.first + NCHILD * q + (lane & 7)) * NR + (row >> 3)) * 8, v);
        else store8(a.out + (q * a.nrow + row) * 8, v);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The harmonic methods: a solid harmonic has a parity under each reflection, so entry i of
// an expansion belongs to one block chi_i, and the translation of child c is that of child 0
// with signs, A_c[i, j] = chi_i(c) chi_j(c) A_0[i, j].  So M2M is
//   out_i = sum_j A_0[i, j] W[chi_i ^ chi_j, j],  W[psi, j] = sum_c (-1)^popcount(psi & c) m_(c, j)
// (block chi: its rows of A_0 against N transformed entries), and L2L
//   y_(c, i) = chi_i(c) sum_psi (-1)^popcount(psi & c) sum_(j in psi) B_0[i, j] l_j:
// N^2 products per column where the dense forms take 8 N^2 (Stokes: 128 N^2 per 4 columns).
// Stokes: the four blocks are columns of the same operator; the coupling of the fourth with
// the child's offset d is applied to the children before M2M (m_4 / 2 + d . m) and to the
// children after L2L (2 y_4 - 2 d . y) (src/operators/harmonics_stokes.jl:112-131).
// 16 columns per workgroup: 16 groups, or 4 groups of 4 blocks.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double child_offset(int c, int a) { return (c >> a) & 1 ? 0.25 : -0.25; }

template <int RT, int NB>
__global__ void __launch_bounds__(SY_TB, 4) k_harm_m2m(const double *__restrict__ B, int N, int KP,
                                                       const uint8_t *__restrict__ chi,
                                                       const uint8_t *__restrict__ rank,
                                                       const int32_t *__restrict__ parent,
                                                       const uint8_t *__restrict__ has_source, int64_t first, int64_t ng,
                                                       double *__restrict__ Mp) {
  constexpr int R = 16 * RT, G = SY_N / NB;
  __shared__ double P[8][SY_K * SY_S];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int64_t g0 = (int64_t)blockIdx.x * G;
  sy_f64x4 acc[RT];
#pragma unroll
  for (int i = 0; i < RT; i++) acc[i] = sy_f64x4{0.0, 0.0, 0.0, 0.0};
  const double *A = B + ((size_t)w * KP + lk) * R + li;
  for (int k0 = 0; k0 < N; k0 += SY_K) {
    const int j = k0 + lane;
    const int cj = j < N ? chi[j] : 0;
    if (k0 > 0) lds_barrier();
    auto put = [&](double v[8], int col) {
      wht8(v);
#pragma unroll
      for (int h = 0; h < 8; h++) P[h ^ cj][lane * SY_S + col] = v[h];
    };
    auto get = [&](int64_t g, int b, double v[8]) {
#pragma unroll
      for (int c = 0; c < 8; c++) {
        const int64_t node = first + NCHILD * g + c;
        v[c] = g < ng && j < N && has_source[node] ? Mp[(node * NB + b) * N + j] : 0.0;
      }
    };
    if constexpr (NB == 1) {
#pragma unroll
      for (int m = 0; m < 2; m++) {
        double v[8];
        get(g0 + w + 8 * m, 0, v);
        put(v, w + 8 * m);
      }
    } else {   // wave w: group w % 4, its blocks 0, 1 or 2, 3
      const int gl = w & 3;
      double v[8], u[8];
      get(g0 + gl, 0, v);
      if (w < 4) {
        put(v, 4 * gl);
        get(g0 + gl, 1, v);
        put(v, 4 * gl + 1);
      } else {
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = child_offset(c, 0) * v[c];
        get(g0 + gl, 1, v);
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = fma(child_offset(c, 1), v[c], u[c]);
        get(g0 + gl, 2, v);
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = fma(child_offset(c, 2), v[c], u[c]);
        put(v, 4 * gl + 2);
        get(g0 + gl, 3, v);
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = fma(0.5, v[c], u[c]);
        put(u, 4 * gl + 3);
      }
    }
    lds_barrier();
    mma_chunk<RT>(acc, A + (size_t)k0 * R, P[w], (min(SY_K, N - k0) + 15) / 16, lk, li);
  }
  wave_lds_fence();
  put_rows<RT>(P[w], acc, lk, li);
  lds_barrier();
  for (int e = t; e < SY_N * N; e += SY_TB) {
    const int col = e / N, i = e % N;
    const int64_t g = g0 + col / NB;
    if (g < ng) Mp[((int64_t)parent[first + NCHILD * g] * NB + col % NB) * N + i] = P[chi[i]][rank[i] * SY_S + col];
  }
}

template <int RT, int NB>
__global__ void __launch_bounds__(SY_TB, 4) k_harm_l2l(const double *__restrict__ B, int N, int RP,
                                                       const uint8_t *__restrict__ chi,
                                                       const uint8_t *__restrict__ rank,
                                                       const int32_t *__restrict__ parent, int64_t first, int64_t ng,
                                                       double *__restrict__ Pl) {
  constexpr int G = SY_N / NB, KS = 4 * RT;
  __shared__ double P[8][SY_K * SY_S];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int64_t g0 = (int64_t)blockIdx.x * G;
  for (int i = lane; i < 4 * KS * SY_S; i += 64) P[w][i] = 0.0;
  lds_barrier();
  for (int e = t; e < SY_N * N; e += SY_TB) {
    const int col = e / N, i = e % N;
    const int64_t g = g0 + col / NB;
    if (g < ng)
      P[chi[i]][rank[i] * SY_S + col] = Pl[((int64_t)parent[first + NCHILD * g] * NB + col % NB) * N + i];
  }
  lds_barrier();
  double b[KS];
#pragma unroll
  for (int s = 0; s < KS; s++) b[s] = P[w][(4 * s + lk) * SY_S + li];
  wave_lds_fence();
  const double *A = B + ((size_t)w * 4 * KS + lk) * RP + li;
  for (int k0 = 0; k0 < N; k0 += SY_K) {
    sy_f64x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = sy_f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
      for (int i = 0; i < 4; i++) acc[i] = mma(A[(size_t)4 * s * RP + k0 + 16 * i], b[s], acc[i]);
    if (k0 > 0) lds_barrier();
    put_rows<4>(P[w], acc, lk, li);
    lds_barrier();
    const int i = k0 + lane;
    const int ci = i < N ? chi[i] : 0;
    auto get = [&](int col, double v[8]) {   // the 8 children's values of a column
#pragma unroll
      for (int h = 0; h < 8; h++) v[h] = P[h][lane * SY_S + col];
      wht8(v);
#pragma unroll
      for (int c = 0; c < 8; c++) v[c] = __builtin_popcount(ci & c) & 1 ? -v[c] : v[c];
    };
    auto put = [&](int64_t g, int bl, const double v[8]) {
      if (g >= ng || i >= N) return;
#pragma unroll
      for (int c = 0; c < 8; c++) Pl[((first + NCHILD * g + c) * NB + bl) * N + i] = v[c];
    };
    if constexpr (NB == 1) {
#pragma unroll
      for (int m = 0; m < 2; m++) {
        double v[8];
        get(w + 8 * m, v);
        put(g0 + w + 8 * m, 0, v);
      }
    } else {
      const int gl = w & 3;
      double v[8], u[8];
      get(4 * gl, v);
      if (w < 4) {
        put(g0 + gl, 0, v);
        get(4 * gl + 1, v);
        put(g0 + gl, 1, v);
      } else {
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = -2.0 * child_offset(c, 0) * v[c];
        get(4 * gl + 1, v);
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = fma(-2.0 * child_offset(c, 1), v[c], u[c]);
        get(4 * gl + 2, v);
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = fma(-2.0 * child_offset(c, 2), v[c], u[c]);
        put(g0 + gl, 2, v);
        get(4 * gl + 3, v);
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = fma(2.0, v[c], u[c]);
        put(g0 + gl, 3, u);
      }
    }
  }
}

// the columns of nodes without sources are zero (nothing writes them)
__global__ void k_sym_zero(const uint8_t *__restrict__ has_source, int64_t nn, int Ns, double *__restrict__ Mp) {
  const int lane = threadIdx.x & 63;
  const int64_t base = ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 64;
  const bool z = base + lane < nn && !has_source[base + lane];
  for (uint64_t m = __ballot(z); m; m &= m - 1) {
    double *__restrict__ p = Mp + (base + __builtin_ctzll(m)) * Ns;
    for (int i = lane; i < Ns; i += 64) p[i] = 0.0;
  }
}

// ---------------------------------------------------------------------------
// host side: the orbits, and the blocks of the operators
// ---------------------------------------------------------------------------
// the boundary points of the n^3 lattice (coordinate 0 fastest), in orbit order: perm[8 r +
// h] = the lattice-order index of orbit r's representative with h's coordinates reflected
std::vector<int32_t> sym_orbits(int n) {
  std::vector<int32_t> id((size_t)n * n * n, -1), perm;
  int32_t m = 0;
  for (int k = 0; k < n * n * n; k++) {
    const int i[3] = {k % n, (k / n) % n, k / (n * n)};
    for (int d = 0; d < 3; d++)
      if (i[d] == 0 || i[d] == n - 1) {
        id[k] = m++;
        break;
      }
  }
  for (int k = 0; k < n * n * n; k++) {
    const int i[3] = {k % n, (k / n) % n, k / (n * n)};
    if (id[k] < 0 || i[0] >= n / 2 || i[1] >= n / 2 || i[2] >= n / 2) continue;
    for (int h = 0; h < 8; h++) {
      int j[3];
      for (int d = 0; d < 3; d++) j[d] = (h >> d) & 1 ? n - 1 - i[d] : i[d];
      perm.push_back(id[j[0] + n * (j[1] + n * j[2])]);
    }
  }
  return perm;
}

// One-sided Jacobi: A (m x n, column major, m >= n) = U diag(s) V^T; A becomes U, V n x n.
// False when U's columns are not orthogonal to 1e-12 after 60 sweeps, or A has no full rank.
static bool jacobi_svd(std::vector<double> &A, int m, int n, std::vector<double> &s, std::vector<double> &V) {
  V.assign((size_t)n * n, 0.0);
  for (int i = 0; i < n; i++) V[(size_t)i * n + i] = 1.0;
  double worst = 0.0;            // the largest cosine that the last sweep met
  for (int sweep = 0; sweep < 60; sweep++) {
    bool done = true;
    worst = 0.0;
    for (int i = 0; i < n - 1; i++)
      for (int j = i + 1; j < n; j++) {
        double *x = &A[(size_t)i * m], *y = &A[(size_t)j * m];
        double aa = 0.0, bb = 0.0, ab = 0.0;
        for (int k = 0; k < m; k++) {
          aa += x[k] * x[k];
          bb += y[k] * y[k];
          ab += x[k] * y[k];
        }
        if (std::abs(ab) <= 1e-15 * std::sqrt(aa * bb)) continue;
        done = false;
        worst = std::max(worst, std::abs(ab) / std::sqrt(aa * bb));
        const double z = (bb - aa) / (2.0 * ab);
        const double tn = (z >= 0.0 ? 1.0 : -1.0) / (std::abs(z) + std::sqrt(1.0 + z * z));
        const double cs = 1.0 / std::sqrt(1.0 + tn * tn), sn = cs * tn;
        auto rot = [&](double *p, double *q, int len) {
          for (int k = 0; k < len; k++) {
            const double u = p[k], v = q[k];
            p[k] = cs * u - sn * v;
            q[k] = sn * u + cs * v;
          }
        };
        rot(x, y, m);
        rot(&V[(size_t)i * n], &V[(size_t)j * n], n);
      }
    if (done) break;
  }
  s.resize(n);
  for (int i = 0; i < n; i++) {
    double q = 0.0;
    for (int k = 0; k < m; k++) q += A[(size_t)i * m + k] * A[(size_t)i * m + k];
    s[i] = std::sqrt(q);
    if (!(s[i] > 0.0)) return false;
    for (int k = 0; k < m; k++) A[(size_t)i * m + k] /= s[i];
  }
  return worst <= 1e-12;
}

static inline double chi_sign(int chi, int h) { return __builtin_popcount(chi & h) & 1 ? -1.0 : 1.0; }

// whether the cube operators of this cache split: even orders within the kernels' sizes,
// pseudo-inverses of full rank (a truncated one keeps its given factors)
bool sym_fits(int p, int pc, int Ns, int r_up, int r_dn) {
  return (p == 2 || p == 4 || p == 6 || p == 8 || p == 10) && pc % 2 == 0 && r_up == Ns && r_dn == Ns;
}

// Whether the given operators are those the blocks stand for, to rounding; a cache given
// others (a regularised inverse, say) keeps them, dense.  Checked on vectors, against the
// Laplace matrix K from the small to the large surface, with everything in the given order:
//   the factors of P_up and P_down are singular value decompositions of K and K^T: U S V^T x
//     = K x to 1e-13 s_1 |x|, U and V orthonormal to 1e-12;
//   M2M and L2L commute with the reflections, M2M in the potentials K M2M x, L2L on
//     potentials K^T y, to 1e-11 (their own entries keep the inverses' amplified rounding,
//     1e-7 at p = 8, which neither sees).
// Operators of level_operators measure 5e-16, 4e-15 and at most 1.6e-13 (p = 2 .. 10, d = 0.01
// .. 0.6).
bool sym_matches(const OpCache &o, const double *small, const double *large, const SymGiven &g) {
  const int Ns = o.Ns, Nl = o.Nl, C = NCHILD;
  const std::vector<int32_t> os = sym_orbits(o.p);
  uint64_t seed = 1;
  auto vec = [&](int n) {
    std::vector<double> x(n);
    for (double &v : x) {
      seed = seed * 6364136223846793005ull + 1442695040888963407ull;
      v = (double)(int64_t)(seed >> 11) / 4503599627370496.0 - 1.0;
    }
    return x;
  };
  // y = A x and A^T x, A (m x n, column major)
  auto mul = [](const double *A, int m, int n, const std::vector<double> &x) {
    std::vector<double> y(m, 0.0);
    for (int j = 0; j < n; j++)
      for (int i = 0; i < m; i++) y[i] += A[(size_t)j * m + i] * x[j];
    return y;
  };
  auto tmul = [](const double *A, int m, int n, const std::vector<double> &x) {
    std::vector<double> y(n, 0.0);
    for (int j = 0; j < n; j++)
      for (int i = 0; i < m; i++) y[j] += A[(size_t)j * m + i] * x[i];
    return y;
  };
  auto norm = [](const std::vector<double> &x) {
    double q = 0.0;
    for (double v : x) q += v * v;
    return std::sqrt(q);
  };
  auto differ = [](const std::vector<double> &x, const std::vector<double> &y) {
    double q = 0.0;
    for (size_t i = 0; i < x.size(); i++) q += (x[i] - y[i]) * (x[i] - y[i]);
    return std::sqrt(q);
  };
  std::vector<double> K((size_t)Nl * Ns);
  for (int r = 0; r < Ns; r++)
    for (int k = 0; k < Nl; k++) {
      double r2 = 0.0;
      for (int d = 0; d < 3; d++) {
        const double e = large[3 * (size_t)k + d] - small[3 * (size_t)r + d];
        r2 += e * e;
      }
      K[(size_t)r * Nl + k] = C4PI / std::sqrt(r2);
    }
  double s1 = 0.0;
  for (int i = 0; i < Ns; i++)
    if (!(g.invS_up[i] > 0.0 && g.invS_dn[i] > 0.0)) return false;
    else s1 = std::max(s1, 1.0 / g.invS_up[i]);
  for (int n = 0; n < 4; n++) {
    const std::vector<double> x = vec(Ns), y = vec(Nl), Kx = mul(K.data(), Nl, Ns, x), Ky = tmul(K.data(), Nl, Ns, y);
    // P_up = V S^-1 U^T: U^T is Uh_up (Ns x Nl), V is V_up (Ns x Ns)
    std::vector<double> t = tmul(g.V_up, Ns, Ns, x);
    if (!(differ(mul(g.V_up, Ns, Ns, t), x) <= 1e-12 * norm(x))) return false;
    for (int i = 0; i < Ns; i++) t[i] /= g.invS_up[i];
    const std::vector<double> u = tmul(g.Uh_up, Ns, Nl, t);
    if (!(differ(mul(g.Uh_up, Ns, Nl, u), t) <= 1e-12 * norm(t))) return false;
    if (!(differ(u, Kx) <= 1e-13 * s1 * norm(x))) return false;
    // P_down = V S^-1 U^T of K^T = U S V^T: V_dn (Nl x Ns), Uh_dn (Ns x Ns)
    t = tmul(g.V_dn, Nl, Ns, y);
    for (int i = 0; i < Ns; i++) t[i] /= g.invS_dn[i];
    const std::vector<double> w = tmul(g.Uh_dn, Ns, Ns, t);
    if (!(differ(mul(g.Uh_dn, Ns, Ns, w), t) <= 1e-12 * norm(t))) return false;
    if (!(differ(tmul(g.V_dn, Nl, Ns, mul(g.V_dn, Nl, Ns, x)), x) <= 1e-12 * norm(x))) return false;
    if (!(differ(w, Ky) <= 1e-13 * s1 * norm(y))) return false;
  }
  for (int f = 1; f < 8; f <<= 1) {   // the reflection of one coordinate
    std::vector<int32_t> at(Ns);
    for (int i = 0; i < Ns; i++) at[os[i]] = os[i ^ f];
    auto points = [&](const std::vector<double> &a) {
      std::vector<double> b(a.size());
      for (int i = 0; i < Ns; i++) b[at[i]] = a[i];
      return b;
    };
    auto children = [&](const std::vector<double> &a) {
      std::vector<double> b(a.size());
      for (int c = 0; c < C; c++)
        for (int i = 0; i < Ns; i++) b[(size_t)(c ^ f) * Ns + at[i]] = a[(size_t)c * Ns + i];
      return b;
    };
    const std::vector<double> x = vec(C * Ns);
    std::vector<double> a = mul(K.data(), Nl, Ns, points(mul(g.M2M, Ns, C * Ns, x)));
    if (!(differ(a, mul(K.data(), Nl, Ns, mul(g.M2M, Ns, C * Ns, children(x)))) <= 1e-11 * norm(a))) return false;
    const std::vector<double> l = tmul(K.data(), Nl, Ns, vec(Nl));
    a = children(mul(g.L2L, C * Ns, Ns, l));
    if (!(differ(a, mul(g.L2L, C * Ns, Ns, points(l))) <= 1e-11 * norm(a))) return false;
  }
  return true;
}

// The blocks' singular value decompositions from the surfaces in orbit order; false when one
// of them did not converge.
bool sym_factor(const OpCache &o, const std::vector<double> &small, const std::vector<double> &large, SymFactors &f) {
  const int nr = o.Ns / 8, nk = o.Nl / 8;
  for (int chi = 0; chi < 8; chi++) {
    // K_chi[k, r] = sum_h chi(h) K(x_(k, h), y_(r, 0))
    std::vector<double> &U = f.U[chi];
    U.assign((size_t)nk * nr, 0.0);
    for (int r = 0; r < nr; r++)
      for (int k = 0; k < nk; k++)
        for (int h = 0; h < 8; h++) {
          double r2 = 0.0;
          for (int d = 0; d < 3; d++) {
            const double e = large[3 * (size_t)(8 * k) + d] * ((h >> d) & 1 ? -1.0 : 1.0) - small[3 * (size_t)(8 * r) + d];
            r2 += e * e;
          }
          U[(size_t)r * nk + k] += chi_sign(chi, h) * C4PI / std::sqrt(r2);
        }
    if (!jacobi_svd(U, nk, nr, f.S[chi], f.V[chi])) return false;
  }
  return true;
}

// The operators' blocks, from those factors and the folded M2M / L2L in orbit order (M2M: Ns
// x 8 Ns, L2L: 8 Ns x Ns, column major), averaged over the reflections (their own rounding
// is not symmetric).
void sym_setup(OpCache &o, const SymFactors &f, const std::vector<double> &large, const std::vector<double> &M2M,
               const std::vector<double> &L2L) {
  const int nr = o.Ns / 8, nk = o.Nl / 8, Ns = o.Ns;
  const int R = (nr + 15) / 16 * 16, KP = (nk + SY_K - 1) / SY_K * SY_K, KP2 = (Ns + SY_K - 1) / SY_K * SY_K;
  const int K4 = (nr + 3) / 4 * 4;
  hipStream_t s = o.ctx->stream;
  o.sym_kp = KP;
  o.sym_kp2 = KP2;
  std::vector<double> rep(3 * (size_t)nk);
  for (int k = 0; k < nk; k++)
    for (int d = 0; d < 3; d++) rep[(size_t)d * nk + k] = large[3 * (size_t)(8 * k) + d];
  // each operator padded by one prefetch group of 16 k
  std::vector<double> u1(8 * (size_t)KP * R + 16 * R, 0.0), u2(8 * (size_t)(R + 16) * R + 16 * R, 0.0), d1 = u2,
      d2(8 * (size_t)K4 * KP, 0.0), mm(8 * (size_t)KP2 * R + 16 * R, 0.0), ll(8 * (size_t)K4 * KP2, 0.0);
  for (int chi = 0; chi < 8; chi++) {
    const std::vector<double> &U = f.U[chi], &S = f.S[chi], &V = f.V[chi];
    for (int i = 0; i < nr; i++) {
      for (int k = 0; k < nk; k++) {
        u1[((size_t)chi * KP + k) * R + i] = U[(size_t)i * nk + k];
        d2[((size_t)chi * K4 + i) * KP + k] = U[(size_t)i * nk + k] / S[i] / 8.0;
      }
      for (int r = 0; r < nr; r++) {
        u2[((size_t)chi * (R + 16) + i) * R + r] = V[(size_t)i * nr + r] / S[i] / 8.0;
        d1[((size_t)chi * (R + 16) + r) * R + i] = V[(size_t)i * nr + r];
      }
    }
    for (int r1 = 0; r1 < nr; r1++)
      for (int r = 0; r < nr; r++)
        for (int d = 0; d < 8; d++) {
          double am = 0.0, al = 0.0;
          for (int h = 0; h < 8; h++) {
            double xm = 0.0, xl = 0.0;   // the mean over the reflections g
            for (int g = 0; g < 8; g++) {
              xm += M2M[((size_t)(d ^ h ^ g) * Ns + 8 * r + (h ^ g)) * Ns + 8 * r1 + g];
              xl += L2L[(size_t)(8 * r1 + (h ^ g)) * (8 * Ns) + (size_t)(d ^ g) * Ns + 8 * r + g];
            }
            am += chi_sign(chi, h) * xm;
            al += chi_sign(chi, h) * xl;
          }
          mm[((size_t)chi * KP2 + 8 * r + d) * R + r1] = am / 64.0;   // 1/8 of the mean, 1/8 of the transform
          ll[((size_t)chi * K4 + r1) * KP2 + 8 * r + d] = al / 64.0;
        }
  }
  o.sym_rep.upload(rep.data(), rep.size(), s);
  o.sym_u1.upload(u1.data(), u1.size(), s);
  o.sym_u2.upload(u2.data(), u2.size(), s);
  o.sym_d1.upload(d1.data(), d1.size(), s);
  o.sym_d2.upload(d2.data(), d2.size(), s);
  o.sym_m2m.upload(mm.data(), mm.size(), s);
  o.sym_l2l.upload(ll.data(), ll.size(), s);
  o.ctx->sync();
  o.sym = true;
}

// The block of each entry of a harmonic expansion of degree p (entry n^2 for order 0, n^2 +
// 2 m - 1 and n^2 + 2 m for the parts of order m: cos and sin) and its place in the block.
void sym_harmonic_entries(OpCache &o) {
  std::vector<uint8_t> chi, rank;
  int cnt[8] = {};
  for (int n = 0; n <= o.p; n++)
    for (int k = 0; k < 2 * n + 1; k++) {
      const int m = (k + 1) / 2, sn = k > 0 && k % 2 == 0;   // sin: even under y -> -y it is not
      const int c = ((m + sn) & 1) | sn << 1 | ((n + m) & 1) << 2;
      chi.push_back((uint8_t)c);
      rank.push_back((uint8_t)cnt[c]++);
    }
  o.hmax = *std::max_element(cnt, cnt + 8);
  if (o.hmax > 64) return;      // more rows than the kernels take: the dense operators
  o.hchi_h = chi;
  o.hrank_h = rank;
  o.hchi.upload(chi.data(), chi.size(), o.ctx->stream);
  o.hrank.upload(rank.data(), rank.size(), o.ctx->stream);
}

// The blocks of a width's scalar M2M (N x 8 N) and L2L (8 N x N, column major), the mean
// over the children; left unset (the dense operators stay) when they are not symmetric.
void sym_harmonic_setup(OpCache &o, HarmonicLevel &lv, const double *M2M, const double *L2L) {
  if (o.hmax > 64) return;
  const int N = o.hN, R = (o.hmax + 15) / 16 * 16, KP = (N + SY_K - 1) / SY_K * SY_K;
  const std::vector<uint8_t> &chi = o.hchi_h, &rank = o.hrank_h;
  std::vector<double> mm(8 * (size_t)KP * R + 16 * R, 0.0), ll(8 * (size_t)R * KP, 0.0);
  double big[2] = {0.0, 0.0}, off[2] = {0.0, 0.0};
  for (int j = 0; j < N; j++)
    for (int i = 0; i < N; i++) {
      double a[2] = {0.0, 0.0}, x[2][8];
      for (int c = 0; c < NCHILD; c++) {
        const double s = chi_sign(chi[i] ^ chi[j], c);
        x[0][c] = s * M2M[((size_t)c * N + j) * N + i];
        x[1][c] = s * L2L[(size_t)j * NCHILD * N + c * N + i];
        for (int k = 0; k < 2; k++) a[k] += x[k][c] / 8.0;
      }
      for (int k = 0; k < 2; k++)
        for (int c = 0; c < NCHILD; c++) {
          big[k] = std::max(big[k], std::abs(x[k][c]));
          off[k] = std::max(off[k], std::abs(x[k][c] - a[k]));
        }
      mm[((size_t)chi[i] * KP + j) * R + rank[i]] = a[0];
      ll[((size_t)chi[j] * R + rank[j]) * KP + i] = a[1];
    }
  if (!(off[0] <= 1e-11 * big[0] && off[1] <= 1e-11 * big[1])) return;
  lv.sym_m2m.upload(mm.data(), mm.size(), o.ctx->stream);
  lv.sym_l2l.upload(ll.data(), ll.size(), o.ctx->stream);
  o.ctx->sync();
}

// ---------------------------------------------------------------------------
// the passes' launches
// ---------------------------------------------------------------------------
template <class F>
static void with_nr(int nr, F &&f) {
  switch (nr) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 19: f(std::integral_constant<int, 19>{}); break;
    case 37: f(std::integral_constant<int, 37>{}); break;
    case 61: f(std::integral_constant<int, 61>{}); break;
    default: fail(FFMM_ERR_STATE, "no symmetric kernel for this order");
  }
}
static unsigned sy_blocks(int64_t n) { return (unsigned)((n + SY_N - 1) / SY_N); }

bool sym_split_s2m(int64_t nq) { return nq < SYM_SPLIT_NODES; }

void sym_s2m_uc2e(Plan &plan, const int32_t *nodes, int64_t nq) {
  OpCache &o = *plan.ops;
  hipStream_t s = plan.ctx->stream;
  const bool mixed = plan.precision == FFMM_PREC_MIXED;
  const SyNodes a{nodes,      nq,         plan.nnodes, plan.centers.p, plan.lam_d.p, plan.level.p,  plan.plo.p,
                  plan.phi.p, plan.sx.p,  plan.sy.p,   plan.sz.p,      plan.tau.p,   o.sym_rep.p,   o.Nl / 8};
  const bool split = sym_split_s2m(nq);
  if (split) {
    const dim3 g((unsigned)nq, (unsigned)(o.sym_kp / SY_K));
    if (mixed) k_sym_s2m<true><<<g, 256, 0, s>>>(a, o.sym_kp, plan.pM.p);
    else k_sym_s2m<false><<<g, 256, 0, s>>>(a, o.sym_kp, plan.pM.p);
    FFMM_LAUNCH_CHECK();
  }
  with_nr(o.Ns / 8, [&](auto NR) {
    constexpr int nr = decltype(NR)::value;
    if (split)
      k_sym_uc2e<2, nr><<<sy_blocks(nq), SY_TB, 0, s>>>(a, o.sym_u1.p, o.sym_u2.p, o.sym_kp, plan.pM.p, plan.Mp.p);
    else if (mixed)
      k_sym_uc2e<1, nr><<<sy_blocks(nq), SY_TB, 0, s>>>(a, o.sym_u1.p, o.sym_u2.p, o.sym_kp, nullptr, plan.Mp.p);
    else
      k_sym_uc2e<0, nr><<<sy_blocks(nq), SY_TB, 0, s>>>(a, o.sym_u1.p, o.sym_u2.p, o.sym_kp, nullptr, plan.Mp.p);
  });
  FFMM_LAUNCH_CHECK();
}

void sym_m2m(Plan &plan, int l) {
  OpCache &o = *plan.ops;
  hipStream_t s = plan.ctx->stream;
  const int64_t first = plan.lo[l + 1], ng = plan.nl[l + 1] / NCHILD;
  if (ng == 0) return;
  with_nr(o.Ns / 8, [&](auto NR) {
    constexpr int nr = decltype(NR)::value;
    k_sym_m2m<nr><<<sy_blocks(ng), SY_TB, 0, s>>>(o.sym_m2m.p, o.sym_kp2, plan.parent.p, plan.has_source.p, first, ng,
                                                 plan.Mp.p);
  });
  FFMM_LAUNCH_CHECK();
}

void sym_l2l(Plan &plan, int l) {
  OpCache &o = *plan.ops;
  const int64_t ng = plan.nl[l] / NCHILD;
  if (ng == 0) return;
  const SyDown a{nullptr, o.sym_l2l.p, o.sym_kp2, o.Ns, plan.parent.p, plan.lo[l], ng, nullptr, nullptr, plan.Pl.p, plan.Pl.p};
  with_nr(o.Ns / 8, [&](auto NR) {
    k_sym_down<0, decltype(NR)::value><<<sy_blocks(ng), SY_TB, 0, plan.ctx->stream>>>(a);
  });
  FFMM_LAUNCH_CHECK();
}

void sym_dc2e(Plan &plan, const int32_t *leaves, int64_t nq, double *Lc) {
  OpCache &o = *plan.ops;
  const SyDown a{o.sym_d1.p,   o.sym_d2.p, o.sym_kp,  o.Nl / 8, leaves, 0, nq, plan.level.p,
                 plan.lam_d.p, plan.Pl.p,  Lc};
  with_nr(o.Ns / 8, [&](auto NR) {
    k_sym_down<1, decltype(NR)::value><<<sy_blocks(nq), SY_TB, 0, plan.ctx->stream>>>(a);
  });
  FFMM_LAUNCH_CHECK();
}

template <class F>
static void with_harmonic(const OpCache &o, F &&f) {
  const int rt = (o.hmax + 15) / 16;
  auto go = [&](auto RT) {
    if (o.nb == 4) f(RT, std::integral_constant<int, 4>{});
    else f(RT, std::integral_constant<int, 1>{});
  };
  if (rt == 1) go(std::integral_constant<int, 1>{});
  else if (rt == 2) go(std::integral_constant<int, 2>{});
  else if (rt == 3) go(std::integral_constant<int, 3>{});
  else go(std::integral_constant<int, 4>{});
}

void sym_harmonic_m2m(Plan &plan, int l) {
  OpCache &o = *plan.ops;
  const int64_t first = plan.lo[l + 1], ng = plan.nl[l + 1] / NCHILD;
  const int KP = (o.hN + SY_K - 1) / SY_K * SY_K;
  if (ng == 0) return;
  with_harmonic(o, [&](auto RT, auto NB) {
    k_harm_m2m<decltype(RT)::value, decltype(NB)::value><<<sy_blocks(ng * o.nb), SY_TB, 0, plan.ctx->stream>>>(
        plan.hl[l]->sym_m2m.p, o.hN, KP, o.hchi.p, o.hrank.p, plan.parent.p, plan.has_source.p, first, ng, plan.Mp.p);
  });
  FFMM_LAUNCH_CHECK();
}

void sym_harmonic_l2l(Plan &plan, int l) {
  OpCache &o = *plan.ops;
  const int64_t ng = plan.nl[l] / NCHILD;
  const int KP = (o.hN + SY_K - 1) / SY_K * SY_K;
  if (ng == 0) return;
  with_harmonic(o, [&](auto RT, auto NB) {
    k_harm_l2l<decltype(RT)::value, decltype(NB)::value><<<sy_blocks(ng * o.nb), SY_TB, 0, plan.ctx->stream>>>(
        plan.hl[l - 1]->sym_l2l.p, o.hN, KP, o.hchi.p, o.hrank.p, plan.parent.p, plan.lo[l], ng, plan.Pl.p);
  });
  FFMM_LAUNCH_CHECK();
}

void sym_zero_unsourced(Plan &plan) {
  k_sym_zero<<<nblocks(plan.nnodes, 256), 256, 0, plan.ctx->stream>>>(plan.has_source.p, plan.nnodes, plan.ops->Ns,
                                                                      plan.Mp.p);
  FFMM_LAUNCH_CHECK();
}

}  // namespace ffmm
