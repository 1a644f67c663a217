// The upward and downward passes on the device.
//
// Upward (levels L-1 .. 2, 0-based): S2M of the childless sourced nodes (check
// potentials on the large surface, one workgroup per node with the node's sources
// staged in LDS), the factored pseudo-inverse UC2E as two FP64 GEMMs, and M2M as one
// GEMM per level straight on the children block of the multipole array (the children
// of a sibling group are consecutive columns).  Downward (levels 2 .. L-1): L2L as one
// GEMM whose output is the level's block of partial locals, the far field (M2L), and
// the pseudo-inverse DC2E of the real leaves, written straight into the compact leaf
// locals.  Follows device_build_expansions! (src/device_passes.jl:511-597) and the
// host passes it restates (src/fmm.jl:170-262).
#include "ffmm_internal.h"

#include <algorithm>
#include <cmath>

namespace ffmm {

constexpr int TB = 256;
constexpr double C4PI = 0.07957747154594767;   // 1 / (4 pi), as 1 / (4 * Float64(pi))

// ---------------------------------------------------------------------------
// S2M: s2m_accumulate! (src/operators/ki_common.jl:256-272), _s2m_kernel!
// (src/device_passes.jl:378-403).  pM[k, q] = sum_j tau_j K(x_j - c, y_k).
// ---------------------------------------------------------------------------
constexpr int S2M_TB = 256;
constexpr int S2M_KP = 6;   // check points per thread; blockIdx.y: blocks of S2M_TB S2M_KP points (1,736 points at p = 9)

__global__ void __launch_bounds__(S2M_TB) k_s2m(const int32_t *__restrict__ nodes, const double *__restrict__ centers,
                                                int64_t nn, const int32_t *__restrict__ level,
                                                const double *__restrict__ lam, const double *__restrict__ surf, int Nl,
                                                const int32_t *__restrict__ plo, const int32_t *__restrict__ phi,
                                                const double *__restrict__ sx, const double *__restrict__ sy,
                                                const double *__restrict__ sz, const double *__restrict__ tau,
                                                double *__restrict__ pM) {
  __shared__ double xs[S2M_TB], ys[S2M_TB], zs[S2M_TB], ts[S2M_TB];
  const int64_t q = blockIdx.x;
  const int node = nodes[q];
  const double c0 = centers[node], c1 = centers[nn + node], c2 = centers[2 * nn + node];
  const double s = lam[level[node]];
  const int t = threadIdx.x, k0 = blockIdx.y * (S2M_TB * S2M_KP);
  double acc[S2M_KP], y0[S2M_KP], y1[S2M_KP], y2[S2M_KP];
#pragma unroll
  for (int m = 0; m < S2M_KP; m++) {
    int k = k0 + t + S2M_TB * m;
    acc[m] = 0.0;
    if (k < Nl) {
      y0[m] = surf[k] * s;
      y1[m] = surf[Nl + k] * s;
      y2[m] = surf[2 * Nl + k] * s;
    } else {
      y0[m] = y1[m] = y2[m] = 1.0;
    }
  }
  const int32_t a = plo[node], b = phi[node];
  for (int32_t j0 = a; j0 <= b; j0 += S2M_TB) {
    int32_t j = j0 + t;
    if (j <= b) {
      xs[t] = sx[j] - c0;
      ys[t] = sy[j] - c1;
      zs[t] = sz[j] - c2;
      ts[t] = tau[j];
    }
    __syncthreads();
    int cnt = min(S2M_TB, b - j0 + 1);
    for (int jj = 0; jj < cnt; jj++) {
      const double xr = xs[jj], yr = ys[jj], zr = zs[jj], tj = ts[jj];
#pragma unroll
      for (int m = 0; m < S2M_KP; m++) {
        double d0 = y0[m] - xr, d1 = y1[m] - yr, d2 = y2[m] - zr;
        double r2 = fma(d2, d2, fma(d1, d1, d0 * d0));
        acc[m] += (C4PI * rsqrt_f64(r2)) * tj;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int m = 0; m < S2M_KP; m++) {
    int k = k0 + t + S2M_TB * m;
    if (k < Nl) pM[q * Nl + k] = acc[m];
  }
}

// The mixed form of S2M: sources relative to the node centre (differences formed in
// FP64, rounded once), surface points scaled and rounded once, v_rsq_f32, FP32 sums over
// each LDS tile folded into FP64 check potentials.  The check surface lies at least
// ~0.9 w from any source of the node, so no pair is close.
__global__ void __launch_bounds__(S2M_TB) k_s2m32(const int32_t *__restrict__ nodes, const double *__restrict__ centers,
                                                  int64_t nn, const int32_t *__restrict__ level,
                                                  const double *__restrict__ lam, const double *__restrict__ surf, int Nl,
                                                  const int32_t *__restrict__ plo, const int32_t *__restrict__ phi,
                                                  const double *__restrict__ sx, const double *__restrict__ sy,
                                                  const double *__restrict__ sz, const double *__restrict__ tau,
                                                  double *__restrict__ pM) {
  __shared__ float4 src[S2M_TB];
  const int64_t q = blockIdx.x;
  const int node = nodes[q];
  const double c0 = centers[node], c1 = centers[nn + node], c2 = centers[2 * nn + node];
  const double s = lam[level[node]];
  const int t = threadIdx.x, k0 = blockIdx.y * (S2M_TB * S2M_KP);
  double acc[S2M_KP];
  float y0[S2M_KP], y1[S2M_KP], y2[S2M_KP];
#pragma unroll
  for (int m = 0; m < S2M_KP; m++) {
    const int k = k0 + t + S2M_TB * m;
    acc[m] = 0.0;
    if (k < Nl) {
      y0[m] = (float)(surf[k] * s);
      y1[m] = (float)(surf[Nl + k] * s);
      y2[m] = (float)(surf[2 * Nl + k] * s);
    } else {
      y0[m] = y1[m] = y2[m] = 1.f;
    }
  }
  const int32_t a = plo[node], b = phi[node];
  for (int32_t j0 = a; j0 <= b; j0 += S2M_TB) {
    const int32_t j = j0 + t;
    if (j <= b) src[t] = make_float4((float)(sx[j] - c0), (float)(sy[j] - c1), (float)(sz[j] - c2), (float)tau[j]);
    __syncthreads();
    const int cnt = min(S2M_TB, b - j0 + 1);
    float part[S2M_KP];
#pragma unroll
    for (int m = 0; m < S2M_KP; m++) part[m] = 0.f;
    for (int jj = 0; jj < cnt; jj++) {
      const float4 v = src[jj];
#pragma unroll
      for (int m = 0; m < S2M_KP; m++) {
        const float d0 = y0[m] - v.x, d1 = y1[m] - v.y, d2 = y2[m] - v.z;
        part[m] = fmaf(__builtin_amdgcn_rsqf(fmaf(d2, d2, fmaf(d1, d1, d0 * d0))), v.w, part[m]);
      }
    }
#pragma unroll
    for (int m = 0; m < S2M_KP; m++) acc[m] += (double)part[m];
    __syncthreads();
  }
#pragma unroll
  for (int m = 0; m < S2M_KP; m++) {
    const int k = k0 + t + S2M_TB * m;
    if (k < Nl) pM[q * Nl + k] = C4PI * acc[m];
  }
}

// dst[i, cols[q]] = alpha * src[i, q]
__global__ void k_scatter_cols(double *__restrict__ dst, const double *__restrict__ src, const int32_t *__restrict__ cols,
                               int rows, int64_t ncols, double alpha) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (int64_t)rows * ncols) return;
  int64_t q = g / rows;
  int i = (int)(g % rows);
  dst[(int64_t)cols[q] * rows + i] = alpha * src[g];
}
// dst[i, q] = src[i, cols[q]]
__global__ void k_gather_cols(double *__restrict__ dst, const double *__restrict__ src, const int32_t *__restrict__ cols,
                              int rows, int64_t ncols) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (int64_t)rows * ncols) return;
  int64_t q = g / rows;
  int i = (int)(g % rows);
  dst[g] = src[(int64_t)cols[q] * rows + i];
}
// dst[i, cols[q]] = lam[level[cols[q]]] * src[i, q]: the columns of several levels at once,
// each scaled by its level's width factor; dst32 (if given) takes the same value in FP32
__global__ void k_scatter_cols_lam(double *__restrict__ dst, const double *__restrict__ src,
                                   const int32_t *__restrict__ cols, int rows, int64_t ncols,
                                   const int32_t *__restrict__ level, const double *__restrict__ lam,
                                   float *__restrict__ dst32) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (int64_t)rows * ncols) return;
  int64_t q = g / rows;
  int i = (int)(g % rows);
  const int32_t c = cols[q];
  const double v = lam[level[c]] * src[g];
  dst[(int64_t)c * rows + i] = v;
  if (dst32) dst32[(int64_t)c * rows + i] = (float)v;
}
// dst[i, q] = lam[level[cols[q]]] * src[i, cols[q]]
__global__ void k_gather_cols_lam(double *__restrict__ dst, const double *__restrict__ src,
                                  const int32_t *__restrict__ cols, int rows, int64_t ncols,
                                  const int32_t *__restrict__ level, const double *__restrict__ lam) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (int64_t)rows * ncols) return;
  int64_t q = g / rows;
  int i = (int)(g % rows);
  const int32_t c = cols[q];
  dst[g] = lam[level[c]] * src[(int64_t)c * rows + i];
}
// the parents of the sibling groups starting at node `first`: dst[i, parent[first + 8g]] =
// alpha src[i, g]; dst32 (if given) takes the same value in FP32
template <class T>
__global__ void k_scatter_parents(double *__restrict__ dst, const T *__restrict__ src,
                                  const int32_t *__restrict__ parent, int64_t first, int rows, int64_t ng, double alpha,
                                  float *__restrict__ dst32) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (int64_t)rows * ng) return;
  int64_t q = g / rows;
  int i = (int)(g % rows);
  const int64_t o = (int64_t)parent[first + NCHILD * q] * rows + i;
  const double v = alpha * (double)src[g];
  dst[o] = v;
  if (dst32) dst32[o] = (float)v;
}
__global__ void k_fill32(float *__restrict__ a, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0.f;
}
__global__ void k_gather_parents(double *__restrict__ dst, const double *__restrict__ src,
                                 const int32_t *__restrict__ parent, int64_t first, int rows, int64_t ng) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (int64_t)rows * ng) return;
  int64_t q = g / rows;
  int i = (int)(g % rows);
  dst[g] = src[(int64_t)parent[first + NCHILD * q] * rows + i];
}
__global__ void k_fill(double *__restrict__ a, int64_t n, double v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

void fill_f64(Context &ctx, double *a, int64_t n, double v) {
  if (n <= 0) return;
  k_fill<<<nblocks(n, TB), TB, 0, ctx.stream>>>(a, n, v);
  FFMM_LAUNCH_CHECK();
}
// the densities into the tree's order: _gather_perm! (src/device_lists.jl:163-171)
__global__ void k_gather_perm(double *__restrict__ dst, const double *__restrict__ src, const int32_t *__restrict__ perm,
                              int64_t n) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) dst[j] = src[perm[j]];
}
// nd components per point, point major
__global__ void k_gather_perm_nd(double *__restrict__ dst, const double *__restrict__ src,
                                 const int32_t *__restrict__ perm, int64_t n, int nd) {
  int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n * nd) return;
  int64_t j = g / nd;
  int c = (int)(g % nd);
  dst[g] = src[(int64_t)perm[j] * nd + c];
}

// ---------------------------------------------------------------------------
// dense M2L by symmetry class: _class_gather! / _class_scatter! (src/device_passes.jl:426-473)
// An expansion column holds nb blocks of N entries (Ns = nb N); the class operator acts
// on each block (nb columns per pair, as the reference lays out the Stokes blocks).
// Gc[i, q nb + b] = sgn[f, i] Mp[b N + idx[f, i], src[q]]  (P_f^T m, block b)
// ---------------------------------------------------------------------------
// One target chunk of a level's class M2L: the chunk-local columns of class c are
// [co[c], co[c + 1]) and hold the class-major pairs cs[c] + (q - co[c]).
struct ChunkArgs {
  int nclass;
  int32_t co[MAX_CLASSES + 1];
  int32_t cs[MAX_CLASSES];
  int32_t to[MAX_CLASSES + 1];   // the fused kernel: first column tile of each class
};

// the class of chunk column q: the last c with co[c] <= q
__device__ __forceinline__ int chunk_class(const ChunkArgs &ca, int32_t q) {
  int c = 0, h = ca.nclass;
  while (h - c > 1) {
    const int m = (c + h) >> 1;
    if (ca.co[m] <= q) c = m;
    else h = m;
  }
  return c;
}

constexpr int GATHER_PAIRS = 8;   // pairs per workgroup of the gather
constexpr int SCATTER_MAXP = 320; // far pairs of one target: at most the 316 far offsets

// Gc[b N + i, q] = sgn[f, i] Mp[b N + idx[f, i], src]  (P_f^T m per block b) for the pairs
// of a chunk, all classes in one launch; one workgroup per GATHER_PAIRS columns, one lane
// per coefficient i with all nb blocks, the pairs' loads independent of each other.  For
// Stokes (nb = 4) the fourth block takes the coupling Psi += o_f . Phi of the translation
// (src/device_passes.jl:465-468, src/operators/harmonics.jl:604-628) before the product:
// the class operator is linear and the same for every block, so T (G_3 + o_f . (G_0, G_1,
// G_2)) is the coupled fourth block of the output.
template <class T>
__global__ void k_chunk_gather(T *__restrict__ Gc, const double *__restrict__ Mp, int Ns, int N, int nb,
                               const int32_t *__restrict__ csrc, const int32_t *__restrict__ cfar, int32_t npk,
                               const int32_t *__restrict__ gsel, const double *__restrict__ offs, ChunkArgs ca) {
  __shared__ int32_t pf[GATHER_PAIRS], ps[GATHER_PAIRS];
  const int nbN = nb * N;
  const int32_t q0 = (int32_t)blockIdx.x * GATHER_PAIRS;
  const int nq = min(GATHER_PAIRS, npk - q0);
  if ((int)threadIdx.x < nq) {
    const int32_t q = q0 + (int32_t)threadIdx.x;
    const int c = chunk_class(ca, q);
    const int32_t p = ca.cs[c] + (q - ca.co[c]);
    pf[threadIdx.x] = cfar[p];
    ps[threadIdx.x] = csrc[p];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < N; i += blockDim.x) {
#pragma unroll
    for (int k = 0; k < GATHER_PAIRS; k++) {
      if (k < nq) {
        const int32_t f = pf[k];
        const int32_t g = gsel[f * N + i];
        const double *__restrict__ m = Mp + (int64_t)ps[k] * Ns + (g & 0x7fffffff);
        T *__restrict__ o = Gc + (int64_t)(q0 + k) * nbN + i;
        const double sg = g < 0 ? -1.0 : 1.0;
        if (nb == 4) {
          const double m0 = m[0], m1 = m[N], m2 = m[2 * N], m3 = m[3 * N];
          o[0] = (T)(sg * m0);
          o[N] = (T)(sg * m1);
          o[2 * N] = (T)(sg * m2);
          o[3 * N] = (T)(sg * (m3 + offs[3 * f] * m0 + offs[3 * f + 1] * m1 + offs[3 * f + 2] * m2));
        } else {
          for (int b = 0; b < nb; b++) o[b * N] = (T)(sg * m[b * N]);
        }
      }
    }
  }
}

constexpr int FM_TB = 512;      // 8 waves: wave w holds the operator's row tile w (rows 16 w .. 16 w + 15)
constexpr int FM_COLS = 64;     // product columns per tile: 4 column tiles of 16
constexpr int FM_BS = FM_MAXN + 1;   // LDS stride of a product column, the last entry for the rows beyond N

// entry i of a wave-uniform array: the address as a scalar base and a 32-bit offset
template <class T>
__device__ __forceinline__ T at32(const T *base, uint32_t i) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + i * (uint32_t)sizeof(T));
}

// The class M2L of the harmonic methods in the mixed form, fused: for each tile of a
// class's pairs in the chunk, the gathered source expansions (P_f^T m per block, signed,
// the Stokes coupling folded into the fourth block, src/device_passes.jl:449-473) go
// straight into LDS and are multiplied by the class operator.  The products are staged in
// each pair's target frame (entry j = fsel position, sign applied), so the scatter adds
// contiguous columns.  N = (p + 1)^2 <= FM_MAXN.
//
// Each FP32 operand is three bfloat16 pieces (the whole FP32 mantissa), the products of
// pieces down to 2^-24 on v_mfma_f32_16x16x32_bf16 with the small ones in accumulators of
// their own: 96 cycles per 16 x 16 block of 32 K where v_mfma_f32_16x16x4_f32 takes 256.
// Values below some 2^-110 lose pieces to bfloat16's range: charges of 2^-112 (2e-34) are as
// exact as larger ones, of 2^-116 4.5e-7, of 2^-120 6.5e-6 (FP32 operands 1.3e-7).
// The form before (FP32 matrix instructions) gathered, multiplied and staged each tile in
// turn behind five barriers.  Here a wave keeps its operator rows while the class lasts, and
// the loads of a tile are in flight during the one before it (the pairs three tiles ahead,
// their permutation bytes one); half of a tile's expansions are loaded behind the products,
// because all of them beside the operator's 48 registers spill.  Loads return in order: a
// tile's own go before the next tile's, or waiting for them waits for all.  Products and
// gathered columns have LDS of their own (two workgroups per CU fill its 160 KB), so that
// two barriers a tile are left.  A column's 16-byte chunks are stored at chunk ^ column:
// reads and writes touch each bank once.  Measured: 1M Stokes points, p = 10, 16.3 -> 8.5 ms
// (10.5 with spilled registers and waits in the wrong order), 200k Yukawa points 3.5 -> 1.9
// with the scatter.  At the larger one the matrix cores are busy 36% of the time and LDS 41%,
// 11.5 GB are fetched and 6.9 GB written beyond the L2 (2.3 TB/s): what is left is latency
// between the two barriers.
// KB: K blocks of 32, ceil(N / 32)
template <int NB, int KB>
__global__ void __launch_bounds__(FM_TB) __attribute__((amdgpu_waves_per_eu(4)))
k_class_m2l32(float *__restrict__ Yc, const double *__restrict__ Mp, int Ns, int N, const bf16x8 *__restrict__ ops,
              const int32_t *__restrict__ csrc, const int32_t *__restrict__ cfar, const uint32_t *__restrict__ gsel8,
              const uint32_t *__restrict__ fsel8, const double *__restrict__ offs, ChunkArgs ca, int32_t ntiles,
              const int32_t *__restrict__ ctgt) {
  constexpr int PPT = FM_COLS / NB;   // pairs per tile
  constexpr int PW = PPT / 8;         // pairs a wave gathers
  constexpr int PLANE = FM_COLS * 64; // words of a plane of pieces: 128 k of each column
  __shared__ __attribute__((aligned(16))) uint32_t Bp[3 * PLANE];
  __shared__ float Ys[FM_COLS * FM_BS];
  __shared__ int32_t pf[2][PPT], pt[2][PPT];   // offsets and targets of a tile's pairs, by its parity
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const bool rows = 16 * w < N;       // this wave's row tile holds operator rows
  const int32_t t0 = (int32_t)((int64_t)blockIdx.x * ntiles / gridDim.x);
  const int32_t t1 = (int32_t)((int64_t)(blockIdx.x + 1) * ntiles / gridDim.x);
  struct Tile {
    int32_t c, p0, q0, npt;           // class, first pair, first chunk column, pairs
  };
  auto next_tile = [&](Tile &t, int32_t tile) {   // tile >= the one t held; the last one again past the end
    tile = min(tile, t1 - 1);
    int c = t.c;
    while (ca.to[c + 1] <= tile) c++;
    const int32_t lp0 = (tile - ca.to[c]) * PPT;
    t.c = c;
    t.p0 = ca.cs[c] + lp0;
    t.q0 = ca.co[c] + lp0;
    t.npt = min(PPT, ca.co[c + 1] - t.q0);
  };
  int32_t f0[PW], f1[PW], s1[PW], f2[PW], s2[PW];
  uint32_t gw[PW], sg, sn = 0;        // permutation words of the next tile; signs of this one and of the next
  double m[PW][2][NB];
  auto load_pairs = [&](const Tile &t, int32_t *f, int32_t *s) {
#pragma unroll
    for (int e = 0; e < PW; e++) {
      const int32_t p = t.p0 + min(w * PW + e, t.npt - 1);
      f[e] = cfar[p];
      s[e] = csrc[p];
    }
  };
  auto load_words = [&](const int32_t *f) {   // entries 2 lane, 2 lane + 1 are half of a word
#pragma unroll
    for (int e = 0; e < PW; e++) gw[e] = at32<uint32_t>(gsel8 + f[e] * 32, lane >> 1);
  };
  auto load_m = [&](const int32_t *s, int e0, int e1) {
#pragma unroll
    for (int e = e0; e < e1; e++) {
      const uint32_t h = gw[e] >> (16 * (lane & 1));
      const double *__restrict__ x = Mp + (int64_t)s[e] * Ns;
      sn |= ((h >> 7) & 1) << (2 * e) | ((h >> 15) & 1) << (2 * e + 1);
#pragma unroll
      for (int b = 0; b < NB; b++) {
        m[e][0][b] = at32<double>(x + b * N, h & 127);
        m[e][1][b] = at32<double>(x + b * N, (h >> 8) & 127);
      }
    }
  };
  // the pairs' columns as pieces: lane k / 2 holds entries k and k + 1, zero beyond N
  auto store_columns = [&]() {
    const bool k0 = 2 * lane < N, k1 = 2 * lane + 1 < N;
#pragma unroll
    for (int e = 0; e < PW; e++) {
      if (NB == 4) {
        const double ox = offs[3 * f0[e]], oy = offs[3 * f0[e] + 1], oz = offs[3 * f0[e] + 2];
#pragma unroll
        for (int z = 0; z < 2; z++)
          m[e][z][NB - 1] += ox * m[e][z][0] + oy * m[e][z][1 % NB] + oz * m[e][z][2 % NB];
      }
      const uint32_t g0 = (sg >> (2 * e)) << 31, g1 = (sg >> (2 * e + 1)) << 31;
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const float a0 = __uint_as_float(__float_as_uint((float)m[e][0][b]) ^ g0);
        const float a1 = __uint_as_float(__float_as_uint((float)m[e][1][b]) ^ g1);
        const f32x2 v = f32x2{k0 ? a0 : 0.f, k1 ? a1 : 0.f};
        const uint32_t h0 = pack_bf16(v);
        const f32x2 r1 = v - unpack_bf16(h0);
        const uint32_t h1 = pack_bf16(r1);
        const uint32_t h2 = pack_bf16(r1 - unpack_bf16(h1));
        const int col = (w * PW + e) * NB + b;
        uint32_t *__restrict__ o = Bp + col * 64 + (((lane >> 2) ^ (col & 15)) << 2) + (lane & 3);
        o[0] = h0;
        o[PLANE] = h1;
        o[2 * PLANE] = h2;
      }
    }
  };
  Tile T0, T1, T3;
  {
    int c = 0, h = ca.nclass;
    while (h - c > 1) {
      const int mid = (c + h) >> 1;
      if (ca.to[mid] <= t0) c = mid;
      else h = mid;
    }
    T0.c = c;
  }
  next_tile(T0, t0);
  T1 = T0;
  next_tile(T1, t0 + 1);
  T3 = T1;
  next_tile(T3, t0 + 2);
  load_pairs(T0, f0, s1);
  load_words(f0);
  load_m(s1, 0, PW);
  sg = sn;
  load_pairs(T1, f1, s1);
  load_words(f1);
  load_pairs(T3, f2, s2);
  Tile T2 = T3;
  int32_t nf, nt;
  if (tid < PPT) {
    pf[0][tid] = cfar[T0.p0 + min(tid, T0.npt - 1)];
    pt[0][tid] = ctgt[T0.p0 + min(tid, T0.npt - 1)];
  }
  nf = cfar[T1.p0 + min(tid, T1.npt - 1)];
  nt = ctgt[T1.p0 + min(tid, T1.npt - 1)];
  lds_barrier();
  bf16x8 A[KB][3];
  int32_t cur = -1;
  for (int32_t tile = t0; tile < t1; tile++) {
    const int par = (tile - t0) & 1;
    const int32_t *__restrict__ ptb = pt[par];
    store_columns();
    // loads return in order: what this tile still needs goes before the next tile's loads
    if (rows && T0.c != cur) {
      cur = T0.c;
      const bf16x8 *__restrict__ Ar = ops + ((size_t)cur * 8 + w) * (4 * 3 * 64) + lane;
#pragma unroll
      for (int kb = 0; kb < KB; kb++)
#pragma unroll
        for (int q = 0; q < 3; q++) A[kb][q] = Ar[(kb * 3 + q) * 64];
      __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0) here, so that no wait is left for the tiles that skip this
    }
    uint32_t fw[FM_COLS / 16];
#pragma unroll
    for (int ct = 0; ct < FM_COLS / 16; ct++) fw[ct] = at32<uint32_t>(fsel8, pf[par][ct * (16 / NB) + li / NB] * 32 + 4 * w + lk);
    // the next tile's expansions: half here, half behind the products (all at once spills)
    sn = 0;
    load_m(s1, 0, PW / 2);
    next_tile(T3, tile + 3);
    int32_t f3[PW], s3[PW];
    load_pairs(T3, f3, s3);
    lds_barrier();
    if (tid < PPT) {   // the next tile's: every wave is past the tile before this one
      pf[par ^ 1][tid] = nf;
      pt[par ^ 1][tid] = nt;
    }
    {
      nf = at32<int32_t>(cfar + T2.p0, min(tid, T2.npt - 1));
      nt = at32<int32_t>(ctgt + T2.p0, min(tid, T2.npt - 1));
    }
    if (rows) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ct = 0; ct < FM_COLS / 16; ct++) {
        f32x4 c0 = f32x4{0.f, 0.f, 0.f, 0.f}, c1 = c0, c2 = c0;
#pragma unroll
        for (int kb = 0; kb < KB; kb++) {
          const uint32_t *p = Bp + (16 * ct + li) * 64 + (((4 * kb + lk) ^ li) << 2);
          const bf16x8 b0 = *reinterpret_cast<const bf16x8 *>(p);
          const bf16x8 b1 = *reinterpret_cast<const bf16x8 *>(p + PLANE);
          const bf16x8 b2 = *reinterpret_cast<const bf16x8 *>(p + 2 * PLANE);
          c0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[kb][0], b0, c0, 0, 0, 0);
          c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[kb][1], b0, c1, 0, 0, 0);
          c2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[kb][2], b0, c2, 0, 0, 0);
          c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[kb][0], b1, c1, 0, 0, 0);
          c2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[kb][1], b1, c2, 0, 0, 0);
          c2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[kb][0], b2, c2, 0, 0, 0);
        }
        // lane (lk, li) holds rows 16 w + 4 lk + r of column 16 ct + li
        const f32x4 v = c0 + (c1 + c2);
        float *__restrict__ y = Ys + (16 * ct + li) * FM_BS;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const uint32_t h = fw[ct] >> (8 * r);
          y[h & 127] = __uint_as_float(__float_as_uint(v[r]) ^ ((h & 128) << 24));
        }
        __builtin_amdgcn_sched_barrier(0);   // a column tile at a time: the registers of one
      }
    }
    load_m(s1, PW / 2, PW);
    sg = sn;
    load_words(f2);
    lds_barrier();   // the products are staged, and every read of the gathered columns is done
    // coalesced copy of the tile's columns (pair column q0 + pl, NB N entries), the products
    // of consecutive pairs of one target summed first: the first pair of each such run
    // carries the run's sum, the others are not written
    float *__restrict__ out = Yc + (int64_t)T0.q0 * NB * N;
    for (int col = w; col < T0.npt * NB; col += FM_TB / 64) {
      const int pl = col / NB, b = col - pl * NB;
      const int32_t tg = ptb[pl];
      if (pl > 0 && tg == ptb[pl - 1]) continue;
      int pe = pl + 1;
      while (pe < T0.npt && ptb[pe] == tg) pe++;
      for (int j = lane; j < N; j += 64) {
        float acc = Ys[col * FM_BS + j];
        for (int r = pl + 1; r < pe; r++) acc += Ys[(r * NB + b) * FM_BS + j];
        out[(int64_t)col * N + j] = acc;
      }
    }
    T0 = T1;
    T1 = T2;
    T2 = T3;
#pragma unroll
    for (int e = 0; e < PW; e++) {
      f0[e] = f1[e];
      f1[e] = f2[e];
      s1[e] = s2[e];
      f2[e] = f3[e];
      s2[e] = s3[e];
    }
  }
}

// The scatter of products already in the target frame: pL[e, t] += alpha sum over the
// target's columns (class by class) of Y'[e, q]; the fused kernel has summed each run of
// the target's pairs within a tile of ppt pairs into the run's first column
__global__ void k_chunk_scatter_framed(double *__restrict__ pL, const float *__restrict__ Yc, int Ns, int nbN,
                                       const int32_t *__restrict__ cstart, int64_t nl, int32_t t0, double alpha,
                                       ChunkArgs ca, int ppt) {
  __shared__ int32_t pq[SCATTER_MAXP];
  __shared__ int32_t npair;
  const int32_t t = t0 + (int32_t)blockIdx.x;
  if (threadIdx.x < 64) {
    // lane c: the columns of class c that carry the target's sums: its first pair's,
    // and each tile start (class-local index a multiple of ppt) among its later pairs
    const int c = threadIdx.x;
    int32_t q0 = 0, f = 0, nh = 0;
    if (c < ca.nclass) {
      const int64_t ec = (int64_t)c * nl + t;
      const int32_t p0 = cstart[ec], n = cstart[ec + 1] - p0;
      if (n > 0) {
        q0 = p0 + ca.co[c] - ca.cs[c];
        f = q0 - ca.co[c];
        nh = 1 + (f + n - 1) / ppt - f / ppt;
      }
    }
    int32_t v = nh;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t u = __shfl_up(v, off, 64);
      if (c >= off) v += u;
    }
    const int32_t start = v - nh;
    if (nh > 0) {
      pq[start] = q0;
      for (int32_t k = 1; k < nh; k++) pq[start + k] = ca.co[c] + (f / ppt + k) * ppt;
    }
    if (c == 63) npair = v;
  }
  __syncthreads();
  const int32_t np = npair;
  for (int e = threadIdx.x; e < nbN; e += blockDim.x) {
    double acc = 0.0;
#pragma unroll 8
    for (int32_t k = 0; k < np; k++) acc += (double)Yc[(int64_t)pq[k] * nbN + e];
    pL[(int64_t)t * Ns + e] += alpha * acc;
  }
}

// As k_chunk_scatter_framed for product columns whose length nbN is a multiple of 4:
// four consecutive entries per lane, 16-byte loads (same summation order per entry)
__global__ void k_chunk_scatter_framed4(double *__restrict__ pL, const float4 *__restrict__ Yc, int Ns, int nbN4,
                                        const int32_t *__restrict__ cstart, int64_t nl, int32_t t0, double alpha,
                                        ChunkArgs ca, int ppt) {
  __shared__ int32_t pq[SCATTER_MAXP];
  __shared__ int32_t npair;
  const int32_t t = t0 + (int32_t)blockIdx.x;
  if (threadIdx.x < 64) {
    // lane c: the columns of class c that carry the target's sums: its first pair's,
    // and each tile start (class-local index a multiple of ppt) among its later pairs
    const int c = threadIdx.x;
    int32_t q0 = 0, f = 0, nh = 0;
    if (c < ca.nclass) {
      const int64_t ec = (int64_t)c * nl + t;
      const int32_t p0 = cstart[ec], n = cstart[ec + 1] - p0;
      if (n > 0) {
        q0 = p0 + ca.co[c] - ca.cs[c];
        f = q0 - ca.co[c];
        nh = 1 + (f + n - 1) / ppt - f / ppt;
      }
    }
    int32_t v = nh;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t u = __shfl_up(v, off, 64);
      if (c >= off) v += u;
    }
    const int32_t start = v - nh;
    if (nh > 0) {
      pq[start] = q0;
      for (int32_t k = 1; k < nh; k++) pq[start + k] = ca.co[c] + (f / ppt + k) * ppt;
    }
    if (c == 63) npair = v;
  }
  __syncthreads();
  const int32_t np = npair;
  for (int e = threadIdx.x; e < nbN4; e += blockDim.x) {
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
#pragma unroll 4
    for (int32_t k = 0; k < np; k++) {
      const float4 y = Yc[(int64_t)pq[k] * nbN4 + e];
      a0 += (double)y.x;
      a1 += (double)y.y;
      a2 += (double)y.z;
      a3 += (double)y.w;
    }
    double2 *o = reinterpret_cast<double2 *>(pL + (int64_t)t * Ns + 4 * e);
    double2 u = o[0], w = o[1];
    u.x += alpha * a0;
    u.y += alpha * a1;
    w.x += alpha * a2;
    w.y += alpha * a3;
    o[0] = u;
    o[1] = w;
  }
}

// Target-owned scatter of the chunk's products, all classes at once: one workgroup per
// target t, one lane per entry (b, j); pL[b N + j, t] += alpha sum over the target's pairs
// (class by class, in pair order) of sgn_t[f, i] Y_b[i, q], i = inv[f, j]
// (src/device_passes.jl:449-473; the Stokes coupling is already in the gathered fourth
// block).  The target's pairs
// (offset, chunk column) are staged in LDS first, so that each lane's loop over them
// issues independent loads.
template <class T>
__global__ void k_chunk_scatter(double *__restrict__ pL, const T *__restrict__ Yc, int Ns, int N, int nb,
                                const int32_t *__restrict__ cstart, int64_t nl, int32_t t0,
                                const int32_t *__restrict__ cfar, const int32_t *__restrict__ ssel, double alpha,
                                ChunkArgs ca) {
  __shared__ int32_t pf[SCATTER_MAXP], pq[SCATTER_MAXP];
  __shared__ int32_t npair;
  const int32_t t = t0 + (int32_t)blockIdx.x;
  const int nbN = nb * N;
  if (threadIdx.x < 64) {
    // lane c: class c's pairs of the target; an exclusive scan over the classes places them
    const int c = threadIdx.x;
    int32_t p0 = 0, n = 0;
    if (c < ca.nclass) {
      const int64_t ec = (int64_t)c * nl + t;
      p0 = cstart[ec];
      n = cstart[ec + 1] - p0;
    }
    int32_t v = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t u = __shfl_up(v, off, 64);
      if (c >= off) v += u;
    }
    const int32_t start = v - n;
    const int32_t qoff = c < ca.nclass ? ca.co[c] - ca.cs[c] : 0;
    for (int32_t k = 0; k < n; k++) {
      pf[start + k] = cfar[p0 + k];
      pq[start + k] = p0 + k + qoff;
    }
    if (c == 63) npair = v;
  }
  __syncthreads();
  const int32_t np = npair;
  for (int e = threadIdx.x; e < nbN; e += blockDim.x) {
    const int b = e / N, j = e - b * N;
    double acc = 0.0;
#pragma unroll 4
    for (int32_t k = 0; k < np; k++) {
      const int32_t f = pf[k];
      const int32_t sv = ssel[f * N + j];
      const int i = sv & 0x7fffffff;
      const double y = (double)Yc[(int64_t)pq[k] * nbN + b * N + i];
      acc += sv < 0 ? -y : y;
    }
    pL[(int64_t)t * Ns + e] += alpha * acc;
  }
}

static void gemm(Context &ctx, int m, int n, int k, double alpha, const double *A, int lda, const double *B, int ldb,
                 double beta, double *C, int ldc) {
  if (m == 0 || n == 0) return;
  FFMM_BLAS(rocblas_dgemm(ctx.blas, rocblas_operation_none, rocblas_operation_none, m, n, k, &alpha, A, lda, B, ldb,
                          &beta, C, ldc));
}

// columns per call of the mixed form's dense M2M (p = 8 with a truncated inverse or an odd
// number of check points per edge; measured there, the odd orders take the same)
constexpr int64_t M2M32_CHUNK = 10240;

static void gemm32(Context &ctx, int m, int n, int k, const float *A, int lda, const float *B, int ldb, float *C,
                   int ldc) {
  if (m == 0 || n == 0) return;
  const float one = 1.0f, zero = 0.0f;
  FFMM_BLAS(rocblas_sgemm(ctx.blas, rocblas_operation_none, rocblas_operation_none, m, n, k, &one, A, lda, B, ldb, &zero,
                          C, ldc));
}

// the harmonic methods in the mixed form with at most FM_MAXN coefficients per block take
// the fused gather + product kernel
static bool fused_m2l(const OpCache &o) {
  return o.method == METHOD_HARMONIC && o.hN <= FM_MAXN && (o.nb == 1 || o.nb == 4);
}

void allocate_pass_buffers(Plan &plan) {
  OpCache &o = *plan.ops;
  const int Ns = o.Ns, Nl = o.Nl;
  int64_t ng = 1, nlmax = 1;
  for (int l = 0; l < plan.L; l++) {
    ng = std::max(ng, plan.nl[l] / NCHILD);
    nlmax = std::max(nlmax, plan.nl[l]);
  }
  int64_t nleaves = plan.leaf_off[plan.L];
  // UC2E and DC2E run once over the leaves of all levels from 2 down
  const int l2 = std::min(2, plan.L);
  const int64_t nq = std::max<int64_t>({1, plan.s2m_off[plan.L] - plan.s2m_off[l2], nleaves - plan.leaf_off[l2]});
  plan.Mp.resize((size_t)Ns * plan.nnodes);
  plan.Pl.resize((size_t)Ns * plan.nnodes);
  plan.Lc.resize((size_t)Nl * std::max<int64_t>(nleaves, 1));
  // the densities, at the widest the method takes: Stokes 9, SphericalHarmonics(Laplace3D())
  // 4 (a charge and a dipole), else 1
  const int ndmax = o.method != METHOD_HARMONIC ? 1 : o.nb == 4 ? 9 : o.kernel == FFMM_KERNEL_LAPLACE ? 4 : 1;
  plan.tau.resize((size_t)plan.N * ndmax);
  if (o.method == METHOD_CUBE) {
    if (o.sym) {
      const int64_t ns2m = plan.s2m_off[plan.L] - plan.s2m_off[l2];
      if (sym_split_s2m(ns2m)) plan.pM.resize((size_t)8 * o.sym_kp * std::max<int64_t>(ns2m, 1));
    } else {
      plan.pM.resize((size_t)Nl * nq);
      plan.tup.resize((size_t)std::max(o.r_up, o.r_dn) * nq);
      plan.Mup.resize((size_t)Ns * nq);
    }
  }
  plan.sym = o.sym;
  plan.rank = std::max(o.r_up, o.r_dn);
  // M2M and L2L as dense products (harmonic levels that do not split; Yukawa's are not known yet)
  const bool harm = o.method == METHOD_HARMONIC;
  bool dense = !harm && !o.sym;
  if (harm)
    for (const HarmonicLevel *h : plan.hl) dense |= !h || !h->sym_m2m.p;
  if (dense) {
    plan.tM.resize((size_t)Ns * ng);
    if (!harm && plan.precision == FFMM_PREC_MIXED) {
      plan.Mp32.resize((size_t)Ns * plan.nnodes);
      plan.tM32.resize((size_t)Ns * ng);
    }
    plan.G.resize((size_t)Ns * (harm ? ng : std::max(nq, ng)));
  }
  int64_t pmax = 1;
  for (auto &li : plan.lists) pmax = std::max(pmax, li.chunk_max);
  if (plan.m2l == FFMM_M2L_DENSE && plan.precision == FFMM_PREC_MIXED) {
    // the mixed form: the class GEMMs in FP32 (FP32 MFMA), gathered from and scattered
    // into the FP64 expansions (the fused form gathers straight into LDS)
    if (!fused_m2l(o)) plan.Gc32.resize((size_t)Ns * pmax);
    plan.Yc32.resize((size_t)Ns * pmax);
  } else if (plan.m2l == FFMM_M2L_DENSE) {
    plan.Gc.resize((size_t)Ns * pmax);
    plan.Yc.resize((size_t)Ns * pmax);
  }
  if (plan.lowrank && plan.m2l == FFMM_M2L_DENSE) {   // Bt_c G of the pairs of one class of a chunk
    if (plan.precision == FFMM_PREC_MIXED)
      plan.Zc32.resize((size_t)plan.lowrank->kmax * pmax);
    else
      plan.Zc.resize((size_t)plan.lowrank->kmax * pmax);
  }
}

void gather_inputs(Plan &plan, const double *tau, int sorted) {
  Context &ctx = *plan.ctx;
  const int nd = plan.nd;
  if (sorted)
    FFMM_HIP(hipMemcpyAsync(plan.tau.p, tau, sizeof(double) * plan.N * nd, hipMemcpyDeviceToDevice, ctx.stream));
  else if (nd == 1)
    k_gather_perm<<<nblocks(plan.N, TB), TB, 0, ctx.stream>>>(plan.tau.p, tau, plan.perm.p, plan.N);
  else
    k_gather_perm_nd<<<nblocks(plan.N * nd, TB), TB, 0, ctx.stream>>>(plan.tau.p, tau, plan.perm.p, plan.N, nd);
  FFMM_LAUNCH_CHECK();
}

// upward pass: src/device_passes.jl:523-547
// whether the plan's buffers and expansions, and its low-rank factors, are of the form of its
// cache's operators, which may have been put again since
void check_operators(const Plan &plan) {
  const OpCache &o = *plan.ops;
  if (o.method != METHOD_CUBE) return;
  if (plan.sym != o.sym || std::max(o.r_up, o.r_dn) > plan.rank || (plan.lowrank && plan.lowrank->sym != o.sym))
    fail(FFMM_ERR_STATE, "the cache's operators were replaced by others of another form since the plan was made");
}

void upward_pass(Plan &plan) {
  check_operators(plan);
  Context &ctx = *plan.ctx;
  OpCache &o = *plan.ops;
  hipStream_t s = ctx.stream;
  const int Ns = o.Ns, Nl = o.Nl;
  const int l2 = std::min(2, plan.L);
  const int64_t nq = plan.s2m_off[plan.L] - plan.s2m_off[l2];
  const int32_t *nodes = plan.s2m_nodes.p + plan.s2m_off[l2];
  const bool harm = o.method == METHOD_HARMONIC;
  if (o.sym || harm) {
    // every sourced column from level 2 down is written before it is read; the others are zero
    const int64_t n01 = l2 < plan.L ? plan.lo[l2] : plan.nnodes;
    k_fill<<<nblocks((int64_t)Ns * n01, TB), TB, 0, s>>>(plan.Mp.p, (int64_t)Ns * n01, 0.0);
    FFMM_LAUNCH_CHECK();
    sym_zero_unsourced(plan);
    if (harm) {
      for (int l = plan.L - 1; l >= 2; l--) {
        // the multipoles directly (partial_to_multipole! is a copy, src/operators/harmonics.jl:441)
        harmonic_s2m_level(plan, l);
        if (l == plan.L - 1) continue;
        if (plan.hl[l]->sym_m2m.p) {
          sym_harmonic_m2m(plan, l);
          continue;
        }
        const int64_t ng = plan.nl[l + 1] / NCHILD;
        gemm(ctx, Ns, (int)ng, NCHILD * Ns, 1.0, plan.hl[l]->M2M.p, Ns, plan.Mp.p + plan.lo[l + 1] * Ns, NCHILD * Ns, 0.0,
             plan.tM.p, Ns);
        k_scatter_parents<double><<<nblocks((int64_t)Ns * ng, TB), TB, 0, s>>>(plan.Mp.p, plan.tM.p, plan.parent.p,
                                                                               plan.lo[l + 1], Ns, ng, 1.0, nullptr);
        FFMM_LAUNCH_CHECK();
      }
      return;
    }
    if (nq > 0) sym_s2m_uc2e(plan, nodes, nq);
    for (int l = plan.L - 2; l >= 2; l--) sym_m2m(plan, l);
    return;
  }
  // every column is written before it is read except by M2M of empty groups: clear.  The
  // cube's mixed form keeps an FP32 mirror of the multipoles, written beside them by the
  // UC2E and M2M scatters, that its FP32 M2M GEMMs read directly
  const bool mirror = plan.precision == FFMM_PREC_MIXED;
  float *Mp32 = mirror ? plan.Mp32.p : nullptr;
  k_fill<<<nblocks(plan.Mp.n, TB), TB, 0, s>>>(plan.Mp.p, plan.Mp.n, 0.0);
  FFMM_LAUNCH_CHECK();
  if (mirror) {
    k_fill32<<<nblocks(plan.Mp32.n, TB), TB, 0, s>>>(Mp32, plan.Mp32.n);
    FFMM_LAUNCH_CHECK();
  }
  if (nq > 0) {
    // the childless sourced nodes of all levels at once (each node's width from its level):
    // S2M into check potentials, then UC2E, M = pinv_scale V diag(invS) (Uh pM)
    // (src/device_passes.jl:496-502), as two GEMMs over all of them.  pinv_scale = lam[l]
    // is a power of two, applied exactly in the scatter.
    const dim3 g((unsigned)nq, (unsigned)((Nl + S2M_TB * S2M_KP - 1) / (S2M_TB * S2M_KP)));
    if (plan.precision == FFMM_PREC_MIXED)
      k_s2m32<<<g, S2M_TB, 0, s>>>(nodes, plan.centers.p, plan.nnodes, plan.level.p, plan.lam_d.p,
                                              o.large.p, Nl, plan.plo.p, plan.phi.p, plan.sx.p, plan.sy.p, plan.sz.p,
                                              plan.tau.p, plan.pM.p);
    else
      k_s2m<<<g, S2M_TB, 0, s>>>(nodes, plan.centers.p, plan.nnodes, plan.level.p, plan.lam_d.p, o.large.p,
                                            Nl, plan.plo.p, plan.phi.p, plan.sx.p, plan.sy.p, plan.sz.p, plan.tau.p,
                                            plan.pM.p);
    FFMM_LAUNCH_CHECK();
    gemm(ctx, o.r_up, (int)nq, Nl, 1.0, o.Uh_up.p, o.r_up, plan.pM.p, Nl, 0.0, plan.tup.p, o.r_up);
    gemm(ctx, Ns, (int)nq, o.r_up, 1.0, o.Vs_up.p, Ns, plan.tup.p, o.r_up, 0.0, plan.Mup.p, Ns);
    k_scatter_cols_lam<<<nblocks((int64_t)Ns * nq, TB), TB, 0, s>>>(plan.Mp.p, plan.Mup.p, nodes, Ns, nq, plan.level.p,
                                                                    plan.lam_d.p, Mp32);
    FFMM_LAUNCH_CHECK();
  }
  for (int l = plan.L - 1; l >= 2; l--) {
    if (l < plan.L - 1) {
      const int64_t ng = plan.nl[l + 1] / NCHILD;
      const double *B = plan.Mp.p + plan.lo[l + 1] * Ns;
      if (mirror) {
        // the mixed form: M2M as an FP32 GEMM over the children's FP32 mirror (its rounding
        // is not amplified: the multipoles feed M2L, never a pseudo-inverse).  Wide levels
        // go in column chunks: for n above ~11k the library takes 256 x 256 tiles, at most
        // 192 workgroups for m = 296, each a 0.5 ms tile on one CU (levels of 14k-25k
        // groups all took ~0.55 ms), where a chunk takes a one-wave grid of smaller tiles
        const float *Bc = Mp32 + plan.lo[l + 1] * Ns;
        for (int64_t c0 = 0; c0 < ng; c0 += M2M32_CHUNK) {
          const int nc = (int)std::min<int64_t>(M2M32_CHUNK, ng - c0);
          gemm32(ctx, Ns, nc, NCHILD * Ns, o.M2M32.p, Ns, Bc + c0 * NCHILD * Ns, NCHILD * Ns, plan.tM32.p + c0 * Ns,
                 Ns);
        }
        k_scatter_parents<float><<<nblocks((int64_t)Ns * ng, TB), TB, 0, s>>>(plan.Mp.p, plan.tM32.p, plan.parent.p,
                                                                              plan.lo[l + 1], Ns, ng, 1.0, Mp32);
      } else {
        gemm(ctx, Ns, (int)ng, NCHILD * Ns, 1.0, o.M2M.p, Ns, B, NCHILD * Ns, 0.0, plan.tM.p, Ns);
        k_scatter_parents<double><<<nblocks((int64_t)Ns * ng, TB), TB, 0, s>>>(plan.Mp.p, plan.tM.p, plan.parent.p,
                                                                               plan.lo[l + 1], Ns, ng, 1.0, nullptr);
      }
      FFMM_LAUNCH_CHECK();
    }
  }
}

void m2l_dense_level(Plan &plan, int l) {
  Context &ctx = *plan.ctx;
  OpCache &o = *plan.ops;
  hipStream_t s = ctx.stream;
  const int Ns = o.Ns;
  const bool harm = o.method == METHOD_HARMONIC;
  const int N = harm ? o.hN : Ns, nb = harm ? o.nb : 1;
  LevelLists &li = plan.lists[l];
  double *pL = plan.Pl.p + plan.lo[l] * Ns;
  // m2l_scale of the level: (w_l / w_ref)^(-1) for the homogeneous kernels, 1 for Yukawa
  const double alpha = harm ? plan.alpha[l] : 1.0 / plan.lam[l];
  const double *reps = harm ? plan.hl[l]->reps.p : o.class_ops.p;
  const float *reps32 = harm ? plan.hl[l]->reps32.p : o.class_ops32.p;
  const bool f32 = plan.precision == FFMM_PREC_MIXED;
  const int nbN = N * nb;
  const unsigned bt = (unsigned)std::min(1024, (nbN + 63) / 64 * 64);   // scatter: a lane per entry
  const unsigned btg = (unsigned)std::min(1024, (N + 63) / 64 * 64);    // gather: a lane per coefficient
  const int64_t nch = (int64_t)li.chunk_t.size() - 1;
  const bool fused = f32 && plan.m2l == FFMM_M2L_DENSE && fused_m2l(o);
  for (int64_t k = 0; k < nch; k++) {
    ChunkArgs ca{};
    ca.nclass = o.nclass;
    for (int c = 0; c < o.nclass; c++) {
      ca.cs[c] = li.chunk_cs[k * o.nclass + c];
      ca.co[c + 1] = ca.co[c] + (li.chunk_cs[(k + 1) * o.nclass + c] - ca.cs[c]);
    }
    const int32_t npk = ca.co[o.nclass];
    const int32_t t0 = li.chunk_t[k], nt = li.chunk_t[k + 1] - t0;
    if (npk == 0 || nt == 0) continue;
    if (fused) {
      const bf16x8 *ops = reinterpret_cast<const bf16x8 *>(plan.hl[l]->repsb.p);
      const uint32_t *g8 = reinterpret_cast<const uint32_t *>(o.gsel8.p), *f8 = reinterpret_cast<const uint32_t *>(o.fsel8.p);
      const int ppt = FM_COLS / nb;
      for (int c = 0; c < o.nclass; c++) ca.to[c + 1] = ca.to[c] + (ca.co[c + 1] - ca.co[c] + ppt - 1) / ppt;
      const int32_t ntiles = ca.to[o.nclass];
      const unsigned grid = (unsigned)std::min<int64_t>(ntiles, 2 * 256);   // two workgroups per CU
      auto go = [&](auto NB, auto KB) {
        k_class_m2l32<decltype(NB)::value, decltype(KB)::value><<<grid, FM_TB, 0, s>>>(
            plan.Yc32.p, plan.Mp.p, Ns, N, ops, li.csrc.p, li.cfar.p, g8, f8, o.offs.p, ca, ntiles, li.ctgt.p);
      };
      auto kb = [&](auto NB) {
        if (N <= 32) go(NB, std::integral_constant<int, 1>{});
        else if (N <= 64) go(NB, std::integral_constant<int, 2>{});
        else if (N <= 96) go(NB, std::integral_constant<int, 3>{});
        else go(NB, std::integral_constant<int, 4>{});
      };
      if (nb == 4) kb(std::integral_constant<int, 4>{});
      else kb(std::integral_constant<int, 1>{});
      FFMM_LAUNCH_CHECK();
      if (nbN % 4 == 0) {
        const unsigned bt4 = (unsigned)std::min(1024, (nbN / 4 + 63) / 64 * 64);
        k_chunk_scatter_framed4<<<(unsigned)nt, bt4, 0, s>>>(pL, reinterpret_cast<const float4 *>(plan.Yc32.p), Ns,
                                                              nbN / 4, li.cstart.p, plan.nl[l], t0, alpha, ca, ppt);
      } else {
        k_chunk_scatter_framed<<<(unsigned)nt, bt, 0, s>>>(pL, plan.Yc32.p, Ns, nbN, li.cstart.p, plan.nl[l], t0,
                                                           alpha, ca, ppt);
      }
      FFMM_LAUNCH_CHECK();
      continue;
    }
    const unsigned gg = (unsigned)((npk + GATHER_PAIRS - 1) / GATHER_PAIRS);
    if (f32) {
      k_chunk_gather<float><<<gg, btg, 0, s>>>(plan.Gc32.p, plan.Mp.p, Ns, N, nb, li.csrc.p, li.cfar.p, npk, o.gsel.p,
                                              o.offs.p, ca);
      FFMM_LAUNCH_CHECK();
      for (int c = 0; c < o.nclass; c++) {
        const int32_t n = ca.co[c + 1] - ca.co[c];
        if (n == 0) continue;
        const size_t off = (size_t)ca.co[c] * nbN;
        if (const ClassFactors *lr = plan.lowrank) {   // A_c (Bt_c G): src/device_passes.jl:570-576
          const int kc = lr->rank[c];
          gemm32(ctx, kc, nb * n, N, lr->Bt32.p + lr->off[c], kc, plan.Gc32.p + off, N, plan.Zc32.p, kc);
          gemm32(ctx, N, nb * n, kc, lr->A32.p + lr->off[c], N, plan.Zc32.p, kc, plan.Yc32.p + off, N);
        } else {
          gemm32(ctx, N, nb * n, N, reps32 + (size_t)c * N * N, N, plan.Gc32.p + off, N, plan.Yc32.p + off, N);
        }
      }
      k_chunk_scatter<float><<<(unsigned)nt, bt, 0, s>>>(pL, plan.Yc32.p, Ns, N, nb, li.cstart.p, plan.nl[l], t0,
                                                         li.cfar.p, o.ssel.p, alpha, ca);
    } else {
      k_chunk_gather<double><<<gg, btg, 0, s>>>(plan.Gc.p, plan.Mp.p, Ns, N, nb, li.csrc.p, li.cfar.p, npk, o.gsel.p,
                                               o.offs.p, ca);
      FFMM_LAUNCH_CHECK();
      for (int c = 0; c < o.nclass; c++) {
        const int32_t n = ca.co[c + 1] - ca.co[c];
        if (n == 0) continue;
        const size_t off = (size_t)ca.co[c] * nbN;
        if (const ClassFactors *lr = plan.lowrank) {   // A_c (Bt_c G): src/device_passes.jl:570-576
          const int kc = lr->rank[c];
          gemm(ctx, kc, nb * n, N, 1.0, lr->Bt.p + lr->off[c], kc, plan.Gc.p + off, N, 0.0, plan.Zc.p, kc);
          gemm(ctx, N, nb * n, kc, 1.0, lr->A.p + lr->off[c], N, plan.Zc.p, kc, 0.0, plan.Yc.p + off, N);
        } else {
          gemm(ctx, N, nb * n, N, 1.0, reps + (size_t)c * N * N, N, plan.Gc.p + off, N, 0.0, plan.Yc.p + off, N);
        }
      }
      k_chunk_scatter<double><<<(unsigned)nt, bt, 0, s>>>(pL, plan.Yc.p, Ns, N, nb, li.cstart.p, plan.nl[l], t0,
                                                          li.cfar.p, o.ssel.p, alpha, ca);
    }
    FFMM_LAUNCH_CHECK();
  }
}

// downward pass: src/device_passes.jl:548-595
void downward_pass(Plan &plan) {
  Context &ctx = *plan.ctx;
  OpCache &o = *plan.ops;
  hipStream_t s = ctx.stream;
  const int Ns = o.Ns, Nl = o.Nl;
  // levels 0 and 1 have no far field: their partial locals and leaf densities are zero
  const int l2 = std::min(2, plan.L);
  const int64_t n01 = l2 < plan.L ? plan.lo[l2] : plan.nnodes;
  k_fill<<<nblocks((int64_t)Ns * n01, TB), TB, 0, s>>>(plan.Pl.p, (int64_t)Ns * n01, 0.0);
  k_fill<<<nblocks((int64_t)Nl * plan.leaf_off[l2], TB), TB, 0, s>>>(plan.Lc.p, (int64_t)Nl * plan.leaf_off[l2], 0.0);
  FFMM_LAUNCH_CHECK();
  for (int l = 2; l < plan.L; l++) {
    const int64_t nl = plan.nl[l], ng = nl / NCHILD;
    double *pL = plan.Pl.p + plan.lo[l] * Ns;
    if (l > 2 && o.sym) {
      sym_l2l(plan, l);
    } else if (l > 2 && o.method == METHOD_HARMONIC && plan.hl[l - 1]->sym_l2l.p) {
      sym_harmonic_l2l(plan, l);
    } else if (l > 2) {
      k_gather_parents<<<nblocks((int64_t)Ns * ng, TB), TB, 0, s>>>(plan.G.p, plan.Pl.p, plan.parent.p, plan.lo[l],
                                                                    Ns, ng);
      FFMM_LAUNCH_CHECK();
      // the stacked children output of L2L is the level's block of partial locals
      const double *L2L = o.method == METHOD_HARMONIC ? plan.hl[l - 1]->L2L.p : o.L2L.p;
      gemm(ctx, NCHILD * Ns, (int)ng, Ns, 1.0, L2L, NCHILD * Ns, plan.G.p, Ns, 0.0, pL, NCHILD * Ns);
    } else {
      k_fill<<<nblocks((int64_t)Ns * nl, TB), TB, 0, s>>>(pL, (int64_t)Ns * nl, 0.0);
      FFMM_LAUNCH_CHECK();
    }
    StageTimer tm(plan, 4, l);
    if (plan.m2l == FFMM_M2L_SPECTRAL) m2l_spectral_level(plan, l);
    else m2l_dense_level(plan, l);
  }
  // the densities of the real leaves of all levels at once: DC2E (src/device_passes.jl:582-593)
  const int64_t nq = plan.leaf_off[plan.L] - plan.leaf_off[l2];
  if (nq == 0) return;
  const int32_t *leaves = plan.leaf_nodes.p + plan.leaf_off[l2];
  double *Lc = plan.Lc.p + plan.leaf_off[l2] * Nl;
  if (o.method == METHOD_HARMONIC) {
    // partial_to_local! is a copy (src/operators/harmonics.jl:442)
    k_gather_cols<<<nblocks((int64_t)Ns * nq, TB), TB, 0, s>>>(Lc, plan.Pl.p, leaves, Ns, nq);
    FFMM_LAUNCH_CHECK();
    return;
  }
  if (o.sym) {
    sym_dc2e(plan, leaves, nq, Lc);
    return;
  }
  // the level's pinv_scale (a power of two) on the gathered check potentials: exact
  k_gather_cols_lam<<<nblocks((int64_t)Ns * nq, TB), TB, 0, s>>>(plan.G.p, plan.Pl.p, leaves, Ns, nq, plan.level.p,
                                                                 plan.lam_d.p);
  FFMM_LAUNCH_CHECK();
  gemm(ctx, o.r_dn, (int)nq, Ns, 1.0, o.Uh_dn.p, o.r_dn, plan.G.p, Ns, 0.0, plan.tup.p, o.r_dn);
  gemm(ctx, Nl, (int)nq, o.r_dn, 1.0, o.Vs_dn.p, Nl, plan.tup.p, o.r_dn, 0.0, Lc, Nl);
}

}  // namespace ffmm
