// The spectral M2L of the cube method on the device.
//
// The small surfaces of all boxes are p-per-edge lattices of one spacing, so M2L at a
// far offset is a convolution of the multipole with a kernel table.  A source index and a
// target index differ by -(p-1) .. p-1 along each axis: 2p - 1 = 15 values, so a circular
// convolution of length 15 gives every output that is kept (length 16 would carry 36%
// more frequencies: 2,304 against 1,688, a real spectrum's unique ones).  Per level:
//   1. forward: every sourced sibling group's multipoles into their spectra, three passes
//      of short DFTs over the 8 nonzero inputs of an axis;
//   2. Hadamard: the products of a frequency, sum over the far pairs of T_f[w] S_s[w], as
//      small matrix products on the matrix cores (below);
//   3. inverse: per group of targets the three inverse DFTs with only the p^3 corner of
//      the output formed, the surface entries scaled and added into the partial locals.
// Spectra are stored by chunks of 512 nodes of the level, frequency-major inside a chunk
// (sp_at): the 8 children of a box are 64 (128 in FP64) contiguous bytes of a frequency,
// which is what the products read, and a box's transform writes into one 7 (14) MB chunk (one
// frequency row for the whole level spread its writes over 1,688 pages: 1.3 times slower).
// Follows _spectral_m2l_level! and _hadamard_block! (src/operators/spectral_m2l.jl:
// 260-286, 328-451); the pair enumeration is that of the interaction lists
// (src/tree/lists.jl:96-124).  p = 8 is fixed here.
#include "ffmm_internal.h"

#include <algorithm>
#include <cmath>
#include <complex>
#include <type_traits>

namespace ffmm {

constexpr int SP_P = 8;                       // points per edge
constexpr int SP_N = 2 * SP_P - 1;            // circular convolution length
constexpr int SP_K1 = SP_P;                   // k1 = 0 .. 7 (the conjugates make up 8 .. 14)
// columns (k1, k2) of the half spectrum: column c < 8 is (0, c), whose partners (0, 15 - c)
// are conjugates; then (k1, k2) at 8 + 15 (k1 - 1) + k2.  Column 0 holds k3 = 0 .. 7 only.
constexpr int SP_COLS = SP_P + (SP_K1 - 1) * SP_N;            // 113
constexpr int SP_NF = SP_P + (SP_COLS - 1) * SP_N;            // 1688 frequencies
static_assert(SP_NF == (SP_N * SP_N * SP_N + 1) / 2, "the unique frequencies of a real 15^3 lattice");
__host__ __device__ constexpr int sp_col(int k1, int k2) { return k1 == 0 ? k2 : SP_P + (k1 - 1) * SP_N + k2; }
__host__ __device__ constexpr int sp_freq(int col, int k3) { return col == 0 ? k3 : SP_P + (col - 1) * SP_N + k3; }

constexpr int SP_CH = 512;                                    // nodes per chunk
__host__ __device__ constexpr int64_t sp_at(int64_t node, int w) {
  return (node / SP_CH * SP_NF + w) * SP_CH + node % SP_CH;
}

template <class T> struct cplx_t;
template <> struct cplx_t<double> { using type = double2; };
template <> struct cplx_t<float> { using type = float2; };

// cos(2 pi j / 15) and sin(2 pi j / 15): every twiddle is one of them, at an index known at
// compile time once the loops are unrolled, so it is an immediate and no table is read.
__device__ constexpr double W15C[SP_N] = {1.0, 0.9135454576426009, 0.6691306063588582, 0.30901699437494745,
    -0.10452846326765333, -0.4999999999999998, -0.8090169943749473, -0.9781476007338057, -0.9781476007338057,
    -0.8090169943749473, -0.4999999999999998, -0.10452846326765333, 0.30901699437494745, 0.6691306063588582,
    0.9135454576426009};
__device__ constexpr double W15S[SP_N] = {0.0, 0.40673664307580015, 0.7431448254773941, 0.9510565162951535,
    0.9945218953682734, 0.8660254037844387, 0.5877852522924732, 0.20791169081775931, -0.20791169081775931,
    -0.5877852522924732, -0.8660254037844387, -0.9945218953682734, -0.9510565162951535, -0.7431448254773941,
    -0.40673664307580015};

// out[k] = sum_{i < 8} a[i] w^(i k), w = exp(-2 pi i / 15): the sums with cosines and with
// sines serve k and 15 - k
template <class C, class T>
__device__ __forceinline__ void dft8to15(const C a[SP_P], C out[SP_N]) {
  C s = a[0];
#pragma unroll
  for (int i = 1; i < SP_P; i++) {
    s.x += a[i].x;
    s.y += a[i].y;
  }
  out[0] = s;
#pragma unroll
  for (int k = 1; k < SP_P; k++) {
    T xc = a[0].x, yc = a[0].y, xs = 0, ys = 0;
#pragma unroll
    for (int i = 1; i < SP_P; i++) {
      const T c = (T)W15C[(i * k) % SP_N], n = (T)W15S[(i * k) % SP_N];
      xc = fma(a[i].x, c, xc);
      yc = fma(a[i].y, c, yc);
      xs = fma(a[i].x, n, xs);
      ys = fma(a[i].y, n, ys);
    }
    out[k] = C{xc + ys, yc - xs};
    out[SP_N - k] = C{xc - ys, yc + xs};
  }
}
// out[i] = sum_{k < 15} u[k] w^(-i k), i < 8, by the pairs k, 15 - k
template <class C, class T>
__device__ __forceinline__ void idft15to8(const C u[SP_N], C out[SP_P]) {
  C p[SP_P], m[SP_P];
#pragma unroll
  for (int k = 1; k < SP_P; k++) {
    p[k] = C{u[k].x + u[SP_N - k].x, u[k].y + u[SP_N - k].y};
    m[k] = C{u[k].x - u[SP_N - k].x, u[k].y - u[SP_N - k].y};
  }
#pragma unroll
  for (int i = 0; i < SP_P; i++) {
    C s = u[0];
#pragma unroll
    for (int k = 1; k < SP_P; k++) {
      const T c = (T)W15C[(i * k) % SP_N], n = (T)W15S[(i * k) % SP_N];
      s.x = fma(p[k].x, c, fma(-m[k].y, n, s.x));
      s.y = fma(p[k].y, c, fma(m[k].x, n, s.y));
    }
    out[i] = s;
  }
}

// ---------------------------------------------------------------------------
// 1. forward and 3. inverse: NB boxes (consecutive nodes) per workgroup, the box index
//    fastest among the lanes, so that a wave's stores of one frequency are 64 contiguous
//    bytes per 8 boxes (FP64: 4 boxes, 64 bytes) and its LDS accesses are free of bank
//    conflicts (the row strides below are 64 modulo 128 bytes).  Bound by the spectra's
//    traffic: 13.5 KB per box in FP32 (18.4 KB with 16^3).
// ---------------------------------------------------------------------------
template <class T> struct SpBoxes;
template <> struct SpBoxes<float> { static constexpr int NB = 8; };
template <> struct SpBoxes<double> { static constexpr int NB = 4; };

template <class T>
__global__ void __launch_bounds__(64 * SpBoxes<T>::NB) k_spec_forward(const double *__restrict__ Mp, int Ns,
                                                                     const int16_t *__restrict__ lat8, int64_t lo,
                                                                     int64_t nl, const uint8_t *__restrict__ has_source,
                                                                     typename cplx_t<T>::type *__restrict__ S) {
  using C = typename cplx_t<T>::type;
  constexpr int NB = SpBoxes<T>::NB, TB = 64 * NB, RS = 9 * NB;   // RS: padded stride of a lattice row
  __shared__ C W[SP_P * SP_COLS * NB];   // [i3 i2][k1][box], then [i3][column][box]
  __shared__ T m[NB * 296];
  const int t = threadIdx.x, b = t % NB, u = t / NB;
  // plain block order: neighbouring boxes write neighbouring bytes of the same rows at the same
  // time from all XCDs (a contiguous range per XCD measured 1.4 times slower)
  const int64_t q0 = (int64_t)blockIdx.x * NB;
  bool any = false;
  for (int i = 0; i < NB; i++) any |= has_source[lo + q0 + i] != 0;
  if (!any) return;
  for (int i = t; i < NB * Ns; i += TB) m[i] = has_source[lo + q0 + i / Ns] ? (T)Mp[(lo + q0) * Ns + i] : (T)0;
  __syncthreads();
  {   // row u = (i3, i2): real inputs over i1
    T x[SP_P];
#pragma unroll
    for (int i1 = 0; i1 < SP_P; i1++) {
      const int s = lat8[u * SP_P + i1];
      x[i1] = s >= 0 ? m[b * Ns + s] : (T)0;
    }
#pragma unroll
    for (int k1 = 0; k1 < SP_K1; k1++) {
      T xc = x[0], xs = 0;
#pragma unroll
      for (int i1 = 1; i1 < SP_P; i1++) {
        xc = fma(x[i1], (T)W15C[(i1 * k1) % SP_N], xc);
        xs = fma(x[i1], (T)W15S[(i1 * k1) % SP_N], xs);
      }
      W[u * RS + k1 * NB + b] = C{xc, -xs};
    }
  }
  __syncthreads();
  {   // u = (i3, k1): over i2
    const int i3 = u / SP_K1, k1 = u % SP_K1;
    C a[SP_P], out[SP_N];
#pragma unroll
    for (int i2 = 0; i2 < SP_P; i2++) a[i2] = W[(i3 * SP_P + i2) * RS + k1 * NB + b];
    __syncthreads();
    dft8to15<C, T>(a, out);
#pragma unroll
    for (int k2 = 0; k2 < SP_N; k2++)
      if (k1 > 0 || k2 < SP_P) W[(i3 * SP_COLS + sp_col(k1, k2)) * NB + b] = out[k2];
  }
  __syncthreads();
  for (int col = u; col < SP_COLS; col += 64) {   // over i3
    C a[SP_P], out[SP_N];
#pragma unroll
    for (int i3 = 0; i3 < SP_P; i3++) a[i3] = W[(i3 * SP_COLS + col) * NB + b];
    dft8to15<C, T>(a, out);
    C *__restrict__ o = S + sp_at(q0 + b, sp_freq(col, 0));
#pragma unroll
    for (int k3 = 0; k3 < SP_N; k3++)
      if (col > 0 || k3 < SP_P) o[k3 * SP_CH] = out[k3];
  }
}

// x = the inverse transform on the [0, p)^3 corner.  The sum over the conjugate half is
// taken by x = 2 Re sum_{stored} u w^-(..), the self-conjugate (0, 0, 0) halved.
template <class T>
__global__ void __launch_bounds__(64 * SpBoxes<T>::NB) k_spec_inverse(const typename cplx_t<T>::type *__restrict__ U,
                                                                     const int32_t *__restrict__ ptr,
                                                                     const int16_t *__restrict__ lat8, int64_t nl, int Ns,
                                                                     double alpha, double *__restrict__ pL) {
  using C = typename cplx_t<T>::type;
  constexpr int NB = SpBoxes<T>::NB, TB = 64 * NB, RS = 9 * NB;
  __shared__ C W[SP_P * SP_COLS * NB];
  __shared__ T x[NB * 296];
  const int t = threadIdx.x, b = t % NB, u = t / NB;
  const int64_t q0 = (int64_t)blockIdx.x * NB;
  if (ptr[q0 + NB] == ptr[q0]) return;      // no far pairs (ghosts included)
  const bool live = ptr[q0 + b + 1] > ptr[q0 + b];
  for (int col = u; col < SP_COLS; col += 64) {   // over k3
    C in[SP_N], out[SP_P];
    const C *__restrict__ p = U + sp_at(q0 + b, sp_freq(col, 0));
#pragma unroll
    for (int k3 = 0; k3 < SP_N; k3++) in[k3] = live && (col > 0 || k3 < SP_P) ? p[k3 * SP_CH] : C{(T)0, (T)0};
    if (col == 0) {
      in[0].x *= (T)0.5;
      in[0].y *= (T)0.5;
    }
    idft15to8<C, T>(in, out);
#pragma unroll
    for (int i3 = 0; i3 < SP_P; i3++) W[(i3 * SP_COLS + col) * NB + b] = out[i3];
  }
  __syncthreads();
  {   // u = (i3, k1): over k2
    const int i3 = u / SP_K1, k1 = u % SP_K1;
    C in[SP_N], out[SP_P];
#pragma unroll
    for (int k2 = 0; k2 < SP_N; k2++)
      in[k2] = k1 > 0 || k2 < SP_P ? W[(i3 * SP_COLS + sp_col(k1, k2)) * NB + b] : C{(T)0, (T)0};
    __syncthreads();
    idft15to8<C, T>(in, out);
#pragma unroll
    for (int i2 = 0; i2 < SP_P; i2++) W[(i3 * SP_P + i2) * RS + k1 * NB + b] = out[i2];
  }
  __syncthreads();
  {   // lattice row u = (i3, i2): the real outputs
    C d[SP_K1];
#pragma unroll
    for (int k1 = 0; k1 < SP_K1; k1++) d[k1] = W[u * RS + k1 * NB + b];
#pragma unroll
    for (int i1 = 0; i1 < SP_P; i1++) {
      const int s = lat8[u * SP_P + i1];
      if (s < 0) continue;
      T y = d[0].x;
#pragma unroll
      for (int k1 = 1; k1 < SP_K1; k1++)
        y = fma(d[k1].x, (T)W15C[(i1 * k1) % SP_N], fma(-d[k1].y, (T)W15S[(i1 * k1) % SP_N], y));
      x[b * Ns + s] = y + y;
    }
  }
  __syncthreads();
  for (int i = t; i < NB * Ns; i += TB) {
    const int64_t q = q0 + i / Ns;
    if (ptr[q + 1] > ptr[q]) pL[q0 * Ns + i] += alpha * (double)x[i];
  }
}

// ---------------------------------------------------------------------------
// 2. Hadamard: U[w][t] = sum over the far pairs (t, s) of T_f[w] S[w][s]
//
// For one frequency the products of a sibling group are a small matrix product: the
// targets a of group g gain sum over the parent's colleagues k and their children c of
// T[F(k, c, a)] S[child c of colleague k], and the 8 x 8 block T[F(k, c, a)] is the same
// for every group (zero where the pair is near).  So 16 groups at a time are the 16 columns
// of the matrix instructions, whose rows are (target a, real / imaginary part) and whose K
// runs over (colleague, child, real / imaginary part).
//
// The 16 groups of a tile are consecutive in the level's order, so their parents lie close
// together and share colleagues: a tile's (group, colleague) entries name about a third as
// many distinct boxes.  Once per plan, each tile's distinct sourced colleagues (its union)
// are found and placed in staging rows; a tile naming more than 192 is cut into halves of 8
// groups or quarters of 4.  A workgroup takes a block of frequencies and up to 64 consecutive
// subtiles; per tile it stages the union's child spectra in LDS (zeros for children without
// sources; zero boxes for missing colleagues), the next tile's loaded into registers
// during this tile's products.  The table operands of a wave's colleagues sit in registers
// for the whole workgroup, read as ready fragments.
//
// FP64: v_mfma_f64_16x16x4, 4 waves each over a quarter of the colleagues, two workgroups per
// CU.  Measured: 300k sources 9.0 -> 4.5 ms (the products on the vector ALUs before, bound by
// LDS); the matrix cores are busy half the time.
// Mixed: each FP32 value as three bfloat16 pieces (8 significant bits each: the whole FP32
// mantissa), the products of pieces down to 2^-24 on v_mfma_f32_16x16x32_bf16 in three FP32
// accumulators: hi hi; mid hi and hi mid; lo hi, mid mid and hi lo.  Six bfloat16 products cost
// 96 cycles per 64 x 16 block of 32 K where v_mfma_f32_16x16x4 takes 256, and a K of 32 per
// instruction rounds the sums less often: against 64 bits the potential's error fell from
// 2.5e-7 to 1.1e-7 at 1M mixture sources.  The pieces of values below some 2^-110 leave
// bfloat16's range: with charges of 2^-112 (2e-34) the error is as above, of 2^-116 2.5e-7,
// of 2^-120 3.6e-6 (FP32 operands 1.4e-7), of 2^-126 2.5e-4 (1.9e-6).
// Measured: 4M sources 17.1 -> 8.0 ms; bound by LDS (active 67% of the cycles, half of that
// counted as bank conflicts), then vector ALU (51%) and matrix cores (33%); 1.78 GB fetched
// and 0.46 GB written a level, 2.8 TB/s.
// ---------------------------------------------------------------------------
constexpr int HM_TILE = 16;          // sibling groups per tile: the matrix instructions' columns
typedef double f64x4 __attribute__((ext_vector_type(4)));

// The levels 2 .. L-1 of a plan: first node, first sibling group and first tile of each.
struct SpLevels {
  int L;
  int64_t lo[MAX_KEY_LEVELS + 3], goff[MAX_KEY_LEVELS + 3], toff[MAX_KEY_LEVELS + 3];   // [l]; goff, toff to L
};
__device__ __forceinline__ int sp_level(const SpLevels &v, const int64_t *off, int64_t x) {
  int l = 2;
  while (l + 1 < v.L && off[l + 1] <= x) l++;
  return l;
}

// gcol[g * 27 + k]: (first child of the parent's colleague k, level-local) << 8 | bit c
// set when that child has sources; -1 when the colleague is missing or has no sourced
// child, and for every k of a ghost group.
__global__ void k_group_cols(SpLevels v, const int32_t *__restrict__ parent, const int32_t *__restrict__ child_first,
                             const int32_t *__restrict__ col, const uint8_t *__restrict__ ghost,
                             const uint8_t *__restrict__ has_source, int64_t ngroups, int64_t nn,
                             int32_t *__restrict__ gcol) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t g = i / NCOLL;
  const int k = (int)(i % NCOLL);
  if (g >= ngroups) return;
  const int l = sp_level(v, v.goff, g);
  const int64_t lo = v.lo[l], first = lo + NCHILD * (g - v.goff[l]);
  int32_t e = -1;
  const int32_t pc = ghost[first] ? -1 : col[(int64_t)k * nn + parent[first]];
  const int32_t cf = pc >= 0 ? child_first[pc] : -1;
  if (cf >= 0) {
    int32_t m = 0;
    for (int c = 0; c < NCHILD; c++) m |= (int32_t)(has_source[cf + c] != 0) << c;
    if (m) e = (int32_t)((cf - lo) << 8) | m;
  }
  gcol[i] = e;
}

constexpr int HU_NK = NCOLL - 1;            // colleagues other than the parent itself
constexpr int HU_B = 192;                   // boxes of a subtile at most (a tile with more is cut)
constexpr int HU_SUB = 4;                   // subtiles of a tile at most (4 groups x 26 boxes fit)
constexpr int HU_NC = 16;                   // colours of the staged boxes
constexpr int HU_CAP = 13;                  // boxes of a colour at most
constexpr int HU_ZROW = HU_NC * HU_CAP;     // the zero boxes, one of each colour
constexpr int HU_NR = HU_ZROW + HU_NC;      // staging rows
constexpr int HU_NS = HM_TILE * HU_NK;      // (group, colleague) slots of a tile
constexpr int HU_R = 64;                    // subtiles per workgroup at most
static_assert(HU_ZROW >= HU_B && HU_NR <= 256, "rows are bytes");
static_assert(HM_TILE / HU_SUB * HU_NK <= HU_B, "a quarter of a tile fits");

// Per tile: the distinct sourced colleagues of its groups (its union), each placed in a row
// of the staging buffer.  A tile whose union has more than HU_B boxes is cut into halves of 8
// groups, a half with more into quarters; sflag of subtile 4 ti + i holds the quarters of
// groups that it covers (bits 0 .. 3; 0: no subtile).  ulist[s][i] = the box's group of children << 10 | whether
// its children 4 .. 7 and 0 .. 3 have sources << 8 | row, 0 past the last; uslot[s][26 j + kk] = the row of group j's colleague
// (a zero box, of a colour that no box of its phase has, when it has none).  The matrix instructions' operand reads take a phase of 8
// groups at one colleague index; a box's row is its colour + 16 x (its place among its
// colour), the colours chosen greedily (in order of first appearance) so that the boxes of
// one (colleague index, half of the groups) have distinct colours: then such a phase
// touches distinct LDS banks (hu_slot).  Where no colour is left, one with room is taken (a
// bank conflict, the result unchanged).  One wave per tile.
__global__ void __launch_bounds__(64) k_tile_union(SpLevels v, const int32_t *__restrict__ gcol,
                                                   uint32_t *__restrict__ ulist,
                                                   uint8_t *__restrict__ uslot, uint8_t *__restrict__ sflag,
                                                   int32_t *__restrict__ cnt) {
  constexpr int HT = 1024;                 // hash table of the tile's boxes (at most 416 distinct)
  __shared__ int32_t e[HU_NS];
  __shared__ int16_t first[HU_NS], slot[HU_NS];
  __shared__ int32_t hkey[HT], hmin[HT];
  __shared__ uint32_t colset[2][HU_B];     // per box: the colleague indices it appears at, per half of the groups
  __shared__ uint8_t row[HU_B], zrow[64];
  const int64_t ti = blockIdx.x;
  const int lane = threadIdx.x;
  const int l = sp_level(v, v.toff, ti);
  const int64_t g0 = v.goff[l] + (ti - v.toff[l]) * HM_TILE;
  const int ng = (int)min((int64_t)HM_TILE, v.goff[l + 1] - g0);
  if (lane < HU_SUB) sflag[HU_SUB * ti + lane] = 0;
  int nsub = 0;
  // the tile's groups from jlo on: as many as fit of 16, 8 or 4 at an aligned start
  for (int jlo = 0, len = HM_TILE; jlo < HM_TILE;) {
    const int jhi = jlo + len;
    const int64_t sub = HU_SUB * ti + nsub;
    __syncthreads();
    for (int i = lane; i < HT; i += 64) {
      hkey[i] = -1;
      hmin[i] = HU_NS;
    }
    for (int i = lane; i < HU_NS; i += 64) {
      const int j = i / HU_NK, kk = i % HU_NK;
      e[i] = j >= jlo && j < jhi && j < ng ? gcol[(g0 + j) * NCOLL + kk + (kk >= SELF_SLOT)] : -1;
    }
    __syncthreads();
    // each box's first entry (the smallest index naming it), by open addressing
    int hs[(HU_NS + 63) / 64];
    for (int n = 0, i = lane; i < HU_NS; i += 64, n++) {
      const int32_t x = e[i];
      hs[n] = -1;
      if (x < 0) continue;
      int h = (int)(((uint32_t)x * 2654435761u) >> 22) & (HT - 1);
      for (;;) {
        const int32_t old = atomicCAS(&hkey[h], -1, x);
        if (old == -1 || old == x) break;
        h = (h + 1) & (HT - 1);
      }
      atomicMin(&hmin[h], i);
      hs[n] = h;
    }
    __syncthreads();
    for (int n = 0, i = lane; i < HU_NS; i += 64, n++) first[i] = (int16_t)(hs[n] >= 0 ? hmin[hs[n]] : i);
    __syncthreads();
    int32_t count = 0;
    for (int base = 0; base < HU_NS; base += 64) {
      const int i = base + lane;
      const bool isfirst = i < HU_NS && e[i] >= 0 && first[i] == i;
      const uint64_t b = __ballot(isfirst);
      if (isfirst) slot[i] = (int16_t)(count + __popcll(b & ((1ull << lane) - 1)));
      count += __popcll(b);
    }
    if (len == HM_TILE && count == 0) return;
    if (count > HU_B) {
      len >>= 1;
      continue;
    }
    for (int u = lane; u < 2 * HU_B; u += 64) colset[u / HU_B][u % HU_B] = 0;
    __syncthreads();
    for (int i = lane; i < HU_NS; i += 64)
      if (e[i] >= 0) atomicOr(&colset[i / HU_NK >= HM_TILE / 2][slot[first[i]]], 1u << (i % HU_NK));
    __syncthreads();
    {   // greedy colouring, one box at a time, the state spread over the wave's lanes: lane
        // 32 h + kk holds the colours taken at colleague kk by half h, lane c < 16 the boxes
        // of colour c so far (the loop is wave-uniform)
      uint32_t cm = 0, nc = 0, avail = (1u << HU_NC) - 1;
      for (int u = 0; u < count; u++) {
        const uint32_t c0 = __builtin_amdgcn_readfirstlane(colset[0][u]);
        const uint32_t c1 = __builtin_amdgcn_readfirstlane(colset[1][u]);
        uint32_t forb = 0;
        for (uint32_t m = c0; m; m &= m - 1) forb |= __builtin_amdgcn_readlane(cm, __builtin_ctz(m));
        for (uint32_t m = c1; m; m &= m - 1) forb |= __builtin_amdgcn_readlane(cm, 32 + __builtin_ctz(m));
        const uint32_t free = avail & ~forb;
        const int pick = __builtin_ctz(free ? free : avail);
        const uint32_t n = __builtin_amdgcn_readlane(nc, pick);
        if (lane == 0) row[u] = (uint8_t)(pick + HU_NC * n);
        if (lane == pick) nc++;
        if (n + 1 == HU_CAP) avail &= ~(1u << pick);
        if (((lane < 32 ? c0 : c1) >> (lane & 31)) & 1) cm |= 1u << pick;
      }
      zrow[lane] = (uint8_t)(HU_ZROW + __builtin_ctz(~cm));   // a phase has at most 8 boxes of the 16 colours
    }
    __syncthreads();
    for (int u = lane; u < HU_B; u += 64)
      if (u >= count) ulist[sub * HU_B + u] = 0;
    for (int i = lane; i < HU_NS; i += 64) {
      const int32_t x = e[i];
      const int s = x >= 0 ? slot[first[i]] : 0;
      if (x >= 0 && first[i] == i)
        ulist[sub * HU_B + s] = (uint32_t)(x >> 11) << 10 | (uint32_t)((x & 15) != 0) << 8 |
                                (uint32_t)((x & 240) != 0) << 9 | row[s];
      uslot[sub * HU_NS + i] = x >= 0 ? row[s] : zrow[(i / HU_NK >= HM_TILE / 2 ? 32 : 0) + i % HU_NK];
    }
    if (lane == 0) {
      sflag[sub] = (uint8_t)(((1 << (len / 4)) - 1) << (jlo / 4));
      atomicAdd(&cnt[l], 1);
    }
    nsub++;
    jlo = jhi;
    len = min(len == 4 && (jlo & 7) ? 4 : HM_TILE / 2, HM_TILE - jlo);
  }
}
__global__ void k_store_counts(const int32_t *__restrict__ cnt, int n, int64_t *__restrict__ host) {
  const int i = threadIdx.x;
  if (i < n) host[i] = cnt[i];
}
__global__ void k_zero_i32(int32_t *__restrict__ a, int n) {
  if ((int)threadIdx.x < n) a[threadIdx.x] = 0;
}

// The table operands as the matrix instructions take them, from T[f][w] (f < 316):
//   mixed: A3[w][pair of colleagues][piece][lane]: 8 bfloat16, lane (q, i) row i, K = 8 q + ..:
//     colleague 2 pair + (q >> 1), children 4 (q & 1) + .., (re, im) each;
//   FP64:  A64[w][colleague][hf][lane]: lane (lk, i) row i, K slot lk: the factor of the
//     real part of child lk + 4 hf (that of its imaginary part is the neighbouring row's,
//     negated in the real rows).
// Row i = (target a = i / 2, part i % 2): the real part takes (T.re, -T.im), the imaginary
// part (T.im, T.re).
__global__ void k_had_fragments(const double2 *__restrict__ T, const int16_t *__restrict__ pairf,
                                __bf16 *__restrict__ A3, double *__restrict__ A64) {
  const int w = blockIdx.x;
  auto table = [&](int kk, int c, int i, int comp) -> double {
    const int k = kk + (kk >= SELF_SLOT), f = pairf[(k * NCHILD + c) * NCHILD + (i >> 1)];
    if (f < 0) return 0.0;
    const double2 x = T[(int64_t)f * SP_NF + w];
    return (i & 1) == comp ? x.x : (i & 1) ? x.y : -x.y;
  };
  for (int n = threadIdx.x; n < HU_NK / 2 * 64; n += blockDim.x) {
    const int pr = n / 64, lane = n % 64, i = lane & 15, q = lane >> 4;
    for (int z = 0; z < 8; z++) {
      double x = table(2 * pr + (q >> 1), 4 * (q & 1) + (z >> 1), i, z & 1);
      for (int pc = 0; pc < 3; pc++) {
        const __bf16 y = (__bf16)(float)x;
        x -= (double)(float)y;
        A3[((((int64_t)w * (HU_NK / 2) + pr) * 3 + pc) * 64 + lane) * 8 + z] = y;
      }
    }
  }
  for (int n = threadIdx.x; n < HU_NK * 2 * 64; n += blockDim.x) {
    const int kk = n / 128, hf = (n / 64) % 2, lane = n % 64;
    A64[(int64_t)w * HU_NK * 128 + n] = table(kk, (lane >> 4) + 4 * hf, lane & 15, 0);
  }
}

// The staging buffer of a frequency.
//   Mixed: piece-major, 32 bytes per row: children 0 .. 3 | 4 .. 7, (re, im) bfloat16 each; the
//   two 16-byte halves swapped by row bit 3.  8 lanes reading 16 bytes of one half at rows of
//   distinct colours (distinct modulo 16) touch distinct banks.
//   FP64: 128 bytes per row, child c at 16-byte place c ^ (row bits 1 .. 3).
// hu_slot: the byte offset of a row with its swizzle bits set; a reader XORs its own place in.
template <bool F64>
__device__ __forceinline__ uint32_t hu_slot(uint32_t row) {
  return F64 ? row * 128 + ((row >> 1) & 7) * 16 : row * 32 + ((row >> 3) & 1) * 16;
}
// the output buffer: one pad slot per 8 targets, so that a write phase touches distinct banks
constexpr int HU_OS = HM_TILE * NCHILD + HM_TILE;   // 144 slots per frequency
__device__ __forceinline__ int hu_opos(int ta, int f) { return f * HU_OS + ta + (ta >> 3); }

// A workgroup is LW loader waves and FB x H product waves (H parts of the colleagues); the
// loaders prefetch DEPTH subtiles into registers (NI half boxes a thread), convert and store
// one into the buffer that the product waves do not read, and write the previous one's
// results out: one barrier per subtile, memory and conversions beside the products.  Mixed:
// one frequency, three workgroups per CU (three frequencies in one workgroup, 6 + 6 waves:
// 9.0 against 8.5 ms at 4M sources; a single staging buffer with loads by all waves: 15.4).
template <bool F64> struct HadForm;
template <> struct HadForm<false> {
  using C = float2;
  using V = float4;                       // a staged load
  static constexpr int FB = 1, H = 2, LW = 2, NI = 3, DEPTH = 2, WPE = 3;
  static constexpr int NV = 2, RB = 32, PIECES = 3;   // loads per slice, bytes per row and piece
};
template <> struct HadForm<true> {
  using C = double2;
  using V = double2;
  static constexpr int FB = 1, H = 4, LW = 4, NI = 2, DEPTH = 2, WPE = 4;
  static constexpr int NV = 4, RB = 128, PIECES = 1;
};

// the neighbouring row's value (lanes 2 m and 2 m + 1 swap: quad_perm [1, 0, 3, 2])
__device__ __forceinline__ double swap_rows(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0xB1, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0xB1, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

struct HadArgs {
  const void *S, *A, *Z;     // spectra, table operands, FB rows of zeros at the spectra's stride
  void *U;
  const int32_t *subs;       // the level's subtiles
  const uint8_t *sflag;
  const uint32_t *ulist;
  const uint8_t *uslot;
  int64_t tile0, nsub, nl, nranges, nreal;
  int R;                     // subtiles per workgroup
};

template <bool F64>
__global__ void __launch_bounds__(64 * (HadForm<F64>::FB * HadForm<F64>::H + HadForm<F64>::LW), HadForm<F64>::WPE)
k_spec_hadamard(HadArgs a) {
  using F = HadForm<F64>;
  using C = typename F::C;
  using V = typename F::V;
  constexpr int FB = F::FB, H = F::H, LT = 64 * F::LW, PLANE = HU_NR * F::RB, BUF = FB * F::PIECES * PLANE;
  constexpr int NT = HM_TILE * NCHILD;                          // targets of a tile
  __shared__ __attribute__((aligned(16))) char Us[2 * BUF];
  __shared__ __attribute__((aligned(16))) C O[2][H][FB * HU_OS];   // the colleague parts' sums
  __shared__ uint32_t Sl[2][HU_NS / 2];                         // the subtile's slots, 16 bits each
  // XCD-aware order: an XCD sweeps all subtiles of its frequencies, whose rows it shares
  const int64_t Lb = xcd_block(blockIdx.x, gridDim.x);
  if (Lb >= a.nreal) return;   // a padding block
  const int f0 = (int)(Lb / a.nranges) * FB;
  const int64_t s0 = (Lb % a.nranges) * a.R;
  const int nm = (int)min((int64_t)a.R, a.nsub - s0);
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // the workgroup's subtiles and their parts, one per lane: no memory round trip per subtile
  const int my = a.subs[s0 + min(lane, nm - 1)], mypart = a.sflag[my];
  auto subtile = [&](int m) { return __builtin_amdgcn_readlane(my, m); };

  if (wave >= FB * H) {
    // ---- the loader waves: thread lt takes NI half boxes, children 4 hf .. 4 hf + 3 of box u[i]
    constexpr int D = F::DEPTH, E = 8, NI = F::NI;   // subtiles of spectra and of entries in registers
    static_assert(NI * LT >= 2 * HU_B && E % D == 0, "an item per half box");
    const int lt = t - 64 * FB * H, hf = lt & 1;
    uint32_t ent[E][NI], sw[D];
    V d[D][NI][FB][F::NV];
    // unconditional loads (of zeros where there is nothing to stage): no branch
    // between them, so that a wait for one subtile's leaves the later ones in flight
    auto entry = [&](int m, int i) -> uint32_t {
      return a.ulist[(int64_t)subtile(min(m, nm - 1)) * HU_B + min((lt + i * LT) >> 1, HU_B - 1)];
    };
    auto valid = [&](int m, int i, uint32_t e) -> uint32_t {   // at the use, not the load
      return m < nm && lt + i * LT < 2 * HU_B ? e : 0;
    };
    auto load = [&](uint32_t e, V x[FB][F::NV]) {
      // no child of this half has sources: zeros (FP64: node 0, zeroed by store; one block of
      // zeros read by every CU took twice the time there)
      const bool on = (e >> (8 + hf)) & 1;
      const C *q = on || F64 ? (const C *)a.S + sp_at((int64_t)(on ? e >> 10 : 0) * NCHILD + 4 * hf, f0) : (const C *)a.Z;
      const V *__restrict__ p = reinterpret_cast<const V *>(q);
#pragma unroll
      for (int y = 0; y < FB; y++)
#pragma unroll
        for (int n = 0; n < F::NV; n++)
          x[y][n] = p[(int64_t)min(y, SP_NF - 1 - f0) * (SP_CH * (int)sizeof(C) / (int)sizeof(V)) + n];
    };
    auto slots = [&](int m) -> uint32_t {
      return reinterpret_cast<const uint32_t *>(a.uslot + (int64_t)subtile(min(m, nm - 1)) * HU_NS)[min(lt, HU_NS / 4 - 1)];
    };
    auto store = [&](uint32_t e, const V x[FB][F::NV], char *buf) {
      if (e == 0) return;
      const uint32_t sl = hu_slot<F64>(e & 255);
#pragma unroll
      for (int y = 0; y < FB; y++) {
        if constexpr (F64) {
#pragma unroll
          for (int c = 0; c < 4; c++)
            *reinterpret_cast<double2 *>(buf + y * PLANE + (sl ^ ((4 * hf + c) * 16))) =
                (e >> (8 + hf)) & 1 ? x[y][c] : make_double2(0.0, 0.0);
        } else {
          // three bfloat16 pieces of each value: round, subtract (exact), round the rest
          const float w[8] = {x[y][0].x, x[y][0].y, x[y][0].z, x[y][0].w, x[y][1].x, x[y][1].y, x[y][1].z, x[y][1].w};
          uint32_t p0[4], p1[4], p2[4];
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const f32x2 v = {w[2 * c], w[2 * c + 1]};
            p0[c] = pack_bf16(v);
            const f32x2 r1 = v - unpack_bf16(p0[c]);
            p1[c] = pack_bf16(r1);
            p2[c] = pack_bf16(r1 - unpack_bf16(p1[c]));
          }
          char *o = buf + y * 3 * PLANE + (sl ^ (hf * 16));
          *reinterpret_cast<uint4 *>(o) = make_uint4(p0[0], p0[1], p0[2], p0[3]);
          *reinterpret_cast<uint4 *>(o + PLANE) = make_uint4(p1[0], p1[1], p1[2], p1[3]);
          *reinterpret_cast<uint4 *>(o + 2 * PLANE) = make_uint4(p2[0], p2[1], p2[2], p2[3]);
        }
      }
    };
    // stage subtile m (its spectra in slot k = m % D, its entry in ent[m % E])
    auto stage = [&](int m, const uint32_t e[NI], const V x[NI][FB][F::NV], uint32_t w) {
#pragma unroll
      for (int i = 0; i < NI; i++) store(valid(m, i, e[i]), x[i], Us + (m & 1) * BUF);
      static_assert(LT >= HU_NS / 4, "four slots per thread");
      if (lt < HU_NS / 4) {
        Sl[m & 1][2 * lt] = hu_slot<F64>(w & 255) | hu_slot<F64>((w >> 8) & 255) << 16;
        Sl[m & 1][2 * lt + 1] = hu_slot<F64>((w >> 16) & 255) | hu_slot<F64>(w >> 24) << 16;
      }
    };
    // a subtile's target rows, out of LDS: 1 KB of each frequency; thread lt the target
    // lt % 128 of frequency lt / 128
    static_assert(LT >= FB * NT, "one target value per thread");
    const int wx = lt / NT, wta = lt % NT;
    auto write_out = [&](int m) {
      const int64_t n0 = ((subtile(m) / HU_SUB) - a.tile0) * NT;
      const int part = __builtin_amdgcn_readlane(mypart, m);
      if (wx >= FB || f0 + wx >= SP_NF || n0 + wta >= a.nl || !((part >> (wta / (NT / 4))) & 1)) return;
      C v = O[m & 1][0][hu_opos(wta, wx)];
#pragma unroll
      for (int h = 1; h < H; h++) {
        const C y = O[m & 1][h][hu_opos(wta, wx)];
        v.x += y.x;
        v.y += y.y;
      }
      ((C *)a.U)[sp_at(n0 + wta, f0 + wx)] = v;
    };
    for (int i = lt; i < 2 * FB * F::PIECES * HU_NC * F::RB / 4; i += LT)   // the zero boxes of both buffers
      *reinterpret_cast<uint32_t *>(Us + (i / (HU_NC * F::RB / 4)) * PLANE + HU_ZROW * F::RB +
                                    (i % (HU_NC * F::RB / 4)) * 4) = 0;
#pragma unroll
    for (int m = 0; m < E; m++)
#pragma unroll
      for (int i = 0; i < NI; i++) ent[m][i] = entry(m, i);
#pragma unroll
    for (int m = 0; m < D; m++) {
#pragma unroll
      for (int i = 0; i < NI; i++) load(valid(m, i, ent[m][i]), d[m][i]);
      sw[m] = slots(m);
    }
    // subtile m is staged while the product waves work on m - 1; no branch around the loads
    // (the compiler would wait for them all at the next use)
    for (int m0 = 0; m0 < nm; m0 += E) {
#pragma unroll
      for (int k = 0; k < E; k++) {
        const int m = m0 + k;
        if (m >= nm) break;
        stage(m, ent[k], d[k % D], sw[k % D]);
#pragma unroll
        for (int i = 0; i < NI; i++) load(valid(m + D, i, ent[(k + D) % E][i]), d[k % D][i]);
        sw[k % D] = slots(m + D);
#pragma unroll
        for (int i = 0; i < NI; i++) ent[k][i] = entry(m + E, i);
        if (m >= 2) write_out(m - 2);
        lds_barrier();
      }
    }
    if (nm >= 2) write_out(nm - 2);
    lds_barrier();
    write_out(nm - 1);
    return;
  }

  // ---- the product waves: frequency f0 + f, part h of the colleagues
  //   (mixed: of the 13 pairs of colleagues; the first parts take one more where H does not divide)
  const int f = wave % FB, h = wave / FB;
  const int j = lane & 15, q = lane >> 4;
  const int64_t fw = min(f0 + f, SP_NF - 1);   // a wave past the last frequency repeats it, unwritten
  constexpr int NU = F64 ? HU_NK : HU_NK / 2, NA = (NU + H - 1) / H;
  const int a0 = h * (NU / H) + min(h, NU % H);
  const bool last = NU % H == 0 || h < NU % H;   // whether it has the NA-th
  bf16x8 A3[F64 ? 1 : NA][3];
  double A64[F64 ? NA : 1][2];
  if constexpr (F64) {
    const double *__restrict__ p = (const double *)a.A + (fw * HU_NK + a0) * 128 + lane;
#pragma unroll
    for (int m = 0; m < NA; m++)
#pragma unroll
      for (int s = 0; s < 2; s++) A64[m][s] = m < NA - 1 || last ? p[(m * 2 + s) * 64] : 0.0;
  } else {
    const bf16x8 *__restrict__ p = (const bf16x8 *)a.A + (fw * (HU_NK / 2) + a0) * 192 + lane;
#pragma unroll
    for (int m = 0; m < NA; m++)
#pragma unroll
      for (int s = 0; s < 3; s++) A3[m][s] = p[((m < NA - 1 || last ? m : 0) * 3 + s) * 64];
  }
  lds_barrier();               // subtile 0 is staged
  for (int s = 0; s < nm; s++) {
    const uint16_t *sl = reinterpret_cast<const uint16_t *>(Sl[s & 1]) + j * HU_NK + (F64 ? a0 : 2 * a0 + (q >> 1));
    C *o = O[s & 1][h];
    if constexpr (F64) {
      const char *Ub = Us + (s & 1) * BUF + f * PLANE;
      f64x4 c0 = f64x4{0, 0, 0, 0}, c1 = c0;
#pragma unroll
      for (int m = 0; m < NA; m++) {
        if (m == NA - 1 && !last) break;
        const uint32_t off = sl[m];
        const double2 x = *reinterpret_cast<const double2 *>(Ub + (off ^ (q * 16)));
        const double2 y = *reinterpret_cast<const double2 *>(Ub + (off ^ ((q + 4) * 16)));
        // the imaginary parts' products unsigned: the real rows subtract them at the end
        c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(A64[m][0], x.x, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(swap_rows(A64[m][0]), x.y, c1, 0, 0, 0);
        c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(A64[m][1], y.x, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(swap_rows(A64[m][1]), y.y, c1, 0, 0, 0);
      }
      // lane (lk, j) holds rows lk + 4 e: target (lk >> 1) + 2 e, part lk & 1
#pragma unroll
      for (int z = 0; z < 4; z++)
        reinterpret_cast<double *>(&o[hu_opos(j * NCHILD + (q >> 1) + 2 * z, f)])[q & 1] =
            q & 1 ? c0[z] + c1[z] : c0[z] - c1[z];
    } else {
      const char *Ub = Us + (s & 1) * BUF + f * 3 * PLANE;
      const uint32_t hx = (q & 1) * 16;
      f32x4 c0 = f32x4{0, 0, 0, 0}, c1 = c0, c2 = c0;
#pragma unroll
      for (int m = 0; m < NA; m++) {
        if (m == NA - 1 && !last) break;
        const char *p = Ub + (sl[2 * m] ^ hx);
        const bf16x8 b0 = *reinterpret_cast<const bf16x8 *>(p);
        const bf16x8 b1 = *reinterpret_cast<const bf16x8 *>(p + PLANE);
        const bf16x8 b2 = *reinterpret_cast<const bf16x8 *>(p + 2 * PLANE);
        c0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A3[m][0], b0, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A3[m][1], b0, c1, 0, 0, 0);
        c2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A3[m][2], b0, c2, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A3[m][0], b1, c1, 0, 0, 0);
        c2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A3[m][1], b1, c2, 0, 0, 0);
        c2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A3[m][0], b2, c2, 0, 0, 0);
      }
      // lane (q, j) holds rows 4 q .. 4 q + 3: targets 2 q and 2 q + 1, (re, im) each
      const f32x4 v = c0 + (c1 + c2);
      const int ta = j * NCHILD + 2 * q;
      o[hu_opos(ta, f)] = make_float2(v[0], v[1]);
      o[hu_opos(ta + 1, f)] = make_float2(v[2], v[3]);
    }
    lds_barrier();
  }
}

// host side -----------------------------------------------------------------
// T[f][w] on the 15^3 lattice from the given tables (numpy rfftn of the kernel on the 16^3
// lattice, [f][k3][k2][k1 <= 8]): the kernel's values at the differences -7 .. 7 by the
// inverse transform, then the length-15 transforms; and the matrix instructions' operands
void spectral_setup(OpCache &o, const double *tables) {
  if (o.p != SP_P) return;
  using cd = std::complex<double>;
  constexpr int M = 16, D = SP_N;
  auto root = [](int j, int n) { return std::polar(1.0, 2.0 * M_PI * (j % n) / n); };
  cd w16[M], w15[D];
  for (int j = 0; j < M; j++) w16[j] = root(j, M);
  for (int j = 0; j < D; j++) w15[j] = root(j, D);
  std::vector<double> T(2 * (size_t)NFAR * SP_NF);
  std::vector<cd> a(D * M * 9), b(D * D * 9), c(D * D * SP_K1), e(D * D * SP_K1);
  std::vector<double> g(D * D * D);
  for (int f = 0; f < NFAR; f++) {
    const cd *t = reinterpret_cast<const cd *>(tables) + (size_t)f * M * M * 9;
    auto at = [](int x) { return (x - (SP_P - 1) + M) % M; };   // place x <-> difference x - 7
    for (int x3 = 0; x3 < D; x3++)
      for (int i = 0; i < M * 9; i++) {
        cd s = 0;
        for (int k = 0; k < M; k++) s += t[k * M * 9 + i] * w16[(k * at(x3)) % M];
        a[x3 * M * 9 + i] = s;
      }
    for (int x3 = 0; x3 < D; x3++)
      for (int x2 = 0; x2 < D; x2++)
        for (int k1 = 0; k1 < 9; k1++) {
          cd s = 0;
          for (int k = 0; k < M; k++) s += a[(x3 * M + k) * 9 + k1] * w16[(k * at(x2)) % M];
          b[(x3 * D + x2) * 9 + k1] = s;
        }
    for (int i = 0; i < D * D; i++)
      for (int x1 = 0; x1 < D; x1++) {
        double s = 0;
        for (int k = 0; k < 9; k++) s += (k == 0 || k == 8 ? 1.0 : 2.0) * (b[i * 9 + k] * w16[(k * at(x1)) % M]).real();
        g[i * D + x1] = s / (M * M * M);
      }
    // forward, place x at difference x - 7: index (x - 7) mod 15
    auto ix = [](int x) { return (x - (SP_P - 1) + D) % D; };
    for (int i = 0; i < D * D; i++)
      for (int k1 = 0; k1 < SP_K1; k1++) {
        cd s = 0;
        for (int x = 0; x < D; x++) s += g[i * D + x] * std::conj(w15[(ix(x) * k1) % D]);
        c[i * SP_K1 + k1] = s;
      }
    for (int x3 = 0; x3 < D; x3++)
      for (int k2 = 0; k2 < D; k2++)
        for (int k1 = 0; k1 < SP_K1; k1++) {
          cd s = 0;
          for (int x = 0; x < D; x++) s += c[(x3 * D + x) * SP_K1 + k1] * std::conj(w15[(ix(x) * k2) % D]);
          e[(x3 * D + k2) * SP_K1 + k1] = s;
        }
    for (int k1 = 0; k1 < SP_K1; k1++)
      for (int k2 = 0; k2 < (k1 == 0 ? SP_P : D); k2++) {
        const int col = sp_col(k1, k2);
        for (int k3 = 0; k3 < (col == 0 ? SP_P : D); k3++) {
          cd s = 0;
          for (int x = 0; x < D; x++) s += e[(x * D + k2) * SP_K1 + k1] * std::conj(w15[(ix(x) * k3) % D]);
          T[2 * ((size_t)f * SP_NF + sp_freq(col, k3))] = s.real();
          T[2 * ((size_t)f * SP_NF + sp_freq(col, k3)) + 1] = s.imag();
        }
      }
  }
  hipStream_t s = o.ctx->stream;
  DBuf<double> dT;
  dT.upload(T.data(), T.size(), s);
  o.had_mixed.resize((size_t)SP_NF * (HU_NK / 2) * 3 * 64 * 8);
  o.had_f64.resize((size_t)SP_NF * HU_NK * 128);
  const std::vector<double> zero(SP_CH * HadForm<false>::FB, 0.0);
  o.had_zero.upload(zero.data(), zero.size(), s);
  k_had_fragments<<<SP_NF, 256, 0, s>>>((const double2 *)dT.p, o.pairf.p, reinterpret_cast<__bf16 *>(o.had_mixed.p),
                                        o.had_f64.p);
  FFMM_LAUNCH_CHECK();
  o.ctx->sync();
}

void spectral_workspace(Plan &plan) {
  int64_t nmax = 1;
  for (int l = 2; l < plan.L; l++) nmax = std::max(nmax, plan.nl[l]);
  const size_t n = (size_t)2 * SP_NF * ((nmax + SP_CH - 1) / SP_CH * SP_CH);
  if (plan.precision == FFMM_PREC_MIXED) {
    plan.spec_S32.resize(n);
    plan.spec_U32.resize(n);
  } else {
    plan.spec_S.resize(n);
    plan.spec_U.resize(n);
  }
}

// once per plan, all levels together: the groups' colleague tables, each tile's union, and
// the subtiles in order (one read back)
void spectral_prepare(Plan &plan) {
  OpCache &o = *plan.ops;
  if (o.p != SP_P) fail(FFMM_ERR_ARGUMENT, "the spectral M2L is built for p = 8");
  spectral_workspace(plan);
  Context &ctx = *plan.ctx;
  hipStream_t s = ctx.stream;
  const int L = plan.L;
  static_assert(MAX_KEY_LEVELS + 3 < NPINNED - 1, "a pinned slot per level");
  plan.spec_nsub.assign(L + 1, 0);
  plan.spec_sub0.assign(L + 1, 0);
  plan.spec_tile0.assign(L + 1, 0);
  if (L <= 2) return;
  SpLevels v{};
  v.L = L;
  for (int l = 2; l < L; l++) {
    const int64_t ng = plan.nl[l] / NCHILD;
    // k_group_cols keeps a box's place in the level in 23 bits (such a level's spectra alone
    // take 226 GB in the mixed form)
    if (plan.nl[l] > (1 << 23)) fail(FFMM_ERR_ARGUMENT, "too many boxes on one level for the spectral M2L");
    v.lo[l] = plan.lo[l];
    v.goff[l + 1] = v.goff[l] + ng;
    v.toff[l + 1] = plan.spec_tile0[l + 1] = v.toff[l] + (ng + HM_TILE - 1) / HM_TILE;
  }
  const int64_t ng = v.goff[L], nt = v.toff[L];
  if (nt == 0) return;
  DBuf<int32_t> gcol, cnt;
  gcol.resize((size_t)ng * NCOLL);
  cnt.resize(L);
  const int64_t ns = HU_SUB * nt;
  plan.spec_ulist.resize((size_t)ns * HU_B);
  plan.spec_uslot.resize((size_t)ns * HU_NS);
  plan.spec_flag.resize(ns);
  plan.spec_subs.resize(ns);
  arm_slots(ctx, 0, L + 1);
  k_zero_i32<<<1, 64, 0, s>>>(cnt.p, L);
  k_group_cols<<<nblocks(ng * NCOLL, 256), 256, 0, s>>>(v, plan.parent.p, plan.child_first.p, plan.col.p, plan.ghost.p,
                                                       plan.has_source.p, ng, plan.nnodes, gcol.p);
  FFMM_LAUNCH_CHECK();
  k_tile_union<<<(unsigned)nt, 64, 0, s>>>(v, gcol.p, reinterpret_cast<uint32_t *>(plan.spec_ulist.p), plan.spec_uslot.p,
                                          plan.spec_flag.p, cnt.p);
  FFMM_LAUNCH_CHECK();
  compact_flags_u8_async(ctx, plan.spec_flag.p, plan.spec_subs.p, ns, L);
  k_store_counts<<<1, 64, 0, s>>>(cnt.p, L, ctx.pinned_dev);
  FFMM_LAUNCH_CHECK();
  for (int l = 0; l < L; l++) {
    plan.spec_nsub[l] = read_slot(ctx, l);
    plan.spec_sub0[l + 1] = plan.spec_sub0[l] + plan.spec_nsub[l];
  }
  read_slot(ctx, L);   // the compaction's own count: its slot is free again
}

// The tiles of level l staged whole, and those cut into parts (a plan with spectral tiles).
bool spectral_tile_counts(const Plan &plan, int l, int64_t &staged, int64_t &cut) {
  staged = cut = 0;
  if (plan.m2l != FFMM_M2L_SPECTRAL || l + 1 >= (int)plan.spec_tile0.size() || plan.spec_nsub[l] == 0) return false;
  std::vector<uint8_t> fl((size_t)HU_SUB * (plan.spec_tile0[l + 1] - plan.spec_tile0[l]));
  FFMM_HIP(hipMemcpy(fl.data(), plan.spec_flag.p + HU_SUB * plan.spec_tile0[l], fl.size(), hipMemcpyDeviceToHost));
  for (size_t i = 0; i < fl.size(); i += HU_SUB) {
    staged += fl[i] == 15;
    cut += fl[i] != 0 && fl[i] != 15;
  }
  return true;
}

template <class T>
static void spectral_level(Plan &plan, int l, typename cplx_t<T>::type *S, typename cplx_t<T>::type *U, const void *A) {
  Context &ctx = *plan.ctx;
  OpCache &o = *plan.ops;
  hipStream_t s = ctx.stream;
  constexpr bool F64 = std::is_same<T, double>::value;
  constexpr int NB = SpBoxes<T>::NB, FB = HadForm<F64>::FB;
  const int64_t lo = plan.lo[l], nl = plan.nl[l];
  if (plan.lists[l].np == 0) return;
  k_spec_forward<T><<<(unsigned)(nl / NB), 64 * NB, 0, s>>>(plan.Mp.p, o.Ns, o.lat8.p, lo, nl, plan.has_source.p, S);
  FFMM_LAUNCH_CHECK();
  {
    StageTimer tm(plan, 8, l);   // the Hadamard launch alone
    HadArgs a{};
    a.S = S;
    a.A = A;
    a.Z = o.had_zero.p;
    a.U = U;
    a.subs = plan.spec_subs.p + plan.spec_sub0[l];
    a.sflag = plan.spec_flag.p;
    a.ulist = reinterpret_cast<const uint32_t *>(plan.spec_ulist.p);
    a.uslot = plan.spec_uslot.p;
    a.tile0 = plan.spec_tile0[l];
    a.nsub = plan.spec_nsub[l];
    a.nl = nl;
    // subtiles per workgroup: enough to hide the first loads, few enough for several
    // workgroups per CU in turn
    const int64_t nfb = (SP_NF + FB - 1) / FB;
    a.nranges = (a.nsub + HU_R - 1) / HU_R;
    while (a.nranges * nfb < 1024 && a.nranges * 8 < a.nsub) a.nranges++;
    a.R = (int)((a.nsub + a.nranges - 1) / a.nranges);
    a.nranges = (a.nsub + a.R - 1) / a.R;
    a.nreal = a.nranges * nfb;
    k_spec_hadamard<F64><<<(unsigned)pad_xcd(a.nreal), 64 * (FB * HadForm<F64>::H + HadForm<F64>::LW), 0, s>>>(a);
    FFMM_LAUNCH_CHECK();
  }
  const double alpha = (1.0 / plan.lam[l]) / (double)(SP_N * SP_N * SP_N);
  k_spec_inverse<T><<<(unsigned)(nl / NB), 64 * NB, 0, s>>>(U, plan.lists[l].ptr.p, o.lat8.p, nl, o.Ns, alpha,
                                                          plan.Pl.p + lo * o.Ns);
  FFMM_LAUNCH_CHECK();
}

void m2l_spectral_level(Plan &plan, int l) {
  OpCache &o = *plan.ops;
  if (plan.precision == FFMM_PREC_MIXED)
    spectral_level<float>(plan, l, (float2 *)plan.spec_S32.p, (float2 *)plan.spec_U32.p, o.had_mixed.p);
  else
    spectral_level<double>(plan, l, (double2 *)plan.spec_S.p, (double2 *)plan.spec_U.p, o.had_f64.p);
}

}  // namespace ffmm
