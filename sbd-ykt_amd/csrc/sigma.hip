// sigma = H c on the alpha x beta product basis (replaces mult, tpb/mult.h:376-632).
//
// In the separated phase order H splits into
//   sigma[ia,ib] = hii*c                                                   (diagonal)
//                + sum_{ja in S(ia)+D(ia)} va(ia,ja) c[ja,ib]             (alpha product)
//                + sum_{jb in S(ib)+D(ib)} vb(ib,jb) c[ia,jb]             (beta product)
//                + sum_{ja in S(ia)} sa [ sum_{k in occ(ib)} (ai|kk) c[ja,ib]
//                                        + sum_{jb in S(ib)} sb (ai|bj) c[ja,jb] ]
//                + sum_{jb in S(ib)} sb [ sum_{k in occ(ia)} (kk|bj) ] c[ia,jb]   (alpha-beta)
// where va, vb are the string-pair values of the excitation tables.  The alpha product
// streams whole rows c[ja,:] (coalesced, one wave per row tile, no atomics); the
// beta product is the same kernel on the transposed vector; the alpha-beta kernel owns
// a segment of one bra row per workgroup, stages the ket row c[ja,:] in LDS chunk by chunk together
// with the (ai|..) slice, and gathers from LDS.  Every output element has one owner.
#include <algorithm>
#include <type_traits>

#include "sbdg_internal.h"

namespace sbdg {

namespace {

template <class T>
struct V16;
template <>
struct V16<double> {
  typedef double u __attribute__((ext_vector_type(2), aligned(8)));  // at element alignment
  static constexpr int n = 2;
};
template <>
struct V16<float> {
  typedef float u __attribute__((ext_vector_type(4), aligned(4)));
  static constexpr int n = 4;
};

constexpr int TS = 256;  // threads of the row-streaming product
// Row products of up to this many elements split each row's list over four waves (k_spmm):
// norb=18, 239^2 strings 26 -> 9 us a product, norb=12, 495^2 19 -> 8; at norb=26, 1,400^2
// (beyond) the plain form fills the chip.
constexpr int64_t SPMM_KS_MAX = 1 << 20;
constexpr int SPMM_ROWS = 4;  // rows per workgroup, one wave each (beyond SPMM_KS_MAX)
constexpr int SPMM_US = 4, SPMM_UD = 4, SPMM_UZ = 8;  // singles, direct pairs, Z rows in flight
constexpr int SPMM_DB = 16;  // direct pairs summed on their own: a short chain of roundings, as a
// core's (norb=36, 3,600 x 3,500 strings in FP32: 3.2e-7 from the exact sigma in one chain, 1.8e-7 so)

// Column range [cb, ce) of one row product:
//   out[r, c] = (DIAG ? hii*X : 0)[r, c] + sum_q (val[q] + sgn_q J[p_q][c]) X[col[q], c]
//             + (ZG ? sum_{s in slots(r)} Z[slot[s], c - cb] : 0)
// jai[q] = +-(p_q) selects the row of the column strings' occupation table J that carries
// the other-spin occupation part of a single; the doubles (entries from mid[r] on) have none
// and are read without it.  Z holds the core-grouped doubles of the same column range
// (k_core_prod).  A work item is one row of one tile of 64 lanes and belongs to one wave, so the
// row's list is read through the scalar path; tiles are outer, rows inner.  Workgroups take
// SPMM_ROWS consecutive items, are dealt to the 8 XCDs in turn, and workgroup L takes items from
// (L % 8) * per + L / 8 (per = ceil(workgroups / 8)): each XCD walks a contiguous run of rows,
// whose strings share many excitation partners, so the rows of X they read meet in that XCD's
// L2.  Bound by the rate of those gathers (two 16-byte rows a lane and single, one a direct
// pair) and by Z, which comes from memory.  With every entry reading a row of J and FP64 rows
// of 512 columns over four waves a sigma at norb=36, 20,000^2 strings took 146.8 ms against 136.0
// (FP32 76.1 / 71.6; the pairs of more cores read directly, CORE_ZMIN: 132.5 and 69.7).  Lanes
// split into groups that take entries in turn over 8, 16 or 32 lanes' columns, so that a tile's
// whole piece of X stays in one L2, were slower (174.4, 159.5, 153.8).
//
// A lane's VN columns are one 16-byte load at the element's own alignment (rows of an odd
// length start anywhere); the lanes past the last whole vector take the row's last VN columns
// again, with the same sums as their neighbour, so no lane leaves the vector path (ncols >= VN;
// VECTOR is false below that, and a lane takes one column).
//
// KS: with few rows and columns the chain of gathers of one row is the time (a row's list,
// four entries per step, one memory latency each), so the four waves of a workgroup take one
// row's columns together, a quarter of its list each, and their sums are added in order.
template <class T, bool DIAG, bool VECTOR, bool ZG, bool KS>
__global__ void __launch_bounds__(TS) k_spmm(int64_t nrows, int64_t ncols, int64_t cb, int64_t ce,
                                             const int64_t* __restrict__ rowptr, const int64_t* __restrict__ mid,
                                             const int32_t* __restrict__ col, const T* __restrict__ val,
                                             const int32_t* __restrict__ jai, const T* __restrict__ J,
                                             const T* __restrict__ X, const T* __restrict__ hii, T* __restrict__ out,
                                             const int32_t* __restrict__ zptr, const int32_t* __restrict__ zslot,
                                             const T* __restrict__ Z, int64_t zcols) {
  constexpr int VN = V16<T>::n;
  constexpr int RW = KS ? 1 : SPMM_ROWS;
  using VT = typename V16<T>::u;
  const int64_t ntl = (ce - cb + 64 * VN - 1) / (64 * VN);
  const int64_t items = ntl * nrows;
  const int64_t per = ((items + RW - 1) / RW + 7) / 8;
  const int64_t bid = (int64_t)(blockIdx.x % 8) * per + blockIdx.x / 8;  // each XCD: a contiguous run of rows
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t item = KS ? bid : bid * RW + wave;
  if (item >= items) return;  // KS: the whole workgroup; otherwise there is no barrier
  const int64_t tile = item / nrows;
  const int64_t r = item - tile * nrows;
  int64_t c0 = cb + (tile * 64 + lane) * VN;
  const bool active = c0 < ce;
  if (VECTOR && !KS && !active) return;
  if (VECTOR) c0 = min(c0, ce - VN);
  T acc[VN];
#pragma unroll
  for (int k = 0; k < VN; ++k) acc[k] = T(0);
  int64_t q = rowptr[r], q1 = rowptr[r + 1], qm = mid[r];
  int32_t z = 0, z1 = 0;
  if (ZG) {
    z = zptr[r];
    z1 = zptr[r + 1];
  }
  if (KS) {
    const int64_t nq = (q1 - q + 3) / 4;
    q = min(q1, q + wave * nq);
    q1 = min(q1, q + nq);
    qm = max(q, min(q1, qm));
    const int32_t nz = (z1 - z + 3) / 4;
    z = min(z1, z + wave * nz);
    z1 = min(z1, z + nz);
  }
  if (VECTOR) {
    if (DIAG && (!KS || wave == 0)) {
      T hv[VN], xv[VN];
      *reinterpret_cast<VT*>(hv) = *reinterpret_cast<const VT*>(hii + r * ncols + c0);
      *reinterpret_cast<VT*>(xv) = *reinterpret_cast<const VT*>(X + r * ncols + c0);
#pragma unroll
      for (int k = 0; k < VN; ++k) acc[k] = hv[k] * xv[k];
    }
    // the entries [e, e + U) of a list, the last step's clamped into it and left out of the sum
    const T* Xc = X + c0;
    const T* Jc = J + c0;
    auto singles = [&](auto tail) {
      constexpr bool TAIL = decltype(tail)::value;
      constexpr int U = SPMM_US;
      T v[U], sg[U], x[U][VN], jv[U][VN];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t e = TAIL ? min(q + u, qm - 1) : q + u;
        const int32_t p = jai[e];
        v[u] = val[e];
        sg[u] = p < 0 ? T(-1) : T(1);
        *reinterpret_cast<VT*>(x[u]) = *reinterpret_cast<const VT*>(Xc + (int64_t)col[e] * ncols);
        *reinterpret_cast<VT*>(jv[u]) = *reinterpret_cast<const VT*>(Jc + (int64_t)(p < 0 ? -p : p) * ncols);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int k = 0; k < VN; ++k) {
          const T s = acc[k] + (v[u] + sg[u] * jv[u][k]) * x[u][k];
          acc[k] = !TAIL || q + u < qm ? s : acc[k];
        }
    };
    auto direct = [&](auto tail, T* sum) {
      constexpr bool TAIL = decltype(tail)::value;
      constexpr int U = SPMM_UD;
      T v[U], x[U][VN];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t e = TAIL ? min(q + u, q1 - 1) : q + u;
        v[u] = val[e];
        *reinterpret_cast<VT*>(x[u]) = *reinterpret_cast<const VT*>(Xc + (int64_t)col[e] * ncols);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int k = 0; k < VN; ++k) {
          const T s = sum[k] + v[u] * x[u][k];
          sum[k] = !TAIL || q + u < q1 ? s : sum[k];
        }
    };
    for (; q + SPMM_US <= qm; q += SPMM_US) singles(std::false_type{});
    if (q < qm) singles(std::true_type{});
    for (q = qm; q < q1;) {
      const int64_t qb = min(q1, q + SPMM_DB);
      T sum[VN];
#pragma unroll
      for (int k = 0; k < VN; ++k) sum[k] = T(0);
      for (; q + SPMM_UD <= qb; q += SPMM_UD) direct(std::false_type{}, sum);
      if (q < qb) {
        direct(std::true_type{}, sum);
        q = qb;
      }
#pragma unroll
      for (int k = 0; k < VN; ++k) acc[k] += sum[k];
    }
    if (ZG) {
      constexpr int U = SPMM_UZ;
      const T* Zc = Z + (c0 - cb);
      for (; z < z1; z += U) {
        T a[U][VN];
#pragma unroll
        for (int u = 0; u < U; ++u)
          *reinterpret_cast<VT*>(a[u]) = *reinterpret_cast<const VT*>(Zc + (int64_t)zslot[min(z + u, z1 - 1)] * zcols);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int k = 0; k < VN; ++k) acc[k] = z + u < z1 ? acc[k] + a[u][k] : acc[k];
      }
    }
    if constexpr (KS) {
      __shared__ T part[3][64][VN];
      if (wave > 0)
#pragma unroll
        for (int k = 0; k < VN; ++k) part[wave - 1][lane][k] = acc[k];
      __syncthreads();
      if (wave > 0 || !active) return;
#pragma unroll
      for (int w = 0; w < 3; ++w)
#pragma unroll
        for (int k = 0; k < VN; ++k) acc[k] += part[w][lane][k];
    }
    *reinterpret_cast<VT*>(out + r * ncols + c0) = *reinterpret_cast<VT*>(acc);
  } else {
    // fewer columns than a vector: a lane takes one column of every 64 / VN th entry, and the
    // lanes of a column are added in a fixed tree.  (A lane that walks the whole list for each
    // column is one chain of memory latencies: norb=20, 3 x 5,918 strings in FP32 543 us a sigma.)
    const int64_t c = min(cb + lane % VN, ce - 1);
    T a = T(0);
    for (int64_t e = q + lane / VN; e < q1; e += 64 / VN) {
      const int32_t p = jai[e];
      a += (val[e] + (p < 0 ? T(-1) : T(1)) * J[(int64_t)(p < 0 ? -p : p) * ncols + c]) * X[(int64_t)col[e] * ncols + c];
    }
    if (ZG)
      for (int32_t e = z + lane / VN; e < z1; e += 64 / VN) a += Z[(int64_t)zslot[e] * zcols + (c - cb)];
    for (int o = 32; o >= VN; o >>= 1) a += __shfl_xor(a, o, 64);
    if (DIAG) a += hii[r * ncols + c] * X[r * ncols + c];
    if (lane < ce - cb) out[r * ncols + c] = a;
  }
}

// Same-spin doubles grouped by core, column range [cb, ce):
//   Z[x, c - cb] = sum_{y in core(x)} eps_x eps_y W[P_x][P_y] X[row_y, c]
// for the members x of one product block (up to CORE_XB members of one core).  Members
// whose pairs overlap have W = 0 (they differ by a single excitation, or are equal), so
// every double pair of the string set is counted exactly once, in the core it shares.
// The block's signed coefficients and member rows are staged in LDS, CORE_YC members at a
// time (every lane reads the same entry: broadcast), and four member rows are loaded
// before they are used.  Each lane owns VN columns.  Bound by the member rows' misses in L2 and
// the Z writes: norb=36, 20,000^2 strings 16.2 ms a spin (FP32 8.3), norb=26, 4,000^2 0.41.  The
// same products on the matrix instructions, 64 members by 256 columns a workgroup, were no faster
// (16.8, 8.1 and 0.46 ms).
// Workgroups are dealt to the 8 XCDs in turn; workgroup L takes work item
// w = (L % 8) * per + L / 8 (per = ceil(items / 8)), so each XCD walks one contiguous range of
// items, and item w is column tile w / ngroups, block group w % ngroups: the blocks of one
// core are neighbours in that range and find the core's member rows in their XCD's L2.
constexpr int CORE_YC = 128;  // members staged per step
// Ranges of up to 128 vectors take 128 threads where there are this many groups of product
// blocks (four a CU): half of 256 threads would only wait at the barriers.  A sigma at norb=58,
// 200 x 40,000 strings 2.53 -> 2.40 ms, FP32 1.64 -> 1.39, norb=26, 100 x 12,000 0.51 -> 0.49.
// With fewer groups the staging of each block is the time, and more threads share it (norb=18,
// 239^2: 62 us with 256 threads, 67 with 128).
constexpr int64_t CORE_NARROW = 1024;

template <class T, bool VECTOR, int NT>
__global__ void __launch_bounds__(NT) k_core_prod(int64_t ncols, int64_t cb, int64_t ce,
                                                  const int32_t* __restrict__ start,
                                                  const int32_t* __restrict__ row,
                                                  const int32_t* __restrict__ pair,
                                                  const int32_t* __restrict__ blk,
                                                  const int32_t* __restrict__ blk_x0,
                                                  const int32_t* __restrict__ grp, int64_t ngroups,
                                                  const T* __restrict__ W, int64_t npair, const T* __restrict__ X,
                                                  T* __restrict__ Z, int64_t zcols) {
  constexpr int VN = V16<T>::n;
  constexpr int XB = CORE_XB;
  using VT = typename V16<T>::u;
  __shared__ __align__(16) T cf[CORE_YC][XB];  // signed coefficients of the staged members
  __shared__ int32_t rw[CORE_YC];              // their rows
  const int64_t ntiles = (ce - cb + NT * VN - 1) / (NT * VN);
  const int64_t ngrp = ngroups;
  const int64_t per = (ntiles * ngrp + 7) / 8;
  const int64_t w = (int64_t)(blockIdx.x % 8) * per + blockIdx.x / 8;
  if (w >= ntiles * ngrp) return;  // whole workgroup: no barrier is skipped by part of it
  const int64_t tile = w / ngrp;
  const int64_t g = w - tile * ngrp;
  int64_t c0 = cb + tile * (NT * VN) + (int64_t)threadIdx.x * VN;
  const bool active = c0 < ce;  // inactive lanes still take part in the barriers
  if (VECTOR) c0 = min(c0, ce - VN);  // the last columns again rather than a part of a vector
  constexpr bool full = VECTOR;
  const int64_t zc = c0 - cb;
  for (int b = grp[g]; b < grp[g + 1]; ++b) {
    const int core = blk[b];
    const int s0 = start[core];
    const int m = start[core + 1] - s0;
    const int x0 = blk_x0[b];
    const int nx = min(XB, m - x0);
    T acc[XB][VN];
#pragma unroll
    for (int xi = 0; xi < XB; ++xi)
#pragma unroll
      for (int k = 0; k < VN; ++k) acc[xi][k] = T(0);
    for (int y0 = 0; y0 < m; y0 += CORE_YC) {
      const int ny = min(CORE_YC, m - y0);
      __syncthreads();  // previous step done with the staged entries
      for (int e = threadIdx.x; e < ny * XB; e += NT) {
        const int yy = e / XB, xi = e - yy * XB;
        T v = T(0);
        if (xi < nx) {
          const int px = pair[s0 + x0 + xi], py = pair[s0 + y0 + yy];
          v = W[(int64_t)(px & 0x7FFFFFFF) * npair + (py & 0x7FFFFFFF)];
          if ((px < 0) != (py < 0)) v = -v;
        }
        cf[yy][xi] = v;
        if (xi == 0) rw[yy] = row[s0 + y0 + yy];
      }
      __syncthreads();
      if (active) {
        int yy = 0;
        for (; yy + 4 <= ny; yy += 4) {
          T xv[4][VN];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const T* x = X + (int64_t)rw[yy + u] * ncols + c0;
            if (full) {
              *reinterpret_cast<VT*>(xv[u]) = *reinterpret_cast<const VT*>(x);
            } else {
#pragma unroll
              for (int k = 0; k < VN; ++k) xv[u][k] = (c0 + k < ce) ? x[k] : T(0);
            }
          }
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int xi = 0; xi < XB; ++xi) {
              const T w = cf[yy + u][xi];
#pragma unroll
              for (int k = 0; k < VN; ++k) acc[xi][k] += w * xv[u][k];
            }
        }
        for (; yy < ny; ++yy) {
          T xv[VN];
          const T* x = X + (int64_t)rw[yy] * ncols + c0;
          if (full) {
            *reinterpret_cast<VT*>(xv) = *reinterpret_cast<const VT*>(x);
          } else {
#pragma unroll
            for (int k = 0; k < VN; ++k) xv[k] = (c0 + k < ce) ? x[k] : T(0);
          }
#pragma unroll
          for (int xi = 0; xi < XB; ++xi) {
            const T w = cf[yy][xi];
#pragma unroll
            for (int k = 0; k < VN; ++k) acc[xi][k] += w * xv[k];
          }
        }
      }
    }
    if (active) {
#pragma unroll
      for (int xi = 0; xi < XB; ++xi) {
        if (xi < nx) {
          T* z = Z + (int64_t)(s0 + x0 + xi) * zcols + zc;
          if (full) {
            *reinterpret_cast<VT*>(z) = *reinterpret_cast<VT*>(acc[xi]);
          } else {
#pragma unroll
            for (int k = 0; k < VN; ++k)
              if (c0 + k < ce) z[k] = acc[xi][k];
          }
        }
      }
    }
  }
}

constexpr int TT = 64;  // transpose tile

// out[c][r] = in[r][c] (ADD 1: out[c][r] += in[r][c]; 2: and add[c][r]).  Every load of a tile is
// issued, at an index held inside the matrix, before the first is used: loads under the edge
// conditions are waited for one by one (16 latencies per tile: 239^2 took 12 us).
template <class T, int ADD>
__global__ void __launch_bounds__(256) k_transpose(int64_t R, int64_t C, const T* __restrict__ in,
                                                   T* __restrict__ out, const T* __restrict__ add) {
  __shared__ T tile[TT][TT + 1];
  const int64_t r0 = (int64_t)blockIdx.y * TT, c0 = (int64_t)blockIdx.x * TT;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  T v[TT / 4], o[TT / 4], a[TT / 4];
#pragma unroll
  for (int u = 0; u < TT / 4; ++u) v[u] = in[min(r0 + ty + 4 * u, R - 1) * C + min(c0 + tx, C - 1)];
  if constexpr (ADD > 0) {
#pragma unroll
    for (int u = 0; u < TT / 4; ++u) {
      const int64_t x = min(c0 + ty + 4 * u, C - 1) * R + min(r0 + tx, R - 1);
      o[u] = out[x];
      a[u] = ADD == 2 ? add[x] : T(0);
    }
  }
#pragma unroll
  for (int u = 0; u < TT / 4; ++u) tile[ty + 4 * u][tx] = v[u];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < TT / 4; ++u) {
    const int64_t c = c0 + ty + 4 * u, r = r0 + tx;
    if (r < R && c < C) {
      if constexpr (ADD > 0) out[c * R + r] = o[u] + (tile[tx][ty + 4 * u] + a[u]);
      else out[c * R + r] = tile[tx][ty + 4 * u];
    }
  }
}

// alpha-beta terms.  The ket rows ja in S(ia) are taken G at a time (G = 2 in FP64, 4 in
// FP32: 16 bytes either way): the G (ai|..) slices and the G rows' current column chunk sit
// in LDS interleaved, so one 16-byte LDS read serves all G rows, and every ELL entry read
// from the L2-resident table serves them too.
template <class T>
struct AbRows {
  static constexpr int G = 16 / (int)sizeof(T);
  struct __align__(16) V {
    T v[G];
  };
  typedef T P2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
  // x with its sign flipped where bit 31 of sbit is set
  __device__ static inline T flip(T x, uint32_t sbit) {
    if constexpr (sizeof(T) == 8)
      return __longlong_as_double(__double_as_longlong(x) ^ ((unsigned long long)(sbit & 0x80000000u) << 32));
    else
      return __int_as_float(__float_as_int(x) ^ (int)(sbit & 0x80000000u));
  }
};

// The LDS vector at byte address a of the workgroup's LDS.  The alpha-beta kernel has no
// static LDS, so its dynamic LDS starts at address 0 (checked at launch) and entries carry
// absolute byte addresses.
typedef unsigned int lds_u32x4 __attribute__((ext_vector_type(4)));
template <class V>
__device__ inline V lds_at(uint32_t a) {
  static_assert(sizeof(V) == 16, "16-byte LDS vectors");
  const lds_u32x4 w = *reinterpret_cast<const __attribute__((address_space(3))) lds_u32x4*>(static_cast<size_t>(a));
  V r;
  __builtin_memcpy(&r, &w, 16);
  return r;
}

// One batch of stream rows of one lane: s[g] += sign_e * V[pair_e][g] * C[jb_e][g] for the G
// rows staged at byte offset off (all LDS reads issued before the products; one sum per row:
// a single chain of dependent FMAs was slower).
template <class T, int B>
__device__ inline void ab_batch(const uint32_t (&p)[B], uint32_t off, T (&s)[AbRows<T>::G]) {
  using R = AbRows<T>;
  using RV = typename R::V;
  constexpr int G = R::G;
  RV v[B], x[B];
#pragma unroll
  for (int u = 0; u < B; ++u) {
    v[u] = lds_at<RV>(((p[u] >> 14) & 0xFFF0u) + off);  // slice vector of pair (b, j)
    x[u] = lds_at<RV>((p[u] & 0x3FFFFu) + off);         // ket vector
  }
#pragma unroll
  for (int u = 0; u < B; ++u) {
#pragma unroll
    for (int g = 0; g < G; ++g) s[g] += R::flip(v[u].v[g], p[u]) * x[u].v[g];
  }
}

template <class T>
struct AbArgs {
  int64_t nb, ntiles, chunk, kbase, groups;
  int L, nch, nseg, assign;
  const int32_t* segrow;  // bra row of each segment
  const int64_t* segq;    // its alpha singles [segq[2s], segq[2s+1])
  const int32_t* segdst;  // -1: sigma's row; else the row of part
  const int32_t* colSa;
  const uint32_t* excSa;
  const int64_t* soff;
  const int32_t* nq;
  const uint32_t* ent;
  const int32_t* colperm;
  const T* Vt;  // (ai|bj) by orbital pairs a > i, b > j
  const T* c;
  T* sigma;
  T* part;
};

// Alpha-beta terms of one segment of a bra row's alpha singles over one column tile:
//   out[ib] += sum_{ja in segment} sa * sum_{entries (jb, b<-j) of ib} sb (ai|bj) c[ja, jb]
// (the other-spin occupation parts of the singles are in the row products).  Chunk by chunk of
// ket columns: S groups of G ket rows of the chunk (signed) and their slices sit in LDS as
// interleaved G-vectors, each lane walks its ELL entries for that chunk (the lane -> column
// map is per chunk, so lanes of a group carry lists of similar length), and the chunk's sums
// are added into the output row before the next chunk (through LDS in column order: scattered
// 8-byte read-modify-writes fetch and write back whole cache lines once the rows in flight
// outgrow the L2).  A wave's entries of a chunk are one stream, four rows per batch; the next
// batch is loaded while the current one is used, across group boundaries, and after the last
// batch the stream's first batch is loaded again for the next ket rows.
//
// Bound: the two 16-byte LDS gathers per entry (their bank conflicts above all); then the
// staging, which the products of the same workgroup wait for.  What the staging costs is the
// number of times a wave waits for memory in it, so no load of a round is under a condition
// and the wave-uniform tables are scalar loads: with each ket value loaded and waited for in
// its own exec region (as a condition on the row and the column compiles) k_ab<double> took
// 83.9 ms at norb=36, 20,000^2 strings (FP32 45.0) and staging alone 29.6 of them; issued
// together 69.5 (37.6), with two columns per load 68.1 (37.1), with the entries ordered over the
// lanes one LDS cycle serves 60.7 (33.9); norb=26, 2,801 x 2,749: 1.56 -> 0.80 ms.  Rows of few columns take S groups per barrier
// (239^2 at norb=18: 25 -> 21 us at S = 4).  Cutting rows into segments of their alpha
// singles (build_segments) took norb=18, 239^2 from 132 to 21 us and norb=58, 200 x 40,000
// from 6.7 to 0.78 ms: the Hartree-Fock row has ten times the singles of the average row.
// Measured and not kept: batches of two rows (the shorter padding is no gain: the
// padding reads one broadcast address), two batches in flight, two column tiles per row with
// two workgroups on a CU at norb=36, 20,000^2 (91.8 ms: the ket rows are staged twice).
template <class T, int M, int NT, int S>
__global__ void __launch_bounds__(NT, NT == 768 ? 3 : 4) k_ab(const AbArgs<T> A) {
  using R = AbRows<T>;
  using RV = typename R::V;
  constexpr int G = R::G;
  constexpr int B = AB_BATCH;
  // 16-byte vectors per thread per staging round: SR ket vectors (4*SR VGPRs beside the
  // accumulators) and SV slice vectors
  constexpr int SR = ab_ket_round((int)sizeof(T), M), SV = ab_slice_round(NT);
  extern __shared__ __align__(16) unsigned char smem[];
  const int64_t nb = A.nb, chunk = A.chunk, kbase = A.kbase;
  const int L = A.L;
  const int NP = L * (L - 1) / 2, NPS = max(NP, 1);  // slice vectors: pairs b > j (at least one)
  const int64_t npos = A.groups * 64;
  const int gvec = (int)(kbase + chunk + 1);  // LDS vectors of one staged group
  const int64_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int64_t tile = slot % A.ntiles;
  const int64_t seg = (slot / A.ntiles) * 8 + xcd;
  if (seg >= A.nseg) return;  // the grid rounds the segments up to a multiple of 8 (whole workgroup)
  const int64_t c0 = tile * (int64_t)NT * M, c1 = min(nb, c0 + (int64_t)NT * M);  // the tile's columns
  const int64_t ia = uniform_at(A.segrow, seg);
  const int64_t q0 = uniform_at(A.segq, 2 * seg), q1 = uniform_at(A.segq, 2 * seg + 1);
  const int dst = uniform_at(A.segdst, seg);
  T* out = dst < 0 ? A.sigma + ia * nb : A.part + (int64_t)dst * nb;
  const bool assign = dst >= 0 || A.assign;
  const int lane = threadIdx.x & 63;
  const int64_t s0 = (tile * (NT >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * A.nch;  // wave-uniform
  if (threadIdx.x < S) {
    RV* z = reinterpret_cast<RV*>(smem) + (int64_t)threadIdx.x * gvec + kbase + chunk;
    for (int g = 0; g < G; ++g) z->v[g] = T(0);
  }
  for (int k = 0; k < A.nch; ++k) {
    const int64_t j0 = (int64_t)k * chunk;
    const int nj = (int)(min(nb, j0 + chunk) - j0);
    // this wave's entry stream of chunk k: `rows` rows (a multiple of B); pn holds the
    // next batch, pf the row after it (wrapping to the start)
    const int64_t so = uniform_at(A.soff, s0 + k);
    const int rows = (int)((uniform_at(A.soff, s0 + k + 1) - so) >> 6);
    const uint32_t* sp = A.ent + so;  // wave-uniform; lanes add their index
    uint32_t pn[B];
    int pf = 0;
#pragma unroll
    for (int u = 0; u < B; ++u) pn[u] = (uint32_t)chunk;
    if (rows > 0) {
#pragma unroll
      for (int u = 0; u < B; ++u) pn[u] = sp[u * 64 + lane];
      pf = rows > B ? B : 0;
    }
    T acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = T(0);
    for (int64_t t = q0; t < q1; t += S * G) {
      __syncthreads();  // previous rows done with LDS (and the previous chunk's sums are stored)
      // The thread index is opaque here so that the addresses are formed per step rather
      // than held in registers through the products.
      int xt = (int)threadIdx.x;
      asm volatile("" : "+v"(xt));
#pragma unroll
      for (int sg = 0; sg < S; ++sg) {
        RV* Vv = reinterpret_cast<RV*>(smem) + sg * gvec;  // slice G-vectors of the pairs b > j
        RV* cbv = Vv + kbase;                               // ket G-vectors
        // rows t..t+G-1 of the group; rows at or past q1 are absent: their ket values are set
        // to zero (their slice is any finite one)
        uint32_t neg[G];
        const T* crow[G];
        const T* srow[G];
        bool has[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int64_t q = min(t + sg * G + g, q1 - 1);
          has[g] = t + sg * G + g < q1;
          const uint32_t e = uniform_at(A.excSa, q);
          neg[g] = ((e >> 24) & 1u) << 31;
          crow[g] = A.c + (int64_t)uniform_at(A.colSa, q) * nb + j0;
          srow[g] = A.Vt + (int64_t)ab_pair((e >> 6) & 63u, e & 63u) * NP;  // (ai|..)
        }
        // the G slices and the G rows' chunk (signed by the alpha single) into LDS: in rounds
        // of SR ket and SV slice vectors per thread.  Every global load of a round is issued,
        // at an index held inside the row, before its first use: a round costs one memory
        // latency (a load under a condition is waited for by itself).
        for (int x0 = 2 * xt, y0 = xt; x0 < nj || y0 < NPS; x0 += SR * NT, y0 += SV * NT) {
          RV sv[SV], kv[SR];
#pragma unroll
          for (int u = 0; u < SV; ++u) {
            const int y = min(y0 + u * NT, NPS - 1);
#pragma unroll
            for (int g = 0; g < G; ++g) sv[u].v[g] = srow[g][y];
          }
#pragma unroll
          for (int u = 0; u < SR; u += 2) {
            const int x = ab_stage_pair(x0 + u * NT, nj);
#pragma unroll
            for (int g = 0; g < G; ++g) {
              const typename R::P2 w = __builtin_nontemporal_load(reinterpret_cast<const typename R::P2*>(crow[g] + x));
              kv[u].v[g] = w.x;
              kv[u + 1].v[g] = w.y;
            }
          }
#pragma unroll
          for (int u = 0; u < SV; ++u) {
            const int y = y0 + u * NT;
            if (y < NPS) Vv[y] = sv[u];
          }
#pragma unroll
          for (int u = 0; u < SR; u += 2) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
              kv[u].v[g] = has[g] ? R::flip(kv[u].v[g], neg[g]) : T(0);
              kv[u + 1].v[g] = has[g] ? R::flip(kv[u + 1].v[g], neg[g]) : T(0);
            }
            const int xx = x0 + u * NT, x = ab_stage_pair(xx, nj);
            if (xx < nj) {
              cbv[x] = kv[u];
              cbv[x + 1] = kv[u + 1];
            }
          }
        }
      }
      __syncthreads();
      // the stream's batch counts, opaque to the compiler here: they are then reloaded for
      // every step instead of being held in M registers
      int qi = (int)((s0 + k) * M);
      asm volatile("" : "+s"(qi));
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int nbt = uniform_at(A.nq, qi + m);  // batches of this wave's m-th group
        T s[G];
#pragma unroll
        for (int g = 0; g < G; ++g) s[g] = T(0);
        for (int b = 0; b < nbt; ++b) {
          uint32_t p[B];
          const uint32_t* rp = sp + pf * 64;
#pragma unroll
          for (int u = 0; u < B; ++u) {
            p[u] = pn[u];
            pn[u] = rp[u * 64 + lane];
          }
          pf = pf + B == rows ? 0 : pf + B;
#pragma unroll
          for (int sg = 0; sg < S; ++sg) ab_batch<T, B>(p, (uint32_t)(sg * gvec) * 16u, s);
        }
        T a = acc[m];
#pragma unroll
        for (int g = 0; g < G; ++g) a += s[g];
        asm volatile("" : "+v"(a));  // formed here, so the group's partial sums die here
        acc[m] = a;
      }
    }
    // opaque again: the column map is read here, not before the products
    int ft = (int)threadIdx.x;
    asm volatile("" : "+v"(ft));
    const bool first = assign && k == 0;  // every column has a position in chunk 0
    // Each column of the tile sits at exactly one position of this chunk: the sums go through
    // LDS (the slices and ket vectors of the first group, idle now; the zero slot after them
    // stays untouched) one block of columns at a time, then into the output row with coalesced
    // read-modify-writes.  Each element is read and written by the same thread in every chunk.
    T* rowbuf = reinterpret_cast<T*>(smem);
    const int64_t cap = (kbase + chunk) * G;
    for (int64_t b0 = c0; b0 < c1; b0 += cap) {
      const int64_t b1 = min(c1, b0 + cap);
      __syncthreads();  // the products, or the previous block's readers, are done with LDS
      int fb = ft;  // opaque per block: the column map is read per block, not held in M registers
      asm volatile("" : "+v"(fb));
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int64_t pos = c0 + (int64_t)m * NT + fb;
        const int32_t ib = A.colperm[(int64_t)k * npos + pos];
        if (ib >= b0 && ib < b1) rowbuf[ib - b0] = acc[m];
      }
      __syncthreads();
      for (int64_t x = threadIdx.x; x < b1 - b0; x += NT) {
        if (first) out[b0 + x] = rowbuf[x];
        else out[b0 + x] += rowbuf[x];
      }
    }
  }
}

// out[row, :] += the partial rows of the row's further segments, in order.  Rows and column
// tiles are one grid dimension: the rows with partial rows are as many as the alpha strings, and
// a second dimension ends at 65,535.
template <class T>
__global__ void __launch_bounds__(256) k_ab_join(int64_t nb, unsigned ntiles, const int32_t* __restrict__ jrow,
                                                 const int32_t* __restrict__ jptr, const T* __restrict__ part,
                                                 T* __restrict__ out) {
  const unsigned j = blockIdx.x / ntiles;
  const int64_t c = (int64_t)(blockIdx.x - j * ntiles) * 256 + threadIdx.x;
  if (c >= nb) return;
  const int64_t r = jrow[j];
  T v = out[r * nb + c];
  for (int e = jptr[j]; e < jptr[j + 1]; ++e) v += part[(int64_t)e * nb + c];
  out[r * nb + c] = v;
}

template <class T>
void launch_spmm(bool diag, int64_t nrows, int64_t ncols, const SpmmTable& tb, const T* J, const T* X,
                 const T* hii, T* out, hipStream_t st, int64_t cb = 0, int64_t ce = -1,
                 const CoreTable* ct = nullptr, const T* Z = nullptr, int64_t zcols = 0) {
  if (ce < 0) ce = ncols;
  if (nrows == 0 || ce <= cb) return;
  constexpr int VN = V16<T>::n;
  const bool ks = nrows * (ce - cb) <= SPMM_KS_MAX && ce - cb >= VN;
  const int RW = ks ? 1 : SPMM_ROWS;
  const int64_t ntiles = (ce - cb + 64 * VN - 1) / (64 * VN);
  const int64_t nblk = ((ntiles * nrows + RW - 1) / RW + 7) / 8 * 8;
  if (nblk > (int64_t)INT32_MAX) throw Error(SBDG_ERR_LIMIT, "grid too large");
  const T* val = nullptr;
  if constexpr (sizeof(T) == 8) val = reinterpret_cast<const T*>(tb.val.p);
  else val = reinterpret_cast<const T*>(tb.val32.p);
  const bool vec = ce - cb >= VN;
  const int32_t* zp = ct ? ct->slot_ptr.p : nullptr;
  const int32_t* zs = ct ? ct->slot.p : nullptr;
  dim3 g((unsigned)nblk), b(TS);
#define SBDG_SPMM(D, V, ZG, KS)                                                                                   \
  hipLaunchKernelGGL((k_spmm<T, D, V, ZG, KS>), g, b, 0, st, nrows, ncols, cb, ce, tb.rowptr.p, tb.mid.p, \
                     tb.col.p, val, tb.jai.p, J, X, hii, out, zp, zs, Z, zcols)
#define SBDG_SPMM_V(D, ZG)                    \
  do {                                        \
    if (ks) SBDG_SPMM(D, true, ZG, true);     \
    else if (vec) SBDG_SPMM(D, true, ZG, false); \
    else SBDG_SPMM(D, false, ZG, false);      \
  } while (0)
  if (ct) {
    if (diag) SBDG_SPMM_V(true, true);
    else SBDG_SPMM_V(false, true);
  } else {
    if (diag) SBDG_SPMM_V(true, false);
    else SBDG_SPMM_V(false, false);
  }
#undef SBDG_SPMM_V
#undef SBDG_SPMM
}

// Z columns per pass over the range of one spin: a multiple of CORE_COLS that fits the
// workspace, at most the whole row length rounded up
template <class T>
int64_t core_zcols(const SigmaPlan& P, const CoreTable& ct, int64_t ncols) {
  const int64_t whole = (ncols + CORE_COLS - 1) / CORE_COLS * CORE_COLS;
  if (ct.zmem == 0) return whole;
  const int64_t fit = (int64_t)(P.zbytes / (sizeof(T) * (size_t)ct.zmem)) / CORE_COLS * CORE_COLS;
  if (fit < CORE_COLS) throw Error(SBDG_ERR_LIMIT, "core workspace too small");
  return std::min(fit, whole);
}

// products of one spin (rows of X are that spin's strings): singles + diagonal by the
// excitation table, doubles by core, one pass per column range of Z
template <class T>
void launch_spin(bool diag, int64_t nrows, int64_t ncols, const SpmmTable& tb, const T* J, const CoreTable* ct,
                 const T* W, int64_t npair, const T* X, const T* hii, T* out, T* Z, const SigmaPlan& P,
                 hipStream_t st) {
  if (!ct) {
    launch_spmm<T>(diag, nrows, ncols, tb, J, X, hii, out, st);
    return;
  }
  if (nrows == 0 || ncols == 0) return;
  constexpr int VN = V16<T>::n;
  const int64_t zcols = core_zcols<T>(P, *ct, ncols);
  for (int64_t cb = 0; cb < ncols; cb += zcols) {
    const int64_t ce = std::min(ncols, cb + zcols);
    if (ct->ngrp > 0) {
      auto prod = [&](auto vec, auto threads) {
        constexpr int NT = decltype(threads)::value;
        const int64_t ntiles = (ce - cb + NT * VN - 1) / (NT * VN);
        const int64_t items = ntiles * ct->ngrp;
        const int64_t nwg = (items + 7) / 8 * 8;
        if (nwg > (int64_t)INT32_MAX) throw Error(SBDG_ERR_LIMIT, "grid too large");
        hipLaunchKernelGGL((k_core_prod<T, decltype(vec)::value, NT>), dim3((unsigned)nwg), dim3(NT), 0, st, ncols, cb,
                           ce, ct->start.p, ct->row.p, ct->pair.p, ct->blk.p, ct->blk_x0.p, ct->grp.p, ct->ngrp, W,
                           npair, X, Z, zcols);
      };
      if (ce - cb < VN) prod(std::false_type{}, std::integral_constant<int, 64>{});
      else if (ce - cb <= 128 * VN && ct->ngrp >= CORE_NARROW) prod(std::true_type{}, std::integral_constant<int, 128>{});
      else prod(std::true_type{}, std::integral_constant<int, TS>{});
    }
    launch_spmm<T>(diag, nrows, ncols, tb, J, X, hii, out, st, cb, ce, ct, Z, zcols);
  }
}

template <class T, int ADD>
void launch_transpose(int64_t R, int64_t C, const T* in, T* out, hipStream_t st, const T* add = nullptr) {
  if (R == 0 || C == 0) return;
  dim3 g((unsigned)((C + TT - 1) / TT), (unsigned)((R + TT - 1) / TT));
  hipLaunchKernelGGL((k_transpose<T, ADD>), g, dim3(256), 0, st, R, C, in, out, add);
}

template <class T, int M, int NT, int S>
void launch_ab_m(const SigmaPlan& P, size_t lds, const T* eri, const T* c, T* sigma, hipStream_t st, int assign) {
  const EllTable& E = *P.ell;
  const AbSegments& G = *P.seg;
  const int64_t nblk = (G.nseg + 7) / 8 * 8 * E.ntiles;
  if (nblk > (int64_t)INT32_MAX) throw Error(SBDG_ERR_LIMIT, "grid too large");
  static const bool lds_at_zero = [] {  // entries hold absolute LDS byte addresses
    hipFuncAttributes fa;
    return hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(&k_ab<T, M, NT, S>)) == hipSuccess &&
           fa.sharedSizeBytes == 0;
  }();
  if (!lds_at_zero) throw Error(SBDG_ERR_STATE, "alpha-beta kernel has static LDS: entry addresses invalid");
  AbArgs<T> A;
  A.nb = P.nb;
  A.ntiles = E.ntiles;
  A.chunk = E.chunk;
  A.kbase = E.kbase;
  A.groups = E.groups;
  A.L = P.L;
  A.nch = E.nch;
  A.nseg = (int)G.nseg;
  A.assign = assign;
  A.segrow = G.row;
  A.segq = G.q;
  A.segdst = G.dst;
  A.colSa = P.sa->col.p;
  A.excSa = P.sa->exc.p;
  A.soff = E.soff;
  A.nq = E.nq;
  A.ent = E.ent;
  A.colperm = E.colperm;
  A.Vt = eri;
  A.c = c;
  A.sigma = sigma;
  A.part = reinterpret_cast<T*>(G.part.p);
  hipLaunchKernelGGL((k_ab<T, M, NT, S>), dim3((unsigned)nblk), dim3(NT), lds, st, A);
}

template <class T>
void launch_ab(const SigmaPlan& P, const T* eri, const T* c, T* sigma, hipStream_t st, int assign) {
  if (P.na == 0 || P.nb == 0) return;
  const EllTable& E = *P.ell;
  if ((int64_t)E.nt * E.m * E.ntiles != E.groups * 64) throw Error(SBDG_ERR_STATE, "alpha-beta table geometry");
  if (P.nb - (int64_t)(E.nch - 1) * E.chunk < 2) throw Error(SBDG_ERR_STATE, "alpha-beta chunk of less than two columns");
  const size_t lds = ab_lds_bytes(E.kbase, E.chunk) * E.s;
  bool done = false;  // the shapes ab_geometry picks
#define SBDG_AB(NT, M, S)                                        \
  if (!done && E.nt == NT && E.m == M && E.s == S) {             \
    launch_ab_m<T, M, NT, S>(P, lds, eri, c, sigma, st, assign); \
    done = true;                                                 \
  }
  SBDG_AB(64, 1, 2)
  SBDG_AB(64, 2, 2)
  SBDG_AB(128, 1, 2)
  SBDG_AB(256, 1, 1)
  SBDG_AB(256, 1, 4)
  SBDG_AB(256, 1, 2)
  SBDG_AB(256, 2, 4)
  SBDG_AB(256, 2, 2)
  SBDG_AB(256, 4, 2)
  SBDG_AB(256, 4, 1)
  SBDG_AB(512, 4, 1)
  SBDG_AB(512, 6, 1)
  SBDG_AB(512, 8, 1)
  SBDG_AB(512, 10, 1)
  SBDG_AB(512, 12, 1)
  SBDG_AB(1024, 8, 1)
  SBDG_AB(1024, 12, 1)
  SBDG_AB(1024, 16, 1)
  SBDG_AB(1024, 20, 1)
  SBDG_AB(1024, 24, 1)
  if constexpr (sizeof(T) == 8) {
    SBDG_AB(768, 40, 1)
    SBDG_AB(768, 48, 1)
    SBDG_AB(768, 53, 1)
  } else {
    SBDG_AB(1024, 40, 1)
    SBDG_AB(1024, 48, 1)
  }
#undef SBDG_AB
  if (!done) throw Error(SBDG_ERR_STATE, "alpha-beta columns per thread");
  const AbSegments& G = *P.seg;
  if (G.njoin > 0) {
    const int64_t tiles = (P.nb + 255) / 256, nblk = tiles * G.njoin;
    if (nblk > (int64_t)INT32_MAX) throw Error(SBDG_ERR_LIMIT, "grid too large");
    hipLaunchKernelGGL(k_ab_join<T>, dim3((unsigned)nblk), dim3(256), 0, st, P.nb, (unsigned)tiles, G.jrow, G.jptr,
                       reinterpret_cast<const T*>(G.part.p), sigma);
  }
}

}  // namespace

void transpose_d(int64_t R, int64_t C, const double* in, double* out, hipStream_t st) {
  launch_transpose<double, 0>(R, C, in, out, st);
  SBDG_CHECK(hipGetLastError());
}

size_t ab_lds_bytes(int64_t kbase, int64_t chunk) {
  return (size_t)16 * ((size_t)chunk + 1 + (size_t)kbase);  // 16-byte row vectors, any precision
}

template <class T>
void sigma_apply(const SigmaPlan& P, const T* c, T* sigma, const SigmaScratch<T>& scr, hipStream_t st,
                 hipEvent_t* ev) {
  T* cT = scr.cT;
  T* sT = scr.sT;
  const T* hii;
  const T* eri;
  if constexpr (sizeof(T) == 8) {
    hii = reinterpret_cast<const T*>(P.hii);
    eri = reinterpret_cast<const T*>(P.Vt);
  } else {
    hii = reinterpret_cast<const T*>(P.hii32);
    eri = reinterpret_cast<const T*>(P.Vt32);
  }
  if (ev) SBDG_CHECK(hipEventRecord(ev[0], st));
  // the alpha-beta terms (LDS-bound) into their own buffer on the second stream, while the
  // spin phases (HBM-bound) run on this one; the transpose-add joins them.  Below 100,000
  // determinants the fork and join cost more than the overlap gains (239^2 strings: 86 us
  // with it, 69 in sequence; 275^2: 95 and 89; 500 x 321: 125 and 152), unless rows are so wide
  // that both sides are long for a few determinants (2 x 13,922: 442 and 490; 4 x 20,000: 445 and
  // 557; 3 x 8,000: 188 and 176).
  T* sab = scr.sab;
  const bool ab = ab_any(P.nb), beside = P.st2 && ab && (P.na * P.nb >= 100000 || P.nb >= 10000);
  if (beside) {
    SBDG_CHECK(hipEventRecord(P.fork, st));
    SBDG_CHECK(hipStreamWaitEvent(P.st2, P.fork, 0));
    launch_ab<T>(P, eri, c, sab, P.st2, 1);
    SBDG_CHECK(hipEventRecord(P.join, P.st2));
  }
  launch_transpose<T, 0>(P.na, P.nb, c, cT, st);
  if (ev) SBDG_CHECK(hipEventRecord(ev[1], st));
  const T* W;
  if constexpr (sizeof(T) == 8) W = reinterpret_cast<const T*>(P.W);
  else W = reinterpret_cast<const T*>(P.W32);
  T* Z = reinterpret_cast<T*>(P.Z);
  const T *Ja, *Jb;
  if constexpr (sizeof(T) == 8) {
    Ja = reinterpret_cast<const T*>(P.Ja);
    Jb = reinterpret_cast<const T*>(P.Jb);
  } else {
    Ja = reinterpret_cast<const T*>(P.Ja32);
    Jb = reinterpret_cast<const T*>(P.Jb32);
  }
  launch_spin<T>(false, P.nb, P.na, *P.mb, Ja, P.cb, W, P.npair, cT, nullptr, sT, Z, P, st);
  if (ev) SBDG_CHECK(hipEventRecord(ev[2], st));
  launch_spin<T>(true, P.na, P.nb, *P.ma, Jb, P.ca, W, P.npair, c, hii, sigma, Z, P, st);
  if (ev) SBDG_CHECK(hipEventRecord(ev[3], st));
  if (beside) {
    SBDG_CHECK(hipStreamWaitEvent(st, P.join, 0));
    if (ev) SBDG_CHECK(hipEventRecord(ev[4], st));
    launch_transpose<T, 2>(P.nb, P.na, sT, sigma, st, sab);
    if (ev) SBDG_CHECK(hipEventRecord(ev[5], st));
  } else {
    launch_transpose<T, 1>(P.nb, P.na, sT, sigma, st);
    if (ev) SBDG_CHECK(hipEventRecord(ev[4], st));
    if (ab) launch_ab<T>(P, eri, c, sigma, st, 0);
    if (ev) SBDG_CHECK(hipEventRecord(ev[5], st));
  }
  SBDG_CHECK(hipGetLastError());
}

template void sigma_apply<double>(const SigmaPlan&, const double*, double*, const SigmaScratch<double>&,
                                  hipStream_t, hipEvent_t*);
template void sigma_apply<float>(const SigmaPlan&, const float*, float*, const SigmaScratch<float>&, hipStream_t,
                                 hipEvent_t*);

}  // namespace sbdg
