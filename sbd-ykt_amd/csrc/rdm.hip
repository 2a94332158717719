// 1- and 2-particle RDMs of a real vector (replaces Correlation, tpb/correlation.h:194-444,
// and feeds the Hellmann-Feynman backward).
//
// Output layout is the reference's: one[s][p + L q] = <c+_{p s} c_{q s}>,
// two[s + 2t][i + L j + L^2 k + L^3 l] = <c+_{i s} c+_{j t} c_{l t} c_{k s}>.
// Mixed-spin blocks are the physical ones.
//
// Work is organised by which string pairs connect bra and ket (separated phase order,
// W real, tables symmetric so both orders of every pair are visited):
//  * alpha pairs (ia,ja), beta fixed: g = sum_ib W[ia,ib] W[ja,ib]; singles also need the
//    beta-occupation-resolved sums gb[k] = sum_ib W[ia,ib] W[ja,ib] n_k(ib), summed over the
//    pairs of one key (a,i).  Beta pairs are the same on the transposed vector.
//  * alpha-beta pairs: T_(a,i)[b,j] = sum sa sb W[ia,ib] W[ja,jb] over alpha singles with
//    orbitals (a<-i) and beta singles (b<-j); one workgroup per segment of the alpha pairs of
//    one key (a,i) and tile of beta pairs, both rows staged in LDS, sums in registers.
//  * the diagonal: density correlators sum_D W_D^2 n_p n_q.
// Every RDM slot is written by exactly one owner (singles by their key (a,i), doubles by
// their orbital quadruple, alpha-beta by (a,i), the diagonal by (p,q)): no global atomics.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <utility>
#include <vector>

#include "sbdg_internal.h"

namespace sbdg {

void transpose_d(int64_t R, int64_t C, const double* in, double* out, hipStream_t st);

namespace {

constexpr int RT = 256;

// first entry of [q0, q1) (partners in ascending order) whose partner lies above r
__device__ inline int64_t first_above(int64_t q0, int64_t q1, const int32_t* __restrict__ col, int64_t r) {
  while (q0 < q1) {
    const int64_t mid = (q0 + q1) >> 1;
    if ((int64_t)col[mid] <= r) q0 = mid + 1;
    else q1 = mid;
  }
  return q0;
}

// The row-pair sums are symmetric in the two rows, and every pair (r, c) of an excitation table has its mirror (c, r), so the
// Gram kernels form only the pairs with c > r; this copies them to the pairs with c < r
// (the same products in the same order: the same bits).
__global__ void k_gram_mirror(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                              double* __restrict__ g) {
  const int64_t r = blockIdx.x;
  const int64_t q1 = first_above(rowptr[r], rowptr[r + 1], col, r);
  for (int64_t q = rowptr[r] + threadIdx.x; q < q1; q += blockDim.x) {
    const int64_t c = col[q];
    const int64_t m = first_above(rowptr[c], rowptr[c + 1], col, r - 1);  // the entry of r in row c
    g[q] = g[m];
  }
}

// entry of partner c in row r of an excitation table (partners ascending); -1 if absent
__device__ inline int64_t find_entry(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                     int64_t r, int64_t c) {
  const int64_t e = first_above(rowptr[r], rowptr[r + 1], col, c - 1);
  return e < rowptr[r + 1] && col[e] == c ? e : -1;
}

// Gram products of the members of one large core of the same-spin doubles (members
// x = core + {A, B}, as sigma groups them): every member row pairs with every other, so a
// workgroup takes a block pair (bi, bj) of one core's members, 16*NB rows each, on the matrix
// cores: G[i][j] += sum_c X[i][c] X[j][c].  Each wave takes 16 columns of every 64: a lane loads
// four neighbouring elements of row l % 16 at column 4 (l / 16), one operand of four products
// (both operands take their columns in the same order), and the four waves' tiles are added in
// order through LDS.  A member pair whose strings differ in four orbitals is a double pair, and
// that pair shares no other core: its sum goes to both entries of the excitation table, (x, y)
// and (y, x), and marks them done.  Rows past the end repeat the last one and are not used.
// Bound: the member rows from L2.  Against a tile of products per thread with both operands read
// from LDS: norb=16 full space (560 cores of 78) 3.6 -> 0.77 ms a spin, norb=36, 4,000 x 20,000
// strings 10.2 -> 1.7.
template <int NB>
__global__ void __launch_bounds__(RT, 4) k_core_gram(int64_t ncols, const int4* __restrict__ items,
                                                     const int32_t* __restrict__ cstart,
                                                     const int32_t* __restrict__ crow,
                                                     const uint64_t* __restrict__ str,
                                                     const int64_t* __restrict__ rowptr,
                                                     const int32_t* __restrict__ col, const double* __restrict__ X,
                                                     double* __restrict__ g, unsigned char* __restrict__ done) {
  typedef double quad __attribute__((ext_vector_type(4), aligned(8)));
  constexpr int BM = 16 * NB;
  __shared__ double sums[RT / 64][NB * NB][256];
  const int4 it = items[blockIdx.x];  // core, block bi, block bj
  const int32_t s0 = cstart[it.x], m = cstart[it.x + 1] - s0;
  const int i0 = it.y * BM, j0 = it.z * BM;
  const bool same = it.y == it.z;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double* ra[NB];
  const double* rb[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    ra[t] = X + (int64_t)crow[s0 + min(i0 + 16 * t + lane % 16, m - 1)] * ncols;
    rb[t] = X + (int64_t)crow[s0 + min(j0 + 16 * t + lane % 16, m - 1)] * ncols;
  }
  Mfma64::acc acc[NB][NB];
#pragma unroll
  for (int u = 0; u < NB; ++u)
#pragma unroll
    for (int v = 0; v < NB; ++v)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[u][v][q] = 0.0;
  auto products = [&](const quad (&a)[NB], const quad (&b)[NB]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int u = 0; u < NB; ++u)
#pragma unroll
        for (int v = 0; v < NB; ++v)
          if (!(same && v < u))  // below the diagonal of a diagonal block
            acc[u][v] = Mfma64::mad(a[u][q], b[v][q], acc[u][v]);
  };
  const int64_t full = ncols / 16 * 16;
  for (int64_t c = 16 * wave; c < full; c += 64) {
    quad a[NB], b[NB];
    const int64_t x = c + 4 * (lane / 16);
#pragma unroll
    for (int t = 0; t < NB; ++t) a[t] = *reinterpret_cast<const quad*>(ra[t] + x);
    if (same) {
#pragma unroll
      for (int t = 0; t < NB; ++t) b[t] = a[t];
    } else {
#pragma unroll
      for (int t = 0; t < NB; ++t) b[t] = *reinterpret_cast<const quad*>(rb[t] + x);
    }
    products(a, b);
  }
  if (full < ncols && wave == RT / 64 - 1) {  // the last columns, zeros past the row
    quad a[NB], b[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t x = full + 4 * (lane / 16) + q;
        a[t][q] = x < ncols ? ra[t][min(x, ncols - 1)] : 0.0;
        b[t][q] = x < ncols ? rb[t][min(x, ncols - 1)] : 0.0;
      }
    products(a, b);
  }
#pragma unroll
  for (int u = 0; u < NB; ++u)
#pragma unroll
    for (int v = 0; v < NB; ++v)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        sums[wave][u * NB + v][Mfma64::row(q, lane) * 16 + lane % 16] = acc[u][v][q];
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NB * NB; ++t) {
    const int i = i0 + 16 * (t / NB) + threadIdx.x / 16, j = j0 + 16 * (t % NB) + threadIdx.x % 16;
    if (i >= m || j >= m || i >= j) continue;
    const int64_t ri = crow[s0 + i], rj = crow[s0 + j];
    if (__popcll(str[ri] ^ str[rj]) != 4) continue;  // pairs sharing an orbital: a single
    const int64_t q1 = find_entry(rowptr, col, ri, rj), q2 = find_entry(rowptr, col, rj, ri);
    if (q1 < 0 || q2 < 0) continue;
    double v = 0.0;
    for (int w = 0; w < RT / 64; ++w) v += sums[w][t][threadIdx.x];
    g[q1] = v;
    g[q2] = v;
    done[q1] = 1;
    done[q2] = 1;
  }
}

// the entries above the diagonal that no core product formed, as a list per row
__global__ void k_pair_flags(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                             const unsigned char* __restrict__ done, int32_t* __restrict__ flag) {
  const int64_t r = blockIdx.x;
  for (int64_t q = rowptr[r] + threadIdx.x; q < rowptr[r + 1]; q += blockDim.x)
    flag[q] = (col[q] > r && !done[q]) ? 1 : 0;
}
__global__ void k_pair_list(int64_t nnz, const int32_t* __restrict__ flag, const int32_t* __restrict__ pos,
                            int32_t* __restrict__ qlist) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < nnz && flag[q]) qlist[pos[q]] = (int32_t)q;
}
__global__ void k_pair_lptr(int64_t n, int64_t nnz, const int64_t* __restrict__ rowptr,
                            const int32_t* __restrict__ flag, const int32_t* __restrict__ pos,
                            int64_t* __restrict__ lptr) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r > n) return;
  const int64_t q = rowptr[r];
  lptr[r] = q < nnz ? pos[q] : (nnz ? (int64_t)pos[nnz - 1] + flag[nnz - 1] : 0);
}

// g[q] = <X[r,:], X[col[q],:]> for the pairs q = qlist[e], e in [lptr[r], lptr[r+1]), of
// row r, GQ pairs per pass: row r is read once per pass for all of them and their sums are
// reduced together (one barrier pair per pass instead of per pair).  Each sum's order is fixed (a thread's columns in order, then
// a shuffle tree, then the waves in order), so g does not depend on timing.  VEC: rows of
// an even length, read two columns at a time.
constexpr int GQ = 8;
template <bool VEC>
__global__ void __launch_bounds__(RT) k_gram_pairs(int64_t ncols, const int64_t* __restrict__ lptr,
                                                   const int32_t* __restrict__ qlist,
                                                   const int32_t* __restrict__ col, const double* __restrict__ X,
                                                   double* __restrict__ g) {
  __shared__ double sh[RT / 64][GQ];
  const int64_t r = blockIdx.x;
  const double* xr = X + r * ncols;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t q1 = lptr[r + 1];
  for (int64_t q0 = lptr[r]; q0 < q1; q0 += GQ) {
    const int nq = (int)min<int64_t>(GQ, q1 - q0);
    const double* xq[GQ];
    double s[GQ];
#pragma unroll
    for (int u = 0; u < GQ; ++u) {
      xq[u] = X + (int64_t)col[qlist[q0 + min(u, nq - 1)]] * ncols;
      s[u] = 0.0;
    }
    if (VEC) {
      for (int64_t cc = 2 * (int64_t)threadIdx.x; cc < ncols; cc += 2 * RT) {
        const double2 x = *reinterpret_cast<const double2*>(xr + cc);
#pragma unroll
        for (int u = 0; u < GQ; ++u)
          if (u < nq) {
            const double2 y = *reinterpret_cast<const double2*>(xq[u] + cc);
            s[u] += x.x * y.x;
            s[u] += x.y * y.y;
          }
      }
    } else {
      for (int64_t cc = threadIdx.x; cc < ncols; cc += RT) {
        const double x = xr[cc];
#pragma unroll
        for (int u = 0; u < GQ; ++u)
          if (u < nq) s[u] += x * xq[u][cc];
      }
    }
#pragma unroll
    for (int u = 0; u < GQ; ++u)
      for (int o = 32; o > 0; o >>= 1) s[u] += __shfl_xor(s[u], o, 64);
    __syncthreads();  // the previous pass's readers of sh are done
    if (lane == 0)
#pragma unroll
      for (int u = 0; u < GQ; ++u) sh[wid][u] = s[u];
    __syncthreads();
    if ((int)threadIdx.x < nq) {
      double t = 0.0;
      for (int w = 0; w < RT / 64; ++w) t += sh[w][threadIdx.x];
      g[qlist[q0 + threadIdx.x]] = t;
    }
  }
}

// Singles of one spin, by key: with the pairs (r, c) of key (a, i) in order, signs s,
//   D[cc] = sum_q s_q X[r_q,cc] X[c_q,cc]   (gocc of the key is sum_cc D[cc] n_k(cc))
//   g_q = <X[r_q,:], X[c_q,:]>
// One workgroup per segment of a key's pairs and tile of columns; a thread keeps its columns'
// D in registers over the segment, each wave adds its part of every g_q once.  The occupation
// sums then need one pass over D per segment (k_occ_contract) instead of one addition per pair,
// column and orbital that differs: those were fixed-point LDS atomics, 16 ms a spin at norb=36,
// 4,000 x 20,000 strings (this form 2) and 7.4 at norb=16 full space (0.7).  Bound: the two
// rows of every pair, from L2.  A key (i, a) holds the pairs of (a, i) read the other way, with
// the same sums, so only a > i is formed.
constexpr int PSU = 4;           // vectors of NV columns per thread
constexpr int PSEG = 256;        // pairs of one segment at most
template <int NV>
__global__ void __launch_bounds__(RT) k_pair_sums(int64_t ncols, int64_t ntiles, int64_t nseg,
                                                  const int32_t* __restrict__ segs, const int32_t* __restrict__ pia,
                                                  const int32_t* __restrict__ pja, int64_t npair,
                                                  const double* __restrict__ X, double* __restrict__ D,
                                                  double* __restrict__ gpart) {
  typedef double vec __attribute__((ext_vector_type(NV), aligned(8)));
  __shared__ double gs[RT / 64][PSEG];
  const int64_t tl = blockIdx.x % ntiles, sg = blockIdx.x / ntiles;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int e0 = segs[2 * sg], e1 = segs[2 * sg + 1];
  int64_t at[PSU];
  bool in[PSU];
  double d[PSU][NV];
#pragma unroll
  for (int u = 0; u < PSU; ++u) {
    const int64_t c = (tl * PSU + u) * (int64_t)(RT * NV) + (int64_t)threadIdx.x * NV;
    at[u] = min(c, ncols - NV);  // NV == 2: the last column of an odd row is taken with its neighbour
    in[u] = c < ncols;
#pragma unroll
    for (int k = 0; k < NV; ++k) d[u][k] = 0.0;
  }
  // columns that a clamped vector repeats count once in g
  auto own = [&](int u, int k) { return in[u] && (tl * PSU + u) * (int64_t)(RT * NV) + (int64_t)threadIdx.x * NV <= at[u] + k; };
  double m[PSU][NV];
#pragma unroll
  for (int u = 0; u < PSU; ++u)
#pragma unroll
    for (int k = 0; k < NV; ++k) m[u][k] = own(u, k) ? 1.0 : 0.0;
  for (int e = e0; e < e1; e += 2) {
    const int f = min(e + 1, e1 - 1);
    const int32_t j0 = pja[e], j1 = pja[f];
    const double* r0 = X + (int64_t)pia[e] * ncols;
    const double* r1 = X + (int64_t)pia[f] * ncols;
    const double* q0 = X + (int64_t)(j0 & 0x7FFFFFFF) * ncols;
    const double* q1 = X + (int64_t)(j1 & 0x7FFFFFFF) * ncols;
    vec a0[PSU], b0[PSU], a1[PSU], b1[PSU];
#pragma unroll
    for (int u = 0; u < PSU; ++u) {
      a0[u] = *reinterpret_cast<const vec*>(r0 + at[u]);
      b0[u] = *reinterpret_cast<const vec*>(q0 + at[u]);
      a1[u] = *reinterpret_cast<const vec*>(r1 + at[u]);
      b1[u] = *reinterpret_cast<const vec*>(q1 + at[u]);
    }
    const double s0 = j0 < 0 ? -1.0 : 1.0, s1 = f == e ? 0.0 : (j1 < 0 ? -1.0 : 1.0);
    double g0 = 0.0, g1 = 0.0;
#pragma unroll
    for (int u = 0; u < PSU; ++u)
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const double p0 = a0[u][k] * b0[u][k], p1 = a1[u][k] * b1[u][k];
        d[u][k] += s0 * p0;
        if (f != e) d[u][k] += s1 * p1;
        g0 += m[u][k] != 0.0 ? p0 : 0.0;
        g1 += m[u][k] != 0.0 ? p1 : 0.0;
      }
    for (int o = 32; o > 0; o >>= 1) {
      g0 += __shfl_xor(g0, o, 64);
      g1 += __shfl_xor(g1, o, 64);
    }
    if (lane == 0) {
      gs[wid][e - e0] = g0;
      gs[wid][f - e0] = f == e ? g0 : g1;
    }
  }
#pragma unroll
  for (int u = 0; u < PSU; ++u)
    if (in[u]) {
#pragma unroll
      for (int k = 0; k < NV; ++k) D[sg * ncols + at[u] + k] = d[u][k];
    }
  __syncthreads();
  for (int x = threadIdx.x; x < e1 - e0; x += RT) {
    double v = 0.0;
    for (int w = 0; w < RT / 64; ++w) v += gs[w][x];
    gpart[tl * npair + e0 + x] = v;
  }
}

// occ[r*64 + k] = sum_c v_c n_k(cstr[c]) over the columns of row r, v = src[r*ncols + c] (SQ:
// its square, and rsq[r] = sum_c v_c): lane k takes orbital k, the waves take quarters of the
// row, v and the string are wave-uniform.  Fixed order, no atomics.
template <bool SQ>
__global__ void __launch_bounds__(RT) k_occ_contract(int64_t ncols, const double* __restrict__ src,
                                                     const uint64_t* __restrict__ cstr, double* __restrict__ occ,
                                                     double* __restrict__ rsq) {
  __shared__ double sh[RT / 64][64], st[RT / 64];
  const int64_t r = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t per = ((ncols + RT / 64 - 1) / (RT / 64) + 63) / 64 * 64;
  const int64_t c0 = min(ncols, wid * per), c1 = min(ncols, c0 + per);
  double a0 = 0.0, a1 = 0.0, t = 0.0;
  for (int64_t b = c0; b < c1; b += 64) {
    const int64_t c = min(b + lane, c1 - 1);
    double v = src[r * ncols + c];
    if (SQ) v *= v;
    if (b + lane >= c1) v = 0.0;
    const uint64_t o = cstr[c];
    if (SQ) t += v;
    const int vl = __double2loint(v), vh = __double2hiint(v), ol = (int)(uint32_t)o, oh = (int)(uint32_t)(o >> 32);
#pragma unroll
    for (int x = 0; x < 64; ++x) {
      const double u = __hiloint2double(__builtin_amdgcn_readlane(vh, x), __builtin_amdgcn_readlane(vl, x));
      const uint64_t w = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(oh, x) << 32) |
                         (uint32_t)__builtin_amdgcn_readlane(ol, x);
      const double add = ((w >> lane) & 1ull) ? u : 0.0;
      if (x & 1) a1 += add;
      else a0 += add;
    }
  }
  sh[wid][lane] = a0 + a1;
  if (SQ) {
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if (lane == 0) st[wid] = t;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    double v = 0.0;
    for (int w = 0; w < RT / 64; ++w) v += sh[w][threadIdx.x];
    occ[r * 64 + threadIdx.x] = v;
    if (SQ && threadIdx.x == 0) {
      double q = 0.0;
      for (int w = 0; w < RT / 64; ++w) q += st[w];
      rsq[r] = q;
    }
  }
}

// D[i][j] = sum_r n_i(rstr[r]) * (Y ? Y[r*64 + j] : w[r] n_j(rstr[r])): rows in CORR_PARTS
// ranges, one workgroup each, and the ranges' sums added in order
constexpr int CORR_PARTS = 128;
__global__ void __launch_bounds__(RT) k_corr(int64_t nrows, int L, const uint64_t* __restrict__ rstr,
                                             const double* __restrict__ w, const double* __restrict__ Y,
                                             double* __restrict__ part) {
  const int64_t per = (nrows + CORR_PARTS - 1) / CORR_PARTS;
  const int64_t r0 = min(nrows, blockIdx.x * per), r1 = min(nrows, r0 + per);
  for (int t = threadIdx.x; t < L * L; t += RT) {
    const int i = t / L, j = t % L;
    const uint64_t need = (1ull << i) | (Y ? 0ull : 1ull << j);
    double v = 0.0;
    for (int64_t r = r0; r < r1; ++r) {
      const double x = Y ? Y[r * 64 + j] : w[r];
      v += (rstr[r] & need) == need ? x : 0.0;
    }
    part[(int64_t)blockIdx.x * L * L + t] = v;
  }
}
__global__ void k_corr_sum(int n, const double* __restrict__ part, double* __restrict__ D) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  double v = 0.0;
  for (int p = 0; p < CORR_PARTS; ++p) v += part[(int64_t)p * n + t];
  D[t] = v;
}

__device__ inline int64_t idx4(int L, int i, int j, int k, int l) {
  return (int64_t)i + (int64_t)L * j + (int64_t)L * L * k + (int64_t)L * L * L * l;
}

// diagonal slots: gamma_s[p,p], Gamma_st[i,j,i,j], Gamma_ss[i,j,j,i]
__global__ void k_diag_slots(int L, const double* __restrict__ dens, const double* __restrict__ Daa,
                             const double* __restrict__ Dbb, const double* __restrict__ Dab,
                             double* __restrict__ one, double* __restrict__ two) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= L * L) return;
  const int i = t / L, j = t % L;
  const int64_t L2 = (int64_t)L * L, L4 = L2 * L2;
  if (i == j) {
    one[i + L * i] = dens[2 * i];
    one[L2 + i + L * i] = dens[2 * i + 1];
  }
  // alpha-beta (block 2) and beta-alpha (block 1): every (i,j)
  two[2 * L4 + idx4(L, i, j, i, j)] = Dab[i * L + j];
  two[1 * L4 + idx4(L, j, i, j, i)] = Dab[i * L + j];
  if (i != j) {
    two[0 * L4 + idx4(L, i, j, i, j)] = Daa[i * L + j];
    two[0 * L4 + idx4(L, i, j, j, i)] = -Daa[i * L + j];
    two[3 * L4 + idx4(L, i, j, i, j)] = Dbb[i * L + j];
    two[3 * L4 + idx4(L, i, j, j, i)] = -Dbb[i * L + j];
  }
}

// singles owners: one workgroup per key (a, i), a > i: its pairs [kseg, kend) of the sorted
// singles, spectators of the same spin from the strings (lane k: orbital k, the waves take the
// pairs in turn), of the other spin from the segments' occupation sums.  Writes the slots of
// (a, i) and of (i, a), whose sums are the same.  blk(s,t) = s + 2t.
__global__ void __launch_bounds__(RT) k_single_slots(int L, int s, const int32_t* __restrict__ keys,
                                                     const int32_t* __restrict__ krange,
                                                     const int32_t* __restrict__ kseg, const int32_t* __restrict__ pia,
                                                     const int32_t* __restrict__ pja,
                                                     const uint64_t* __restrict__ str, int64_t npair, int64_t ntiles,
                                                     const double* __restrict__ gpart, const double* __restrict__ occ,
                                                     double* __restrict__ one, double* __restrict__ two) {
  __shared__ double shS[RT / 64][64], shg[RT / 64];
  const int key = keys[blockIdx.x], a = key / L, i = key % L;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double accS = 0.0, gam = 0.0;
  for (int e = krange[2 * blockIdx.x] + wid; e < krange[2 * blockIdx.x + 1]; e += RT / 64) {
    double g = 0.0;
    for (int64_t t = 0; t < ntiles; ++t) g += gpart[t * npair + e];
    const int32_t jw = pja[e];
    const double v = jw < 0 ? -g : g;
    const uint64_t both = str[pia[e]] & str[jw & 0x7FFFFFFF];
    gam += v;
    accS += ((both >> lane) & 1ull) ? v : 0.0;
  }
  shS[wid][lane] = accS;
  if (lane == 0) shg[wid] = gam;
  __syncthreads();
  const int k = threadIdx.x;
  if (k >= L) return;
  double vs = 0.0, vo = 0.0, g = 0.0;
  for (int w = 0; w < RT / 64; ++w) {
    vs += shS[w][k];
    g += shg[w];
  }
  for (int q = kseg[blockIdx.x]; q < kseg[blockIdx.x + 1]; ++q) vo += occ[(int64_t)q * 64 + k];
  const int64_t L2 = (int64_t)L * L, L4 = L2 * L2;
  const int ss = s + 2 * s;        // same-spin block
  const int so = s + 2 * (1 - s);  // (s, other)
  const int os = (1 - s) + 2 * s;  // (other, s)
  if (k == 0) one[s * L2 + a + L * i] = one[s * L2 + i + L * a] = g;
  for (int turn = 0; turn < 2; ++turn) {
    const int p = turn ? i : a, q = turn ? a : i;
    if (k != a && k != i) {
      two[ss * L4 + idx4(L, p, k, q, k)] = vs;
      two[ss * L4 + idx4(L, k, p, k, q)] = vs;
      two[ss * L4 + idx4(L, p, k, k, q)] = -vs;
      two[ss * L4 + idx4(L, k, p, q, k)] = -vs;
    }
    two[so * L4 + idx4(L, p, k, q, k)] = vo;
    two[os * L4 + idx4(L, k, p, k, q)] = vo;
  }
}

// doubles owners: one thread per distinct quadruple (segment of sorted keys)
__global__ void k_double_slots(int L, int s, int64_t nseg, const int32_t* __restrict__ seg,
                               const int32_t* __restrict__ perm, const uint32_t* __restrict__ keys,
                               const uint32_t* __restrict__ exc, const double* __restrict__ g,
                               double* __restrict__ two) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nseg) return;
  const int64_t L2 = (int64_t)L * L, L4 = L2 * L2;
  double v = 0.0;
  for (int32_t e = seg[t]; e < seg[t + 1]; ++e) {
    const int32_t q = perm[e];
    v += (((exc[q] >> 24) & 1u) ? -1.0 : 1.0) * g[q];
  }
  const uint32_t key = keys[seg[t]];
  const int J = key % L, I = (key / L) % L, B = (key / L / L) % L, A = key / L / L / L;
  const int ss = s + 2 * s;
  two[ss * L4 + idx4(L, A, B, I, J)] = v;
  two[ss * L4 + idx4(L, B, A, J, I)] = v;
  two[ss * L4 + idx4(L, A, B, J, I)] = -v;
  two[ss * L4 + idx4(L, B, A, I, J)] = -v;
}

__global__ void k_single_keys(int64_t nnz, int L, const uint32_t* __restrict__ exc, uint32_t* __restrict__ keys,
                              int32_t* __restrict__ idx) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nnz) return;
  const uint32_t e = exc[q];
  keys[q] = ((e >> 6) & 63u) * (uint32_t)L + (e & 63u);  // a*L + i
  idx[q] = (int32_t)q;
}

__global__ void k_double_keys(int64_t nnz, int L, const uint32_t* __restrict__ exc, uint32_t* __restrict__ keys,
                              int32_t* __restrict__ idx) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nnz) return;
  const uint32_t e = exc[q];
  const uint32_t I = e & 63u, J = (e >> 6) & 63u, A = (e >> 12) & 63u, B = (e >> 18) & 63u;
  keys[q] = ((A * L + B) * L + I) * L + J;
  idx[q] = (int32_t)q;
}

// segment starts of sorted keys: flag[e] = (e==0 || key[e] != key[e-1])
__global__ void k_flag(int64_t n, const uint32_t* __restrict__ keys, int32_t* __restrict__ flag) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  flag[e] = (e == 0 || keys[e] != keys[e - 1]) ? 1 : 0;
}

__global__ void k_segstart(int64_t n, const int32_t* __restrict__ flag, const int32_t* __restrict__ pos,
                           int32_t* __restrict__ seg, int32_t nseg) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n && flag[e]) seg[pos[e]] = (int32_t)e;
  if (e == 0) seg[nseg] = (int32_t)n;
}

// per key (a,i) dense segment table: kseg[key] = first sorted entry with key >= key
__global__ void k_keyseg(int64_t n, int nkeys, const uint32_t* __restrict__ keys, int32_t* __restrict__ kseg) {
  const int key = blockIdx.x * blockDim.x + threadIdx.x;
  if (key > nkeys) return;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int)keys[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  kseg[key] = (int32_t)lo;
}

// alpha-beta pair sums.  A beta pair is a pair of columns (x, y) one excitation apart, x
// holding the upper orbital b and y the lower j; it contributes to T_(a,i)[b,j] (bra x, ket y)
// and to T_(a,i)[j,b] (bra y, ket x).  Workgroup: one tile of beta pairs against one segment of
// the alpha pairs of one key (a, i).  Each thread keeps its pairs' two sums and their LDS
// addresses in registers through the whole segment; per alpha pair the columns the tile needs
// of the two rows are staged as (bra, ket) vectors, so a beta pair costs two 16-byte LDS reads
// and two FMAs, and no table is read.  At the end the sums go through LDS and each run of pairs
// with one (b, j) is summed in a fixed order by one wave: no atomics, the same bits every time.
//
// Bound: the 16-byte LDS gathers (ordered by order_pairs they spend 0.38 bank-conflict cycles an
// LDS instruction at norb=16, full space, and 0.62 at norb=36, 4,000 x 20,000 strings) and the
// latency of the next rows, about evenly.  Before, every product was a fixed-point 64-bit LDS
// atomic into the L^2 sums of one key, with the pairs re-read from their table for each alpha
// pair: those two sets 108 ms and 57; now 11.0 and 8.6.  On the way, the same two sets: two
// workgroups of 512 threads and 8,192 pairs on a CU 14.4 and 9.1 ms, of 6,144 pairs 19.8 and 9.1
// (an alpha pair costs its staging latency, not its pairs); one of 1,024 threads with the next
// rows in registers 14.3 and 10.4; ordered pairs, empty rounds skipped, one column per load
// 11.7 and 8.8.
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

struct AbRdmArgs {
  int64_t nb, nruns, ntiles, nseg;
  const int4* tile;
  const int64_t* entoff;
  const uint32_t* ent;
  const uint16_t* rank;
  const int32_t* runptr;
  const int32_t* runstart;
  const int32_t* segptr;
  const int32_t* pia;
  const int32_t* pja;
  const double* W;
  double* part;
};

// the tile and segment of a workgroup: one XCD takes the tiles of one segment after another,
// they read the same rows
__device__ inline bool ab_rdm_item(const AbRdmArgs& A, int64_t& tl, int64_t& sg) {
  const int64_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  tl = slot % A.ntiles;
  sg = (slot / A.ntiles) * 8 + xcd;
  return sg < A.nseg;
}

// column pairs x, x + 1 of rows wi and wj (x within the tile's staged columns, the last pair
// again for the threads past it)
template <int SR, int NT>
struct AbRdmRows {
  d2u i[SR / 2], j[SR / 2];
  __device__ inline void load(const double* wi, const double* wj, const int4& ti, int nc, int x0) {
#pragma unroll
    for (int u = 0; u < SR / 2; ++u) {
      const int x = min(x0 + 2 * u * NT, nc - 2);
      const int64_t c = x < ti.y ? ti.x + x : ti.z + (x - ti.y);
      i[u] = *reinterpret_cast<const d2u*>(wi + c);
      j[u] = *reinterpret_cast<const d2u*>(wj + c);
    }
  }
  __device__ inline void store(double2* to, bool has, double sa, int nc, int x0) const {
#pragma unroll
    for (int u = 0; u < SR / 2; ++u) {
      const int xx = x0 + 2 * u * NT, x = min(xx, nc - 2);
      if (xx < nc) {
        to[x] = has ? make_double2(i[u].x, sa * j[u].x) : make_double2(0.0, 0.0);
        to[x + 1] = has ? make_double2(i[u].y, sa * j[u].y) : make_double2(0.0, 0.0);
      }
    }
  }
};

// rounds: of the U pairs per thread, the first that the tile fills (wave-uniform)
template <int U>
__device__ inline void ab_rdm_products(const double2* buf, int rounds, const uint32_t (&en)[U], double (&s0)[U],
                                       double (&s1)[U]) {
  constexpr int QB = 3 - (U % 3 != 0);  // pairs whose LDS reads are issued before their products
#pragma unroll
  for (int u = 0; u < U; u += QB) {
    if (u >= rounds) break;
    double2 x[QB], y[QB];
#pragma unroll
    for (int k = 0; k < QB; ++k) {
      uint32_t w = en[u + k];
      asm volatile("" : "+v"(w));  // decoded here, not held as two addresses through the segment
      x[k] = buf[w & 0x7FFFu];
      y[k] = buf[(w >> 15) & 0x7FFFu];
    }
#pragma unroll
    for (int k = 0; k < QB; ++k) {
      s0[u + k] += x[k].x * y[k].y;
      s1[u + k] += y[k].x * x[k].y;
      // formed here: left to the end of the block, the products would hold every pair's reads
      asm volatile("" : "+v"(s0[u + k]), "+v"(s1[u + k]));
    }
  }
}

// the runs of one (b, j): ranks [runstart[r], runstart[r + 1]) of the tile's pairs, in order; a
// tile's list ends with its number of pairs
template <int NT, int U>
__device__ inline void ab_rdm_runs(const AbRdmArgs& A, int64_t tl, int64_t sg, double* sums, const uint32_t (&en)[U],
                                   const double (&s0)[U], const double (&s1)[U]) {
  const uint16_t* rank = A.rank + A.entoff[tl];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int r0 = A.runptr[tl], r1 = A.runptr[tl + 1] - 1;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double v = d ? s1[u] : s0[u];
      sums[rank[u * NT + threadIdx.x]] = (en[u] >> 30) & 1u ? -v : v;
    }
    __syncthreads();
    for (int r = r0 + wid; r < r1; r += NT / 64) {
      double v = 0.0;
      for (int x = A.runstart[r] + lane; x < A.runstart[r + 1]; x += 64) v += sums[x];
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      if (lane == 0) A.part[(sg * A.nruns + r) * 2 + d] = v;
    }
  }
}

// Many beta pairs: one workgroup of 1,024 threads on a CU, the rows of the next alpha pair
// loaded into registers while the current one is used, two LDS buffers, one barrier per alpha
// pair.  What a thread loads and where it goes is the same for every alpha pair (offsets held
// in registers, rows as scalar bases; a thread past the last columns loads and stores them
// again).
constexpr int ABR_NT = 1024, ABR_U = 12;
__global__ void __launch_bounds__(ABR_NT, 4) k_ab_rdm(const AbRdmArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int SH = 5;  // columns per thread
  static_assert(SH * ABR_NT >= AB_PAIR_COLS, "one staging round");
  int64_t tl, sg;
  if (!ab_rdm_item(A, tl, sg)) return;  // whole workgroup
  const int4 ti = make_int4(uniform_at(&A.tile[tl].x, 0), uniform_at(&A.tile[tl].y, 0), uniform_at(&A.tile[tl].z, 0),
                            uniform_at(&A.tile[tl].w, 0));  // first column and number of columns of the two chunks
  const int nc = ti.y + ti.w, stride = nc + 1;
  double2* buf = reinterpret_cast<double2*>(smem);
  uint32_t en[ABR_U], off[SH];
  double s0[ABR_U], s1[ABR_U];
#pragma unroll
  for (int u = 0; u < ABR_U; ++u) {
    en[u] = A.ent[uniform_at(A.entoff, tl) + u * ABR_NT + threadIdx.x];
    s0[u] = s1[u] = 0.0;
  }
#pragma unroll
  for (int u = 0; u < SH; ++u) {
    const int x = min((int)threadIdx.x + u * ABR_NT, nc - 1);
    off[u] = (uint32_t)(x < ti.y ? ti.x + x : ti.z + (x - ti.y)) * 8u;
  }
  if (threadIdx.x < 2) buf[(int)threadIdx.x * stride + nc] = make_double2(0.0, 0.0);  // padding reads this
  const int e0 = uniform_at(A.segptr, 2 * sg), e1 = uniform_at(A.segptr, 2 * sg + 1);
  const int rounds = (uniform_at(A.runstart, uniform_at(A.runptr, tl + 1) - 1) + ABR_NT - 1) / ABR_NT;
  double vi[SH], vj[SH];
  uint32_t neg = 0;
  // the rows of the pair to load next: read one alpha pair ahead of its loads
  int32_t ni = uniform_at(A.pia, e0), nj = uniform_at(A.pja, e0);
  auto load = [&](int next) {
    neg = (uint32_t)nj & 0x80000000u;
    const char* wi = reinterpret_cast<const char*>(A.W + (int64_t)ni * A.nb);
    const char* wj = reinterpret_cast<const char*>(A.W + (int64_t)(nj & 0x7FFFFFFF) * A.nb);
#pragma unroll
    for (int u = 0; u < SH; ++u) {
      vi[u] = *reinterpret_cast<const double*>(wi + off[u]);
      vj[u] = *reinterpret_cast<const double*>(wj + off[u]);
    }
    ni = uniform_at(A.pia, min(next, e1 - 1));
    nj = uniform_at(A.pja, min(next, e1 - 1));
  };
  auto flip = [&](double v) { return __hiloint2double(__double2hiint(v) ^ (int)neg, __double2loint(v)); };
  auto store = [&](double2* b) {
#pragma unroll
    for (int u = 0; u < SH; ++u) {
      const int x = (int)threadIdx.x + u * ABR_NT;
      if (x < nc) b[x] = make_double2(vi[u], flip(vj[u]));
    }
  };
  load(e0 + 1);
  store(buf);
  load(e0 + 2);
  __syncthreads();
  for (int e = e0; e < e1; ++e) {
    const int cur = (e - e0) & 1;
    ab_rdm_products<ABR_U>(buf + cur * stride, rounds, en, s0, s1);
    store(buf + (cur ^ 1) * stride);
    load(e + 3);
    __syncthreads();  // the next rows are in place, the current ones done with
  }
  ab_rdm_runs<ABR_NT, ABR_U>(A, tl, sg, reinterpret_cast<double*>(smem), en, s0, s1);
}

// Few beta pairs: 256 threads of 4 pairs, SP alpha pairs staged per barrier, several workgroups
// on a CU.
constexpr int ABR_NT_S = 256, ABR_U_S = 4;
template <int SP>
__global__ void __launch_bounds__(ABR_NT_S) k_ab_rdm_small(const AbRdmArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int SR = 4;
  int64_t tl, sg;
  if (!ab_rdm_item(A, tl, sg)) return;  // whole workgroup
  const int4 ti = make_int4(uniform_at(&A.tile[tl].x, 0), uniform_at(&A.tile[tl].y, 0), uniform_at(&A.tile[tl].z, 0),
                            uniform_at(&A.tile[tl].w, 0));
  const int nc = ti.y + ti.w, stride = nc + 1;
  double2* buf = reinterpret_cast<double2*>(smem);
  uint32_t en[ABR_U_S];
  double s0[ABR_U_S], s1[ABR_U_S];
#pragma unroll
  for (int u = 0; u < ABR_U_S; ++u) {
    en[u] = A.ent[uniform_at(A.entoff, tl) + u * ABR_NT_S + threadIdx.x];
    s0[u] = s1[u] = 0.0;
  }
  if ((int)threadIdx.x < SP) buf[(int)threadIdx.x * stride + nc] = make_double2(0.0, 0.0);
  const int e0 = uniform_at(A.segptr, 2 * sg), e1 = uniform_at(A.segptr, 2 * sg + 1);
  for (int e = e0; e < e1; e += SP) {
    __syncthreads();  // the previous rows are done with
#pragma unroll
    for (int sp = 0; sp < SP; ++sp) {
      const int q = min(e + sp, e1 - 1);
      const int32_t jw = uniform_at(A.pja, q);
      const double* wi = A.W + (int64_t)uniform_at(A.pia, q) * A.nb;
      const double* wj = A.W + (int64_t)(jw & 0x7FFFFFFF) * A.nb;
      for (int x0 = 2 * (int)threadIdx.x; x0 < nc; x0 += SR * ABR_NT_S) {
        AbRdmRows<SR, ABR_NT_S> rows;
        rows.load(wi, wj, ti, nc, x0);
        rows.store(buf + sp * stride, e + sp < e1, jw < 0 ? -1.0 : 1.0, nc, x0);  // absent: zeros
      }
    }
    __syncthreads();
#pragma unroll
    for (int sp = 0; sp < SP; ++sp) ab_rdm_products<ABR_U_S>(buf + sp * stride, ABR_U_S, en, s0, s1);
  }
  ab_rdm_runs<ABR_NT_S, ABR_U_S>(A, tl, sg, reinterpret_cast<double*>(smem), en, s0, s1);
}

// the alpha pairs of the sorted singles: bra row, and ket row with the sign in bit 31
__global__ void k_alpha_pairs(int64_t n, const int32_t* __restrict__ perm, const int64_t* __restrict__ rowof,
                              const int32_t* __restrict__ col, const uint32_t* __restrict__ exc,
                              int32_t* __restrict__ pia, int32_t* __restrict__ pja) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int32_t q = perm[e];
  pia[e] = (int32_t)rowof[q];
  pja[e] = (int32_t)((uint32_t)col[q] | (((exc[q] >> 24) & 1u) << 31));
}

// sum the partials of one key (a, i), a > i, over its segments and each pair's runs, and write
// T_(a,i)[b,j] and T_(a,i)[j,b] with their images: Gamma_ab[a,b,i,j], Gamma_ba[b,a,j,i], and
// key (i, a), whose pairs are the same pairs read the other way: T_(i,a)[j,b] = T_(a,i)[b,j]
__global__ void k_ab_slots(int L, const int32_t* __restrict__ keys, const int32_t* __restrict__ kseg, int64_t seg0,
                           int64_t nruns, const int32_t* __restrict__ pairptr, const int32_t* __restrict__ pairrun,
                           const double* __restrict__ part, double* __restrict__ two) {
  const int a = keys[blockIdx.x] / L, i = keys[blockIdx.x] % L;
  const int NP = L * (L - 1) / 2;
  const int64_t L2 = (int64_t)L * L, L4 = L2 * L2;
  for (int p = threadIdx.x; p < NP; p += blockDim.x) {
    int b = 1;
    while ((b + 1) * b / 2 <= p) ++b;
    const int j = p - b * (b - 1) / 2;
    double v0 = 0.0, v1 = 0.0;
    for (int32_t s = kseg[blockIdx.x]; s < kseg[blockIdx.x + 1]; ++s)
      for (int32_t e = pairptr[p]; e < pairptr[p + 1]; ++e) {
        const double* x = part + ((s - seg0) * nruns + pairrun[e]) * 2;
        v0 += x[0];
        v1 += x[1];
      }
    two[2 * L4 + idx4(L, a, b, i, j)] = v0;
    two[1 * L4 + idx4(L, b, a, j, i)] = v0;
    two[2 * L4 + idx4(L, i, j, a, b)] = v0;
    two[1 * L4 + idx4(L, j, i, b, a)] = v0;
    two[2 * L4 + idx4(L, a, j, i, b)] = v1;
    two[1 * L4 + idx4(L, j, a, b, i)] = v1;
    two[2 * L4 + idx4(L, i, b, a, j)] = v1;
    two[1 * L4 + idx4(L, b, i, j, a)] = v1;
  }
}

__global__ void k_rowof(int64_t n, const int64_t* __restrict__ rowptr, int64_t* __restrict__ rowof) {
  const int64_t r = blockIdx.x;
  for (int64_t q = rowptr[r] + threadIdx.x; q < rowptr[r + 1]; q += blockDim.x) rowof[q] = r;
  (void)n;
}

__global__ void k_backward(int L, const double* __restrict__ one, const double* __restrict__ two, double g,
                           double* __restrict__ dh, double* __restrict__ deri) {
  const int64_t L2 = (int64_t)L * L, L4 = L2 * L2;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < L4 && deri) {
    const int s_ = (int)(t % L), r = (int)((t / L) % L), q = (int)((t / L2) % L), p = (int)(t / L2 / L);
    const int64_t x = idx4(L, p, r, q, s_);
    deri[t] = 0.5 * g * (two[x] + two[L4 + x] + two[2 * L4 + x] + two[3 * L4 + x]);
  }
  if (t < L2 && dh) {
    const int q = (int)(t % L), p = (int)(t / L);
    dh[t] = g * (one[p + L * q] + one[L2 + p + L * q]);
  }
}

inline unsigned nb_for(int64_t n, int t) { return (unsigned)std::max<int64_t>(1, (n + t - 1) / t); }

// sort (key, index) pairs; returns sorted keys/indices in the out buffers
void sort_pairs(int64_t n, WBuf<uint32_t>& keys, WBuf<int32_t>& idx, WBuf<uint32_t>& keys_out,
                WBuf<int32_t>& idx_out, int end_bit, Arena& ar, hipStream_t st) {
  keys_out.alloc(std::max<int64_t>(n, 1));
  idx_out.alloc(std::max<int64_t>(n, 1));
  if (n == 0) return;
  size_t tmp = 0;
  SBDG_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, keys.p, keys_out.p, idx.p, idx_out.p, (int)n, 0,
                                                end_bit, st));
  WBuf<unsigned char> t(ar);
  t.alloc(tmp + 1);
  SBDG_CHECK(hipcub::DeviceRadixSort::SortPairs(t.p, tmp, keys.p, keys_out.p, idx.p, idx_out.p, (int)n, 0, end_bit,
                                                st));
  SBDG_CHECK(hipStreamSynchronize(st));
}

int bits_for(uint64_t v) {
  int b = 1;
  while ((1ull << b) <= v) ++b;
  return b;
}

// The singles of one spin sorted by key: pia/pja as k_alpha_pairs writes them, hk[key] the
// first of key (host; L^2 + 1 of them).
struct SortedSingles {
  explicit SortedSingles(Arena& ar) : pia(ar), pja(ar) {}
  WBuf<int32_t> pia, pja;
  std::vector<int32_t> hk;
};

void sort_singles(const Table& t, int L, SortedSingles& ss, Arena& ar, hipStream_t st) {
  const int L2 = L * L;
  ss.hk.assign(L2 + 1, 0);
  if (t.nnz == 0) return;
  WBuf<int64_t> rowof(ar);
  WBuf<uint32_t> keys(ar), ks(ar);
  WBuf<int32_t> idx(ar), perm(ar), kseg(ar);
  rowof.alloc(t.nnz);
  keys.alloc(t.nnz);
  idx.alloc(t.nnz);
  ss.pia.alloc(t.nnz);
  ss.pja.alloc(t.nnz);
  kseg.alloc(L2 + 1);
  hipLaunchKernelGGL(k_rowof, dim3((unsigned)t.n), dim3(256), 0, st, t.n, t.rowptr.p, rowof.p);
  hipLaunchKernelGGL(k_single_keys, dim3(nb_for(t.nnz, 256)), dim3(256), 0, st, t.nnz, L, t.exc.p, keys.p, idx.p);
  sort_pairs(t.nnz, keys, idx, ks, perm, bits_for((uint64_t)L2), ar, st);
  hipLaunchKernelGGL(k_alpha_pairs, dim3(nb_for(t.nnz, 256)), dim3(256), 0, st, t.nnz, perm.p, rowof.p, t.col.p,
                     t.exc.p, ss.pia.p, ss.pja.p);
  hipLaunchKernelGGL(k_keyseg, dim3(nb_for(L2 + 1, 256)), dim3(256), 0, st, t.nnz, L2, ks.p, kseg.p);
  SBDG_CHECK(hipMemcpyAsync(ss.hk.data(), kseg.p, sizeof(int32_t) * (L2 + 1), hipMemcpyDeviceToHost, st));
  SBDG_CHECK(hipStreamSynchronize(st));
}

// Keys (a, i), a > i, with pairs, cut into segments of at most len pairs, and batches of whole
// keys of at most `most` segments (at least one key).
struct KeySegments {
  std::vector<int32_t> keys, krange, kseg, segs;
  std::vector<std::pair<size_t, size_t>> batch;
  int64_t widest = 0;  // segments of the largest batch
  const int32_t *dkeys = nullptr, *dkrange = nullptr, *dkseg = nullptr, *dsegs = nullptr;
  std::vector<int32_t> lists;  // the four, copied at once
  WBuf<int32_t> dlists;
  explicit KeySegments(Arena& ar) : dlists(ar) {}
};

void key_segments(const std::vector<int32_t>& hk, int L, int64_t len, int64_t most, KeySegments& K, hipStream_t st) {
  for (int key = 0; key < L * L; ++key) {
    if (key / L <= key % L || hk[key] == hk[key + 1]) continue;
    K.keys.push_back(key);
    K.krange.push_back(hk[key]);
    K.krange.push_back(hk[key + 1]);
    K.kseg.push_back((int32_t)(K.segs.size() / 2));
    for (int64_t e = hk[key]; e < hk[key + 1]; e += len) {
      K.segs.push_back((int32_t)e);
      K.segs.push_back((int32_t)std::min<int64_t>(e + len, hk[key + 1]));
    }
  }
  K.kseg.push_back((int32_t)(K.segs.size() / 2));
  for (size_t k = 0; k < K.keys.size();) {
    size_t f = k + 1;
    while (f < K.keys.size() && K.kseg[f + 1] - K.kseg[k] <= most) ++f;
    K.batch.emplace_back(k, f);
    K.widest = std::max<int64_t>(K.widest, K.kseg[f] - K.kseg[k]);
    k = f;
  }
  const std::vector<int32_t>* all[] = {&K.keys, &K.krange, &K.kseg, &K.segs};
  for (const auto* h : all) K.lists.insert(K.lists.end(), h->begin(), h->end());
  K.dlists.alloc(K.lists.size());
  SBDG_CHECK(hipMemcpyAsync(K.dlists.p, K.lists.data(), sizeof(int32_t) * K.lists.size(), hipMemcpyHostToDevice, st));
  K.dkeys = K.dlists.p;
  K.dkrange = K.dkeys + K.keys.size();
  K.dkseg = K.dkrange + K.krange.size();
  K.dsegs = K.dkseg + K.kseg.size();
}

// singles of one spin: pair sums by key segment, their occupation parts, then key owners
void singles_part(const Table& t, const SortedSingles& ss, int L, int s, const double* X, int64_t ncols,
                  const uint64_t* rstr, const uint64_t* cstr, double* one, double* two, Arena& ar,
                  hipStream_t st) {
  if (t.nnz == 0) return;
  const int NV = ncols >= 2 ? 2 : 1;
  const int64_t tw = (int64_t)RT * NV * PSU, ntiles = (ncols + tw - 1) / tw;
  const int64_t len = std::min<int64_t>(PSEG, std::max<int64_t>(16, t.nnz / 2 * ntiles / 4096));
  KeySegments K(ar);
  key_segments(ss.hk, L, len, std::max<int64_t>(1, RDM_PART_BYTES / (8 * ncols)), K, st);
  WBuf<double> D(ar), gpart(ar), occ(ar);
  D.alloc((size_t)(K.widest * ncols));
  gpart.alloc((size_t)(ntiles * t.nnz));
  occ.alloc(K.segs.size() / 2 * 64);
  for (const auto& bt : K.batch) {
    const int64_t s0 = K.kseg[bt.first], ns = K.kseg[bt.second] - s0;
    if (ns * ntiles > (int64_t)INT32_MAX) throw Error(SBDG_ERR_LIMIT, "grid too large");
    if (NV == 2)
      hipLaunchKernelGGL(k_pair_sums<2>, dim3((unsigned)(ns * ntiles)), dim3(RT), 0, st, ncols, ntiles, ns,
                         K.dsegs + 2 * s0, ss.pia.p, ss.pja.p, t.nnz, X, D.p, gpart.p);
    else
      hipLaunchKernelGGL(k_pair_sums<1>, dim3((unsigned)(ns * ntiles)), dim3(RT), 0, st, ncols, ntiles, ns,
                         K.dsegs + 2 * s0, ss.pia.p, ss.pja.p, t.nnz, X, D.p, gpart.p);
    hipLaunchKernelGGL(k_occ_contract<false>, dim3((unsigned)ns), dim3(RT), 0, st, ncols, D.p, cstr, occ.p + s0 * 64,
                       nullptr);
  }
  hipLaunchKernelGGL(k_single_slots, dim3((unsigned)K.keys.size()), dim3(RT), 0, st, L, s, K.dkeys, K.dkrange,
                     K.dkseg, ss.pia.p, ss.pja.p, rstr, t.nnz, ntiles, gpart.p, occ.p, one, two);
  SBDG_CHECK(hipGetLastError());
  SBDG_CHECK(hipStreamSynchronize(st));
}

// Row-pair sums of the doubles table t: by core block for the cores of ct (the larger
// cores, when sigma built them), by pair for the rest of the entries above the diagonal,
// then mirrored to the entries below it.
void doubles_gram(const Table& t, const CoreTable* ct, const uint64_t* strs, const double* X, int64_t ncols,
                  double* g, Arena& ar, hipStream_t st) {
  WBuf<unsigned char> done(ar);
  done.alloc(t.nnz);
  SBDG_CHECK(hipMemsetAsync(done.p, 0, t.nnz, st));
  if (ct && ct->ncore > 0) {
    std::vector<int32_t> hs(ct->ncore + 1);
    SBDG_CHECK(hipMemcpyAsync(hs.data(), ct->start.p, sizeof(int32_t) * hs.size(), hipMemcpyDeviceToHost, st));
    SBDG_CHECK(hipStreamSynchronize(st));
    std::vector<int4> items[2];  // blocks of 16 and of 32 members
    for (int64_t k = 0; k < ct->ncore; ++k) {
      const int m = hs[k + 1] - hs[k];
      if (m < 2) continue;
      const int w = m <= 16 ? 0 : 1, bm = 16 << w, nbk = (m + bm - 1) / bm;
      for (int bi = 0; bi < nbk; ++bi)
        for (int bj = bi; bj < nbk; ++bj) items[w].push_back(make_int4((int)k, bi, bj, 0));
    }
    WBuf<int4> ditems[2] = {WBuf<int4>(ar), WBuf<int4>(ar)};
    for (int w = 0; w < 2; ++w) {
      if (items[w].empty()) continue;
      ditems[w].alloc(items[w].size());
      SBDG_CHECK(hipMemcpyAsync(ditems[w].p, items[w].data(), sizeof(int4) * items[w].size(), hipMemcpyHostToDevice,
                                st));
    }
#define SBDG_CG(W)                                                                                             \
  if (!items[W].empty())                                                                                       \
  hipLaunchKernelGGL(k_core_gram<W + 1>, dim3((unsigned)items[W].size()), dim3(RT), 0, st, ncols, ditems[W].p, \
                     ct->start.p, ct->row.p, strs, t.rowptr.p, t.col.p, X, g, done.p)
    SBDG_CG(0);
    SBDG_CG(1);
#undef SBDG_CG
    SBDG_CHECK(hipGetLastError());
    SBDG_CHECK(hipStreamSynchronize(st));  // the item lists on the host stay alive until here
  }
  WBuf<int32_t> flag(ar), pos(ar), qlist(ar);
  WBuf<int64_t> lptr(ar);
  flag.alloc(t.nnz);
  pos.alloc(t.nnz);
  qlist.alloc(t.nnz);
  lptr.alloc(t.n + 1);
  hipLaunchKernelGGL(k_pair_flags, dim3((unsigned)t.n), dim3(RT), 0, st, t.rowptr.p, t.col.p, done.p, flag.p);
  size_t tmp = 0;
  SBDG_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, flag.p, pos.p, (int)t.nnz, st));
  WBuf<unsigned char> tb(ar);
  tb.alloc(tmp + 1);
  SBDG_CHECK(hipcub::DeviceScan::ExclusiveSum(tb.p, tmp, flag.p, pos.p, (int)t.nnz, st));
  hipLaunchKernelGGL(k_pair_list, dim3(nb_for(t.nnz, 256)), dim3(256), 0, st, t.nnz, flag.p, pos.p, qlist.p);
  hipLaunchKernelGGL(k_pair_lptr, dim3(nb_for(t.n + 1, 256)), dim3(256), 0, st, t.n, t.nnz, t.rowptr.p, flag.p, pos.p,
                     lptr.p);
  if (ncols % 2 == 0)
    hipLaunchKernelGGL(k_gram_pairs<true>, dim3((unsigned)t.n), dim3(RT), 0, st, ncols, lptr.p, qlist.p, t.col.p, X,
                       g);
  else
    hipLaunchKernelGGL(k_gram_pairs<false>, dim3((unsigned)t.n), dim3(RT), 0, st, ncols, lptr.p, qlist.p, t.col.p,
                       X, g);
  hipLaunchKernelGGL(k_gram_mirror, dim3((unsigned)t.n), dim3(RT), 0, st, t.rowptr.p, t.col.p, g);
  SBDG_CHECK(hipGetLastError());
  SBDG_CHECK(hipStreamSynchronize(st));
}

void doubles_part(const Table& t, int L, int s, const double* X, int64_t ncols, const CoreTable* ct,
                  const uint64_t* strs, double* two, Arena& ar, hipStream_t st) {
  if (t.nnz == 0) return;
  WBuf<double> g(ar);
  g.alloc(t.nnz);
  doubles_gram(t, ct, strs, X, ncols, g.p, ar, st);
  WBuf<uint32_t> keys(ar), ks(ar);
  WBuf<int32_t> idx(ar), perm(ar), flag(ar), pos(ar), seg(ar);
  keys.alloc(t.nnz);
  idx.alloc(t.nnz);
  hipLaunchKernelGGL(k_double_keys, dim3(nb_for(t.nnz, 256)), dim3(256), 0, st, t.nnz, L, t.exc.p, keys.p, idx.p);
  sort_pairs(t.nnz, keys, idx, ks, perm, bits_for((uint64_t)L * L * L * L), ar, st);
  flag.alloc(t.nnz);
  pos.alloc(t.nnz);
  hipLaunchKernelGGL(k_flag, dim3(nb_for(t.nnz, 256)), dim3(256), 0, st, t.nnz, ks.p, flag.p);
  size_t tmp = 0;
  SBDG_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, flag.p, pos.p, (int)t.nnz, st));
  WBuf<unsigned char> tb(ar);
  tb.alloc(tmp + 1);
  SBDG_CHECK(hipcub::DeviceScan::ExclusiveSum(tb.p, tmp, flag.p, pos.p, (int)t.nnz, st));
  int32_t lastpos = 0, lastflag = 0;
  SBDG_CHECK(hipMemcpyAsync(&lastpos, pos.p + t.nnz - 1, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  SBDG_CHECK(hipMemcpyAsync(&lastflag, flag.p + t.nnz - 1, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  SBDG_CHECK(hipStreamSynchronize(st));
  const int32_t nseg = lastpos + lastflag;
  seg.alloc(nseg + 1);
  hipLaunchKernelGGL(k_segstart, dim3(nb_for(t.nnz, 256)), dim3(256), 0, st, t.nnz, flag.p, pos.p, seg.p, nseg);
  hipLaunchKernelGGL(k_double_slots, dim3(nb_for(nseg, 256)), dim3(256), 0, st, L, s, (int64_t)nseg, seg.p, perm.p,
                     ks.p, t.exc.p, g.p, two);
  SBDG_CHECK(hipGetLastError());
  SBDG_CHECK(hipStreamSynchronize(st));
}

}  // namespace

// Order of a tile's n pairs over the lanes: in sets of 16 whose two columns each fall into 16
// different 16-byte LDS slots where the pairs allow it, a set on the lanes that a read serves
// together (LDS16_LANE).  Per set and slot of the first column, the largest class of
// pairs (by their two slots) whose second slot is still free in the set; a slot left without
// one takes the largest class of any.  out and rank: the pairs in order and their places in
// the sorted list.  The sixteen classes of a first slot are compared as one vector of 16-bit
// counts (3.5M pairs, all strings of 7 electrons in 20 orbitals: 180 -> 70 ms on the host; 2.9M of
// 200,000 sampled strings at norb=36, whose 1,543 tiles leave more to the fills: 210 -> 64).
static void order_pairs(const uint32_t* in, int n, uint32_t* out, uint16_t* rank) {
  typedef int16_t v16 __attribute__((vector_size(32)));
  alignas(32) int16_t left[256] = {0};  // pairs left per class (n is at most a tile's: 12,288)
  std::vector<int> next(256, 0), cls(n);
  auto slots = [](uint32_t w) { return (int)((w & 15u) * 16 + ((w >> 15) & 15u)); };
  for (int e = 0; e < n; ++e) ++left[slots(in[e])];
  for (int k = 1; k < 256; ++k) next[k] = next[k - 1] + left[k - 1];
  {
    std::vector<int> at(next);
    for (int e = 0; e < n; ++e) cls[at[slots(in[e])]++] = e;
  }
  int pos = 0;
  auto take = [&](int k) {
    const int e = cls[next[k]++];
    --left[k];
    const int at = pos - (pos & 31) + LDS16_LANE[pos & 31];
    out[at] = in[e];
    rank[at] = (uint16_t)e;
    ++pos;
  };
  const v16* rows = reinterpret_cast<const v16*>(left);
  while (pos < n) {
    v16 open = v16{} - 1;  // second slots still free in the set
    for (int t = 0; t < 16 && pos < n; ++t) {
      const int i = (t + pos / 16) & 15;  // no slot always chooses last
      const v16 c = rows[i] & open;
      const int16_t most = __builtin_reduce_max(c);
      if (most == 0) continue;
      int j = 0;
      while (c[j] != most) ++j;
      open[j] = 0;
      take(16 * i + j);
    }
    // fill the set to a multiple of 16 with what is left over
    while (pos < n && (pos & 15)) {
      v16 m = rows[0];
      for (int i = 1; i < 16; ++i) m = __builtin_elementwise_max(m, rows[i]);
      const int16_t most = __builtin_reduce_max(m);
      int i = 0, j = 0;
      while (!__builtin_reduce_or(rows[i] == most)) ++i;
      while (rows[i][j] != most) ++j;
      take(16 * i + j);
    }
  }
}

// Tiles of beta pairs for k_ab_rdm, on the host.  Columns are cut into chunks (two fit the
// LDS share; one where the whole row fits it), pairs are grouped by the chunks of their two
// columns and sorted by orbital pair inside a group, and a group is cut into tiles.  Many
// pairs: tiles of 12,288 (1,024 threads of 12); below 32,768 of them tiles of 1,024 (256
// threads of 4), so that a small set has several per key, with four alpha pairs staged at once
// while their rows fit 40 KiB.
void build_ab_pairs(const Table& sb, int L, AbPairs& ab, hipStream_t st) {
  const int64_t nb = sb.n;
  if (nb > (1 << 18)) throw Error(SBDG_ERR_LIMIT, "beta string set beyond 2^18 strings");
  const int64_t nnz = sb.nnz;
  std::vector<int64_t> rp(nb + 1, 0);
  std::vector<int32_t> col(nnz);
  std::vector<uint32_t> exc(nnz);
  SBDG_CHECK(hipMemcpyAsync(rp.data(), sb.rowptr.p, sizeof(int64_t) * (nb + 1), hipMemcpyDeviceToHost, st));
  if (nnz) {
    SBDG_CHECK(hipMemcpyAsync(col.data(), sb.col.p, sizeof(int32_t) * nnz, hipMemcpyDeviceToHost, st));
    SBDG_CHECK(hipMemcpyAsync(exc.data(), sb.exc.p, sizeof(uint32_t) * nnz, hipMemcpyDeviceToHost, st));
  }
  SBDG_CHECK(hipStreamSynchronize(st));
  const int64_t NP = std::max<int64_t>(1, (int64_t)L * (L - 1) / 2);
  const bool small = nnz / 2 < 32768;
  ab.nt = small ? ABR_NT_S : ABR_NT;
  ab.u = small ? ABR_U_S : ABR_U;
  constexpr int64_t CAP = AB_PAIR_COLS;  // columns of one staged alpha pair
  // equal chunks of an even number of columns (column pairs are loaded together)
  const int64_t nch = nb <= CAP ? 1 : (nb + CAP / 2 - 1) / (CAP / 2);
  const int64_t chunk = nch == 1 ? nb : ((nb + nch - 1) / nch + 1) / 2 * 2;
  ab.maxcols = nch == 1 ? nb : 2 * chunk;
  ab.sp = small && 4 * 16 * (ab.maxcols + 1) <= 40 * 1024 ? 4 : 1;
  auto group = [&](int64_t lo, int64_t hi) { return hi * (hi + 1) / 2 + lo; };  // chunks lo <= hi
  const int64_t ngroup = nch * (nch + 1) / 2;
  std::vector<int32_t> cnt((size_t)(ngroup * NP + 1), 0);
  auto each = [&](auto&& f) {  // every beta pair once: the entry whose bra holds the upper orbital
    for (int64_t x = 0; x < nb; ++x)
      for (int64_t q = rp[x]; q < rp[x + 1]; ++q) {
        const uint32_t e = exc[q], j = e & 63u, b = (e >> 6) & 63u;
        if (b < j) continue;
        const int64_t y = col[q], cx = x / chunk, cy = y / chunk;
        const int64_t lo = std::min(cx, cy), hi = std::max(cx, cy);
        // column -> LDS vector: the lower chunk first, then the upper one
        auto at = [&](int64_t c, int64_t k) { return (uint32_t)(c - k * chunk + (k == hi && hi != lo ? chunk : 0)); };
        f(group(lo, hi) * NP + ab_pair(b, j), at(x, cx) | (at(y, cy) << 15) | (((e >> 24) & 1u) << 30));
      }
  };
  each([&](int64_t k, uint32_t) { ++cnt[k + 1]; });
  for (size_t k = 1; k < cnt.size(); ++k) cnt[k] += cnt[k - 1];
  std::vector<uint32_t> sorted(std::max<int64_t>(nnz / 2, 1));
  {
    std::vector<int32_t> at(cnt.begin(), cnt.end() - 1);
    each([&](int64_t k, uint32_t w) { sorted[at[k]++] = w; });
  }
  const int64_t T = (int64_t)ab.nt * ab.u;
  std::vector<int4> tile;
  std::vector<int64_t> entoff;
  std::vector<uint32_t> ent;
  std::vector<uint16_t> rank;
  std::vector<int32_t> runptr(1, 0), runstart, runpair;
  for (int64_t hi = 0; hi < nch; ++hi)
    for (int64_t lo = 0; lo <= hi; ++lo) {
      const int64_t g = group(lo, hi);
      const int32_t nlo = (int32_t)(std::min(nb, (lo + 1) * chunk) - lo * chunk);
      const int32_t nhi = hi == lo ? 0 : (int32_t)(std::min(nb, (hi + 1) * chunk) - hi * chunk);
      int64_t p = 0;
      for (int64_t e = cnt[g * NP]; e < cnt[(g + 1) * NP]; e += T) {
        const int64_t f = std::min<int64_t>(e + T, cnt[(g + 1) * NP]);
        tile.push_back(make_int4((int)(lo * chunk), nlo, (int)(hi * chunk), nhi));
        entoff.push_back((int64_t)ent.size());
        const uint32_t z = (uint32_t)(nlo + nhi);
        ent.resize(entoff.back() + T, z | (z << 15));  // padding: the zero vector
        rank.resize(entoff.back() + T, 0xFFFF);
        order_pairs(sorted.data() + e, (int)(f - e), ent.data() + entoff.back(), rank.data() + entoff.back());
        for (int64_t x = 0, free = f - e; x < T; ++x)  // padding goes after the pairs
          if (rank[entoff.back() + x] == 0xFFFF) rank[entoff.back() + x] = (uint16_t)free++;
        for (int64_t x = e; x < f;) {
          while (cnt[g * NP + p + 1] <= x) ++p;
          runstart.push_back((int32_t)(x - e));
          runpair.push_back((int32_t)p);
          x = std::min<int64_t>(f, cnt[g * NP + p + 1]);
        }
        runstart.push_back((int32_t)(f - e));
        runpair.push_back(-1);
        runptr.push_back((int32_t)runstart.size());
      }
    }
  std::vector<int32_t> pairptr(NP + 1, 0), pairrun(std::max<size_t>(runpair.size(), 1));
  for (int32_t p : runpair)
    if (p >= 0) ++pairptr[p + 1];
  for (int64_t p = 0; p < NP; ++p) pairptr[p + 1] += pairptr[p];
  {
    std::vector<int32_t> at(pairptr.begin(), pairptr.end() - 1);
    for (size_t r = 0; r < runpair.size(); ++r)
      if (runpair[r] >= 0) pairrun[at[runpair[r]]++] = (int32_t)r;
  }
  ab.ntiles = (int64_t)tile.size();
  ab.nruns = (int64_t)runstart.size();
  ab.mem.put({{&ab.tile, tile}, {&ab.entoff, entoff}, {&ab.ent, ent}, {&ab.rank, rank}, {&ab.runptr, runptr},
              {&ab.runstart, runstart}, {&ab.pairptr, pairptr}, {&ab.pairrun, pairrun}});
  ab.built = true;
}

void rdm_compute(const RdmPlan& P, const double* W, double* WT, double* one, double* two, Arena& ar,
                 hipStream_t st) {
  const int L = P.L;
  const int64_t na = P.na, nb = P.nb, N = na * nb;
  const int64_t L2 = (int64_t)L * L, L4 = L2 * L2;
  SBDG_CHECK(hipMemsetAsync(one, 0, sizeof(double) * 2 * L2, st));
  SBDG_CHECK(hipMemsetAsync(two, 0, sizeof(double) * 4 * L4, st));
  if (N == 0) return;
  transpose_d(na, nb, W, WT, st);

  // diagonal: density correlators
  {
    WBuf<double> rsa(ar), Pa(ar), rsb(ar), Daa(ar), Dbb(ar), Dab(ar), dens(ar), part(ar);
    rsa.alloc(na);
    Pa.alloc(na * 64);
    rsb.alloc(nb);
    part.alloc(CORR_PARTS * L2);
    Daa.alloc(L2);
    Dbb.alloc(L2);
    Dab.alloc(L2);
    dens.alloc(2 * L);
    // rows of W: rsa[ia] = sum W^2, Pa[ia][j] = sum_ib W^2 n_j(ib)  (beta occupations)
    hipLaunchKernelGGL(k_occ_contract<true>, dim3((unsigned)na), dim3(RT), 0, st, nb, W, P.b, Pa.p, rsa.p);
    row_sumsq(WT, nb, na, rsb.p, st);
    auto corr = [&](int64_t n, const uint64_t* str, const double* w, const double* Y, double* D) {
      hipLaunchKernelGGL(k_corr, dim3(CORR_PARTS), dim3(RT), 0, st, n, L, str, w, Y, part.p);
      hipLaunchKernelGGL(k_corr_sum, dim3(nb_for(L2, 64)), dim3(64), 0, st, (int)L2, part.p, D);
    };
    corr(na, P.a, rsa.p, nullptr, Daa.p);
    corr(nb, P.b, rsb.p, nullptr, Dbb.p);
    corr(na, P.a, nullptr, Pa.p, Dab.p);
    // densities: diagonal of Daa/Dbb
    std::vector<double> hdaa(L2), hdbb(L2), hd(2 * L);
    SBDG_CHECK(hipMemcpyAsync(hdaa.data(), Daa.p, sizeof(double) * L2, hipMemcpyDeviceToHost, st));
    SBDG_CHECK(hipMemcpyAsync(hdbb.data(), Dbb.p, sizeof(double) * L2, hipMemcpyDeviceToHost, st));
    SBDG_CHECK(hipStreamSynchronize(st));
    for (int i = 0; i < L; ++i) {
      hd[2 * i] = hdaa[i * L + i];
      hd[2 * i + 1] = hdbb[i * L + i];
    }
    SBDG_CHECK(hipMemcpyAsync(dens.p, hd.data(), sizeof(double) * 2 * L, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_diag_slots, dim3(nb_for(L2, 64)), dim3(64), 0, st, L, dens.p, Daa.p, Dbb.p, Dab.p, one, two);
    SBDG_CHECK(hipGetLastError());
    SBDG_CHECK(hipStreamSynchronize(st));
  }
  // alpha pairs (beta spectators from the beta strings of the columns)
  SortedSingles ssa(ar), ssb(ar);
  sort_singles(*P.sa, L, ssa, ar, st);
  sort_singles(*P.sb, L, ssb, ar, st);
  singles_part(*P.sa, ssa, L, 0, W, nb, P.a, P.b, one, two, ar, st);
  doubles_part(*P.da, L, 0, W, nb, P.ca, P.a, two, ar, st);
  // beta pairs on the transposed vector (alpha spectators from the alpha strings)
  singles_part(*P.sb, ssb, L, 1, WT, na, P.b, P.a, one, two, ar, st);
  doubles_part(*P.db, L, 1, WT, na, P.cb, P.b, two, ar, st);

  // alpha-beta
  const Table& sa = *P.sa;
  const AbPairs& ab = *P.ab;
  if (sa.nnz > 0 && P.sb->nnz > 0) {
    // segments of at most plen alpha pairs: about 4,096 workgroups where there is work for them
    int64_t plen = std::min<int64_t>(1024, std::max<int64_t>(32, sa.nnz / 2 * ab.ntiles / 4096));
    int64_t longest = 0;
    for (int key = 0; key < (int)L2; ++key) longest = std::max<int64_t>(longest, ssa.hk[key + 1] - ssa.hk[key]);
    while (plen < longest && (longest + plen - 1) / plen * ab.nruns * 16 > RDM_PART_BYTES) plen *= 2;
    KeySegments K(ar);
    key_segments(ssa.hk, L, plen, std::max<int64_t>(1, RDM_PART_BYTES / (16 * std::max<int64_t>(1, ab.nruns))), K, st);
    WBuf<double> part(ar);
    part.alloc((size_t)K.widest * ab.nruns * 2);
    const bool many = ab.nt == ABR_NT;
    const size_t lds = std::max<size_t>(16 * (size_t)(many ? 2 : ab.sp) * (size_t)(ab.maxcols + 1),
                                        8 * (size_t)ab.nt * ab.u);
    AbRdmArgs A{nb, ab.nruns, ab.ntiles, 0, ab.tile, ab.entoff, ab.ent, ab.rank, ab.runptr, ab.runstart,
                nullptr, ssa.pia.p, ssa.pja.p, W, part.p};
    for (const auto& bt : K.batch) {
      const int64_t s0 = K.kseg[bt.first], ns = K.kseg[bt.second] - s0;
      const int64_t nblk = (ns + 7) / 8 * 8 * ab.ntiles;
      if (nblk > (int64_t)INT32_MAX) throw Error(SBDG_ERR_LIMIT, "grid too large");
      A.nseg = ns;
      A.segptr = K.dsegs + 2 * s0;
      const dim3 g((unsigned)nblk), t(ab.nt);
      if (many) hipLaunchKernelGGL(k_ab_rdm, g, t, lds, st, A);
      else if (ab.sp > 1) hipLaunchKernelGGL(k_ab_rdm_small<4>, g, t, lds, st, A);
      else hipLaunchKernelGGL(k_ab_rdm_small<1>, g, t, lds, st, A);
      hipLaunchKernelGGL(k_ab_slots, dim3((unsigned)(bt.second - bt.first)), dim3(256), 0, st, L,
                         K.dkeys + bt.first, K.dkseg + bt.first, s0, ab.nruns, ab.pairptr, ab.pairrun, part.p, two);
    }
    SBDG_CHECK(hipGetLastError());
    SBDG_CHECK(hipStreamSynchronize(st));
  }
}

void rdm_backward(const double* d_one, const double* d_two, int L, double g, double* d_dh, double* d_deri,
                  hipStream_t st) {
  const int64_t L4 = (int64_t)L * L * L * L;
  hipLaunchKernelGGL(k_backward, dim3(nb_for(L4, 256)), dim3(256), 0, st, L, d_one, d_two, g, d_dh, d_deri);
  SBDG_CHECK(hipGetLastError());
}

}  // namespace sbdg
