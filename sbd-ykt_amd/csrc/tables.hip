// Excitation tables and the diagonal, built on the device.
//
// Tables (replacing GenerateExcitation + MakeSmartHelper, tpb/helper.h:132-197,367-437):
// for every bra string the kets at XOR-popcount 2 (singles) and 4 (doubles), ascending.
// One workgroup per bra row scans the string set twice (count, then fill with a
// ballot/prefix so the ascending order survives), then a per-entry pass derives the
// orbitals with ctz and the separated-order sign with a masked popcount, and evaluates
// the spin-string-only part of the Slater-Condon element (determinants.h:423-465).
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "sbdg_internal.h"

namespace sbdg {

namespace {

constexpr int TB = 256;  // threads per row workgroup

__device__ inline uint64_t between_mask(int x, int y) {
  // bits strictly between orbitals x and y (x != y)
  int lo = x < y ? x : y, hi = x < y ? y : x;
  uint64_t below_hi = (hi >= 64) ? ~0ull : ((1ull << hi) - 1ull);
  uint64_t upto_lo = (lo + 1 >= 64) ? ~0ull : ((1ull << (lo + 1)) - 1ull);
  return below_hi & ~upto_lo;
}

__device__ inline int block_sum(int v, int* sh) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  int t = 0;
  if (threadIdx.x == 0) {
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += sh[w];
    sh[0] = t;
  }
  __syncthreads();
  t = sh[0];
  __syncthreads();
  return t;
}

__global__ void __launch_bounds__(TB) k_count(const uint64_t* __restrict__ s, int64_t n,
                                              int64_t* __restrict__ cs, int64_t* __restrict__ cd) {
  __shared__ int sh[TB / 64];
  const int64_t i = blockIdx.x;
  const uint64_t si = s[i];
  int ns = 0, nd = 0;
  for (int64_t j = threadIdx.x; j < n; j += TB) {
    int d = __popcll(si ^ s[j]);
    ns += (d == 2);
    nd += (d == 4);
  }
  ns = block_sum(ns, sh);
  nd = block_sum(nd, sh);
  if (threadIdx.x == 0) {
    cs[i] = ns;
    cd[i] = nd;
  }
}

// exclusive scan of cnt[0..n) into rp[0..n] (one workgroup, fixed order)
__global__ void __launch_bounds__(1024) k_scan(const int64_t* __restrict__ cnt, int64_t n,
                                               int64_t* __restrict__ rp) {
  __shared__ int64_t part[1024];
  const int t = threadIdx.x;
  const int64_t per = (n + 1023) / 1024;
  const int64_t b = t * per, e = min(n, b + per);
  int64_t s = 0;
  for (int64_t k = b; k < e; ++k) s += cnt[k];
  part[t] = s;
  __syncthreads();
  if (t == 0) {
    int64_t acc = 0;
    for (int k = 0; k < 1024; ++k) {
      int64_t v = part[k];
      part[k] = acc;
      acc += v;
    }
  }
  __syncthreads();
  int64_t acc = part[t];
  for (int64_t k = b; k < e; ++k) {
    rp[k] = acc;
    acc += cnt[k];
  }
  if (e == n && b < e) rp[n] = acc;
  if (n == 0 && t == 0) rp[0] = 0;
}

__global__ void __launch_bounds__(TB) k_fill(const uint64_t* __restrict__ s, int64_t n,
                                             const int64_t* __restrict__ rps,
                                             const int64_t* __restrict__ rpd,
                                             int32_t* __restrict__ cols, int32_t* __restrict__ cold) {
  __shared__ int wcs[TB / 64], wcd[TB / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t i = blockIdx.x;
  const uint64_t si = s[i];
  int64_t ps = rps[i], pd = rpd[i];
  const uint64_t lt = (1ull << lane) - 1ull;
  for (int64_t base = 0; base < n; base += TB) {
    const int64_t j = base + threadIdx.x;
    int d = (j < n) ? __popcll(si ^ s[j]) : 0;
    uint64_t ms = __ballot(d == 2), md = __ballot(d == 4);
    if (lane == 0) {
      wcs[wid] = __popcll(ms);
      wcd[wid] = __popcll(md);
    }
    __syncthreads();
    int offs = 0, offd = 0, tots = 0, totd = 0;
    for (int w = 0; w < TB / 64; ++w) {
      if (w < wid) {
        offs += wcs[w];
        offd += wcd[w];
      }
      tots += wcs[w];
      totd += wcd[w];
    }
    if (d == 2) cols[ps + offs + __popcll(ms & lt)] = (int32_t)j;
    if (d == 4) cold[pd + offd + __popcll(md & lt)] = (int32_t)j;
    ps += tots;
    pd += totd;
    __syncthreads();
  }
}

__device__ inline double eri4(const double* __restrict__ eri, int L, int p, int q, int r, int s) {
  return eri[(((int64_t)p * L + q) * L + r) * L + s];
}

// singles: bra-only a, ket-only i; sign from the ket string between them;
// value sign*(h_ai + sum over occ(ket)\{i} of [(ai|kk) - (ak|ki)])
__global__ void __launch_bounds__(TB) k_single(const uint64_t* __restrict__ s, int L,
                                               const double* __restrict__ h1,
                                               const double* __restrict__ eri,
                                               const int64_t* __restrict__ rp,
                                               const int32_t* __restrict__ col,
                                               uint32_t* __restrict__ exc, double* __restrict__ val,
                                               float* __restrict__ val32) {
  const int64_t r = blockIdx.x;
  const uint64_t bra = s[r];
  for (int64_t q = rp[r] + threadIdx.x; q < rp[r + 1]; q += TB) {
    const uint64_t ket = s[col[q]];
    const uint64_t bo = bra & ~ket, ko = ket & ~bra;
    const int a = __builtin_ctzll(bo), i = __builtin_ctzll(ko);
    const int neg = __popcll(ket & between_mask(i, a)) & 1;
    double v = h1[a * L + i];
    uint64_t occ = ket & ~(1ull << i);
    while (occ) {
      int k = __builtin_ctzll(occ);
      occ &= occ - 1;
      v += eri4(eri, L, a, i, k, k) - eri4(eri, L, a, k, k, i);
    }
    v = neg ? -v : v;
    exc[q] = (uint32_t)i | ((uint32_t)a << 6) | ((uint32_t)neg << 24);
    val[q] = v;
    val32[q] = (float)v;
  }
}

// doubles: ket-only I<J, bra-only A<B; sign by the two-pair rule of TwoExcite
// (determinants.h:447-465) applied to the ket string; value sign*((AI|BJ)-(AJ|BI))
__global__ void __launch_bounds__(TB) k_double(const uint64_t* __restrict__ s, int L,
                                               const double* __restrict__ eri,
                                               const int64_t* __restrict__ rp,
                                               const int32_t* __restrict__ col,
                                               uint32_t* __restrict__ exc, double* __restrict__ val,
                                               float* __restrict__ val32) {
  const int64_t r = blockIdx.x;
  const uint64_t bra = s[r];
  for (int64_t q = rp[r] + threadIdx.x; q < rp[r + 1]; q += TB) {
    const uint64_t ket = s[col[q]];
    uint64_t bo = bra & ~ket, ko = ket & ~bra;
    const int A = __builtin_ctzll(bo);
    bo &= bo - 1;
    const int B = __builtin_ctzll(bo);
    const int I = __builtin_ctzll(ko);
    ko &= ko - 1;
    const int J = __builtin_ctzll(ko);
    int neg = (__popcll(ket & between_mask(I, A)) + __popcll(ket & between_mask(J, B))) & 1;
    if (A > J || B < I) neg ^= 1;
    double v = eri4(eri, L, A, I, B, J) - eri4(eri, L, A, J, B, I);
    v = neg ? -v : v;
    exc[q] = (uint32_t)I | ((uint32_t)J << 6) | ((uint32_t)A << 12) | ((uint32_t)B << 18) |
             ((uint32_t)neg << 24);
    val[q] = v;
    val32[q] = (float)v;
  }
}

__device__ inline int32_t single_jai(uint32_t e, int L) {
  const int32_t p = (int32_t)((e >> 6) & 63u) * L + (int32_t)(e & 63u);  // bra-only * L + ket-only
  return ((e >> 24) & 1u) ? -(p + 1) : (p + 1);
}

__global__ void k_jai(int64_t nnz, int L, const uint32_t* __restrict__ exc, int32_t* __restrict__ jai) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < nnz) jai[q] = single_jai(exc[q], L);
}

__global__ void k_merge(int64_t n, int L, const int64_t* __restrict__ rps, const int32_t* __restrict__ cs,
                        const double* __restrict__ vs, const float* __restrict__ vs32,
                        const uint32_t* __restrict__ es,
                        const int64_t* __restrict__ rpd, const int32_t* __restrict__ cd,
                        const double* __restrict__ vd, const float* __restrict__ vd32,
                        int64_t* __restrict__ rpm, int64_t* __restrict__ mid, int32_t* __restrict__ cm,
                        double* __restrict__ vm, float* __restrict__ vm32, int32_t* __restrict__ jm) {
  const int64_t r = blockIdx.x;
  const int64_t b = rps[r] + rpd[r];
  const int64_t ns = rps[r + 1] - rps[r], nd = rpd[r + 1] - rpd[r];
  if (threadIdx.x == 0) {
    rpm[r] = b;
    mid[r] = b + ns;
    if (r == n - 1) rpm[n] = rps[n] + rpd[n];
  }
  for (int64_t k = threadIdx.x; k < ns + nd; k += blockDim.x) {
    if (k < ns) {
      cm[b + k] = cs[rps[r] + k];
      vm[b + k] = vs[rps[r] + k];
      vm32[b + k] = vs32[rps[r] + k];
      jm[b + k] = single_jai(es[rps[r] + k], L);
    } else {
      cm[b + k] = cd[rpd[r] + k - ns];
      vm[b + k] = vd[rpd[r] + k - ns];
      vm32[b + k] = vd32[rpd[r] + k - ns];
      jm[b + k] = 0;
    }
  }
}

// J[(p+1)*n + r] = sum_{o in occ(s[r])} eri[p*L^2 + o*L + o]; row 0 zero
__global__ void k_occ_table(const uint64_t* __restrict__ s, int64_t n, int L, const double* __restrict__ eri,
                            double* __restrict__ J, float* __restrict__ J32) {
  const int64_t LL = (int64_t)L * L;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (LL + 1) * n) return;
  const int64_t p = t / n, r = t - p * n;
  double v = 0.0;
  if (p > 0) {
    const double* e = eri + (p - 1) * LL;
    uint64_t y = s[r];
    while (y) {
      const int o = __builtin_ctzll(y);
      y &= y - 1;
      v += e[(int64_t)o * L + o];
    }
  }
  J[t] = v;
  J32[t] = (float)v;
}

// memberships: thread t -> (string r, electron pair q); key = core bits, value =
// r | P(a,b) << 32 | neg << 63 with eps = (-1)^(#core below a + #core below b)
__global__ void k_core_enum(const uint64_t* __restrict__ s, int64_t n, int nel, uint64_t* __restrict__ key,
                            uint64_t* __restrict__ val) {
  const int64_t npp = (int64_t)nel * (nel - 1) / 2;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * npp) return;
  const int64_t r = t / npp;
  int q = (int)(t % npp);
  int j = 1;
  while ((j + 1) * j / 2 <= q) ++j;  // positions i < j of the occupied orbitals
  const int i = q - j * (j - 1) / 2;
  uint64_t x = s[r];
  int a = -1, b = -1;
  for (int pos = 0; x; ++pos) {
    const int o = __builtin_ctzll(x);
    x &= x - 1;
    if (pos == i) a = o;
    if (pos == j) b = o;
  }
  const uint64_t core = s[r] & ~(1ull << a) & ~(1ull << b);
  const int neg = (__popcll(core & ((1ull << a) - 1ull)) + __popcll(core & ((1ull << b) - 1ull))) & 1;
  key[t] = core;
  val[t] = (uint64_t)r | ((uint64_t)(b * (b - 1) / 2 + a) << 32) | ((uint64_t)neg << 63);
}

// W[P*npair+Q] = (AI|BJ) - (AJ|BI) for P=(A<B), Q=(I<J) disjoint, 0 otherwise
__global__ void k_pair_int(const double* __restrict__ eri, int L, int64_t npair, double* __restrict__ W,
                           float* __restrict__ W32) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= npair * npair) return;
  const int64_t P = t / npair, Q = t % npair;
  auto unpair = [](int64_t p, int& lo, int& hi) {
    int b = 1;
    while ((int64_t)(b + 1) * b / 2 <= p) ++b;
    hi = b;
    lo = (int)(p - (int64_t)b * (b - 1) / 2);
  };
  int A, B, I, J;
  unpair(P, A, B);
  unpair(Q, I, J);
  double v = 0.0;
  if (A != I && A != J && B != I && B != J) v = eri4(eri, L, A, I, B, J) - eri4(eri, L, A, J, B, I);
  W[t] = v;
  W32[t] = (float)v;
}

// The direct pairs of member z of a small core, from its place in the table on: every member of the
// core, in order, whose pair shares no orbital with z's; value eps_x eps_y W[P_x][P_y].  mem: row,
// orbitals of the pair (six bits each, bit 31 the sign), first member of the core and their number.
__global__ void k_direct_fill(const int4* __restrict__ mem, const int64_t* __restrict__ at, int64_t n, int L,
                              const double* __restrict__ eri, int32_t* __restrict__ col, double* __restrict__ val,
                              float* __restrict__ val32) {
  const int64_t z = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (z >= n) return;
  const int4 x = mem[z];
  const int A = x.y & 63, B = (x.y >> 6) & 63;
  int64_t q = at[z];
  for (int k = 0; k < x.w; ++k) {
    const int4 y = mem[x.z + k];
    const int I = y.y & 63, J = (y.y >> 6) & 63;
    if (A == I || A == J || B == I || B == J) continue;
    double v = eri4(eri, L, A, I, B, J) - eri4(eri, L, A, J, B, I);
    if ((x.y ^ y.y) < 0) v = -v;
    col[q] = y.x;
    val[q] = v;
    val32[q] = (float)v;
    ++q;
  }
}

__global__ void k_pair_slices(const double* __restrict__ eri, int L, int64_t npair, double* __restrict__ Vt,
                              float* __restrict__ Vt32) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= npair * npair) return;
  auto unpair = [](int64_t p, int& lo, int& hi) {
    int b = 1;
    while ((int64_t)(b + 1) * b / 2 <= p) ++b;
    hi = b;
    lo = (int)(p - (int64_t)b * (b - 1) / 2);
  };
  int a, i, b, j;
  unpair(t / npair, i, a);
  unpair(t % npair, j, b);
  const double v = eri4(eri, L, a, i, b, j);
  Vt[t] = v;
  Vt32[t] = (float)v;
}

// per-string diagonal parts: E[s] = sum_{i in s} h_ii + sum_{i<j in s} [(ii|jj)-(ij|ji)]
__global__ void k_strdiag(const uint64_t* __restrict__ s, int64_t n, int L,
                          const double* __restrict__ h1, const double* __restrict__ eri,
                          double* __restrict__ E) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  uint64_t x = s[t];
  double e = 0.0;
  while (x) {
    int i = __builtin_ctzll(x);
    x &= x - 1;
    e += h1[i * L + i];
    uint64_t y = x;
    while (y) {
      int j = __builtin_ctzll(y);
      y &= y - 1;
      e += eri4(eri, L, i, i, j, j) - eri4(eri, L, i, j, j, i);
    }
  }
  E[t] = e;
}

// hii[ia,ib] = core + Ea[ia] + Eb[ib] + sum_{i in a, j in b} (ii|jj)
__global__ void __launch_bounds__(TB) k_hii(const uint64_t* __restrict__ a, const uint64_t* __restrict__ b,
                                            int64_t nb, int L, double core,
                                            const double* __restrict__ Ea,
                                            const double* __restrict__ Eb,
                                            const double* __restrict__ eri, double* __restrict__ hii) {
  __shared__ double J[64];
  const int64_t ia = blockIdx.x;
  const uint64_t A = a[ia];
  if (threadIdx.x < L) {
    double v = 0.0;
    uint64_t x = A;
    while (x) {
      int i = __builtin_ctzll(x);
      x &= x - 1;
      v += eri4(eri, L, i, i, threadIdx.x, threadIdx.x);
    }
    J[threadIdx.x] = v;
  }
  __syncthreads();
  const double base = core + Ea[ia];
  for (int64_t ib = threadIdx.x; ib < nb; ib += TB) {
    uint64_t x = b[ib];
    double v = base + Eb[ib];
    while (x) {
      int j = __builtin_ctzll(x);
      x &= x - 1;
      v += J[j];
    }
    hii[ia * nb + ib] = v;
  }
}

inline unsigned blocks_for(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

}  // namespace

void build_table(const uint64_t* d_str, int64_t n, int L, const double* d_h1, const double* d_eri,
                 Table& ts, Table& td, hipStream_t st) {
  ts.n = td.n = n;
  DBuf<int64_t> cs, cd;
  cs.alloc(n);
  cd.alloc(n);
  ts.rowptr.alloc(n + 1);
  td.rowptr.alloc(n + 1);
  if (n > 0) {
    hipLaunchKernelGGL(k_count, dim3((unsigned)n), dim3(TB), 0, st, d_str, n, cs.p, cd.p);
    SBDG_CHECK(hipGetLastError());
  }
  hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, st, cs.p, n, ts.rowptr.p);
  hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, st, cd.p, n, td.rowptr.p);
  SBDG_CHECK(hipGetLastError());
  SBDG_CHECK(hipMemcpyAsync(&ts.nnz, ts.rowptr.p + n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  SBDG_CHECK(hipMemcpyAsync(&td.nnz, td.rowptr.p + n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  SBDG_CHECK(hipStreamSynchronize(st));
  if (ts.nnz >= (int64_t)INT32_MAX || td.nnz >= (int64_t)INT32_MAX)
    throw Error(SBDG_ERR_LIMIT, "excitation table beyond 2^31 entries");
  for (Table* t : {&ts, &td}) {
    t->col.alloc(std::max<int64_t>(t->nnz, 1));
    t->exc.alloc(std::max<int64_t>(t->nnz, 1));
    t->val.alloc(std::max<int64_t>(t->nnz, 1));
    t->val32.alloc(std::max<int64_t>(t->nnz, 1));
  }
  if (n > 0) {
    hipLaunchKernelGGL(k_fill, dim3((unsigned)n), dim3(TB), 0, st, d_str, n, ts.rowptr.p, td.rowptr.p,
                       ts.col.p, td.col.p);
    hipLaunchKernelGGL(k_single, dim3((unsigned)n), dim3(TB), 0, st, d_str, L, d_h1, d_eri, ts.rowptr.p,
                       ts.col.p, ts.exc.p, ts.val.p, ts.val32.p);
    hipLaunchKernelGGL(k_double, dim3((unsigned)n), dim3(TB), 0, st, d_str, L, d_eri, td.rowptr.p, td.col.p,
                       td.exc.p, td.val.p, td.val32.p);
    SBDG_CHECK(hipGetLastError());
  }
  SBDG_CHECK(hipStreamSynchronize(st));
}

void build_spmm(const Table& s, const Table& d, SpmmTable& m, int L, hipStream_t st, bool with_doubles) {
  if (!with_doubles) {  // singles only: copy the singles CSR
    m.n = s.n;
    m.nnz = s.nnz;
    m.rowptr.alloc(m.n + 1);
    m.mid.alloc(std::max<int64_t>(m.n, 1));
    m.col.alloc(std::max<int64_t>(m.nnz, 1));
    m.val.alloc(std::max<int64_t>(m.nnz, 1));
    m.val32.alloc(std::max<int64_t>(m.nnz, 1));
    m.jai.alloc(std::max<int64_t>(m.nnz, 1));
    SBDG_CHECK(hipMemcpyAsync(m.rowptr.p, s.rowptr.p, sizeof(int64_t) * (m.n + 1), hipMemcpyDeviceToDevice, st));
    SBDG_CHECK(hipMemcpyAsync(m.mid.p, s.rowptr.p + 1, sizeof(int64_t) * m.n, hipMemcpyDeviceToDevice, st));
    if (m.nnz) {
      SBDG_CHECK(hipMemcpyAsync(m.col.p, s.col.p, sizeof(int32_t) * m.nnz, hipMemcpyDeviceToDevice, st));
      SBDG_CHECK(hipMemcpyAsync(m.val.p, s.val.p, sizeof(double) * m.nnz, hipMemcpyDeviceToDevice, st));
      SBDG_CHECK(hipMemcpyAsync(m.val32.p, s.val32.p, sizeof(float) * m.nnz, hipMemcpyDeviceToDevice, st));
      hipLaunchKernelGGL(k_jai, dim3(blocks_for(m.nnz, 256)), dim3(256), 0, st, m.nnz, L, s.exc.p, m.jai.p);
      SBDG_CHECK(hipGetLastError());
    }
    SBDG_CHECK(hipStreamSynchronize(st));
    return;
  }
  m.n = s.n;
  m.nnz = s.nnz + d.nnz;
  m.rowptr.alloc(m.n + 1);
  m.mid.alloc(std::max<int64_t>(m.n, 1));
  m.col.alloc(std::max<int64_t>(m.nnz, 1));
  m.val.alloc(std::max<int64_t>(m.nnz, 1));
  m.val32.alloc(std::max<int64_t>(m.nnz, 1));
  m.jai.alloc(std::max<int64_t>(m.nnz, 1));
  if (m.n > 0) {
    hipLaunchKernelGGL(k_merge, dim3((unsigned)m.n), dim3(TB), 0, st, m.n, L, s.rowptr.p, s.col.p, s.val.p,
                       s.val32.p, s.exc.p, d.rowptr.p, d.col.p, d.val.p, d.val32.p, m.rowptr.p, m.mid.p, m.col.p,
                       m.val.p, m.val32.p, m.jai.p);
    SBDG_CHECK(hipGetLastError());
  } else {
    SBDG_CHECK(hipMemsetAsync(m.rowptr.p, 0, sizeof(int64_t), st));
  }
}

// Alpha-beta launch geometry for rows of nb columns: nt threads, m columns per thread, so that
// one workgroup covers a whole row where it can (a second column tile stages every ket row
// again: norb=36, 4,000 x 24,000 9.2 ms with one tile, 11.7 with two), s groups of ket rows
// staged per barrier, and the ket columns cut into equal chunks that fill the LDS share.
//  * up to 128 columns the slices are most of what is staged: 64 threads for up to 400 slice
//    vectors, 128 up to 1,000, 256 beyond, and many workgroups on a CU (256 threads of four groups
//    against one workgroup of 64 threads per whole row and these: norb=26, 20,000 x 64 FP64 1,054 /
//    654 / 420 us, FP32 769 / 355 / 252, 20,000 x 4 800 / 537 / 274 and 611 / 290 / 161; norb=16,
//    4,368 x 20 193 / 101 / 93; norb=36, 5,000 x 64 164 / 772 / 102; norb=58, 3,000 x 20
//    170 / 700 / 133);
//  * up to 1,024 columns: 256 threads and several groups per barrier while a few workgroups
//    still fit a CU (norb=26, 2,000 x 1,000: 259 us with one group, 214 with two; norb=58,
//    600 x 400: 115 / 104 / 249 us with one, two and four);
//  * up to 6,000: 512 threads and half the LDS, so that two workgroups share a CU and one
//    stages while the other computes (FP64, against 1,024 threads and all of it: norb=26,
//    2,801 x 2,749 0.93 and 1.21 ms, norb=36, 5,001 x 4,999 1.65 and 1.97 ms, 1,000 x 7,000
//    equal, 800 x 10,000 0.72 and 0.71, 500 x 15,000 1.01 and 0.82: more chunks, each with its
//    slices and part-filled batches);
//  * beyond: one workgroup per CU with all of its LDS.  FP64 accumulators bound the columns
//    per thread: 1,024 threads (four waves per SIMD, 128 VGPRs) hold 24, 768 threads (three
//    waves, 168 VGPRs) 53 (norb=58, 40,000^2 in one tile 256 ms, in two tiles of 1,024 threads
//    316); FP32 holds 48 at 1,024 threads.  Wider rows take several tiles.
AbGeometry ab_geometry(int64_t nb, int L, int elem) {
  AbGeometry g;
  const int64_t kb = ab_slice_span(L);
  const bool half = nb <= 6000;
  g.nt = nb <= 1024 ? 256 : half ? 512 : 1024;
  g.s = 1;
  if (nb <= 128) {
    g.nt = kb <= 400 ? 64 : kb <= 1000 ? 128 : 256;
    g.s = kb <= 1000 ? 2 : 1;
  } else if (nb <= 1024) {
    const int64_t grp = 16 * (kb + nb + 1);
    g.s = nb <= 512 && 4 * grp <= 48 * 1024 ? 4 : 2 * grp <= 80 * 1024 ? 2 : 1;
  }
  if (elem == 8 && nb > 24 * 1024) g.nt = 768;
  const int64_t maxchunk = (half ? 80 : 160) * 1024 / 16 / g.s - kb - 1;
  const int64_t nch = std::max<int64_t>(1, (nb + maxchunk - 1) / maxchunk);
  g.chunk = std::max<int64_t>(1, (nb + nch - 1) / nch);
  static const int m64[] = {1, 2, 0}, m128[] = {1, 0}, m256[] = {1, 2, 4, 0}, m512[] = {4, 6, 8, 10, 12, 0},
                   m1024d[] = {8, 12, 16, 20, 24, 0}, m1024f[] = {8, 12, 16, 20, 24, 40, 48, 0},
                   m768[] = {40, 48, 53, 0};
  const int* ms = g.nt == 64 ? m64 : g.nt == 128 ? m128 : g.nt == 256 ? m256 : g.nt == 512 ? m512 : g.nt == 768 ? m768
                  : elem == 4 ? m1024f : m1024d;
  g.m = 0;
  for (int i = 0; ms[i]; ++i) {
    g.m = ms[i];
    if (nb <= (int64_t)ms[i] * g.nt) break;
  }
  return g;
}

// Segment length: an equal share of all alpha singles (times column tiles) over two workgroups
// per CU, between 8 and 64 singles, in multiples of 8 (whole staging groups in both precisions);
// longer where the partial rows would outgrow AB_PART_BYTES.  Longest first, so that the last
// workgroups to start are short.  Lengths of 16, 32 and 64 measure alike at norb=26, 4,000^2
// (2.63 / 2.63 / 2.61 ms); one segment per row 2.61 there, but 0.68 against 1.63 ms at norb=36,
// 3,600 x 3,500 in FP32.
void build_segments(const Table& sa, int64_t nb, int64_t ntiles, AbSegments& g, hipStream_t st) {
  const int64_t na = sa.n;
  std::vector<int64_t> rp(na + 1, 0);
  SBDG_CHECK(hipMemcpyAsync(rp.data(), sa.rowptr.p, sizeof(int64_t) * (na + 1), hipMemcpyDeviceToHost, st));
  SBDG_CHECK(hipStreamSynchronize(st));
  int64_t len = std::min<int64_t>(64, std::max<int64_t>(8, (rp[na] * ntiles / 512 + 7) / 8 * 8));
  auto extra = [&](int64_t l) {
    int64_t e = 0;
    for (int64_t r = 0; r < na; ++r) e += std::max<int64_t>(0, (rp[r + 1] - rp[r] - 1) / l);
    return e;
  };
  while (extra(len) * nb * (int64_t)sizeof(double) > AB_PART_BYTES) len *= 2;
  // every row's segments of l singles, the last one shorter: the row's first writes sigma (dst -1)
  auto each = [&](auto&& f) {
    int32_t np = 0;
    for (int64_t r = 0; r < na; ++r) {
      int64_t q = rp[r];
      do {
        const int64_t end = std::min(rp[r + 1], q + len);
        f(r, q, end, q == rp[r] ? -1 : np++);
        q = end;
      } while (q < rp[r + 1]);
    }
  };
  std::vector<int64_t> at(std::min<int64_t>(len, rp[na]) + 2, 0);  // by decreasing length
  auto place = [&](int64_t l) -> int64_t& { return at[at.size() - 1 - l]; };
  int32_t np = 0;
  std::vector<int32_t> jrow, jptr(1, 0);
  each([&](int64_t r, int64_t q, int64_t end, int32_t dst) {
    ++place(end - q);
    if (dst < 0) return;
    np = dst + 1;
    if (jrow.empty() || jrow.back() != r) {
      jrow.push_back((int32_t)r);
      jptr.push_back(0);
    }
    jptr.back() = np;
  });
  int64_t nseg = 0;
  for (int64_t& x : at) {
    const int64_t k = x;
    x = nseg;
    nseg += k;
  }
  std::vector<int32_t> row(nseg), to(nseg);
  std::vector<int64_t> q(2 * nseg);
  each([&](int64_t r, int64_t q0, int64_t q1, int32_t dst) {
    const int64_t k = place(q1 - q0)++;
    row[k] = (int32_t)r;
    to[k] = dst;
    q[2 * k] = q0;
    q[2 * k + 1] = q1;
  });
  g.nseg = nseg;
  g.npart = np;
  g.njoin = (int64_t)jrow.size();
  g.mem.put({{&g.row, row}, {&g.dst, to}, {&g.q, q}, {&g.jrow, jrow}, {&g.jptr, jptr}});
  g.part.alloc(std::max<int64_t>((int64_t)np * nb, 1));
}

// Order of the entries of the lanes of one (group, chunk) block, step by step, so that the 16
// lanes that a 16-byte read serves together (LDS16_LANE) read distinct LDS slots of 16 in both
// the ket-row array and the integral array; equal addresses broadcast and cost nothing.
// (Against 32 contiguous lanes over the 16 slots: norb=36, 20,000^2 FP64 68.1 -> 64.4 ms, FP32
// 37.1 -> 35.8, norb=26, 2,801 x 2,749 0.91 -> 0.81.)  Padding (the zero slot, pair 0) may be
// placed at any step while a lane has slack.  Greedy: at each step the lanes with least slack choose first,
// each taking the entry that adds the fewest new addresses to slots already in use.
// lists[l] holds lane l's entries (ket byte address | pair << 18 | sign << 31); out gets
// K*64.  Slots count 16-byte LDS vectors: the pair's slice vector is the pair index, the
// ket's is its byte address / 16.
static void schedule_block(std::vector<std::vector<uint32_t>>& lists, int K, uint32_t pad, uint32_t* out) {
  constexpr int P = 16, S = 16;
  struct Use {
    uint32_t addr[8];
    int n;
  };
  std::vector<int> rem(64), order(P);
  for (int l = 0; l < 64; ++l) rem[l] = (int)lists[l].size();
  auto cost1 = [](const Use& u, uint32_t a) {
    for (int i = 0; i < u.n; ++i)
      if (u.addr[i] == a) return 0;
    return u.n;
  };
  auto add1 = [](Use& u, uint32_t a) {
    for (int i = 0; i < u.n; ++i)
      if (u.addr[i] == a) return;
    if (u.n < 8) u.addr[u.n++] = a;
  };
  std::vector<Use> uc(S), uv(S);
  for (int p0 = 0; p0 < 64; p0 += P) {
    for (int e = 0; e < K; ++e) {
      for (int x = 0; x < S; ++x) uc[x].n = uv[x].n = 0;
      for (int i = 0; i < P; ++i) order[i] = (p0 & 32) + LDS16_LANE[(p0 & 31) + i];
      std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return rem[a] > rem[b]; });
      for (int l : order) {
        const int slack = (K - e) - rem[l];
        auto& ls = lists[l];
        int best = -1, bc = 1 << 30;
        for (int j = 0; j < rem[l]; ++j) {
          const uint32_t w = ls[j];
          const uint32_t ca = (w & 0x3FFFFu) >> 4;
          const uint32_t va = (w >> 18) & 0xFFFu;
          const int cst = cost1(uc[ca % S], ca) + cost1(uv[va % S], va);
          if (cst < bc) {
            bc = cst;
            best = j;
            if (cst == 0) break;
          }
        }
        uint32_t w = pad;
        if (slack > 0) {
          const uint32_t ca = (pad & 0x3FFFFu) >> 4, va = (pad >> 18) & 0xFFFu;
          const int cst = cost1(uc[ca % S], ca) + cost1(uv[va % S], va);
          if (best < 0 || cst < bc) best = -1;
        }
        if (best >= 0) {
          w = ls[best];
          ls[best] = ls[rem[l] - 1];  // order of the rest does not matter
          --rem[l];
        }
        const uint32_t ca = (w & 0x3FFFFu) >> 4, va = (w >> 18) & 0xFFFu;
        add1(uc[ca % S], ca);
        add1(uv[va % S], va);
        out[(size_t)e * 64 + l] = w;
      }
    }
  }
}

void build_ell(const Table& sb, int L, int prec_bytes, EllTable& e, hipStream_t st) {
  const int64_t nb = sb.n;
  const AbGeometry geo = ab_geometry(nb, L, prec_bytes);
  const int64_t chunk = geo.chunk;
  if (L > 64) throw Error(SBDG_ERR_LIMIT, "norb beyond 64");
  e.kbase = ab_slice_span(L);
  if (16 * (e.kbase + chunk + 1) > (1 << 18)) throw Error(SBDG_ERR_LIMIT, "alpha-beta LDS beyond 256 KiB");
  e.chunk = chunk;
  e.nch = (int)std::max<int64_t>(1, (nb + chunk - 1) / chunk);
  e.nt = geo.nt;
  e.m = geo.m;
  e.s = geo.s;
  const int64_t tw = (int64_t)e.nt * e.m;
  e.ntiles = std::max<int64_t>(1, (nb + tw - 1) / tw);
  const int64_t npos = e.ntiles * tw;
  e.groups = npos / 64;
  const int nch = e.nch;
  const int64_t ng = e.groups * nch;
  // host copies of the beta singles
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
  // entries of column ib in chunk k: its singles with ket in the chunk
  std::vector<int32_t> cnt((size_t)nb * nch, 0);
  for (int64_t ib = 0; ib < nb; ++ib)
    for (int64_t q = rp[ib]; q < rp[ib + 1]; ++q) ++cnt[(size_t)ib * nch + col[q] / chunk];
  // column tiles: contiguous ranges of tw columns; inside a tile, each chunk orders its
  // columns by decreasing count in that chunk, so the 64 lanes of a group carry similar
  // lists (little padding).  A column stays in its tile for every chunk: one workgroup owns
  // it, and the workgroup's output is a contiguous piece of the row.
  std::vector<int32_t> perm((size_t)std::max<int64_t>(npos * nch, 1), -1);
  for (int k = 0; k < nch; ++k) {
    for (int64_t t = 0; t < e.ntiles; ++t) {
      const int64_t lo = t * tw, hi = std::min<int64_t>(nb, lo + tw);
      if (lo >= hi) break;
      std::vector<int32_t> cols(hi - lo);
      for (int64_t i = lo; i < hi; ++i) cols[i - lo] = (int32_t)i;
      std::stable_sort(cols.begin(), cols.end(), [&](int32_t x, int32_t y) {
        return cnt[(size_t)x * nch + k] > cnt[(size_t)y * nch + k];
      });
      // groups of 64 columns in count order; each goes to the wave with the fewest rows so
      // far that still has a free slot (the kernel walks slot j of wave w as group w + j*W)
      const int Wv = e.nt / 64;
      std::vector<int> load(Wv, 0), used(Wv, 0);
      for (int j = 0; j < Wv * e.m; ++j) {
        const size_t i0 = (size_t)j * 64;
        const int mx = i0 < cols.size() ? cnt[(size_t)cols[i0] * nch + k] : 0;  // first lane holds the most
        int best = -1;
        for (int w = 0; w < Wv; ++w)
          if (used[w] < e.m && (best < 0 || load[w] < load[best])) best = w;
        const int64_t slot = (int64_t)best + (int64_t)used[best] * Wv;
        ++used[best];
        load[best] += (mx + AB_BATCH - 1) / AB_BATCH * AB_BATCH;
        for (size_t l = 0; l < 64 && i0 + l < cols.size(); ++l) perm[(size_t)k * npos + lo + slot * 64 + l] = cols[i0 + l];
      }
    }
  }
  // rows of each (group, chunk) block: the longest list of its lanes, rounded up to whole batches
  std::vector<int32_t> K((size_t)std::max<int64_t>(ng, 1), 0);
  for (int64_t g = 0; g < e.groups; ++g)
    for (int k = 0; k < nch; ++k) {
      int mx = 0;
      for (int l = 0; l < 64; ++l) {
        const int32_t ib = perm[(size_t)k * npos + g * 64 + l];
        if (ib >= 0) mx = std::max(mx, cnt[(size_t)ib * nch + k]);
      }
      K[g * nch + k] = (mx + AB_BATCH - 1) / AB_BATCH * AB_BATCH;
    }
  // one stream per (tile, wave, chunk): the wave's groups j = 0..m-1 one after another
  const int W = e.nt / 64;
  const int64_t nstream = e.ntiles * W * nch;
  std::vector<int64_t> soff((size_t)nstream + 1, 0), off((size_t)std::max<int64_t>(ng, 1), 0);
  std::vector<int32_t> nq((size_t)std::max<int64_t>(nstream * e.m, 1), 0);
  for (int64_t t = 0; t < e.ntiles; ++t)
    for (int w = 0; w < W; ++w)
      for (int k = 0; k < nch; ++k) {
        const int64_t s = (t * W + w) * nch + k;
        int64_t o = soff[s];
        for (int j = 0; j < e.m; ++j) {
          const int64_t g = t * W * e.m + w + (int64_t)j * W;
          off[g * nch + k] = o;
          nq[s * e.m + j] = K[g * nch + k] / AB_BATCH;
          o += (int64_t)K[g * nch + k] * 64;
        }
        soff[s + 1] = o;
      }
  const int64_t total = soff[nstream];
  const uint32_t pad = ((uint32_t)e.kbase + (uint32_t)chunk) << 4;  // zero slot, pair 0
  std::vector<uint32_t> ent((size_t)std::max<int64_t>(total, 1), pad);
  const uint32_t kbase = (uint32_t)e.kbase;  // ket vectors follow the slice vectors
  std::vector<std::vector<uint32_t>> lists(64);
  for (int64_t g = 0; g < e.groups; ++g)
    for (int k = 0; k < nch; ++k) {
      const int64_t j0 = (int64_t)k * chunk;
      const int64_t base = off[g * nch + k];
      for (int l = 0; l < 64; ++l) {
        auto& lst = lists[l];
        lst.clear();
        const int32_t ib = perm[(size_t)k * npos + g * 64 + l];
        if (ib < 0) continue;
        for (int64_t q = rp[ib]; q < rp[ib + 1]; ++q) {
          if (col[q] < j0 || col[q] >= j0 + chunk) continue;
          const uint32_t x = exc[q];
          const uint32_t j = x & 63u, b = (x >> 6) & 63u, neg = (x >> 24) & 1u;
          lst.push_back(((kbase + (uint32_t)(col[q] - j0)) << 4) | (ab_pair(b, j) << 18) | (neg << 31));
        }
      }
      schedule_block(lists, K[g * nch + k], pad, ent.data() + base);
    }
  e.mem.put({{&e.soff, soff}, {&e.nq, nq}, {&e.ent, ent}, {&e.colperm, perm}});
}

void build_cores(const uint64_t* d_str, int64_t n, int L, int nel, const double* d_eri, int64_t ncols,
                 CoreTable& ct, Table& direct, hipStream_t st) {
  ct.ncore = ct.nmem = ct.zmem = ct.small = ct.nblk = 0;
  const int64_t npp = (int64_t)nel * (nel - 1) / 2;
  const int64_t total = n * npp;
  std::vector<int32_t> start(1, 0), row, pair, blk, blk_x0, grp, slot_ptr(n + 1, 0), slot;
  // members of the small cores as k_direct_fill takes them, and the pairs of each.  Only counted
  // here: pairs listed and valued on the host were most of this function's time (norb=16, 2,703
  // strings, half a million pairs: 2 of 2.4 ms).
  std::vector<int4> dmem;
  std::vector<int32_t> dcnt;
  // orbitals of every pair index (six bits each), and their bits
  std::vector<uint32_t> porb;
  std::vector<uint64_t> pbits;
  for (uint32_t b = 1; b < (uint32_t)L; ++b)
    for (uint32_t a = 0; a < b; ++a) {
      porb.push_back(a | (b << 6));
      pbits.push_back((1ull << a) | (1ull << b));
    }
  if (total > 0) {
    if (total >= (int64_t)INT32_MAX) throw Error(SBDG_ERR_LIMIT, "too many core memberships");
    DBuf<uint64_t> key, val, key2, val2;
    key.alloc(total);
    val.alloc(total);
    key2.alloc(total);
    val2.alloc(total);
    hipLaunchKernelGGL(k_core_enum, dim3(blocks_for(total, 256)), dim3(256), 0, st, d_str, n, nel, key.p, val.p);
    SBDG_CHECK(hipGetLastError());
    size_t tmp = 0;
    SBDG_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, key.p, key2.p, val.p, val2.p, (int)total, 0,
                                                  std::max(1, L), st));
    DBuf<unsigned char> tb;
    tb.alloc(tmp + 1);
    SBDG_CHECK(hipcub::DeviceRadixSort::SortPairs(tb.p, tmp, key.p, key2.p, val.p, val2.p, (int)total, 0,
                                                  std::max(1, L), st));
    std::vector<uint64_t> hk(total), hv(total);
    SBDG_CHECK(hipMemcpyAsync(hk.data(), key2.p, sizeof(uint64_t) * total, hipMemcpyDeviceToHost, st));
    SBDG_CHECK(hipMemcpyAsync(hv.data(), val2.p, sizeof(uint64_t) * total, hipMemcpyDeviceToHost, st));
    SBDG_CHECK(hipStreamSynchronize(st));
    // keep, core by core, the members whose pair is disjoint from some other member's pair:
    // any other member is a single excitation away (or the same string), contributes
    // nothing and receives nothing.  Radix sort is stable: members ascend by string.
    // Cores of CORE_ZMIN members and more come first: the product goes over those, the RDMs'
    // over all that are kept.
    struct Member {
      uint64_t bits;
      int32_t row, pair;  // pair as in CoreTable
    };
    std::vector<Member> all, keep, mids;
    std::vector<int32_t> midsize;
    auto push = [&](const Member* q, int64_t m) {
      for (int64_t x = 0; x < m; ++x) {
        row.push_back(q[x].row);
        pair.push_back(q[x].pair);
      }
      start.push_back((int32_t)row.size());
    };
    for (int64_t e = 0; e < total;) {
      int64_t f = e + 1;
      while (f < total && hk[f] == hk[e]) ++f;
      if (f - e < 2) {
        e = f;
        continue;
      }
      all.clear();
      keep.clear();
      for (int64_t q = e; q < f; ++q) {
        const int32_t P = (int32_t)((hv[q] >> 32) & 0x7FFFFFFFull);
        all.push_back({pbits[P], (int32_t)(hv[q] & 0xFFFFFFFFull), P | (int32_t)((hv[q] >> 63) << 31)});
      }
      for (const Member& x : all)
        for (const Member& y : all)
          if ((x.bits & y.bits) == 0) {
            keep.push_back(x);
            break;
          }
      const int64_t m = (int64_t)keep.size();
      if (m >= 2 && m < CORE_ZMIN) {
        const int32_t base = (int32_t)dmem.size();
        int64_t pairs = 0;
        for (const Member& x : keep) {
          int32_t with = 0;
          for (const Member& y : keep) with += (x.bits & y.bits) == 0;  // else W = 0 (and x == y)
          dmem.push_back(make_int4(x.row, (int)(porb[x.pair & 0x7FFFFFFF] | ((uint32_t)x.pair & 0x80000000u)), base, (int)m));
          dcnt.push_back(with);
          pairs += with;
        }
        if (m < CORE_KMIN) {
          ct.small += pairs;
        } else {
          mids.insert(mids.end(), keep.begin(), keep.end());
          midsize.push_back((int32_t)m);
        }
      } else if (m >= 2) {
        const int32_t c = (int32_t)(start.size() - 1);
        for (int64_t x0 = 0; x0 < m; x0 += CORE_XB) {
          blk.push_back(c);
          blk_x0.push_back((int32_t)x0);
        }
        push(keep.data(), m);
      }
      e = f;
    }
    ct.zmem = (int64_t)row.size();
    const Member* next = mids.data();
    for (int32_t m : midsize) {
      push(next, m);
      next += m;
    }
    // workgroups: consecutive product blocks until about CORE_WORK member rows, fewer where
    // the pass would then have less than CORE_WGS workgroups (a small problem's blocks one
    // after another in a few workgroups took 84-96 us at 239^2 and 495^2 strings)
    grp.push_back(0);
    int64_t work = 0, total_work = 0;
    for (int32_t c : blk) total_work += start[c + 1] - start[c];
    const int64_t tiles = std::max<int64_t>(1, (ncols + CORE_COLS - 1) / CORE_COLS);
    const int64_t target = std::min<int64_t>(CORE_WORK, total_work * tiles / CORE_WGS);
    for (size_t q = 0; q < blk.size(); ++q) {
      work += start[blk[q] + 1] - start[blk[q]];
      if (work >= target || q + 1 == blk.size()) {
        grp.push_back((int32_t)(q + 1));
        work = 0;
      }
    }
    // per-string slots (counting sort by row)
    for (int64_t q = 0; q < ct.zmem; ++q) ++slot_ptr[row[q] + 1];
    for (int64_t r = 0; r < n; ++r) slot_ptr[r + 1] += slot_ptr[r];
    slot.resize(ct.zmem);
    std::vector<int32_t> fillp(slot_ptr.begin(), slot_ptr.end() - 1);
    for (int64_t q = 0; q < ct.zmem; ++q) slot[fillp[row[q]]++] = (int32_t)q;
  }
  // the direct pairs as a CSR table (rows ascending, a row's by core)
  {
    std::vector<int64_t> rp(n + 1, 0), at(dmem.size());
    for (size_t z = 0; z < dmem.size(); ++z) rp[dmem[z].x + 1] += dcnt[z];
    for (int64_t r = 0; r < n; ++r) rp[r + 1] += rp[r];
    std::vector<int64_t> fill(rp.begin(), rp.end() - 1);
    for (size_t z = 0; z < dmem.size(); ++z) {
      at[z] = fill[dmem[z].x];
      fill[dmem[z].x] += dcnt[z];
    }
    direct.n = n;
    direct.nnz = rp[n];
    const size_t nnz = (size_t)std::max<int64_t>(rp[n], 1);
    direct.rowptr.alloc(n + 1);
    direct.col.alloc(nnz);
    direct.exc.alloc(1);
    direct.val.alloc(nnz);
    direct.val32.alloc(nnz);
    SBDG_CHECK(hipMemcpy(direct.rowptr.p, rp.data(), sizeof(int64_t) * (n + 1), hipMemcpyHostToDevice));
    if (direct.nnz > 0) {
      TableMem t;
      const int4* mem;
      const int64_t* place;
      t.put({{&mem, dmem}, {&place, at}});
      hipLaunchKernelGGL(k_direct_fill, dim3(blocks_for((int64_t)dmem.size(), 256)), dim3(256), 0, st, mem, place,
                         (int64_t)dmem.size(), L, d_eri, direct.col.p, direct.val.p, direct.val32.p);
      SBDG_CHECK(hipGetLastError());
      SBDG_CHECK(hipStreamSynchronize(st));
    }
  }
  ct.ncore = (int64_t)start.size() - 1;
  ct.nmem = (int64_t)row.size();
  ct.nblk = (int64_t)blk.size();
  ct.ngrp = grp.empty() ? 0 : (int64_t)grp.size() - 1;
  auto up = [&](DBuf<int32_t>& d, const std::vector<int32_t>& h) {
    d.alloc(std::max<size_t>(h.size(), 1));
    if (!h.empty()) SBDG_CHECK(hipMemcpy(d.p, h.data(), sizeof(int32_t) * h.size(), hipMemcpyHostToDevice));
  };
  up(ct.start, start);
  up(ct.row, row);
  up(ct.pair, pair);
  up(ct.blk, blk);
  up(ct.blk_x0, blk_x0);
  up(ct.slot_ptr, slot_ptr);
  up(ct.slot, slot);
  up(ct.grp, grp);
}

void build_occ_table(const uint64_t* d_str, int64_t n, int L, const double* d_eri, double* J, float* J32,
                     hipStream_t st) {
  const int64_t total = ((int64_t)L * L + 1) * n;
  if (total == 0) return;
  hipLaunchKernelGGL(k_occ_table, dim3(blocks_for(total, 256)), dim3(256), 0, st, d_str, n, L, d_eri, J, J32);
  SBDG_CHECK(hipGetLastError());
}

void build_pair_integrals(const double* d_eri, int L, double* W, float* W32, hipStream_t st) {
  const int64_t npair = (int64_t)L * (L - 1) / 2;
  if (npair == 0) return;
  hipLaunchKernelGGL(k_pair_int, dim3(blocks_for(npair * npair, 256)), dim3(256), 0, st, d_eri, L, npair, W, W32);
  SBDG_CHECK(hipGetLastError());
  SBDG_CHECK(hipStreamSynchronize(st));
}

void build_pair_slices(const double* d_eri, int L, double* Vt, float* Vt32, hipStream_t st) {
  const int64_t npair = (int64_t)L * (L - 1) / 2;
  if (npair == 0) return;
  hipLaunchKernelGGL(k_pair_slices, dim3(blocks_for(npair * npair, 256)), dim3(256), 0, st, d_eri, L, npair, Vt, Vt32);
  SBDG_CHECK(hipGetLastError());
}

void compute_hii(const uint64_t* d_a, int64_t na, const uint64_t* d_b, int64_t nb, int L, double core,
                 const double* d_h1, const double* d_eri, double* d_hii, hipStream_t st) {
  DBuf<double> Ea, Eb;
  Ea.alloc(std::max<int64_t>(na, 1));
  Eb.alloc(std::max<int64_t>(nb, 1));
  if (na > 0) hipLaunchKernelGGL(k_strdiag, dim3(blocks_for(na, 256)), dim3(256), 0, st, d_a, na, L, d_h1, d_eri, Ea.p);
  if (nb > 0) hipLaunchKernelGGL(k_strdiag, dim3(blocks_for(nb, 256)), dim3(256), 0, st, d_b, nb, L, d_h1, d_eri, Eb.p);
  if (na > 0 && nb > 0)
    hipLaunchKernelGGL(k_hii, dim3((unsigned)na), dim3(TB), 0, st, d_a, d_b, nb, L, core, Ea.p, Eb.p, d_eri, d_hii);
  SBDG_CHECK(hipGetLastError());
  SBDG_CHECK(hipStreamSynchronize(st));
}

}  // namespace sbdg
