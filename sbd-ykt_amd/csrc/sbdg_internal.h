// Internal declarations of the MI355X selected-basis diagonalization library.
//
// Conventions used on the device (the C-ABI converts at its boundary):
//  * alpha strings index rows, beta strings columns: a wavefunction is row-major
//    [ia][ib], beta fastest, exactly the reference layout (tpb/qcham.h:359, mult.h:487);
//  * determinants are phased in the separated order (all alpha creators, ascending, then
//    all beta creators, ascending).  The reference phases them in interleaved order
//    (alpha p -> spin-orbital 2p, beta q -> 2q+1; determinants.h:96-142).  The two differ
//    by the diagonal sign s(A,B) = (-1)^(sum over p in A of #{q in B : q < p}), so
//    H_ref = S H_sep S, sigma_ref(c) = S sigma_sep(S c), and every matrix element keeps
//    its magnitude.  In the separated order an alpha-alpha element depends on the beta
//    string only through the beta occupation (singles) or not at all (doubles).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <initializer_list>
#include <string>
#include <vector>

#include "../../include/sbdg.h"

#define SBDG_CHECK(expr)                                                         \
  do {                                                                           \
    hipError_t _e = (expr);                                                      \
    if (_e != hipSuccess) throw sbdg::Error(SBDG_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
  } while (0)

namespace sbdg {

struct Error {
  int code;
  std::string msg;
  Error(int c, std::string m) : code(c), msg(std::move(m)) {}
};

// Device bytes held by the library's buffers (all devices of the process) and their
// high-water mark since the last reset; sbdg_stats reports them.
struct MemCount {
  std::atomic<int64_t> now{0}, peak{0};
  void add(int64_t b) {
    const int64_t v = now.fetch_add(b) + b;
    int64_t p = peak.load();
    while (v > p && !peak.compare_exchange_weak(p, v)) {
    }
  }
  void reset_peak() { peak.store(now.load()); }
};
inline MemCount& mem_count() {
  static MemCount m;
  return m;
}

// Device buffer owned by the context.
template <class T>
struct DBuf {
  T* p = nullptr;
  size_t n = 0;
  void alloc(size_t count) {
    if (count == n && p) return;
    free();
    if (count) {
      SBDG_CHECK(hipMalloc(&p, sizeof(T) * count));
      n = count;
      mem_count().add((int64_t)(sizeof(T) * count));
    }
  }
  void free() {
    if (p) {
      (void)hipFree(p);
      mem_count().add(-(int64_t)(sizeof(T) * n));
    }
    p = nullptr;
    n = 0;
  }
  ~DBuf() { free(); }
  DBuf() = default;
  DBuf(const DBuf&) = delete;
  DBuf& operator=(const DBuf&) = delete;
};

// Tables made on the host, together in one device buffer: one allocation, and one copy where they
// are small (each takes some 10 us, which a set of a few strings feels).
class TableMem {
 public:
  struct Part {
    void* at;  // const T*: set to the table's place
    void (*set)(void*, const void*);
    const void* src;
    size_t bytes;
    template <class T>
    Part(const T** a, const std::vector<T>& h)
        : at(a), set([](void* d, const void* p) { *static_cast<const T**>(d) = static_cast<const T*>(p); }),
          src(h.data()), bytes(sizeof(T) * h.size()) {}
  };
  void put(std::initializer_list<Part> parts) {
    size_t total = 0;
    for (const Part& x : parts) total += room(x);
    mem_.alloc(total);
    std::vector<unsigned char> host(total <= SMALL ? total : 0);
    size_t o = 0;
    for (const Part& x : parts) {
      x.set(x.at, mem_.p + o);
      if (x.bytes && !host.empty()) std::memcpy(host.data() + o, x.src, x.bytes);
      else if (x.bytes) SBDG_CHECK(hipMemcpy(mem_.p + o, x.src, x.bytes, hipMemcpyHostToDevice));
      o += room(x);
    }
    if (!host.empty()) SBDG_CHECK(hipMemcpy(mem_.p, host.data(), total, hipMemcpyHostToDevice));
  }
  void free() { mem_.free(); }

 private:
  static constexpr size_t SMALL = 1 << 20;
  static size_t room(const Part& x) { return (x.bytes + 255) / 256 * 256 + (x.bytes ? 0 : 256); }
  DBuf<unsigned char> mem_;
};

// Workspace carved out of device memory that lies idle (the RDMs' out of the Davidson vectors):
// first fit over a list of pieces, everything on one stream, which orders a piece's next use
// after its last.  Memory not found there is allocated.
class Arena {
 public:
  void add(void* p, size_t bytes) {
    const uintptr_t a = ((uintptr_t)p + 255) & ~(uintptr_t)255, e = ((uintptr_t)p + bytes) & ~(uintptr_t)255;
    if (p && e > a) pieces_.push_back({a, e - a, false, true});
  }
  void* take(size_t bytes) {  // null: no piece is large enough
    bytes = (bytes + 255) & ~(size_t)255;
    for (size_t k = 0; k < pieces_.size(); ++k) {
      if (pieces_[k].used || pieces_[k].bytes < bytes) continue;
      const Piece rest{pieces_[k].at + bytes, pieces_[k].bytes - bytes, false, false};
      pieces_[k].bytes = bytes;
      pieces_[k].used = true;
      const uintptr_t at = pieces_[k].at;
      if (rest.bytes) pieces_.insert(pieces_.begin() + (int64_t)k + 1, rest);
      return reinterpret_cast<void*>(at);
    }
    return nullptr;
  }
  void give(void* p) {
    for (size_t k = 0; k < pieces_.size(); ++k) {
      if (pieces_[k].at != (uintptr_t)p) continue;
      pieces_[k].used = false;
      if (k + 1 < pieces_.size() && !pieces_[k + 1].used && !pieces_[k + 1].first) join(k);
      if (k > 0 && !pieces_[k - 1].used && !pieces_[k].first) join(k - 1);
      return;
    }
  }

 private:
  struct Piece {
    uintptr_t at;
    size_t bytes;
    bool used, first;  // first: start of a region
  };
  void join(size_t k) {
    pieces_[k].bytes += pieces_[k + 1].bytes;
    pieces_.erase(pieces_.begin() + (int64_t)k + 1);
  }
  std::vector<Piece> pieces_;
};

// A buffer from the arena, or of its own where the arena has no room.
template <class T>
struct WBuf {
  T* p = nullptr;
  explicit WBuf(Arena& a) : ar(a) {}
  void alloc(size_t count) {
    free();
    if (!count) return;
    p = static_cast<T*>(ar.take(sizeof(T) * count));
    lent = p != nullptr;
    if (lent) return;
    own.alloc(count);
    p = own.p;
  }
  void free() {
    if (lent) ar.give(p);
    own.free();
    p = nullptr;
    lent = false;
  }
  ~WBuf() { free(); }
  WBuf(const WBuf&) = delete;
  WBuf& operator=(const WBuf&) = delete;

 private:
  Arena& ar;
  DBuf<T> own;
  bool lent = false;
};

// A table the kernel never writes, read at wave-uniform indices: through the constant address
// space, so that the reads are scalar loads.  (As vector loads they share a counter with the
// other loads in flight, and using one waits for all issued before it.)
template <class I>
__device__ inline I uniform_at(const I* p, int64_t i) {
  return reinterpret_cast<const __attribute__((address_space(4))) I*>(reinterpret_cast<uintptr_t>(p))[i];
}

// The lanes of each half wave that one cycle of a 16-byte LDS read serves together: the first 16
// entries are one such group, the others the second (lanes 32-63 alike).  Each group reads 16
// slots of 16 bytes at once; different addresses in one slot (address / 16 mod 16) take a cycle
// each, equal addresses none.  Measured with every lane on one address but two lanes on one
// slot, for all pairs of lanes: 4.4 clocks per read, 5.5 where the two share a group.
constexpr int LDS16_LANE[32] = {0, 1, 2, 3, 12, 13, 14, 15, 20, 21, 22, 23, 24, 25, 26, 27,
                                4, 5, 6, 7, 8,  9,  10, 11, 16, 17, 18, 19, 28, 29, 30, 31};

// The 16 x 16 x 4 FP64 matrix instruction.  Operands: lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16]; of the product, element q of lane l is row(q, l), column l % 16.
struct Mfma64 {
  typedef double acc __attribute__((ext_vector_type(4)));
  __device__ static inline acc mad(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static inline int row(int q, int lane) { return 4 * q + lane / 16; }
};
// Excitation table of one string set, CSR with ket indices ascending per bra row
// (membership and order of chemistry/tpb/helper.h:132-197).
//  exc word (singles): bits 0-5 ket-only orbital i, 6-11 bra-only orbital a,
//                      bit 24 set when the separated-order sign is negative.
//  exc word (doubles): bits 0-5 I, 6-11 J (ket-only, I<J), 12-17 A, 18-23 B (bra-only,
//                      A<B), bit 24 sign.
//  val: the spin-string-only part of the element in the separated order:
//       singles  sign * (h_ai + sum_{k in occ(ket)\{i}} [(ai|kk) - (ak|ki)])
//       doubles  sign * ((AI|BJ) - (AJ|BI))
struct Table {
  int64_t n = 0, nnz = 0;
  DBuf<int64_t> rowptr;  // n+1
  DBuf<int32_t> col;     // nnz
  DBuf<uint32_t> exc;    // nnz
  DBuf<double> val;      // nnz
  DBuf<float> val32;     // nnz
};

// Row-merged (singles then doubles) table feeding the row-streaming product.
struct SpmmTable {
  int64_t n = 0, nnz = 0;
  DBuf<int64_t> rowptr;
  DBuf<int64_t> mid;  // n: where the row's doubles start
  DBuf<int32_t> col;
  DBuf<double> val;
  DBuf<float> val32;
  // other-spin occupation term of a single: +-(p + 1) with p = a*L + i its orbital pair
  // and the sign of the single; 0 for a double.  The product adds sign * J[p + 1][c] per
  // column (J: occupation table of the column strings, row 0 zero).
  DBuf<int32_t> jai;
};

// Beta pairs (columns one excitation apart, each once) in tiles for the alpha-beta RDM kernel
// (build_ab_pairs): entry = LDS vector of the column with the upper orbital | of the other one
// << 15 | negative sign << 30, a tile's entries ordered for the LDS and padded to nt*u; rank is
// their place when sorted by orbital pair.  runstart lists, per tile, the first place of each
// orbital pair's run and then the tile's number of entries (runptr delimits the tiles' lists); pairptr/pairrun list each orbital
// pair's runs.
constexpr int64_t AB_PAIR_COLS = 80 * 1024 / 16 - 4;         // columns of one staged alpha pair: half a CU's LDS, a multiple of 4
constexpr int64_t RDM_PART_BYTES = (int64_t)256 << 20;  // partial sums of one batch of orbital-pair keys
struct AbPairs {
  bool built = false;
  int nt = 0, u = 0, sp = 1;  // threads, pairs per thread, alpha pairs staged at once
  int64_t maxcols = 0, ntiles = 0, nruns = 0;
  TableMem mem;
  const int4* tile;      // first column and number of columns of the tile's two chunks
  const int64_t* entoff;
  const uint32_t* ent;
  const uint16_t* rank;  // place of each entry in its tile's sorted list
  const int32_t *runptr, *runstart, *pairptr, *pairrun;
};

// Beta singles in an ELL layout for the alpha-beta sigma kernel.  Columns are cut into
// contiguous tiles of nt*m lane positions (one workgroup each); in ket chunk k, colperm[k*npos + pos]
// is the column at lane position pos (-1: none).  Per chunk, a tile's columns are sorted by
// their entry count in that chunk and cut into 64-lane groups (lists of similar length);
// wave w of tile t walks the groups at slots g = t*W*m + w + j*W, j < m (W = nt/64), and
// the groups are dealt to the slots longest first, each to the wave with the fewest rows
// so far, so the waves of a workgroup reach its barriers together.  Per chunk k a wave's
// groups form one stream starting at soff[(t*W + w)*nch + k], group after group, each a
// multiple of four rows of 64 lane-interleaved entries (nq[stream*m + j] batches of four
// rows) padded with a zero-weight entry: the wave reads its stream coalesced, four rows
// at a time, with the next four rows in flight across group boundaries.
// Entry: bits 0-17 LDS byte address of the ket vector (16 * (kbase + column offset inside
// the chunk); offset `chunk` is a zero vector: padding), bits 18-29 the slice vector of
// orbital pair (b, j) (ab_pair(b, j)), bit 31 sign.  Within a lane the entries are ordered
// so that lanes read distinct LDS slots where possible.
constexpr int AB_BATCH = 4;  // ELL rows per batch of the alpha-beta kernel
struct EllTable {
  int nch = 0;
  int nt = 0, m = 0, s = 1;  // alpha-beta launch: threads per workgroup, columns per thread, groups staged at once
  int64_t chunk = 0, groups = 0, ntiles = 0;
  int64_t kbase = 0;        // first ket vector (16-byte units): after the slice vectors
  TableMem mem;
  const int64_t* soff;      // ntiles*(nt/64)*nch + 1: start of each wave's entry stream per chunk
  const int32_t* nq;        // ntiles*(nt/64)*nch*m: four-row batches of each group of the stream
  const uint32_t* ent;
  const int32_t* colperm;   // nch * groups*64: column of each lane position in each chunk (-1: none)
  void release() {
    mem.free();
    nch = nt = m = 0;
  }
};

// Bra rows of the alpha-beta kernel cut into segments of their alpha singles (longest
// first): one workgroup per segment and column tile.  A row's first segment writes sigma's
// row, the others rows of `part`, which k_ab_join adds in order.
constexpr int64_t AB_PART_BYTES = (int64_t)256 << 20;  // at most this much in partial rows
struct AbSegments {
  int64_t nseg = 0, npart = 0, njoin = 0;
  TableMem mem;
  const int32_t* row;   // nseg
  const int64_t* q;     // 2*nseg: first and past-the-end alpha single
  const int32_t* dst;   // nseg: -1 or the row of part
  const int32_t* jrow;  // njoin rows with partial rows
  const int32_t* jptr;  // njoin + 1
  DBuf<double> part;    // npart rows of nb
};

// Double excitations of one spin grouped by their (n-2)-electron core: a double pair
// (x, y) shares exactly one core k = x & y (two electrons fewer than x), and its element
// in the separated order is eps_x * eps_y * W[P_x][P_y], with P_x = (a < b) the pair added
// to k to make x, eps_x = <x| c+_a c+_b |k> and W[(A,B)][(I,J)] = (AI|BJ) - (AJ|BI)
// (zero when the pairs overlap).  Members are stored core by core, the cores of CORE_ZMIN
// members and more first: those go through the product and its workspace (row slots list, per
// string, the member entries it owns there).  Cores down to CORE_KMIN members follow for the
// RDMs' Gram products.  The pairs of all cores below CORE_ZMIN (two members and up) are cheaper
// read directly: they go to a CSR table of their own that the row-streaming product merges with
// the singles.
struct CoreTable {
  int64_t ncore = 0, nmem = 0, nblk = 0;  // cores and members down to CORE_KMIN, product blocks
  int64_t zmem = 0;                       // members of the cores that go through the workspace
  int64_t small = 0;                      // direct pairs of the cores below CORE_KMIN
  DBuf<int32_t> start;    // ncore + 1
  DBuf<int32_t> row;      // nmem
  DBuf<int32_t> pair;     // nmem: P(a,b) = b(b-1)/2 + a, bit 31 set when eps is negative
  DBuf<int32_t> blk;      // nblk: core of each product block
  DBuf<int32_t> blk_x0;   // nblk: first member of the block
  DBuf<int32_t> slot_ptr; // n + 1
  DBuf<int32_t> slot;     // zmem
  int64_t ngrp = 0;
  DBuf<int32_t> grp;      // ngrp + 1: product blocks of each workgroup
};
constexpr int CORE_XB = 16;     // output members per product block
constexpr int CORE_COLS = 512;  // column granularity of the core-product passes
constexpr int CORE_WORK = 256;  // member rows streamed per core-product workgroup (at most, when several blocks share one)
constexpr int CORE_WGS = 4096;  // workgroups a core pass should have before blocks are grouped
// Smallest core taken through the workspace.  A core of k members costs 3k row transfers there
// (member rows in, Z out, Z gathered), of which the 2k of Z go to memory and back; read directly
// it costs at most k(k-1), fewer where members' pairs overlap, but of k rows that the next rows
// of the same core find in cache.  FP64 sigma with the cut at
// 10 / 13 / 20 / 28 / 40 members: norb=36, 20,000^2 strings 136.1 / 133.1 / 132.7 / 132.9 / 132.9
// ms; norb=26, 4,000^2 4.59 / 4.57 / 4.43 / 4.39 / 4.40; norb=36, 5,001 x 4,999 5.24 / 5.09 / 4.96 / 4.68 /
// 4.69; norb=58, 200 x 40,000 2.65 / 2.63 / 2.55 / 2.54 / 2.84.
constexpr int CORE_ZMIN = 28;
// Smallest core of the RDMs' Gram products (k_core_gram): one 16-row tile filled to more than
// half; smaller cores' pairs one by one.
constexpr int CORE_KMIN = 10;

// kernels (tables.hip)
void build_table(const uint64_t* d_str, int64_t n, int L, const double* d_h1, const double* d_eri,
                 Table& t_single, Table& t_double, hipStream_t st);
void build_spmm(const Table& s, const Table& d, SpmmTable& m, int L, hipStream_t st, bool with_doubles = true);
// d_eri: the integrals (full L^4), for the values of the direct pairs
void build_cores(const uint64_t* d_str, int64_t n, int L, int nel, const double* d_eri, int64_t ncols,
                 CoreTable& ct, Table& direct, hipStream_t st);
// J[(p+1)*n + r] = sum_{o in occ(s[r])} eri[p*L^2 + o*L + o] for p < L^2 (row 0 zero):
// the occupation part of the other spin's singles, (ai|oo) summed over the string's orbitals
void build_occ_table(const uint64_t* d_str, int64_t n, int L, const double* d_eri, double* J, float* J32,
                     hipStream_t st);
// W[P*npair + Q] (FP64 and FP32), npair = L(L-1)/2
void build_pair_integrals(const double* d_eri, int L, double* W, float* W32, hipStream_t st);
// Vt[ab_pair(a,i)*npair + ab_pair(b,j)] = (ai|bj): one alpha single's slice is contiguous
void build_pair_slices(const double* d_eri, int L, double* Vt, float* Vt32, hipStream_t st);
// prec_bytes: 8 (FP64) or 4 (FP32) -- the launch geometry depends on the accumulator size
void build_ell(const Table& sb, int L, int prec_bytes, EllTable& e, hipStream_t st);
// Launch geometry of the alpha-beta kernel: threads, columns per thread, ket-row groups staged
// at once, ket columns per chunk.
struct AbGeometry {
  int nt, m, s;
  int64_t chunk;
};
AbGeometry ab_geometry(int64_t nb, int L, int prec_bytes);
void build_segments(const Table& sa, int64_t nb, int64_t ntiles, AbSegments& g, hipStream_t st);
void compute_hii(const uint64_t* d_a, int64_t na, const uint64_t* d_b, int64_t nb, int L, double core,
                 const double* d_h1, const double* d_eri, double* d_hii, hipStream_t st);

// sigma (sigma.hip)
struct SigmaPlan {
  int64_t na = 0, nb = 0;
  int L = 0;
  const uint64_t* a = nullptr;
  const uint64_t* b = nullptr;
  const SpmmTable* ma = nullptr;  // alpha merged
  const SpmmTable* mb = nullptr;  // beta merged
  const Table* sa = nullptr;      // alpha singles (exc, col)
  const EllTable* ell = nullptr;
  const AbSegments* seg = nullptr;
  const double* Vt = nullptr;  // (ai|bj) over orbital pairs a > i, b > j (alpha-beta slices)
  const float* Vt32 = nullptr;
  const double* hii = nullptr;
  const float* hii32 = nullptr;
  const double* Jb = nullptr;  // beta-occupation table (columns of c), alpha singles
  const float* Jb32 = nullptr;
  const double* Ja = nullptr;  // alpha-occupation table (columns of c^T), beta singles
  const float* Ja32 = nullptr;
  const CoreTable* ca = nullptr;  // alpha doubles by core (null: doubles in ma/mb)
  const CoreTable* cb = nullptr;
  const double* W = nullptr;
  const float* W32 = nullptr;
  int64_t npair = 0;
  void* Z = nullptr;    // core-product workspace of zbytes
  size_t zbytes = 0;
  hipStream_t st2 = nullptr;  // when set: the alpha-beta terms run there, beside the spin phases
  hipEvent_t fork = nullptr, join = nullptr;
};
// sigma = H c in the separated convention.  Scratch: three vectors of na*nb elements of T
// (c transposed, the beta product on it, the alpha-beta terms when they run on the second
// stream), any device memory the caller does not use while sigma runs; none may overlap
// c or sigma.
template <class T>
struct SigmaScratch {
  T* cT = nullptr;
  T* sT = nullptr;
  T* sab = nullptr;
};
template <class T>
void sigma_apply(const SigmaPlan& P, const T* c, T* sigma, const SigmaScratch<T>& scr, hipStream_t st,
                 hipEvent_t* ev = nullptr);
size_t ab_lds_bytes(int64_t kbase, int64_t chunk);

// The alpha-beta kernel's LDS in 16-byte vectors: one integral slice vector per orbital pair
// b > j at ab_pair(b, j) = b(b-1)/2 + j (a single moves an electron between two different
// orbitals, and (ai|bj) = (ai|jb) for the 8-fold symmetric integrals the library takes), at
// least one vector; then the ket vectors of one chunk.
inline int64_t ab_pairs(int L) {
  return std::max<int64_t>(1, (int64_t)L * (L - 1) / 2);
}
__host__ __device__ inline uint32_t ab_pair(uint32_t b, uint32_t j) {
  const uint32_t h = b > j ? b : j, l = b > j ? j : b;
  return h * (h - 1) / 2 + l;
}
// A set of one beta string has no singles, so there are no alpha-beta terms.
inline bool ab_any(int64_t nb) { return nb >= 2; }
// Vectors that a thread of the alpha-beta kernel stages per round.  Ket vectors: what its m columns
// need, up to eight, four where the FP64 accumulators take the registers; more would only load the
// row's last pair again.  Slice vectors: 512 of a workgroup of up to 256 threads.
constexpr int ab_ket_round(int elem, int m) { return m <= 2 ? 2 : m <= 4 || elem * m > 160 ? 4 : 8; }
constexpr int ab_slice_round(int nt) { return nt <= 256 ? 512 / nt : 2; }
// First of the two neighbouring columns that place x of the alpha-beta kernel's staging loads of
// a chunk of nj columns (nj >= 2: ab_any): the places past the last two take them again.
__host__ __device__ inline int ab_stage_pair(int x, int nj) { return x < nj - 2 ? x : nj - 2; }
inline int64_t ab_slice_span(int L) {
  return ab_pairs(L);
}

// vector kernels (linalg.hip)
void sign_transform(const uint64_t* a, int64_t na, const uint64_t* b, int64_t nb, const double* in,
                    double* out, hipStream_t st);
void cast_d2f(const double* in, float* out, int64_t n, hipStream_t st);
void fill_test_vector(double* x, int64_t n, uint64_t seed, hipStream_t st);
void cast_f2d(const float* in, double* out, int64_t n, hipStream_t st);
// Basis vectors are contiguous: X_k = X + k*ldx.
// out[k] = <X_k, y> for k < m (deterministic two-stage reduction); y FP64 or FP32.
void multi_dot_impl(const double* X, int64_t ldx, int m, const double* y, int64_t n, double* out, double* part,
                    hipStream_t st);
void multi_dot_rows_impl(const float* Y, int64_t ldy, int m, const double* x, const double* z, int64_t n,
                         double* out, double* part, hipStream_t st);
void multi_dot_impl(const double* X, int64_t ldx, int m, const float* y, int64_t n, double* out, double* part,
                    hipStream_t st);
// W = sum_k u[k] V_k ; R = sum_k u[k] HV_k - theta W ; out[0] = |W|^2, out[1] = |R|^2
template <class TH>
void ritz_combine_impl(const double* V, int64_t ldv, const TH* HV, int64_t ldh, int m, const double* u,
                       const double* theta, double* W, double* R, int64_t n, double* out, double* part,
                       hipStream_t st);
// fused Ritz step (m <= 32): out[0..m) = V_k . t, out[m] = |r|^2, out[m+1] = |t|^2, t -> T
template <class TH>
void ritz_expand_impl(const double* V, int64_t ldv, const TH* HV, int64_t ldh, int m, const double* u,
                      const double* theta, const double* hii, double* T, int64_t n, double* out, double* part,
                      hipStream_t st);
void scale_impl(double* x, const double* n2, int64_t n, hipStream_t st);  // x /= sqrt(n2[0])
// x /= sqrt(n2[0]) and y = (float)x in the same pass
void scale_cast_impl(double* x, const double* n2, float* y, int64_t n, hipStream_t st);
// out[k] = <Y_k, x> for k < m (Y FP32, Y_k = Y + k*ldy), and out[m] = <z, x> when z is set:
// one pass that reads x once
// t = (R/|R|) / (theta - d), with the 1e-12 regularisation of davidson.h:855-862
void precond_impl(const double* R, const double* rn2, const double* hii, const double* theta, double* t, int64_t n,
                  hipStream_t st);
// t -= sum_k s[k] V_k; out[0] = |t|^2
void gs_impl(const double* V, int64_t ldv, int m, const double* s, double* t, int64_t n, double* out, double* part,
             hipStream_t st);
// in place: X_j = sum_k U[k + ld*j] X_k for j < mk (thick-restart rotation)
template <class T>
void rotate_impl(T* X, int64_t ldx, int m, const double* U, int ld, int mk, int64_t n, hipStream_t st);
// Order of eigenvalues x at place i and y at place j: ascending, NaN last, equal ones by place.  A
// strict order whatever the values, so that counting the places before each gives every rank once.
__host__ __device__ inline bool eigen_before(double x, int i, double y, int j) {
  if (x != x || y != y) return (x != x) == (y != y) ? i < j : y != y;
  return x < y || (x == y && i < j);
}
// symmetric eigensolve of the m x m column-major d_H (ld) on the device: ascending
// eigenvalues in d_E, eigenvectors in the columns of d_U (ld).
void syev_device(const double* d_H, int m, int ld, double* d_E, double* d_U, hipStream_t st);
// d_part: density_part(na, nb) doubles of scratch
int64_t density_part(int64_t na, int64_t nb);
void density(const double* W, const uint64_t* a, int64_t na, const uint64_t* b, int64_t nb, int L,
             double* d_dens, double* d_part, hipStream_t st);
// d_rs[ia] = sum_ib W[ia,ib]^2 (fixed-order block sums)
void row_sumsq(const double* W, int64_t na, int64_t nb, double* d_rs, hipStream_t st);

// RDMs (rdm.hip)
struct RdmPlan {
  int64_t na = 0, nb = 0;
  int L = 0;
  const uint64_t* a = nullptr;
  const uint64_t* b = nullptr;
  const Table* sa = nullptr;
  const Table* da = nullptr;
  const Table* sb = nullptr;
  const Table* db = nullptr;
  const AbPairs* ab = nullptr;
  const CoreTable* ca = nullptr;  // larger cores of the same-spin doubles (row-pair sums by block), or null
  const CoreTable* cb = nullptr;
};
void build_ab_pairs(const Table& sb, int L, AbPairs& ab, hipStream_t st);
// one[2][L^2], two[4][L^4] in the reference layout (correlation.h:194-444) from the
// separated-convention vector W; WT: scratch of na*nb doubles (W transposed).  Bitwise
// reproducible: every sum is taken in a fixed order.
// Transient buffers come out of ar where they fit.
void rdm_compute(const RdmPlan& P, const double* W, double* WT, double* d_one, double* d_two, Arena& ar,
                 hipStream_t st);
// Hellmann-Feynman gradient: dh[p*L+q] = g*(one_a+one_b)[p+L*q];
// deri[((p*L+q)*L+r)*L+s] = g/2 * sum_blk two[blk][p + L*r + L^2*q + L^3*s]
void rdm_backward(const double* d_one, const double* d_two, int L, double g, double* d_dh,
                  double* d_deri, hipStream_t st);

}  // namespace sbdg
