// Batched sparse LDL^T and QR with sixteen lanes per instance.
//
// The one-lane-per-instance programs (jit.hip) need thousands of wavefronts'
// worth of instances to fill the chip: 8192 KKT systems are 128 wavefronts on
// 1024 SIMDs, each streaming its own 685 KB straight line (318 us for the
// n = 274 LDL, 700 us for the QR).  The factorisations themselves are
// parallel: once row r of L is final, every row c below it that has an entry
// in column r can take its entry (c, r) at the same time.  So here an
// instance owns one 16-lane DPP row of a wavefront, a lane owns an active row
// of L (LDL) or an active column of A and the right-hand side (QR), and the
// pivots run in order:
//
//   LDL, pivot r (owner lane q)   v(c) = A(c,r) - sum_k L(r,k) W(c,k), k in the
//                                 order of L^T's column r; L(c,r) = v / D(r);
//                                 D(c) -= v L(c,r);  y(c) -= L(c,r) y(r)
//   QR, pivot r (owner lane q)    casadi_house on the owner's column; every
//                                 column (and the right-hand side) with an
//                                 entry in row r of R takes the reflection
//   back substitution, r = n-1..0 x(r) = z(r) - sum_c L(c,r) x(c)   or
//                                 x(r) = (w(r) - sum_c R(r,c) x(c)) / R(r,r),
//                                 c descending
//
// which are the updates of casadi_ldl / casadi_qr (casadi/core/runtime/
// casadi_ldl.hpp:24-109, casadi_qr.hpp:24-230) in another interleaving: every
// value sees the same operations on the same operands in the same order, the
// products with structural zeros of the work vector included, so the bits
// are those of the other programs.  The owner's values reach the other lanes
// through v_mov_b64_dpp row_newbcast (one instruction, no LDS); the values an
// active row or column holds live in registers whose slots are interval
// coloured over the pivots.
//
// Memory.  A wavefront gather of 16 rows costs the vector L1 one lookup per
// lane (64), which bounded a first version (25 lookups per access, 174 us and
// 336 us).  So what a program reads from the caller's arrays is staged
// through an LDS ring, 16 entries x 4 instances per access (16 lookups, every
// byte used), in the order the pivots consume it, and a pivot reads its
// entries from consecutive ring rows.  What it keeps between the forward and
// the backward sweep (a pivot's L or R entries and z or w, one block per pivot
// and instance) is written and read back as consecutive doubles.
//
// Measured (n = 274, horizon-30 control KKT, 8192 instances, a whole
// solve_batch call): LDL 350 -> 141 us, QR 805 -> 271 us; a single instance's
// chain (64 instances) 278 -> 110 and 630 -> 186 us.  What bounds it now is
// VALU issue and the pivots' dependent chain together (two wavefronts per
// SIMD, 73% of the issue cycles in VALU).
//
// A pattern fits when at most 16 rows (LDL) or 15 columns (QR) are active at
// once and their values fit kMaxSlots registers; the horizon-30 control KKT
// has 9 rows of 13 values, and 13 columns of 18.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <set>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/casadi_hip.h"
#include "capi_common.hpp"
#include "jit_common.hpp"
#include "linsol_rows.hpp"
#include "tape_internal.hpp"

namespace sxh {

namespace {

constexpr int kLanes = 16;
constexpr int kMaxSlots = 40;  // values per lane: 2 x 40 doubles (LDL's W and L) leave room for the rest
constexpr int kChunk = 8;      // pivots per chunk of the generated program
constexpr int kBatch = 16;     // entries staged by one access
constexpr int kRing = 128;     // entries of the LDS ring (a gather never wraps: kLanes more are readable)
constexpr int kLand = 2;       // batches written to the ring ahead of the first that needs them
constexpr int kFlight = 8;     // batches in flight from memory beyond those
constexpr int kBack = 16;      // blocks in flight in the back substitution (written long before: they come from HBM)
constexpr int kIdx = 4;        // table rows of the factor's scattered stores read ahead

// The generated program's vocabulary.  A test that runs it on the host
// defines CXR_EMULATED and its own (vd: the sixteen lanes of one instance).
const char kRowsPrologue[] = R"CXR(
struct CxrArgs {
  const char* a; char* x;      // A's nonzeros; right-hand side / solution
  char* f; char* d; char* z;   // factor rows, D or beta rows, intermediate rows
  char* w;                     // blocks kept from the forward to the backward sweep, [instance][pivot]
  const int* tab;              // staged entries, then store rows of 16
  int* status;
  long long a_t, x_t;          // bytes per instance of a, x
  unsigned a_s, x_s, ld, w_t;  // bytes per nonzero of a, x; per row of f, d, z; per instance of w
  double eps;
  long long n;
};
#ifndef CXR_EMULATED
typedef double vd;
typedef int vi;
#define CXR_IN(m) ((lanebit & (unsigned)(m)) != 0)
#define CXR_WHERE(m) if (CXR_IN(m))
#define CXR_BC(v, q) __longlong_as_double(__builtin_amdgcn_mov_dpp(__double_as_longlong(v), 0x150 + (q), 0xf, 0xf, true))
// a in the lanes of m, b in the others: two v_cndmask with the mask, a
// constant of the program, in an SGPR pair
__device__ __forceinline__ double cxr_sel(unsigned long long m, double a, double b) {
  union { double d; unsigned u[2]; } x, y, r;
  x.d = a;
  y.d = b;
  asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(r.u[0]) : "v"(y.u[0]), "v"(x.u[0]), "s"(m));
  asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(r.u[1]) : "v"(y.u[1]), "v"(x.u[1]), "s"(m));
  return r.d;
}
#define CXR_SEL(m, a, b) cxr_sel((m) * 0x0001000100010001ull, a, b)
// rank of this lane among the lanes of m
#define CXR_RANK(m) (unsigned)__builtin_popcount((unsigned)(m) & below)
// Staging: lane = 4 * entry + instance of the wavefront's four.  An entry's
// table word is its nonzero and, in the top three bits, the array.
#define CXR_ENTRY(b) A.tab[(b) * 16 + (lane64 >> 2)]
#define CXR_FETCH(e_) cxr_fetch(A, e_, ics, is)
#define CXR_LAND(b, v) do { __builtin_amdgcn_wave_barrier(); ring[((b) % 8) * 64 + lane64] = (v); __builtin_amdgcn_wave_barrier(); } while (0)
#define CXR_RING(start, m) *(const double*)((const char*)ring + (start) * 32 + (CXR_RANK(m) * 32u + ring_at))
__device__ __forceinline__ double cxr_fetch(const CxrArgs& A, int e, long long ic, long long i) {
  const unsigned k = (unsigned)e & 0x1fffffffu, what = (unsigned)e >> 29;
  // the arrays the program stages (CXR_STAGED), each through an opaque copy:
  // a choice between kernel arguments would otherwise become a choice between
  // their addresses, and the arguments a copy in scratch
#define CXR_FROM(c, base, at, stride) \
  if ((CXR_STAGED >> c) & 1) { \
    unsigned long long b_ = (unsigned long long)(base); unsigned s_ = (stride); \
    asm("" : "+s"(b_), "+s"(s_)); \
    if (what == c) { p = b_ + (unsigned long long)(at); s = s_; } \
  }
  unsigned long long p = 0;
  unsigned s = 0;
  CXR_FROM(0, A.a, ic * A.a_t, A.a_s)
  CXR_FROM(1, A.x, ic * A.x_t, A.x_s)
  CXR_FROM(2, A.f, i * 8, A.ld)
  CXR_FROM(3, A.d, i * 8, A.ld)
  return *(const double*)(p + (unsigned long long)k * (unsigned long long)s);
}
// a pivot's block.  Every lane reads, a lane above those of the mask one value
// past them: the next block's first, which must be there.  A block of one
// value is read by all lanes alike (the last one is: nothing follows it).
#define CXR_KEPT1(off) *(const double*)(A.w + (off) * 8 + w_at)
#define CXR_KEPT(off, m) *(const double*)(A.w + (off) * 8 + (CXR_RANK(m) * 8u + w_at))
#define CXR_KEEP_BLOCK(off, m, v) do { if (CXR_IN(m)) *(double*)(A.w + (off) * 8 + (CXR_RANK(m) * 8u + w_at)) = (v); } while (0)
// scattered stores of the factor's rows, instance i
#define CXR_IDX(j) A.tab[(j) * 16 + lane]
#define CXR_PUT_f(m, i_, v) do { if (CXR_IN(m)) *(double*)(pf + (unsigned long long)(unsigned)(i_) * (unsigned long long)A.ld) = (v); } while (0)
#define CXR_PUT_d(m, i_, v) do { if (CXR_IN(m)) *(double*)(pd + (unsigned long long)(unsigned)(i_) * (unsigned long long)A.ld) = (v); } while (0)
#define CXR_PUT_z(m, i_, v) do { if (CXR_IN(m)) *(double*)(pz + (unsigned long long)(unsigned)(i_) * (unsigned long long)A.ld) = (v); } while (0)
#define CXR_PUT_x(m, i_, v) do { if (CXR_IN(m) && valid) *(double*)(px + (unsigned long long)(i_) * (unsigned long long)A.x_s) = (v); } while (0)
#define CXR_BAD(v) ((v) != 0 && (v) - (v) == 0 ? 0 : 1)
#define CXR_SMALL(v, e) (__builtin_fabs(v) >= (e) ? 0 : 1)
#define CXR_SQRT(v) sqrt(v)
#define CXR_EQ0(c, a, b) ((c) == 0 ? (a) : (b))
#define CXR_LE0(c, a, b) ((c) <= 0 ? (a) : (b))
// counted here: left to the compiler, every pivot is held to the program's end
#define CXR_KEEP(c) asm volatile("" : "+v"(c))
// the wavefront's rows and blocks are written before its lanes read them back
#define CXR_SYNC() do { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup"); __builtin_amdgcn_s_barrier(); \
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup"); } while (0)
#define CXR_COUNT(c) do { if (lane0 == 0 && valid && A.status) A.status[i] = (c); } while (0)
#define CXR_BODY(name) __device__ __forceinline__ void name(const CxrArgs& A, const long long i, const int lane0, double* const ring)
#define CXR_SETUP() \
  const bool valid = i < A.n; \
  const long long ic = valid ? i : A.n - 1; \
  const long long is0 = (i & ~3ll) + (threadIdx.x & 3), ics0 = is0 < A.n ? is0 : A.n - 1
// Opaque copies for one chunk: what is derived from them (addresses, lane
// masks) is computed where it is used, not once for every chunk at the top of
// the program (hundreds of registers).
#define CXR_CHUNK() \
  int lane = lane0; asm volatile("" : "+v"(lane)); \
  const unsigned lanebit = 1u << lane, below = lanebit - 1u; \
  int lane64 = (int)(threadIdx.x & 63); asm volatile("" : "+v"(lane64)); \
  const unsigned sub = (unsigned)lane64 >> 4, ring_at = sub * 8u; \
  unsigned inst = (unsigned)i; asm volatile("" : "+v"(inst)); \
  const unsigned w_at = inst * A.w_t; \
  long long is = is0; asm volatile("" : "+v"(is)); long long ics = ics0; asm volatile("" : "+v"(ics)); \
  char* const pf = A.f + (long long)inst * 8; char* const pd = A.d + (long long)inst * 8; \
  char* const pz = A.z + (long long)inst * 8; \
  char* const px = A.x + (valid ? (long long)inst : A.n - 1) * A.x_t; \
  (void)lanebit; (void)below; (void)ring_at; (void)w_at; (void)is; (void)ics; (void)pf; (void)pd; (void)pz; (void)px
#endif
)CXR";

std::string S(int64_t v) { return std::to_string(v); }

std::string hexmask(unsigned m) {
  char b[24];
  std::snprintf(b, sizeof b, "0x%04xull", m);
  return b;
}

int popcount(unsigned m) { return __builtin_popcount(m); }

// Text of a program.  entries() names the value of staged entries, one per
// lane of a mask; the ring's batches are landed and fetched where the pivots
// reach them.  The backward phase starts staging from nothing (it may read
// what the forward one wrote).
struct RowsEmit {
  std::vector<int> entry;               // staged table words of all phases, whole batches
  std::vector<int> rows;                // store rows, [row][16], after the entries in the table
  std::string body;                     // text of the current chunk
  std::string out;                      // finished text
  size_t phase0 = 0;                    // first entry of the current phase
  int reached = -1;                     // last batch of the phase whose turn has come
  std::vector<std::string> chunks;
  std::vector<int> puts;                // store rows of the phase, in order

  static int word(char base, int nz) {
    const int what = base == 'a' ? 0 : base == 'x' ? 1 : base == 'f' ? 2 : 3;
    return static_cast<int>(static_cast<unsigned>(what) << 29 | static_cast<unsigned>(nz));
  }
  // words[l]: table word of lane l, for the lanes of mask
  std::string entries(unsigned mask, const std::vector<int>& words) {
    const int need = popcount(mask);
    size_t at = entry.size() - phase0;
    if (at % kRing + static_cast<size_t>(need) > static_cast<size_t>(kRing)) {  // not across the ring's end
      entry.resize(phase0 + (at / kRing + 1) * kRing, last_word());
      at = entry.size() - phase0;
    }
    for (int l = 0; l < kLanes; ++l)
      if (mask >> l & 1u) entry.push_back(words[l]);
    // the batches this gather reaches
    const int hi = static_cast<int>((entry.size() - phase0 - 1) / kBatch);
    while (reached < hi) body += "\x01" + S(++reached) + "\x02";
    return "CXR_RING(" + S(static_cast<int64_t>(at % kRing)) + ", " + hexmask(mask) + ")";
  }
  int last_word() const { return entry.empty() ? 0 : entry.back(); }
  // stores through table rows (the factor's own layout)
  void put(char base, unsigned mask, const std::vector<int>& idx, const std::string& v) {
    const int j = static_cast<int>(puts.size());
    puts.push_back(static_cast<int>(rows.size()) / kLanes);
    for (int l = 0; l < kLanes; ++l) rows.push_back(std::max(idx[l], 0));
    body += "  CXR_PUT_" + std::string(1, base) + "(" + hexmask(mask) + ", p" + S(j % kIdx) + ", " + v + ");\n\x03" + S(j) +
            "\x02";
  }
  // var = value in the lanes of mask
  void set(unsigned mask, const std::string& var, const std::string& value) {
    if (mask == 0) return;
    if (mask == 0xffffu) body += "  " + var + " = " + value + ";\n";
    else body += "  " + var + " = CXR_SEL(" + hexmask(mask) + ", " + value + ", " + var + ");\n";
  }
  void end_chunk() {
    if (!body.empty()) chunks.push_back(std::move(body));
    body.clear();
  }
  void end_phase() {
    end_chunk();
    while ((entry.size() - phase0) % kBatch) entry.push_back(last_word());
    const int b0 = static_cast<int>(phase0) / kBatch, nb = static_cast<int>((entry.size() - phase0) / kBatch);
    auto load_entry = [&](int b) {  // the table words of batch b
      return b < nb ? "  e" + S(b % 2) + " = CXR_ENTRY(" + S(b0 + b) + ");\n" : std::string();
    };
    auto fetch = [&](int b) {  // batch b from memory, then the words of the batch after next
      return b < nb ? "  s" + S(b % kFlight) + " = CXR_FETCH(e" + S(b % 2) + ");\n" + load_entry(b + 2) : std::string();
    };
    auto land = [&](int b) {  // batch b to the ring, its register to batch b + kFlight
      return b < nb ? "  CXR_LAND(" + S(b) + ", s" + S(b % kFlight) + ");\n" + fetch(b + kFlight) : std::string();
    };
    auto issue_put = [&](int j) {
      return j < static_cast<int>(puts.size()) ? "  p" + S(j % kIdx) + " = CXR_IDX(@" + S(puts[j]) + "@);\n" : std::string();
    };
    out += "  { CXR_CHUNK();\n" + load_entry(0) + load_entry(1);
    for (int b = 0; b < kFlight; ++b) out += fetch(b);
    for (int b = 0; b < kLand; ++b) out += land(b);
    for (int j = 0; j < kIdx; ++j) out += issue_put(j);
    out += "  }\n";
    for (const std::string& c : chunks) {
      out += "  { CXR_CHUNK();\n";
      for (size_t p = 0; p < c.size();) {
        const size_t q = c.find_first_of("\x01\x03", p);
        if (q == std::string::npos) {
          out += c.substr(p);
          break;
        }
        out += c.substr(p, q - p);
        const int j = std::atoi(c.c_str() + q + 1);
        out += c[q] == '\x01' ? land(j + kLand) : issue_put(j + kIdx);
        p = c.find('\x02', q) + 1;
      }
      out += "  }\n";
    }
    chunks.clear();
    puts.clear();
    phase0 = entry.size();
    reached = -1;
  }
};

// Lowest free lane, or -1.
int take(std::set<int>& free_set) {
  if (free_set.empty()) return -1;
  const int l = *free_set.begin();
  free_set.erase(free_set.begin());
  return l;
}

std::set<int> lanes_upto(int n) {
  std::set<int> s;
  for (int l = 0; l < n; ++l) s.insert(l);
  return s;
}

void finish(RowsEmit& E, const std::string& decl, const std::string& tail, RowsProgram& P) {
  // store rows follow the staged entries in the table
  const int64_t base = static_cast<int64_t>(E.entry.size()) / kLanes;
  std::string text;
  for (size_t p = 0; p < E.out.size();) {
    const size_t q = E.out.find('@', p);
    if (q == std::string::npos) {
      text += E.out.substr(p);
      break;
    }
    const size_t e = E.out.find('@', q + 1);
    text += E.out.substr(p, q - p) + S(base + std::atoll(E.out.c_str() + q + 1));
    p = e + 1;
  }
  unsigned staged = 0;
  for (int w : E.entry) staged |= 1u << (static_cast<unsigned>(w) >> 29);
  std::string o = "// batches up to " + S(P.limit) + "\n#define CXR_STAGED " + S(staged) + "\n";
  o += kRowsPrologue;
  o += "CXR_BODY(cxr_body) {\n  CXR_SETUP();\n" + decl;
  for (int j = 0; j < kFlight; ++j) o += "  vd s" + S(j) + " = 0.0;\n";
  o += "  vi e0 = 0, e1 = 0;\n";
  for (int j = 0; j < kIdx; ++j) o += "  vi p" + S(j) + " = 0;\n";
  o += text + tail + "}\n";
  // one block: 16 instances, whose rows of f, d and z fill whole 128-byte lines
  o += "#ifndef CXR_EMULATED\nextern \"C\" __global__ void __launch_bounds__(256) " + std::string(P.kernel) +
       "(const CxrArgs A) {\n  __shared__ double ring[4][" + S(4 * (kRing + kLanes)) + "];\n"
       "  cxr_body(A, (long long)blockIdx.x * 16 + (threadIdx.x >> 4), (int)(threadIdx.x & 15), ring[threadIdx.x >> 6]);\n}\n"
       "#endif\n";
  P.source = std::move(o);
  P.tab = std::move(E.entry);
  P.tab.insert(P.tab.end(), E.rows.begin(), E.rows.end());
}

// Largest batch of a program whose pivots hold `values` values in all, `wide`
// a pivot or more being worth kRowsMost.  The sixteen-lane programs spend the
// same instructions on a pivot however many of the lanes hold something, on four
// times the wavefronts: ahead while the one-lane programs leave SIMDs idle,
// behind once those fill the chip, and the sooner the fewer values there are.
// 274 rows, us per call, sixteen-lane / one-lane:
//   LDL factor + solve, 2.0 values a pivot (tridiagonal): 103 / 124 at 8192
//   instances, 133 / 126 at 12288, 319 / 237 at 32768; 3.0: 157 / 164 at 12288,
//   186 / 175 at 14336; 5.0: 262 / 304 at 16384, 479 / 421 at 32768; 6.7 (control
//   KKT): 155 / 336 at 8192, 537 / 576 at 32768; 8.9: 696 / 810 at 32768
//   LDL factor alone: 2.0: 96 / 96 at 12288; 5.0: 205 / 280 at 16384, 375 / 336
//   at 32768; 6.7: 439 / 489 at 32768
//   LDL solve alone (little to do per pivot): 2.0: 82 / 98 at 8192, 102 / 98 at
//   10240; 5.0: 167 / 167 at 12288, 235 / 195 at 16384; 6.7: 197 / 242 at 12288,
//   566 / 393 at 32768
//   QR factor + solve, 6.0: 372 / 434 at 16384, 677 / 606 at 32768 (factor alone
//   355 / 506, 643 / 620); 9.9: 876 / 989 at 32768; 12.0 (control KKT): 1132 / 1251 at 32768, 1613 / 1558 at 49152
int64_t batch_limit(int64_t values, int pivots, double wide, int64_t most) {
  const double per_pivot = static_cast<double>(values) / pivots;
  return std::min(most, per_pivot >= wide ? kRowsMost : static_cast<int64_t>(4096 * per_pivot));
}

using Idx = std::vector<int>;
Idx none() { return Idx(kLanes, -1); }

}  // namespace

// The LDL^T of one pattern; false when it does not fit sixteen lanes.
bool rows_ldl_source(int n, const std::vector<int>& a_colind, const std::vector<int>& a_row,
                     const std::vector<int>& lt_colind, const std::vector<int>& lt_row, const std::vector<int>& p,
                     int part, RowsProgram& P) {
  if (n <= 0) return false;
  // members[r]: the rows c > r of L with an entry in column r, with its nonzero
  std::vector<std::vector<std::pair<int, int>>> members(n);
  std::vector<int> first(n), last(n);
  for (int c = 0; c < n; ++c) first[c] = last[c] = c;
  for (int c = 0; c < n; ++c)
    for (int k = lt_colind[c]; k < lt_colind[c + 1]; ++k) {
      const int r = lt_row[k];
      if (k > lt_colind[c] && lt_row[k - 1] >= r) return false;  // rows of a column in increasing order
      members[r].push_back({c, k});
      first[c] = std::min(first[c], r);
      last[r] = std::max(last[r], c);
    }
  std::map<std::pair<int, int>, int> a_at;  // (permuted row, column) -> nonzero of A: the last one wins, as in the scatter
  std::vector<int> pinv(n);
  for (int i = 0; i < n; ++i) pinv[p[i]] = i;
  for (int c1 = 0; c1 < n; ++c1)
    for (int k = a_colind[c1]; k < a_colind[c1 + 1]; ++k) a_at[{pinv[a_row[k]], pinv[c1]}] = k;
  auto a_nz = [&](int r, int c) {  // entry (p[r], p[c]) as column c's scatter reads it
    auto it = a_at.find({r, c});
    return it == a_at.end() ? -1 : it->second;
  };
  const bool factor = part != LS_SOLVE, solve = part != LS_FACTOR;
  RowsEmit E;
  // ---- forward: the factor, and the solve with L
  std::vector<std::vector<int>> act(n);
  for (int c = 0; c < n; ++c) act[first[c]].push_back(c);
  // A row's lane is free again once the columns it has entries in are dead:
  // a new row then finds the zeros it starts from.  Where that takes more
  // than sixteen lanes, lanes are reused from the row's own pivot on, its
  // entries cleared there.
  std::vector<int> until(n);
  for (int c = 0; c < n; ++c) {
    until[c] = c;
    for (int k = lt_colind[c]; k < lt_colind[c + 1]; ++k) until[c] = std::max(until[c], last[lt_row[k]]);
  }
  std::vector<int> lane(n, -1);
  bool clear = false;
  for (int pass = 0; pass < 2; ++pass, clear = true) {
    std::set<int> free_lane = lanes_upto(kLanes);
    std::vector<std::vector<int>> ends(n);
    bool ok = true;
    for (int r = 0; r < n && ok; ++r) {
      for (int c : act[r]) {
        ok = ok && (lane[c] = take(free_lane)) >= 0;
        ends[clear ? c : until[c]].push_back(c);
      }
      for (int c : ends[r]) free_lane.insert(lane[c]);
    }
    if (ok) break;
    if (clear) return false;
  }
  std::set<int> free_slot;
  int n_slot = 0;
  unsigned active = 0;  // lanes whose row is not final
  std::vector<int> slot(n, -1);
  std::vector<std::vector<int>> dies(n);  // columns whose slot is free after pivot r
  std::vector<unsigned> mem(n, 0);        // lanes of column r's entries
  std::vector<int64_t> block(n + 1, 0);   // first kept value of pivot r
  for (int r = 0; r < n; ++r) {
    const int q = lane[r];
    const unsigned own = 1u << q;
    const std::string rs = S(r), qs = S(q);
    if (!act[r].empty()) {
      Idx dw = none(), bw = none();
      unsigned am = 0, dm = 0;
      for (int c : act[r]) {
        const int l = lane[c];
        am |= 1u << l;
        bw[l] = RowsEmit::word('x', p[c]);
        if (a_nz(c, c) >= 0) {
          dw[l] = RowsEmit::word('a', a_nz(c, c));
          dm |= 1u << l;
        }
      }
      active |= am;
      if (factor) {
        if (dm) E.set(dm, "d", E.entries(dm, dw));
        E.set(am & ~dm, "d", "vd(0.0)");
      }
      if (solve) E.set(am, "y", E.entries(am, bw));
    }
    for (const auto& m : members[r]) mem[r] |= 1u << lane[m.first];
    block[r + 1] = block[r] + popcount(mem[r] | own);
    // lanes that must keep their row's d and y; the others (the owner, free
    // lanes) are set before they are read again
    const unsigned upd = (active & ~mem[r] & ~own) ? mem[r] : 0xffffu;
    if (!factor) {  // the pivots are stored: the owner's D, the members' L
      Idx dw = none(), lw = none();
      dw[q] = RowsEmit::word('d', r);
      for (const auto& m : members[r]) lw[lane[m.first]] = RowsEmit::word('f', m.second);
      E.body += "  const vd c" + rs + " = " + E.entries(own, dw) + ";\n  vd t" + rs + " = y / c" + rs + ";\n";
      if (mem[r]) {
        E.body += "  const vd l" + rs + " = " + E.entries(mem[r], lw) + ";\n  const vd y" + rs + " = CXR_BC(y, " + qs + ");\n";
        E.set(upd, "y", "y - l" + rs + " * y" + rs);
        E.set(mem[r], "t" + rs, "l" + rs);
      }
      E.body += "  CXR_KEEP_BLOCK(" + S(block[r]) + ", " + hexmask(mem[r] | own) + ", t" + rs + ");\n";
    } else {
      E.body += "  const vd d" + rs + " = CXR_BC(d, " + qs + ");\n  cnt = cnt + CXR_BAD(d" + rs + ");\n  CXR_KEEP(cnt);\n";
      std::string num = "y";
      if (mem[r]) {
        Idx aw = none();
        unsigned am = 0;
        for (const auto& m : members[r]) {
          // L^T(r, c) starts from A(p[r], p[c]) as column c's scatter left it
          const int l = lane[m.first], nz = a_nz(r, m.first);
          if (nz < 0) continue;
          aw[l] = RowsEmit::word('a', nz);
          am |= 1u << l;
        }
        num = "v" + rs;
        E.body += "  vd " + num + " = 0.0;\n";
        // the lanes outside the column compute alongside; nothing reads them
        if (am) E.set(am == mem[r] ? 0xffffu : am, num, E.entries(am, aw));
        for (int k = lt_colind[r]; k < lt_colind[r + 1]; ++k) {
          const std::string s = S(slot[lt_row[k]]);
          E.body += "  " + num + " = " + num + " - CXR_BC(l" + s + ", " + qs + ") * w" + s + ";\n";
        }
        if (solve) {  // the owner divides its y: z = y / d
          E.body += "  vd n" + rs + " = " + num + ";\n";
          num = "n" + rs;
          E.set(own, num, "y");
        }
      }
      if (mem[r] || solve) E.body += "  const vd t" + rs + " = " + num + " / d" + rs + ";\n";
      if (clear)  // the owner's row is final: its entries leave the lane as zeros
        for (int k = lt_colind[r]; k < lt_colind[r + 1]; ++k)
          if (last[lt_row[k]] > r) E.set(own, "w" + S(slot[lt_row[k]]), "vd(0.0)");
      if (mem[r]) {
        if (free_slot.empty()) free_slot.insert(n_slot++);
        if (n_slot > kMaxSlots) return false;
        slot[r] = take(free_slot);
        dies[last[r]].push_back(r);
        const std::string s = S(slot[r]);
        if (solve) E.body += "  const vd y" + rs + " = CXR_BC(y, " + qs + ");\n";
        E.set(upd, "d", "d - v" + rs + " * t" + rs);
        if (solve) E.set(upd, "y", "y - t" + rs + " * y" + rs);
        E.body += "  w" + s + " = CXR_SEL(" + hexmask(mem[r]) + ", v" + rs + ", vd(0.0));\n  l" + s + " = t" + rs + ";\n";
      }
      if (solve) {  // the members' L and the owner's z
        E.body += "  CXR_KEEP_BLOCK(" + S(block[r]) + ", " + hexmask(mem[r] | own) + ", t" + rs + ");\n";
      } else {
        Idx li = none(), ri = none();
        for (const auto& m : members[r]) li[lane[m.first]] = m.second;
        ri[q] = r;
        if (mem[r]) E.put('f', mem[r], li, "t" + rs);
        E.put('d', own, ri, "d" + rs);
      }
      for (int s : dies[r]) free_slot.insert(slot[s]);
    }
    active &= ~own;
    if (r % kChunk == kChunk - 1) E.end_chunk();
  }
  E.end_phase();
  // ---- back substitution with L^T: x(r) in row r's lane
  if (solve) {
    E.out += "  CXR_SYNC();\n";
    for (int j = 0; j < kBack; ++j) E.out += "  vd k" + S(j) + " = 0.0;\n";
    auto kept = [&](int r) {
      if (r < 0) return std::string();
      const std::string v = "  k" + S(r % kBack) + " = ", at = S(block[r]);
      return v + (mem[r] ? "CXR_KEPT(" + at + ", " + hexmask(mem[r] | 1u << lane[r]) + ");\n" : "CXR_KEPT1(" + at + ");\n");
    };
    for (int j = 1; j <= kBack; ++j) E.body += kept(n - j);
    for (int r = n - 1; r >= 0; --r) {
      const std::string rs = S(r);
      E.body += "  const vd b" + rs + " = k" + S(r % kBack) + ";\n" + kept(r - kBack) + "  vd x" + rs + " = CXR_BC(b" + rs + ", " +
                S(lane[r]) + ");\n";
      if (mem[r]) {
        E.body += "  const vd m" + rs + " = b" + rs + " * y;\n";
        for (auto m = members[r].rbegin(); m != members[r].rend(); ++m)
          E.body += "  x" + rs + " = x" + rs + " - CXR_BC(m" + rs + ", " + S(lane[m->first]) + ");\n";
      }
      E.set(1u << lane[r], "y", "x" + rs);
      E.body += "  CXR_PUT_x(1, " + S(p[r]) + ", x" + rs + ");\n";
      if (r % kChunk == 0) E.end_chunk();
    }
    E.end_phase();
  }
  std::string decl = "  vd y = 0.0;\n  (void)y;\n";
  if (factor) {
    decl += "  vd d = 0.0;\n  vi cnt = 0;\n";
    for (int s = 0; s < n_slot; ++s) decl += "  vd w" + S(s) + " = 0.0, l" + S(s) + " = 0.0;\n";
  }
  P.kernel = part == LS_FUSED ? "cxj_ldl_rows" : part == LS_FACTOR ? "cxj_ldl_rows_fact" : "cxj_ldl_rows_solve";
  P.kept = solve ? block[n] : 0;
  P.limit = batch_limit(block[n], n, 6.0, part == LS_SOLVE ? 12288 : kRowsMost);
  finish(E, decl, factor ? "  CXR_COUNT(cnt);\n" : "", P);
  return true;
}

// The QR of one pattern: factor and solve (one right-hand side, not
// transposed) or the factor alone.
bool rows_qr_source(int ncol, int nrow, const std::vector<int>& a_colind, const std::vector<int>& a_row,
                    const std::vector<int>& v_colind, const std::vector<int>& v_row, const std::vector<int>& r_colind,
                    const std::vector<int>& r_row, const std::vector<int>& prinv, const std::vector<int>& pc, int part,
                    RowsProgram& P) {
  if (ncol <= 0 || part == LS_SOLVE) return false;
  const bool solve = part == LS_FUSED;
  const int rhs = kLanes - 1;  // the right-hand side's lane (fused)
  std::vector<std::vector<std::pair<int, int>>> members(ncol);  // row r of R: (column c > r, nonzero)
  std::vector<int> first(ncol), diag(ncol);
  std::vector<std::map<int, int>> acol(ncol);  // column c of the permuted A: row -> nonzero (the last one wins)
  for (int c = 0; c < ncol; ++c) {
    first[c] = c;
    std::set<int> fill;
    for (int k = a_colind[pc[c]]; k < a_colind[pc[c] + 1]; ++k) {
      acol[c][prinv[a_row[k]]] = k;
      fill.insert(prinv[a_row[k]]);
    }
    int before = -1;
    for (int k = r_colind[c]; k < r_colind[c + 1]; ++k) {
      const int r = r_row[k];
      if (r <= before || r > c) return false;
      before = r;
      if (r == c) {
        diag[c] = k;
        continue;
      }
      members[r].push_back({c, k});
      first[c] = std::min(first[c], r);
      for (int q = v_colind[r]; q < v_colind[r + 1]; ++q) fill.insert(v_row[q]);
      fill.erase(r);
    }
    if (before != c || v_colind[c + 1] <= v_colind[c] || v_row[v_colind[c]] != c) return false;
    std::set<int> mine;
    for (int k = v_colind[c]; k < v_colind[c + 1]; ++k) {
      if (v_row[k] < c || !mine.insert(v_row[k]).second) return false;
    }
    // what the reflections leave in the work vector must lie in V's column
    // (else it would reach the next column of the sequential algorithm)
    if (!std::includes(mine.begin(), mine.end(), fill.begin(), fill.end())) return false;
  }
  // rows: live from the first column or reflection that holds them to their
  // pivot (rows past the last column: to their last reflection)
  std::vector<int> entry(nrow, ncol), death(nrow, -1);
  for (int c = 0; c < ncol; ++c) {
    for (const auto& kv : acol[c]) entry[kv.first] = std::min(entry[kv.first], first[c]);
    for (int k = v_colind[c]; k < v_colind[c + 1]; ++k) {
      const int i = v_row[k];
      entry[i] = std::min(entry[i], c);
      death[i] = std::max(death[i], c);
    }
  }
  for (int i = 0; i < nrow; ++i)
    if (entry[i] < ncol && death[i] < entry[i]) return false;
  std::vector<int> b_of(nrow, -1);  // row i starts from the right-hand side's entry b_of[i]
  for (int c = 0; c < ncol; ++c) b_of[prinv[c]] = c;
  std::vector<std::vector<int>> act(ncol), enter(ncol), leave(ncol);
  for (int c = 0; c < ncol; ++c) act[first[c]].push_back(c);
  for (int i = 0; i < nrow; ++i)
    if (entry[i] < ncol) {
      enter[entry[i]].push_back(i);
      leave[death[i]].push_back(i);
    }
  RowsEmit E;
  std::set<int> free_lane = lanes_upto(solve ? kLanes - 1 : kLanes), free_slot;
  int n_slot = 0;
  std::vector<int> lane(ncol, -1), slot(nrow, -1);
  std::set<int> live;
  unsigned active = 0;  // lanes whose column is not final
  std::vector<unsigned> mems(ncol, 0);
  std::vector<int64_t> block(ncol + 1, 0);
  for (int r = 0; r < ncol; ++r) {
    const std::string rs = S(r);
    for (int c : act[r])
      if ((lane[c] = take(free_lane)) < 0) return false;
    unsigned am = 0;
    for (int c : act[r]) am |= 1u << lane[c];
    active |= am;
    std::vector<char> fresh(nrow, 0);
    for (int i : enter[r]) {
      if (free_slot.empty()) free_slot.insert(n_slot++);
      if (n_slot > kMaxSlots) return false;
      slot[i] = take(free_slot);
      live.insert(i);
      fresh[i] = 1;
    }
    for (int i : live) {  // the new columns' entries of the live rows; new rows are zero in every other lane
      if (!am && !fresh[i]) continue;
      Idx gw = none();
      unsigned gm = 0;
      for (int c : act[r]) {
        auto it = acol[c].find(i);
        if (it == acol[c].end()) continue;
        gw[lane[c]] = RowsEmit::word('a', it->second);
        gm |= 1u << lane[c];
      }
      if (solve && fresh[i] && b_of[i] >= 0) {
        gw[rhs] = RowsEmit::word('x', b_of[i]);
        gm |= 1u << rhs;
      }
      const std::string x = "x_" + S(slot[i]);
      const unsigned zm = (fresh[i] ? 0xffffu : am) & ~gm;
      E.set(zm, x, "vd(0.0)");
      if (gm) E.set(gm, x, E.entries(gm, gw));
    }
    // casadi_house on the owner's column (the other lanes compute alongside)
    const int q = lane[r];
    const std::string qs = S(q);
    const unsigned own = 1u << q;
    std::vector<std::string> xs;
    for (int k = v_colind[r]; k < v_colind[r + 1]; ++k) xs.push_back("x_" + S(slot[v_row[k]]));
    E.body += "  vd sg" + rs + " = 0.0;\n";
    for (size_t k = 1; k < xs.size(); ++k) E.body += "  sg" + rs + " = sg" + rs + " + " + xs[k] + " * " + xs[k] + ";\n";
    // both branches of each selection are computed: a branch around a division
    // costs more than the division
    E.body += "  const vd sq" + rs + " = CXR_SQRT(" + xs[0] + " * " + xs[0] + " + sg" + rs + ");\n" +
              "  const vd va" + rs + " = " + xs[0] + " - sq" + rs + ", vb" + rs + " = -sg" + rs + " / (" + xs[0] + " + sq" + rs +
              ");\n  const vd vc" + rs + " = CXR_LE0(" + xs[0] + ", va" + rs + ", vb" + rs + ");\n" +
              "  const vd vn" + rs + " = CXR_EQ0(sg" + rs + ", vd(1.0), vc" + rs + ");\n" +
              "  const vd ba" + rs + " = CXR_LE0(" + xs[0] + ", vd(2.0), vd(0.0)), bb" + rs + " = vd(-1.0) / (sq" + rs + " * vn" +
              rs + ");\n  const vd be" + rs + " = CXR_EQ0(sg" + rs + ", ba" + rs + ", bb" + rs + ");\n" +
              "  cnt = cnt + CXR_SMALL(CXR_BC(sq" + rs + ", " + qs + "), A.eps);\n  CXR_KEEP(cnt);\n";
    unsigned mem = 0;
    Idx si = none();
    for (const auto& m : members[r]) {
      mem |= 1u << lane[m.first];
      si[lane[m.first]] = m.second;
    }
    if (solve) mem |= 1u << rhs;
    mems[r] = mem | own;
    block[r + 1] = block[r] + popcount(mem | own);
    const bool keep = !solve;  // the factor alone stores V and beta
    if (mem || keep) {
      E.body += "  const vd h" + rs + "_0 = CXR_BC(vn" + rs + ", " + qs + ");\n";
      for (size_t k = 1; k < xs.size(); ++k)
        E.body += "  const vd h" + rs + "_" + S(k) + " = CXR_BC(" + xs[k] + ", " + qs + ");\n";
      E.body += "  const vd hb" + rs + " = CXR_BC(be" + rs + ", " + qs + ");\n";
    }
    if (mem) {
      std::string t = "vd al = 0.0;";
      for (size_t k = 0; k < xs.size(); ++k) t += " al = al + h" + rs + "_" + S(k) + " * " + xs[k] + ";";
      t += " al = al * hb" + rs + ";";
      for (size_t k = 0; k < xs.size(); ++k) t += " " + xs[k] + " = " + xs[k] + " - al * h" + rs + "_" + S(k) + ";";
      // columns outside row r of R keep their entries; the owner's and free
      // lanes are set before they are read again
      const bool all = !(active & ~mem & ~own);
      E.body += (all ? std::string("  { ") : "  CXR_WHERE(" + hexmask(mem) + ") { ") + t + " }\n";
    }
    // row r of R (and of Q'b)
    E.body += "  vd ro" + rs + " = " + xs[0] + ";\n";
    E.set(own, "ro" + rs, "sq" + rs);
    si[q] = diag[r];
    if (solve) E.body += "  CXR_KEEP_BLOCK(" + S(block[r]) + ", " + hexmask(mem | own) + ", ro" + rs + ");\n";
    else E.put('f', mem | own, si, "ro" + rs);
    if (keep) {
      // V's column, sixteen entries to a store
      for (size_t k0 = 0; k0 < xs.size(); k0 += kLanes) {
        const std::string nm = "vs" + rs + "_" + S(k0);
        E.body += "  vd " + nm + " = h" + rs + "_" + S(k0) + ";\n";
        Idx vi = none();
        unsigned vm = 0;
        for (size_t k = k0; k < std::min(xs.size(), k0 + kLanes); ++k) {
          vi[k - k0] = v_colind[r] + static_cast<int>(k);
          vm |= 1u << (k - k0);
          if (k > k0) E.set(1u << (k - k0), nm, "h" + rs + "_" + S(k));
        }
        E.put('z', vm, vi, nm);
      }
      Idx bi = none();
      bi[0] = r;
      E.put('d', 1u, bi, "hb" + rs);
    }
    for (int i : leave[r]) {
      live.erase(i);
      free_slot.insert(slot[i]);
    }
    free_lane.insert(q);
    active &= ~own;
    if (r % kChunk == kChunk - 1) E.end_chunk();
  }
  E.end_phase();
  if (solve) {  // back substitution with R: x(r) in column r's lane
    E.out += "  CXR_SYNC();\n";
    for (int j = 0; j < kBack; ++j) E.out += "  vd k" + S(j) + " = 0.0;\n";
    auto kept = [&](int r) {  // lane 15 is in every mask: no lane reads past a block
      return r >= 0 ? "  k" + S(r % kBack) + " = CXR_KEPT(" + S(block[r]) + ", " + hexmask(mems[r]) + ");\n" : std::string();
    };
    for (int j = 1; j <= kBack; ++j) E.body += kept(ncol - j);
    for (int r = ncol - 1; r >= 0; --r) {
      const std::string rs = S(r);
      E.body += "  const vd b" + rs + " = k" + S(r % kBack) + ";\n" + kept(r - kBack) + "  vd x" + rs + " = CXR_BC(b" + rs + ", " +
                S(rhs) + ");\n";
      if (!members[r].empty()) {
        E.body += "  const vd m" + rs + " = b" + rs + " * y;\n";
        for (auto m = members[r].rbegin(); m != members[r].rend(); ++m)
          E.body += "  x" + rs + " = x" + rs + " - CXR_BC(m" + rs + ", " + S(lane[m->first]) + ");\n";
      }
      E.body += "  const vd z" + rs + " = x" + rs + " / CXR_BC(b" + rs + ", " + S(lane[r]) + ");\n";
      E.set(1u << lane[r], "y", "z" + rs);
      E.body += "  CXR_PUT_x(1, " + S(pc[r]) + ", z" + rs + ");\n";
      if (r % kChunk == 0) E.end_chunk();
    }
    E.end_phase();
  }
  std::string decl = "  vi cnt = 0;\n";
  if (solve) decl += "  vd y = 0.0;\n";
  for (int s = 0; s < n_slot; ++s) decl += "  vd x_" + S(s) + " = 0.0;\n";
  P.kernel = solve ? "cxj_qr_rows" : "cxj_qr_rows_fact";
  P.kept = solve ? block[ncol] : 0;
  P.limit = batch_limit(block[ncol] + (solve ? 0 : ncol), ncol, 8.0, kRowsMost);  // the right-hand side's lane in both
  finish(E, decl, "  CXR_COUNT(cnt);\n", P);
  return true;
}

bool rows_ready(RowsProgram& P) {
  if (!P.fn) {
    hipFunction_t f = jit_function(P.source, P.kernel);
    if (scratch_bytes(f) > 0) return false;  // not launched, as no generated kernel that spills is
    P.fn = f;
    P.d_tab.upload(P.tab.data(), P.tab.size() * sizeof(int));
  }
  return true;
}

void rows_launch(RowsProgram& P, int64_t n_inst, const RowsIO& io, hipStream_t s) {
  struct {
    const void* a;
    void *x, *f, *d, *z, *w;
    const int* tab;
    int* status;
    long long a_t, x_t;
    uint32_t a_s, x_s, ld, w_t;
    double eps;
    long long n;
  } A{io.a, io.x, io.f, io.d, io.z, io.w, P.d_tab.as<int>(), io.status, static_cast<long long>(io.a_t * 8),
      static_cast<long long>(io.x_t * 8), static_cast<uint32_t>(io.a_s * 8), static_cast<uint32_t>(io.x_s * 8),
      static_cast<uint32_t>(io.ld * 8), static_cast<uint32_t>(P.kept * 8), io.eps, n_inst};
  void* params[] = {&A};
  hip_check(hipModuleLaunchKernel(P.fn, static_cast<unsigned>((n_inst + 15) / 16), 1, 1, 256, 1, 1, 0, s, params, nullptr),
            "linsol rows launch");
}

}  // namespace sxh
