// Host vocabulary of the sixteen-lanes-per-instance programs, for the tests:
// a vd is the sixteen lanes of one instance, an assignment inside CXR_WHERE
// reaches only the lanes of its mask, a broadcast reads one lane.  Every
// gather and scatter is checked against the registered buffers, and a lane's
// store must not meet another lane's store of the same phase.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <map>
#include <vector>

#define CXR_EMULATED

namespace rows_emu {
static unsigned mask = 0xffffu;
static long long errors = 0;
struct Region {
  uintptr_t lo, hi;
};
static std::vector<Region> regions;
static bool inside(const void* p) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  for (const Region& r : regions)
    if (a >= r.lo && a + 8 <= r.hi) return true;
  if (errors++ < 8) std::fprintf(stderr, "[rows] access outside every buffer: %p\n", p);
  return false;
}
struct Where {
  unsigned old;
  bool run = true;
  explicit Where(unsigned m) : old(mask) { mask &= m; }
  ~Where() { mask = old; }
  bool once() { return run ? (run = false, true) : false; }
};
}  // namespace rows_emu

template <class T>
struct lanes16 {
  T v[16];
  lanes16(T x = T()) {
    for (T& e : v) e = x;
  }
  lanes16(const lanes16& o) {
    for (int l = 0; l < 16; ++l) v[l] = o.v[l];
  }
  lanes16& operator=(const lanes16& o) {
    for (int l = 0; l < 16; ++l)
      if (rows_emu::mask >> l & 1u) v[l] = o.v[l];
    return *this;
  }
};
typedef lanes16<double> vd;
typedef lanes16<int> vi;
#define ROWS_OP(op)                                    \
  static vd operator op(const vd& a, const vd& b) {    \
    vd r;                                              \
    for (int l = 0; l < 16; ++l) r.v[l] = a.v[l] op b.v[l]; \
    return r;                                          \
  }
ROWS_OP(+) ROWS_OP(-) ROWS_OP(*) ROWS_OP(/)
static vd operator-(const vd& a) {
  vd r;
  for (int l = 0; l < 16; ++l) r.v[l] = -a.v[l];
  return r;
}
static vi operator+(const vi& a, const vi& b) {
  vi r;
  for (int l = 0; l < 16; ++l) r.v[l] = a.v[l] + b.v[l];
  return r;
}
static vd rows_map(const vd& a, double (*f)(double)) {
  vd r;
  for (int l = 0; l < 16; ++l) r.v[l] = f(a.v[l]);
  return r;
}
static vd rows_pick(const vd& c, bool le, const vd& a, const vd& b) {
  vd r;
  for (int l = 0; l < 16; ++l) r.v[l] = (le ? c.v[l] <= 0 : c.v[l] == 0) ? a.v[l] : b.v[l];
  return r;
}
static vi rows_flag(const vd& a, double e, bool small) {
  vi r;
  for (int l = 0; l < 16; ++l)
    r.v[l] = small ? !(std::fabs(a.v[l]) >= e) : !(a.v[l] != 0 && std::isfinite(a.v[l]));
  return r;
}
static vd rows_bc(const vd& a, int q) { return vd(a.v[q]); }
// the entry of staged word e for instance i
template <class Args>
static double rows_fetch(const Args& A, int e, long long i) {
  const unsigned k = static_cast<unsigned>(e) & 0x1fffffffu, what = static_cast<unsigned>(e) >> 29;
  const char* p = what == 0 ? A.a + i * A.a_t : what == 1 ? A.x + i * A.x_t : (what == 2 ? A.f : what == 3 ? A.d : A.z) + i * 8;
  p += static_cast<long long>(k) * (what == 0 ? A.a_s : what == 1 ? A.x_s : A.ld);
  return rows_emu::inside(p) ? *reinterpret_cast<const double*>(p) : 0.0;
}
static int rows_rank(unsigned m, int l) { return __builtin_popcount(m & ((1u << l) - 1u)); }
// a ring slot that was never written reads as NaN
static vd rows_ring(const double* ring, int start, unsigned m) {
  vd r(NAN);
  for (int l = 0; l < 16; ++l)
    if (m >> l & 1u) r.v[l] = ring[start + rows_rank(m, l)];
  return r;
}
// every lane of the wavefront reads, the lanes outside the mask a value that
// nothing uses
static vd rows_kept(const char* w, unsigned m) {
  vd r(NAN);
  for (int l = 0; l < 16; ++l) {
    const char* p = w + rows_rank(m, l) * 8;
    if (rows_emu::inside(p) && (m >> l & 1u)) r.v[l] = *reinterpret_cast<const double*>(p);
  }
  return r;
}
static void rows_keep(char* w, unsigned m, const vd& x) {
  for (int l = 0; l < 16; ++l) {
    char* p = w + rows_rank(m, l) * 8;
    if ((m >> l & 1u) && rows_emu::inside(p)) *reinterpret_cast<double*>(p) = x.v[l];
  }
}
static void rows_put(unsigned m, char* base, const vi& idx, long long stride, const vd& x) {
  std::map<const void*, int> seen;
  for (int l = 0; l < 16; ++l) {
    if (!(m >> l & 1u)) continue;
    char* p = base + idx.v[l] * stride;
    if (!seen.emplace(p, l).second && rows_emu::errors++ < 8) std::fprintf(stderr, "[rows] two lanes store to %p\n", (void*)p);
    if (rows_emu::inside(p)) *reinterpret_cast<double*>(p) = x.v[l];
  }
}
static vi rows_idx(const int* tab, long long j) {
  vi r;
  for (int l = 0; l < 16; ++l) r.v[l] = tab[j * 16 + l];
  return r;
}

#define CXR_WHERE(m) for (rows_emu::Where w_(static_cast<unsigned>(m)); w_.once();)
static vd rows_sel(unsigned m, const vd& a, const vd& b) {
  vd r;
  for (int l = 0; l < 16; ++l) r.v[l] = (m >> l & 1u) ? a.v[l] : b.v[l];
  return r;
}
#define CXR_SEL(m, a, b) rows_sel(static_cast<unsigned>(m), a, b)
#define CXR_BC(v, q) rows_bc(v, q)
#define CXR_IDX(j) rows_idx(A.tab, j)
// a batch's words and values: sixteen entries in the sixteen elements
#define CXR_ENTRY(b) rows_idx(A.tab, b)
#define CXR_FETCH(e_) rows_batch(A, e_, i)
#define CXR_LAND(b, x) do { for (int l = 0; l < 16; ++l) ring[((b) % 8) * 16 + l] = (x).v[l]; } while (0)
#define CXR_RING(start, m) rows_ring(ring, start, static_cast<unsigned>(m))
#define CXR_KEPT1(off) (rows_emu::inside(A.w + i * A.w_t + (off) * 8) ? vd(*(const double*)(A.w + i * A.w_t + (off) * 8)) : vd(NAN))
#define CXR_KEPT(off, m) rows_kept(A.w + i * A.w_t + (off) * 8, static_cast<unsigned>(m))
#define CXR_KEEP_BLOCK(off, m, v) rows_keep(A.w + i * A.w_t + (off) * 8, static_cast<unsigned>(m), v)
template <class Args>
static vd rows_batch(const Args& A, const vi& e, long long i) {
  vd r;
  for (int l = 0; l < 16; ++l) r.v[l] = rows_fetch(A, e.v[l], i);
  return r;
}
#define CXR_PUT_f(m, i_, v) rows_put(m, pf, i_, A.ld, v)
#define CXR_PUT_d(m, i_, v) rows_put(m, pd, i_, A.ld, v)
#define CXR_PUT_z(m, i_, v) rows_put(m, pz, i_, A.ld, v)
#define CXR_PUT_x(m, i_, v) rows_put(m, px, vi(i_), A.x_s, v)
#define CXR_BAD(v) rows_flag(v, 0.0, false)
#define CXR_SMALL(v, e) rows_flag(v, e, true)
#define CXR_SQRT(v) rows_map(v, [](double t) { return std::sqrt(t); })
#define CXR_EQ0(c, a_, b_) rows_pick(c, false, a_, b_)
#define CXR_LE0(c, a_, b_) rows_pick(c, true, a_, b_)
#define CXR_KEEP(c) ((void)0)
#define CXR_SYNC() ((void)0)
#define CXR_COUNT(c) do { if (A.status) A.status[i] = (c).v[0]; } while (0)
#define CXR_BODY(name) static void name(const CxrArgs& A, const long long i)
#define CXR_SETUP()                                        \
  char* const px = A.x ? A.x + i * A.x_t : nullptr;         \
  char* const pf = A.f ? A.f + i * 8 : nullptr;             \
  char* const pd = A.d ? A.d + i * 8 : nullptr;             \
  char* const pz = A.z ? A.z + i * 8 : nullptr;             \
  double ring[128];                                         \
  for (double& r_ : ring) r_ = NAN;                         \
  (void)px; (void)pf; (void)pd; (void)pz
#define CXR_CHUNK() ((void)0)

extern "C" {
void rows_clear() {
  rows_emu::regions.clear();
  rows_emu::errors = 0;
}
void rows_region(const void* p, long long bytes) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  rows_emu::regions.push_back({a, a + static_cast<uintptr_t>(bytes)});
}
long long rows_errors() { return rows_emu::errors; }
}
