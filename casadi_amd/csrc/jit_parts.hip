// Independent parts of a Jacobian or Hessian sweep.
//
// The gradient of a multiple-shooting Lagrangian (and any Function that
// evaluates one expression on many slices of its inputs) is a tape whose
// values fall into sets that never meet: stage k's terms depend on x_k, u_k
// and lam_k only.  Run as one program per instance, the tape costs its whole
// length in code (the 20-stage quadrotor gradient is 14 589 instructions:
// eight kernels of four direction groups, every stage streamed through the
// instruction cache once per wavefront) and in latency, on n / 64 wavefronts
// per group.
//
// Here the tape is taken apart into those sets.  Parts whose instructions,
// constants, seeds and scatter agree up to the rows they touch are one class:
// one program, run side by side over instances and parts.  The rows of its
// inputs, outputs and nonzeros are computed from the part's number where they
// advance by a fixed step from part to part, and read from a table where not.  Every value is computed by the same operations
// on the same operands as before, so the bits do not change.
//
// Measured, quadrotor Lagrangian Hessian, whole-tape kernels / parts: horizon
// 20 at 16384 instances 636 / 249 us, at 1001 302 / 29, at 64 234 / 14; horizon
// 3 at 16384 59 / 44.  First-call compile 37 / 2 s.  What bounds it now is VALU
// issue and the chains of about one wavefront per SIMD (3280 VALU instructions per
// wavefront of a stage's group, VALU active in 54% of the wavefronts' cycles, 424 MB
// of traffic against 398), four groups computing a stage's primal again.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cstdint>
#include <cstring>
#include <map>
#include <numeric>
#include <set>
#include <string>
#include <utility>
#include <vector>

#include "jit_parts.hpp"
#include "sx_ops.h"

namespace sxh {

namespace {

constexpr int64_t kMaxPart = 4096;  // instructions of one part's program, its inputs and constants included: one kernel
constexpr int64_t kSmall = 512;    // classes with fewer instructions in all run together as one part

struct Part {
  std::vector<int64_t> instr;  // its instructions, in tape order
};

int64_t root(std::vector<int64_t>& up, int64_t k) {
  while (up[k] != k) k = up[k] = up[up[k]];
  return k;
}

// One part as a plan over local rows; `sign` receives what its class is
// known by.
std::unique_ptr<PartClass> localise(const cxh_jac_s* j, const std::vector<int64_t>& instr, const std::vector<int64_t>& d1,
                                    const std::vector<int64_t>& d2, std::vector<int>& rows, std::string& sign) {
  const cxh_tape_s* t = j->tape;
  const int nd = j->ndir;
  auto P = std::make_unique<PartClass>();
  std::vector<Instr>& alg = P->tape.alg;
  int ws = 0;
  std::map<int64_t, int> slot;                     // instruction -> local slot
  std::map<std::pair<int, int>, int> in_slot;      // (block, row) -> local slot
  std::map<uint64_t, int> const_slot;
  std::vector<std::pair<int, int>> ins, outs;      // (block, row) in local order
  auto konst = [&](double v) {
    uint64_t bits;
    std::memcpy(&bits, &v, sizeof bits);
    auto it = const_slot.find(bits);
    if (it != const_slot.end()) return it->second;
    Instr e{};
    e.op = OP_CONST;
    e.i0 = ws++;
    e.d = v;
    alg.push_back(e);
    const_slot.emplace(bits, e.i0);
    return e.i0;
  };
  auto operand = [&](int64_t u) {
    if (u < 0) return konst(0.0);  // a slot never written
    const Instr& e = t->alg[u];
    if (e.op == OP_CONST) return konst(e.d);
    if (e.op != OP_INPUT) return slot.at(u);
    const std::pair<int, int> key{e.i1, e.i2};
    auto it = in_slot.find(key);
    if (it != in_slot.end()) return it->second;
    Instr x{};
    x.op = OP_INPUT;
    x.i0 = ws++;
    x.i1 = e.i1;
    x.i2 = static_cast<int>(ins.size());
    alg.push_back(x);
    ins.push_back(key);
    in_slot.emplace(key, x.i0);
    return x.i0;
  };
  for (int64_t k : instr) {
    const Instr& e = t->alg[k];
    Instr x{};
    x.op = e.op;
    if (e.op == OP_OUTPUT) {
      x.i1 = operand(d1[k]);
      x.i0 = e.i0;
      x.i2 = static_cast<int>(outs.size());
      outs.push_back({e.i0, e.i2});
    } else {
      x.i1 = operand(d1[k]);
      x.i2 = op_is_binary(e.op) ? operand(d2[k]) : x.i1;
      x.i0 = ws++;
      slot[k] = x.i0;
    }
    alg.push_back(x);
  }
  // directions that seed one of the part's inputs or scatter one of its
  // outputs, ordered by what they do here (their own numbers differ from
  // part to part)
  std::vector<std::pair<std::string, int>> dirs;
  for (int d = 0; d < nd; ++d) {
    std::string key;
    bool any = false;
    for (const auto& in : ins) {
      const double v = j->seedval[(j->in_off[in.first] + in.second) * static_cast<int64_t>(nd) + d];
      key.append(reinterpret_cast<const char*>(&v), sizeof v);
      any |= v != 0.0;
    }
    for (const auto& o : outs) {
      const int2 tg = j->scatter[(j->out_off[o.first] + o.second) * static_cast<int64_t>(nd) + d];
      key += static_cast<char>((tg.x >= 0) + 2 * (tg.y >= 0));
      any |= tg.x >= 0 || tg.y >= 0;
    }
    if (any) dirs.push_back({key, d});
  }
  std::stable_sort(dirs.begin(), dirs.end(), [](const auto& x, const auto& y) { return x.first > y.first; });
  const int ld = static_cast<int>(dirs.size());
  P->n_in = static_cast<int>(ins.size());
  P->n_out = static_cast<int>(outs.size());
  for (const auto& in : ins) rows.push_back(in.second);
  for (const auto& o : outs) rows.push_back(o.second);
  cxh_jac_s& J = P->jac;
  J.ndir = ld;
  J.seedval.assign(static_cast<size_t>(std::max(P->n_in, 1)) * std::max(ld, 1), 0.0);
  J.scatter.assign(static_cast<size_t>(std::max(P->n_out, 1)) * std::max(ld, 1), int2{-1, -1});
  for (int d = 0; d < ld; ++d) {
    for (int i = 0; i < P->n_in; ++i)
      J.seedval[static_cast<size_t>(i) * ld + d] =
          j->seedval[(j->in_off[ins[i].first] + ins[i].second) * static_cast<int64_t>(nd) + dirs[d].second];
    for (int o = 0; o < P->n_out; ++o) {
      const int2 tg = j->scatter[(j->out_off[outs[o].first] + outs[o].second) * static_cast<int64_t>(nd) + dirs[d].second];
      int2& l = J.scatter[static_cast<size_t>(o) * ld + d];
      for (int h = 0; h < 2; ++h) {
        const int q = h ? tg.y : tg.x;
        if (q < 0) continue;
        (h ? l.y : l.x) = P->n_q++;
        rows.push_back(q);
      }
    }
  }
  P->tape.ws = std::max(ws, 1);
  P->tape.nnz_in.assign(t->nnz_in.size(), 0);
  P->tape.nnz_out.assign(t->nnz_out.size(), 0);
  J.nnz_jac = P->n_q;
  J.in_off.assign(t->nnz_in.size(), 0);
  J.out_off.assign(t->nnz_out.size(), 0);
  sign.assign(reinterpret_cast<const char*>(alg.data()), alg.size() * sizeof(Instr));
  sign += "/" + std::to_string(P->n_in) + "/" + std::to_string(ld) + "/";
  for (const auto& d : dirs) sign += d.first;
  return P;
}

}  // namespace

std::vector<std::unique_ptr<PartClass>> find_parts(const cxh_jac_s* j, std::vector<int>& rows) {
  const cxh_tape_s* t = j->tape;
  const int64_t n = static_cast<int64_t>(t->alg.size());
  std::vector<std::unique_ptr<PartClass>> out;
  rows.clear();
  if (j->ndir == 0 || n < 2 * kSmall) return out;
  // operands as defining instructions; sets of operations that meet
  std::vector<int64_t> cur(t->ws, -1), d1(n, -1), d2(n, -1), up(n);
  std::iota(up.begin(), up.end(), int64_t{0});
  auto meets = [&](int64_t k, int64_t u) {
    if (u >= 0 && t->alg[u].op != OP_CONST && t->alg[u].op != OP_INPUT) up[root(up, u)] = root(up, k);
  };
  std::set<std::pair<int, int>> written;
  for (int64_t k = 0; k < n; ++k) {
    const Instr& e = t->alg[k];
    if (e.op == OP_CONST || e.op == OP_INPUT) {
      cur[e.i0] = k;
      continue;
    }
    meets(k, d1[k] = cur[e.i1]);
    if (e.op == OP_OUTPUT) {
      if (!written.insert({e.i0, e.i2}).second) return out;  // the last write counts, and parts have no order
      continue;
    }
    if (op_is_binary(e.op)) meets(k, d2[k] = cur[e.i2]);
    cur[e.i0] = k;
  }
  std::vector<Part> parts;
  std::map<int64_t, size_t> at;
  for (int64_t k = 0; k < n; ++k) {
    if (t->alg[k].op == OP_CONST || t->alg[k].op == OP_INPUT) continue;
    auto it = at.emplace(root(up, k), parts.size());
    if (it.second) parts.emplace_back();
    parts[it.first->second].instr.push_back(k);
  }
  if (parts.size() < 2) return out;
  // classes, before the small ones are gathered
  std::map<std::string, std::vector<size_t>> classes;
  std::vector<std::string> sign(parts.size());
  for (size_t p = 0; p < parts.size(); ++p) {
    std::vector<int> unused;
    localise(j, parts[p].instr, d1, d2, unused, sign[p]);
    classes[sign[p]].push_back(p);
  }
  std::vector<std::vector<size_t>> groups;  // the parts of each class, in tape order
  Part rest;                                // every class with little to do, as one part
  for (const auto& c : classes) {
    int64_t work = 0;
    for (size_t p : c.second) work += static_cast<int64_t>(parts[p].instr.size());
    if (work >= kSmall) {
      groups.push_back(c.second);
    } else {
      for (size_t p : c.second) rest.instr.insert(rest.instr.end(), parts[p].instr.begin(), parts[p].instr.end());
    }
  }
  if (!rest.instr.empty()) {
    std::sort(rest.instr.begin(), rest.instr.end());
    parts.push_back(rest);
    groups.push_back({parts.size() - 1});
  }
  auto work = [&](const std::vector<size_t>& g) {
    return static_cast<int64_t>(g.size() * parts[g[0]].instr.size());
  };
  std::sort(groups.begin(), groups.end(), [&](const auto& x, const auto& y) {
    return work(x) != work(y) ? work(x) > work(y) : x[0] < y[0];
  });
  // Worth it when the longest part is at most half of the tape: the parts run
  // side by side, so that is what the chain of one instance shrinks to.  Many
  // classes are many programs in one kernel.
  int64_t longest = 0, ops = 0;
  for (const auto& g : groups) {
    longest = std::max(longest, static_cast<int64_t>(parts[g[0]].instr.size()));
    ops += work(g);
  }
  if (longest * 2 > ops || longest > kMaxPart || groups.size() > 16) return out;  // and the localised part, below
  for (const auto& g : groups) {
    const int64_t first = static_cast<int64_t>(rows.size());
    std::unique_ptr<PartClass> C;
    std::string s;
    for (size_t p : g) {
      auto L = localise(j, parts[p].instr, d1, d2, rows, s);
      if (!C) C = std::move(L);
    }
    if (static_cast<int64_t>(C->tape.alg.size()) > kMaxPart) {
      rows.clear();
      return {};
    }
    C->count = static_cast<int>(g.size());
    C->first_row = first;
    C->jac.tape = &C->tape;
    C->jac.seg_len = kMaxPart;  // one kernel
    out.push_back(std::move(C));
  }
  return out;
}

}  // namespace sxh
