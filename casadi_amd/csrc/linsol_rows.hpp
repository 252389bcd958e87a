// Batched LDL^T / QR with sixteen lanes per instance (linsol_rows.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "tape_internal.hpp"

namespace sxh {

constexpr int64_t kRowsMost = 32768;  // no sixteen-lane program serves a larger batch

// A generated program, its index table and, once compiled, its kernel.
struct RowsProgram {
  const char* kernel = "";
  std::string source;
  std::vector<int> tab;
  int64_t kept = 0;  // doubles per instance kept between the sweeps (RowsIO::w)
  int64_t limit = 0;  // largest batch it serves by choice (batch_limit)
  DeviceBuffer d_tab;
  hipFunction_t fn = nullptr;
};

// Operands of a launch, strides in doubles: nonzero k of A for instance j at
// a[k*a_s + j*a_t], entry i of the right-hand side and solution at
// x[i*x_s + j*x_t]; f, d, z hold rows of ld doubles (ld a multiple of 64, at
// least n_inst): the factors as the other programs lay them out.  LDL: f =
// L^T's nonzeros, d = D.  QR: f = R's nonzeros, d = beta, z = V's nonzeros.
// w: round_up(n_inst, 16) * RowsProgram::kept doubles (fused, solve alone).
struct RowsIO {
  const double* a = nullptr;
  int64_t a_s = 0, a_t = 0;
  double* x = nullptr;
  int64_t x_s = 0, x_t = 0;
  double *f = nullptr, *d = nullptr, *z = nullptr, *w = nullptr;
  int64_t ld = 0;
  int32_t* status = nullptr;
  double eps = 0;
};

// The program of one part (LinsolPart) of a pattern's factor and solve; false
// when the pattern does not fit (the one-lane programs serve it).
bool rows_ldl_source(int n, const std::vector<int>& a_colind, const std::vector<int>& a_row,
                     const std::vector<int>& lt_colind, const std::vector<int>& lt_row, const std::vector<int>& p,
                     int part, RowsProgram& P);
bool rows_qr_source(int ncol, int nrow, const std::vector<int>& a_colind, const std::vector<int>& a_row,
                    const std::vector<int>& v_colind, const std::vector<int>& v_row, const std::vector<int>& r_colind,
                    const std::vector<int>& r_row, const std::vector<int>& prinv, const std::vector<int>& pc, int part,
                    RowsProgram& P);
// Compiles and loads the program; false when its kernel would need scratch.
bool rows_ready(RowsProgram& P);
void rows_launch(RowsProgram& P, int64_t n_inst, const RowsIO& io, hipStream_t s);

}  // namespace sxh
