// Independent parts of a Jacobian sweep (jit_parts.hip).
#pragma once
#include <memory>
#include <vector>

#include "tape_internal.hpp"

namespace sxh {

// One class of isomorphic parts: a tape and Jacobian plan of its own over
// local inputs, outputs and nonzeros.  Local input li of the plan is row
// rows[li] of its block, local output lo row rows[n_in + lo], local nonzero q
// nonzero rows[n_in + n_out + q], with the part's rows at
// first_row + part * row_len of the table.
struct PartClass {
  cxh_tape_s tape;
  cxh_jac_s jac;
  int count = 0;  // parts of this class
  int n_in = 0, n_out = 0, n_q = 0;
  int64_t first_row = 0;
  const std::vector<int>* rows = nullptr;  // the table
  int row_len() const { return n_in + n_out + n_q; }
};

// The parts of a plan by class, the one with the most work first, and their
// row table; empty when the tape does not split into repeated parts.
std::vector<std::unique_ptr<PartClass>> find_parts(const cxh_jac_s* j, std::vector<int>& rows);

}  // namespace sxh
