// Window-only and dense compressed forward over runs of consecutive tokens
// (sas_fwd_win.hip).
#pragma once

#include "sas_kern.h"

namespace sas {

constexpr int kRunTokens = 64;       // tokens of a run, at most
constexpr int kDenseWinRows = 192;   // dense compressed scenario: win_left + run, at most
constexpr int kDenseCmpRows = 128;   // and its compressed rows

// Cache rows in the query dtype, one split, `run` tokens per workgroup. SWA:
// windows of at most 128 rows. CFA: H a multiple of 64 (fp.nhg = H / 64),
// within the limits above.
int launch_fwd_win(const FwdParams& fp, int D, int q_dtype, int run, hipStream_t st);

}  // namespace sas
