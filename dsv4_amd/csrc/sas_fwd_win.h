// Window-only forward over runs of consecutive tokens (sas_fwd_win.hip).
#pragma once

#include "sas_kern.h"

namespace sas {

// Windows of at most 128 rows, cache rows in the query dtype, one split, `run`
// tokens per workgroup.
int launch_fwd_win(const FwdParams& fp, int D, int q_dtype, int run, hipStream_t st);

}  // namespace sas
