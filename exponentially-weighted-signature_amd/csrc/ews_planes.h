// Host entry points of the wave-per-chunk plane kernels (ews_planes.hip), called by the C ABI in ews_diag.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "ews_args.h"

namespace ews {

// True if the configuration has wave-per-chunk kernels: rotation planes at depth 2, 3 to 16 of them, rows of every step
// (prefix or log rows), per-interval flows, chunk length at most 64, and a leaf whose coefficients are those of the
// closed forms.
bool planes_eligible(const DiagArgs& a);
// Every chunk's class (a.cflag, a.chbar) and the summaries of the strictly uniform ones.
int planes_summary(const DiagArgs& a, hipStream_t st);
// Their prefix rows from the chunk carries (a.log unset: the log rows are the generic kernels').
int planes_rows(const DiagArgs& a, hipStream_t st);
// Strictly uniform chunks of the backward: the cotangent on the carry-in state of the chunk's own rows.
int planes_local(const DiagArgs& a, hipStream_t st);
// The full adjoint of the invertible ones among them, without the clock gradient.
int planes_full(const DiagArgs& a, hipStream_t st);

}  // namespace ews
