// capi_internal.h -- descriptor checks and derived constants shared by the
// single-box (capi.hip) and multi-box (capi_batch.hip) entry points.
#pragma once

#include <string>

#include "../../include/nmhd.h"
#include "nmhd_kernels.h"

namespace nmhd {

// Validate a box descriptor; on failure `why` names the offending field.
bool desc_valid(const nmhd_desc *d, std::string &why);

// Derived constants, in FP32 exactly as the reference's constant
// expressions (simulation_config_default.h:79-103).
void derive_box(const nmhd_desc *d, Box &b, nmhd_geometry &g);

// The frozen-dt step W_out = S(W_in; dt) of a periodic box with the
// production stage kernels, enqueued on s: Wstar holds the midpoint stage
// state (unused for NMHD_EULER1).  F: the 11 arrays that the face march hands
// to the update (tiled::stage_buf), the others null, or all 21, which the
// kernels of small boxes (direct_stage) need.
void enqueue_frozen_step(hipStream_t s, const Box &b, int integrator, FieldPtrs Win,
                         FieldPtrs Wstar, FieldPtrs Wout, const FluxSet &F, float dt);

// Floats from one field-sized array to the next in a block of them: an odd
// number of 256-byte lines, so that a cell's values in the arrays a kernel
// streams side by side lie in different memory channels.  As separate
// allocations, a multiple of 2 MiB apart each, the update took 398 / 432 us at
// 256^3 against 388 / 421, and 801 / 876 at 512x520x128 against 775 / 848.
inline size_t array_stride(long ncell) { return (((size_t)ncell + 63) / 64 | 1) * 64; }

// The CFL minimum of a record read back.
float cfl_minimum(const StepRec &r);

// The message nmhd_adj_last_error(NULL) returns (failures of calls that
// have no nmhd_adj object).
void set_adj_global_error(const std::string &msg);

}  // namespace nmhd
