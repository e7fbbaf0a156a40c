// Bit-exact parallel ranlxs2 stream and ziggurat Gaussians.
#pragma once
#include "gic_common.h"
#include "rng_plan.h"
#include <vector>

namespace gic {

// Draw the stream's Gaussians into the listed targets in order, as the
// reference's serial loop does: a padded real field (n > 0, count n^3, cell
// order x, y, z) or a dense array (n == 0, count values).  Each value is
// stored as T(v * scale).
struct RngLevelOut {
  void *field;       // T*
  int n;
  size_t count;
};
template <typename T>
void rng_draw_real(const RngPlan &plan, const std::vector<RngLevelOut> &levels, void *workspace, size_t ws_bytes,
                   hipStream_t st, struct TimingHook *hook, double scale = 1.0, uint32_t *cover_flag = nullptr,
                   int flag_stride = 0, const void *dev_plan = nullptr);
// With cover_flag the draw has no host synchronisation: a device check sets
// cover_flag[i * flag_stride] to 1 if stream i held too few Gaussians (the
// cells past the end are then left as they were); without, the call waits
// for the draw and raises an error.
// dev_plan: the plan already in device memory (rng_dev_pack'd, rng_dev_bytes
// long, copied there by the caller); otherwise the call puts it into the
// workspace.

// Draws into a caller's device array with the fixed per-device workspace:
// rng_scratch_setup(device) once per device with that device current, then
// rng_gaussians_noalloc (no device allocation; at most
// rng_noalloc_max_gaussians() values; overlapping calls on one GPU race).
void rng_scratch_setup(int device);
size_t rng_noalloc_max_gaussians();
void rng_gaussians_noalloc(int device, unsigned long seed, double *dev_out, size_t n, hipStream_t st);

// Raw 24-bit stream (testing / bit-exactness checks): the first n numbers.
void rng_raw(const RngPlan &plan, uint32_t *d_out, size_t n, hipStream_t st);

}  // namespace gic
