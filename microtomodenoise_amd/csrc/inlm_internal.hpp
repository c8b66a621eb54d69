// Library-internal helpers shared between translation units.
#pragma once
#include <cstddef>
#include <cstdint>
#include <functional>
#include <string>

#include <hip/hip_runtime.h>

#include "inlm_capi.h"

namespace inlm {

// message returned by inlm_last_error(NULL)
void set_global_error(const std::string &msg);

// The host half of get_noiselevel (noiselevel.cpp:9-95): sigma per slice
// from the per-sample patch stds sd[0..n) of the sorted sample list, in the
// parameters' noise mode.  which = 0: first estimate; semi_ref keeps the
// semimanual reference sample between estimates.
inlm_status sigma_from_std(const inlm_params &p, const int shape[3], const int64_t *samples, const double *sd,
                           int64_t n, int which, int64_t &semi_ref, float *sig, std::string &err);

// Whether sigma_from_std is the quicker one: no clustering, or one of few
// samples.  Its time goes with the samples of all windows, times their
// iterations, which grow with a window: samples times their count's bits.  The
// GPU takes 10 to 30 us more than the host for a few samples.  An estimate by
// the host and the GPU, us: one window of 300 samples (cost 2700) 38 / 54, of
// 700 (7000) 48 / 56, of 1000 (10000) 57 to 70 / 60 to 68; 64 windows of about
// 24 (7800) 51 / 62, 256 of 5 (3900) 39 / 49, 16 of 94 (10600) 65 / 62, 16 of
// 100 (11300) 88 / 59.
constexpr int64_t kHostClusterCost = 9000;
bool clusters_on_host(const inlm_params &p, const int shape[3], const int64_t *samples, int64_t n);

// The same in the global and z-adaptive modes from standard deviations on the
// device (n >= 1), clustered there; work: cluster_bytes(nz) of device memory.
// Returns when sig is written.
size_t cluster_bytes(int nz);
inlm_status sigma_on_device(const inlm_params &p, const int shape[3], const int64_t *samples, int64_t n,
                            const double *std_dev, void *work, hipStream_t st, float *sig, std::string &err);

// Elements of a padded volume's allocation behind its guard (flat: the patch
// has no z radius).
struct Geometry;
size_t padded_elems(const Geometry &g, bool flat);

// Device bytes a handle of these parameters allocates for `shape`.
size_t handle_bytes(const inlm_params &p, const int32_t shape[3]);

// Anscombe transform and its algebraic inverse (Color/colorspace.h:87-123)
void anscombe(float *v, size_t n);
void inverse_anscombe(float *v, size_t n);

// The colour schedule; on_iteration(iter, channels) sees (and may change)
// each iteration's result on the host before it is used further.
inlm_status denoise_rgb(const inlm_params *p, const inlm_rgb_options *c, const int32_t shape[2], int32_t device,
                        const float *in, float *out, float *sigma_log,
                        const std::function<bool(int, float *)> &on_iteration);

}  // namespace inlm
