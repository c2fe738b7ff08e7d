// The recurrent kernels of the library, whose workgroups wait for one another, behind a plain launch: the reference side of
// recurrent_solo_check.hip.  (The runtime grants cooperative launches to one process at a time, and the process that starts the check
// may hold them: the library would then take a launch per step, which sums in another order.)  The check leaves the rest of the
// chip idle, and its grid is smaller than the chip, so all workgroups run at once; every wait is bounded all the same.
#define slayer slayer_waiting                                // its names are not the library's
#include <hip/hip_runtime.h>
#define hipLaunchCooperativeKernel hipLaunchKernel
#include "../../lava-dl_amd/csrc/recurrent_grid.hip"
#include <cstring>

namespace slayer {
unsigned* range_flag_device() { return nullptr; }
void range_flag_raise_from_host() {}
}  // namespace slayer

// step: the StepFwd of the check
bool waiting_fwd(const void* step, bool alif, float* spk, float* vol, float* theta, const float* z, const float* rec, float* ws,
                 int64_t floats, int* error) {
    slayer::StepFwd p;
    memcpy(&p, step, sizeof p);
    return slayer::grid_fwd(p, alif, true, spk, vol, theta, z, rec, ws, floats, nullptr, error);
}
bool waiting_bwd(float* gz, const float* g, const float* v, const float* theta, const float* rec, int64_t N, int64_t C, int64_t T,
                 float* ws, int64_t floats, int* error) {
    return slayer::grid_bwd(gz, g, v, theta, rec, 1.25f, 1.0f, 0.1f, 0, N, C, T, ws, floats, nullptr, error);
}
