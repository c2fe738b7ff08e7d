// The recurrent layer when its workgroups give up waiting for one another: this copy of the kernels polls once
// (SLAYER_GRID_POLLS = 0), so every workgroup leaves at its first wait that is not already over and the layer is computed
// by the kernels behind.  Compared with the copy in recurrent_waiting.hip, whose workgroups do wait: forward bit for bit, also with
// weights that have all their 24 bits, backward to the order of summation.
#define SLAYER_GRID_POLLS 0
#define slayer slayer_solo                                   // its names are not the library's
// No workgroup waits for another here, so they need not all be on the chip at once (and the runtime grants
// cooperative launches to one process at a time).
#include <hip/hip_runtime.h>
#define hipLaunchCooperativeKernel hipLaunchKernel
#include "../../lava-dl_amd/csrc/recurrent_grid.hip"
#include <cmath>
#include <cstdio>
#include <vector>

namespace slayer {
unsigned* range_flag_device() { return nullptr; }
void range_flag_raise_from_host() {}
}  // namespace slayer

bool waiting_fwd(const void* step, bool alif, float* spk, float* vol, float* theta, const float* z, const float* rec, float* ws,
                 int64_t floats, int* error);
bool waiting_bwd(float* gz, const float* g, const float* v, const float* theta, const float* rec, int64_t N, int64_t C, int64_t T,
                 float* ws, int64_t floats, int* error);

static int check(hipError_t e, const char* what) {
    if (e != hipSuccess) { printf("%s: %s\n", what, hipGetErrorString(e)); exit(1); }
    return 0;
}
static float* device(const std::vector<float>& v) {
    float* d = nullptr;
    check(hipMalloc(&d, v.size() * 4), "hipMalloc");
    check(hipMemcpy(d, v.data(), v.size() * 4, hipMemcpyHostToDevice), "upload");
    return d;
}
static std::vector<float> host(const float* d, size_t n) {
    std::vector<float> v(n);
    check(hipMemcpy(v.data(), d, n * 4, hipMemcpyDeviceToHost), "download");
    return v;
}

int main() {
    using namespace slayer;
    const int N = 18, C = 1300, T = 20;                      // two sample tiles, two neurons per thread of the solo kernels
    const size_t nct = (size_t)N * C * T, nc = (size_t)N * C;
    unsigned state = 12345u;
    auto uniform = [&]() { state = state * 1664525u + 1013904223u; return (float)(state >> 8) / (1 << 24) * 2.0f - 1.0f; };
    std::vector<float> z(nct), g(nct), rec((size_t)C * C);
    for (auto& x : z) x = 2.5f * uniform();
    for (auto& x : g) x = uniform();
    const float par[] = {1024.f, 512.f, 256.f, 2048.f, 0.f, 1.25f};   // decays; states at rest; threshold state
    float *dz = device(z), *dg = device(g), *dr = device(rec), *dp = device(std::vector<float>(par, par + 6));
    const int64_t floats = slayer_recurrent_steps_workspace(N, C, T, 1);
    float* ws = device(std::vector<float>((size_t)floats));
    float* out[2][3];                                        // spikes, voltage, theta: waiting, solo
    float* last[2][4];
    float* gz[2];
    for (int k = 0; k < 2; ++k) {
        for (auto& p : out[k]) p = device(std::vector<float>(nct));
        for (auto& p : last[k]) p = device(std::vector<float>(nc));
        gz[k] = device(std::vector<float>(nct));
    }
    int bad = 0;
    auto gave_up = [&](const char* what, int k) {            // the mark is the integer 1
        if ((host(ws, 1)[0] != 0.0f) != (k == 1)) { printf("%s %d: workgroups that should %s\n", what, k, k ? "give up" : "wait"); ++bad; }
    };
    for (int form = 0; form < 4; ++form) {
        const int alif = form & 1, real = form >> 1;
        // real weights: a scale that shows every bit of a sum in the voltage
        const int scale = real ? 1 << 20 : 64;
        const int64_t th0 = 5 * scale / 4;
        for (auto& x : rec) x = real ? uniform() / 8 : std::rint(8.0f * uniform()) / 64.0f;
        check(hipMemcpy(dr, rec.data(), rec.size() * 4, hipMemcpyHostToDevice), "weights");
        StepFwd p{};
        p.i_decay = dp; p.v_decay = dp + 1; p.th_decay = dp + 2; p.ref_decay = dp + 3;
        p.i_state = p.v_state = p.ref_state = dp + 4; p.th_state = dp + 5;
        p.n_id = p.n_vd = p.n_td = p.n_rd = p.n_is = p.n_vs = p.n_ts = p.n_rs = 1;
        p.w = (float)scale; p.inv_w = 1.0f / p.w; p.spike_thr = 1.25f; p.spike_scale = 1.0f; p.th_step_f = 0.5f; p.base = (int)th0;
        p.N = N; p.C = C; p.T = T;
        for (int k = 0; k < 2; ++k) {
            p.cur_last = last[k][0]; p.vol_last = last[k][1]; p.th_last = last[k][2]; p.ref_last = last[k][3];
            int error = 0;
            const bool taken = k == 0 ? waiting_fwd(&p, alif != 0, out[k][0], out[k][1], out[k][2], dz, dr, ws, floats, &error)
                                      : grid_fwd(p, alif != 0, true, out[k][0], out[k][1], out[k][2], dz, dr, ws, floats, nullptr, &error);
            if (!taken || error) { printf("forward %d not taken: %d\n", k, error); return 1; }
            check(hipDeviceSynchronize(), "forward");
            gave_up("forward", k);
        }
        double spikes = 0;
        for (int o = 0; o < 2 + alif; ++o) {
            const auto a = host(out[0][o], nct), b = host(out[1][o], nct);
            for (size_t i = 0; i < nct; ++i) { bad += a[i] != b[i]; if (o == 0) spikes += a[i]; }
        }
        for (int o = 0; o < (alif ? 4 : 2); ++o) {
            const auto a = host(last[0][o], nc), b = host(last[1][o], nc);
            for (size_t i = 0; i < nc; ++i) bad += a[i] != b[i];
        }
        if (spikes < 0.01 * nct || spikes > 0.9 * nct) { printf("spike rate %g\n", spikes / nct); ++bad; }
        const float* theta = alif ? out[0][2] : nullptr;
        for (int k = 0; k < 2; ++k) {
            int error = 0;
            const bool taken = k == 0 ? waiting_bwd(gz[k], dg, out[0][1], theta, dr, N, C, T, ws, floats, &error)
                                      : grid_bwd(gz[k], dg, out[0][1], theta, dr, 1.25f, 1.0f, 0.1f, 0, N, C, T, ws, floats, nullptr, &error);
            if (!taken || error) { printf("backward %d not taken: %d\n", k, error); return 1; }
            check(hipDeviceSynchronize(), "backward");
            gave_up("backward", k);
        }
        const auto a = host(gz[0], nct), b = host(gz[1], nct);
        double diff = 0, most = 0;
        for (size_t i = 0; i < nct; ++i) { diff = std::max(diff, (double)std::fabs(a[i] - b[i])); most = std::max(most, (double)std::fabs(a[i])); }
        if (!(diff <= 1e-5 * most) || most == 0) { printf("backward: %g of %g\n", diff, most); ++bad; }
    }
    printf(bad ? "%d differences\n" : "solo kernels agree\n", bad);
    return bad != 0;
}
