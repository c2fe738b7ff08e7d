// What the two multi-workgroup forms of the recurrent layer share (recurrent_grid.hip: the whole time loop in one
// launch; recurrent_steps.hip: a launch per time step): their arguments and one step of one neuron.
#pragma once
#include "common.h"
#include "tile.h"

namespace slayer {

struct StepFwd {
    float *spk_t, *vol_t, *theta_t;                           // [T][N][C]; theta: ALIF only
    const float* z_t;                                         // [T][N][C]
    int* carried;                                             // [4][N][C]: current, voltage, threshold, refractory
    float *cur_last, *vol_last, *th_last, *ref_last;          // [N*C]; th / ref: ALIF only
    const float4* rec_packed;                                 // see pack_weights_kernel
    float4* spk_packed;                                       // two buffers of [KB][S][64] quads, written in turn
    int KB, S;                                                // blocks of 16 neurons, sample tiles
    const float *i_decay, *v_decay, *th_decay, *ref_decay, *i_state, *v_state, *th_state, *ref_state;
    int64_t n_id, n_vd, n_td, n_rd, n_is, n_vs, n_ts, n_rs;
    float w, inv_w, spike_thr, spike_scale, th_step_f;
    int base;
    int N, C, T;
    unsigned* range_flag;                                     // see raise_range_flag in tile.h
};

struct StepValues { float spike, current, voltage, theta, threshold, refractory; };

// The carried states of one neuron and its step: that of recurrent_fwd_kernel (recurrent.hip), state by state -- each
// starts from the float32 value the previous step left and hands a float32 value on, as between two one-step
// neuron calls.
template <bool ALIF, bool GRADED, bool POW2>
struct StepNeuron {
    int yc, yv, th, r;                                        // current, voltage, threshold, refractory state
    int mi, mv, mt, mr;                                       // their multipliers
    unsigned acc_lif, acc_th;                                 // range of the states, see range_bits in tile.h

    __device__ __forceinline__ void track() {
        if (ALIF) acc_th |= ((unsigned)th + (1u << 28)) | ((unsigned)r + (1u << 28));
    }
    // the initial states and the multipliers against their bounds
    __device__ __forceinline__ void check(unsigned* flag) {
        check_multiplier(mi, flag); check_multiplier(mv, flag);
        if (ALIF) { check_multiplier(mt, flag); check_multiplier(mr, flag); }
        acc_lif |= ((unsigned)yc + (1u << 30)) | ((unsigned)yv + (1u << 30));
        track();
    }
    __device__ __forceinline__ void load_decays(const StepFwd& p, int c) {
        mi = 4096 - trunc_i32(rintf(p.i_decay[p.n_id == 1 ? 0 : c]));
        mv = 4096 - trunc_i32(rintf(p.v_decay[p.n_vd == 1 ? 0 : c]));
        if (ALIF) {
            mt = 4096 - trunc_i32(rintf(p.th_decay[p.n_td == 1 ? 0 : c]));
            mr = 4096 - trunc_i32(rintf(p.ref_decay[p.n_rd == 1 ? 0 : c]));
        }
    }
    __device__ __forceinline__ void load_states(const StepFwd& p, int64_t m) {
        yc = trunc_i32(p.i_state[p.n_is == 1 ? 0 : m] * p.w);
        yv = trunc_i32(p.v_state[p.n_vs == 1 ? 0 : m] * p.w);
        if (ALIF) {
            th = trunc_i32(p.th_state[p.n_ts == 1 ? 0 : m] * p.w);
            r = trunc_i32(p.ref_state[p.n_rs == 1 ? 0 : m] * p.w);
        }
    }
    // A step in three parts, so that what the feedback is waited for with is as short as can be: what depends on the
    // carried states alone; the spike; the states the next step starts from.
    int cd, vd;                                               // decayed current and voltage
    float cur, vol, theta, thf, rf;
    static __device__ __forceinline__ float from(int y, const StepFwd& p) { const float f = (float)y; return POW2 ? f * p.inv_w : f / p.w; }
    __device__ __forceinline__ void decay(const StepFwd& p) {
        cd = rs0_12(yc, mi);
        vd = rs0_12(yv, mv);
        theta = p.spike_thr; thf = 0.f; rf = 0.f;
        if (ALIF) {
            r = rs0_12(r, mr);
            th = rs0_12(th - p.base, mt) + p.base;
            track();
            thf = from(th, p);
            rf = from(r, p);
            theta = thf + rf;
        }
    }
    __device__ __forceinline__ float fire(float dend, const StepFwd& p) {
        yc = add_sat(cd, trunc_i32(p.w * dend));
        cur = from(yc, p);
        yc = trunc_i32(p.w * cur);
        yv = add_sat(vd, yc);
        vol = from(yv, p);
        const bool fired = vol >= theta;
        return GRADED ? ((fired ? 1.0f : 0.0f) * vol) / p.spike_scale : (fired ? 1.0f : 0.0f);
    }
    __device__ __forceinline__ void carry(float s, const StepFwd& p) {
        acc_lif |= ((unsigned)yc + (1u << 30)) | ((unsigned)yv + (1u << 30));
        const bool spiked = s > 0.0f;                          // what the carried states see
        if (ALIF) {
            yv = trunc_i32(p.w * vol);
            r = trunc_i32((spiked ? rf + 2.0f * thf : rf) * p.w);
            th = trunc_i32((spiked ? thf + p.th_step_f : thf) * p.w);
        } else {
            yv = spiked ? 0 : trunc_i32(p.w * vol);
        }
    }
    __device__ __forceinline__ StepValues step(float dend, const StepFwd& p) {
        decay(p);
        const float s = fire(dend, p);
        carry(s, p);
        return StepValues{s, cur, vol, theta, thf, rf};
    }
};

// recurrent_grid.hip.  Both return true when the call is done (*error: 0, or what went wrong) and false when it is not one
// for them: a layer, a batch or a sequence of another size, a stream under capture, a device that does not hold the grid.
bool grid_fwd(StepFwd p, bool alif, bool pow2, float* spk, float* vol, float* theta, const float* z, const float* rec,
              float* workspace, int64_t workspace_floats, hipStream_t st, int* error);
bool grid_bwd(float* gz, const float* grad_spikes, const float* voltage, const float* theta, const float* rec,
              float spike_thr, float tau, float rho, int graded, int64_t N, int64_t C, int64_t T,
              float* workspace, int64_t workspace_floats, hipStream_t st, int* error);

}  // namespace slayer
