// Recurrent layer of CUBA or ALIF neurons: the whole time loop of
//   feedback[t] = R s[t-1];  s[t] = neuron(z[t] + feedback[t])
// in one launch per direction.  The reference runs this loop in Python with one neuron call per
// time step (utils/recurrent.py:45-112), i.e. a dozen launches per step; here one workgroup owns
// one batch sample, one thread one neuron, and a step costs one barrier: the neurons that fired at
// step t-1 travel as per-wave index lists through LDS and the feedback is the sum of the columns of
// R they select (times the spike's value for graded spikes), read as rows of R^T so that
// neighbouring threads read neighbouring addresses.  rec_t carries one extra all-zero row: the lists
// are padded with its index.  Layers of up to kRegisterNeurons take the register form further down.
//
// A neuron called one step at a time carries its state between the calls as float32 (CUBA: current,
// voltage * (1 - spike); ALIF: current, voltage, threshold + spike * step, refractory + 2 * spike *
// threshold); the kernel makes the same round trip, so it matches that loop bit for bit whenever the
// feedback sum is exact in float32 (quantised weights, and for graded spikes quantised voltages that
// keep the products exact), and to float32 summation order otherwise.
#include "common.h"
#include "tile.h"

namespace slayer {

constexpr int kMaxRecurrent = 1024;      // neurons per sample = threads per workgroup
constexpr int kGather = 16;              // rows of the weight matrix a thread keeps in flight

struct RecurrentFwd {
    float *spk, *vol, *theta;                                 // [N][C][T]; theta: ALIF only
    float *cur_last, *vol_last, *th_last, *ref_last;          // [N*C]; th / ref: ALIF only
    const float *z, *rec_t;
    const float *i_decay, *v_decay, *th_decay, *ref_decay, *i_state, *v_state, *th_state, *ref_state;
    int64_t n_id, n_vd, n_td, n_rd, n_is, n_vs, n_ts, n_rs;
    float w, inv_w, spike_thr, spike_scale, th_step_f;
    int base;
    int C, T;
    unsigned* range_flag;                                     // see raise_range_flag in tile.h
};

// Any workgroup of whole waves with at least C threads.
template <bool ALIF, bool GRADED, bool POW2, bool VEC4>
__device__ __forceinline__ void recurrent_fwd_gather(const RecurrentFwd& p) {
    // spikes of the previous step: per wave a count and the indices of its neurons that fired, padded
    // to a multiple of kGather with C, the index of the all-zero row that ends rec_t; graded spikes
    // bring their values along (0 in the padding)
    __shared__ int counts[2][kMaxRecurrent / kWave];
    __shared__ __attribute__((aligned(16))) int fired_list[2][kMaxRecurrent];
    __shared__ __attribute__((aligned(16))) float fired_value[GRADED ? 2 : 1][GRADED ? kMaxRecurrent : 4];
    const int C = p.C, T = p.T;
    const float w = p.w, inv_w = p.inv_w;
    const float* __restrict__ rec_t = p.rec_t;
    const int c = threadIdx.x;
    const int waves = (blockDim.x + kWave - 1) / kWave;
    const bool live = c < C;
    const int64_t m = (int64_t)blockIdx.x * C + (live ? c : 0);
    const float* zrow = p.z + m * (int64_t)T;
    float* srow = p.spk + m * (int64_t)T;
    float* vrow = p.vol + m * (int64_t)T;
    float* trow = ALIF ? p.theta + m * (int64_t)T : nullptr;
    auto from = [&](int y) -> float { const float f = (float)y; return POW2 ? f * inv_w : f / w; };

    int yc = 0, yv = 0, th = 0, r = 0, mi = 0, mv = 0, mt = 0, mr = 0;
    unsigned acc_lif = 0u, acc_th = 0u;                       // range of the states, see range_bits in tile.h
    if (live) {
        yc = trunc_i32(p.i_state[p.n_is == 1 ? 0 : m] * w);
        yv = trunc_i32(p.v_state[p.n_vs == 1 ? 0 : m] * w);
        mi = 4096 - trunc_i32(rintf(p.i_decay[param_index(m, C, p.n_id)]));
        mv = 4096 - trunc_i32(rintf(p.v_decay[param_index(m, C, p.n_vd)]));
        if (ALIF) {
            th = trunc_i32(p.th_state[p.n_ts == 1 ? 0 : m] * w);
            r = trunc_i32(p.ref_state[p.n_rs == 1 ? 0 : m] * w);
            mt = 4096 - trunc_i32(rintf(p.th_decay[param_index(m, C, p.n_td)]));
            mr = 4096 - trunc_i32(rintf(p.ref_decay[param_index(m, C, p.n_rd)]));
            check_multiplier(mt, p.range_flag); check_multiplier(mr, p.range_flag);
        }
        check_multiplier(mi, p.range_flag); check_multiplier(mv, p.range_flag);
        acc_lif = ((unsigned)yc + (1u << 30)) | ((unsigned)yv + (1u << 30));
        acc_th = ((unsigned)th + (1u << 28)) | ((unsigned)r + (1u << 28));
    }
    float cur = 0.f, vol = 0.f, thf = 0.f, rf = 0.f;
    float4 zq = make_float4(0.f, 0.f, 0.f, 0.f), sq = zq, vq = zq, tq = zq;

    for (int t = 0; t < T; ++t) {
        // feedback from the spikes of step t-1 (none before the first step)
        float fb = 0.f;
        if (t > 0) {
            for (int wv = 0; wv < waves; ++wv) {
                const int cnt = __builtin_amdgcn_readfirstlane(counts[(t - 1) & 1][wv]);
                const int4* seg = reinterpret_cast<const int4*>(&fired_list[(t - 1) & 1][wv * kWave]);
                const float4* val = reinterpret_cast<const float4*>(&fired_value[GRADED ? (t - 1) & 1 : 0][GRADED ? wv * kWave : 0]);
                for (int k = 0; k < cnt; k += kGather) {           // kGather rows of R^T in flight at a time
                    int row[kGather];
                    float sv[kGather];
#pragma unroll
                    for (int q = 0; q < kGather / 4; ++q) {
                        const int4 i4 = seg[k / 4 + q];
                        row[4 * q] = i4.x; row[4 * q + 1] = i4.y; row[4 * q + 2] = i4.z; row[4 * q + 3] = i4.w;
                        if (GRADED) {
                            const float4 f4 = val[k / 4 + q];
                            sv[4 * q] = f4.x; sv[4 * q + 1] = f4.y; sv[4 * q + 2] = f4.z; sv[4 * q + 3] = f4.w;
                        }
                    }
                    float v[kGather];
#pragma unroll
                    for (int q = 0; q < kGather; ++q) v[q] = live ? rec_t[row[q] * C + c] : 0.f;
#pragma unroll
                    for (int q = 0; q < kGather; ++q) fb += GRADED ? sv[q] * v[q] : v[q];
                }
            }
        }
        float zt;
        if (VEC4) {
            if ((t & 3) == 0 && live) zq = *reinterpret_cast<const float4*>(zrow + t);
            zt = (t & 3) == 0 ? zq.x : (t & 3) == 1 ? zq.y : (t & 3) == 2 ? zq.z : zq.w;
        } else {
            zt = live ? zrow[t] : 0.f;
        }
        const float dend = zt + fb;
        // one step of every state, each starting from the float32 value the previous call left and
        // handing a float32 value to the next operator
        yc = add_sat(rs0_12(yc, mi), trunc_i32(w * dend));
        cur = from(yc);
        yc = trunc_i32(w * cur);
        const int yn = add_sat(rs0_12(yv, mv), yc);
        acc_lif |= ((unsigned)yc + (1u << 30)) | ((unsigned)yn + (1u << 30));
        vol = from(yn);
        float theta = p.spike_thr;
        if (ALIF) {
            r = rs0_12(r, mr);
            th = rs0_12(th - p.base, mt) + p.base;
            acc_th |= ((unsigned)th + (1u << 28)) | ((unsigned)r + (1u << 28));
            thf = from(th);
            rf = from(r);
            theta = thf + rf;
        }
        const bool fired = live && vol >= theta;
        const float s = GRADED ? ((fired ? 1.0f : 0.0f) * vol) / p.spike_scale : (fired ? 1.0f : 0.0f);
        const bool spiked = live && s > 0.0f;           // what the carried states and the feedback see
        if (ALIF) {
            yv = trunc_i32(w * vol);
            r = trunc_i32((spiked ? rf + 2.0f * thf : rf) * w);
            th = trunc_i32((spiked ? thf + p.th_step_f : thf) * w);
        } else {
            yv = spiked ? 0 : trunc_i32(w * vol);
        }
        {
            // a graded spike that is not positive still takes part in the feedback with its value
            const bool listed = GRADED ? (live && s != 0.0f) : fired;
            const unsigned long long ballot = __ballot(listed);
            const int lane = c & (kWave - 1);
            const int cnt = __builtin_popcountll(ballot);
            const int below = __builtin_popcountll(ballot & ((1ull << lane) - 1ull));   // listed lanes below this one
            int* seg = &fired_list[t & 1][(c / kWave) * kWave];
            if (listed) {
                seg[below] = c;
                if (GRADED) fired_value[t & 1][(c / kWave) * kWave + below] = s;
            } else {                                   // the other lanes write the padding
                const int slot = cnt + (lane - below);
                if (slot < ((cnt + kGather - 1) & ~(kGather - 1))) {
                    seg[slot] = C;
                    if (GRADED) fired_value[t & 1][(c / kWave) * kWave + slot] = 0.0f;
                }
            }
            if (lane == 0) counts[t & 1][c / kWave] = cnt;
        }
        if (VEC4) {
            if ((t & 3) == 0) { sq.x = s; vq.x = vol; tq.x = theta; }
            else if ((t & 3) == 1) { sq.y = s; vq.y = vol; tq.y = theta; }
            else if ((t & 3) == 2) { sq.z = s; vq.z = vol; tq.z = theta; }
            else {
                sq.w = s; vq.w = vol; tq.w = theta;
                if (live) {
                    *reinterpret_cast<float4*>(srow + t - 3) = sq;
                    *reinterpret_cast<float4*>(vrow + t - 3) = vq;
                    if (ALIF) *reinterpret_cast<float4*>(trow + t - 3) = tq;
                }
            }
        } else if (live) {
            srow[t] = s;
            vrow[t] = vol;
            if (ALIF) trow[t] = theta;
        }
        __syncthreads();
    }
    if (live && (range_exceeded(acc_lif, 30) || range_exceeded(acc_th, 28))) raise_range_flag(p.range_flag);
    if (live) {
        p.cur_last[m] = cur;
        p.vol_last[m] = vol;
        if (ALIF) {
            p.th_last[m] = thf;
            p.ref_last[m] = rf;
        }
    }
}

template <bool ALIF, bool GRADED, bool POW2, bool VEC4>
__global__ __launch_bounds__(kMaxRecurrent) void recurrent_fwd_kernel(const RecurrentFwd p) {
    recurrent_fwd_gather<ALIF, GRADED, POW2, VEC4>(p);
}

// Backward through the loop as the reference differentiates it (utils/recurrent.py:83-112): the
// state carried between the one-step neuron calls is a constant, so a step contributes the spike
// surrogate only, and the gradient reaches step t-1 through R.
template <bool THETA, bool GRADED, bool VEC4>
__global__ __launch_bounds__(kMaxRecurrent) void recurrent_bwd_kernel(
    float* __restrict__ grad_z, const float* __restrict__ grad_spikes, const float* __restrict__ voltage,
    const float* __restrict__ theta, const float* __restrict__ rec, float spike_thr, float tau, float rho, int C,
    int T) {
    __shared__ float gd_s[2][kMaxRecurrent];
    const int c = threadIdx.x;
    const bool live = c < C;
    const int64_t m = (int64_t)blockIdx.x * C + (live ? c : 0);
    const float* grow = grad_spikes + m * (int64_t)T;
    const float* vrow = voltage + m * (int64_t)T;
    const float* trow = THETA ? theta + m * (int64_t)T : nullptr;
    float* orow = grad_z + m * (int64_t)T;
    const float lead = (rho / 2.0f) / tau;
    const float inv_tau = 1.0f / tau;
    float carry = 0.f;
    float4 gq = make_float4(0.f, 0.f, 0.f, 0.f), vq = gq, oq = gq, tq = gq;

    for (int t = T - 1; t >= 0; --t) {
        float g, v, th = spike_thr;
        if (VEC4) {
            if ((t & 3) == 3 && live) {
                gq = *reinterpret_cast<const float4*>(grow + t - 3);
                vq = *reinterpret_cast<const float4*>(vrow + t - 3);
                if (THETA) tq = *reinterpret_cast<const float4*>(trow + t - 3);
            }
            g = (t & 3) == 0 ? gq.x : (t & 3) == 1 ? gq.y : (t & 3) == 2 ? gq.z : gq.w;
            v = (t & 3) == 0 ? vq.x : (t & 3) == 1 ? vq.y : (t & 3) == 2 ? vq.z : vq.w;
            if (THETA) th = (t & 3) == 0 ? tq.x : (t & 3) == 1 ? tq.y : (t & 3) == 2 ? tq.z : tq.w;
        } else {
            g = live ? grow[t] : 0.f;
            v = live ? vrow[t] : 0.f;
            if (THETA) th = live ? trow[t] : 0.f;
        }
        const float gs = carry + g;
        const float d = v - th;
        const float factor = GRADED ? rho * expf(fminf(d, 0.0f) * inv_tau) : lead * expf(-fabsf(d) * inv_tau);
        const float gd = live ? factor * gs : 0.f;
        if (VEC4) {
            if ((t & 3) == 3) oq.w = gd;
            else if ((t & 3) == 2) oq.z = gd;
            else if ((t & 3) == 1) oq.y = gd;
            else {
                oq.x = gd;
                if (live) *reinterpret_cast<float4*>(orow + t) = oq;
            }
        } else if (live) {
            orow[t] = gd;
        }
        gd_s[t & 1][c] = gd;
        __syncthreads();
        // gradient handed to step t-1: (grad of the feedback) R, this thread's column
        carry = 0.f;
        if (live && t > 0) {
            const float* col = rec + c;
            const float* gd = gd_s[t & 1];
            int cc = 0;
            for (; cc + 16 <= C; cc += 16) {       // sixteen rows of R in flight at a time
                float r[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) r[k] = col[(int64_t)(cc + k) * C];
#pragma unroll
                for (int k = 0; k < 16; ++k) carry = __fmaf_rn(gd[cc + k], r[k], carry);
            }
            for (; cc < C; ++cc) carry = __fmaf_rn(gd[cc], col[(int64_t)cc * C], carry);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------------
// Narrow layers (C <= kRegisterNeurons): the matrix stays in the registers of the sample's workgroup.
//
// What bounds a step is one chain -- the spikes out of LDS, the products, their sum, the neuron, the barrier -- so the
// matrix must not be fetched inside it.  The kernels above read it from the L2 in every step ([32, 128, 300]: 859 us
// forward, 555 us backward for ALIF neurons; a training step of the layer 1480 -> 396 us).  Here four threads serve a neuron and a row of sixteen lanes four neurons: lane j of
// the row holds the columns k = 64 i + 4 j + {0..3} of its four rows, 16 registers for every 64 neurons (64 at most: 16
// waves of 128 registers are what a CU holds), so a step reads the vector of spikes with one or a few ds_read_b128 a
// thread, sixteen lanes contiguously, and every value read serves four products.  The sixteen partial sums of a neuron
// are added with four DPP steps that halve the neurons a lane keeps until a quad of lanes holds one neuron's sum.  All
// four compute its step, and lane q of the quad moves the samples of time 4 i + q: any row length and alignment with
// dword accesses that fill 16 bytes a neuron, loaded four steps ahead.
//
// A row sum is dense here: a neuron that did not fire contributes weight * 0.  Forward, where that is a NaN for a
// weight that is not finite and would cost the receiving neuron its input, a workgroup with such a weight takes the
// form above, which adds the weights of firing neurons only; backward that form is dense, too.
constexpr int kRegisterNeurons = 256;

template <int CTRL>
__device__ inline float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int E>
__device__ inline float of_quad(float x) { return dpp<E * 0x55>(x); }      // lane E of the quad, in all four

template <int KQ>
struct RegisterMatrix {
    float w[4][4 * KQ];      // [neuron of the row of lanes][column]

    // element (row n, column k) lies at mat[k * C + n]; false if one of this thread's elements is not finite
    __device__ bool load(const float* __restrict__ mat, int C) {
        const int j = threadIdx.x & 15, n = (int)(threadIdx.x >> 4) * 4;
        float zero = 0.f;                                     // a NaN after an element that is not finite
#pragma unroll
        for (int i = 0; i < KQ; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k = 64 * i + 4 * j + e;
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    w[a][4 * i + e] = (k < C && n + a < C) ? mat[k * C + n + a] : 0.f;
                    zero = __fmaf_rn(w[a][4 * i + e], 0.f, zero);
                }
            }
        return zero == 0.f;
    }
    // product with the vector at x; the result for neuron 4 * (thread / 16) + (thread / 4) % 4
    __device__ float times(const float4* x) const {
        const int j = threadIdx.x & 15;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        float4 q[KQ];
#pragma unroll
        for (int i = 0; i < KQ; ++i) q[i] = x[16 * i + j];
#pragma unroll
        for (int i = 0; i < KQ; ++i)
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                v[a] = __fmaf_rn(w[a][4 * i], q[i].x, v[a]);
                v[a] = __fmaf_rn(w[a][4 * i + 1], q[i].y, v[a]);
                v[a] = __fmaf_rn(w[a][4 * i + 2], q[i].z, v[a]);
                v[a] = __fmaf_rn(w[a][4 * i + 3], q[i].w, v[a]);
            }
        const bool b3 = j & 8, b2 = j & 4;
        const float k0 = (b3 ? v[2] : v[0]) + dpp<0x128>(b3 ? v[0] : v[2]);      // row_ror:8, lane ^ 8
        const float k1 = (b3 ? v[3] : v[1]) + dpp<0x128>(b3 ? v[1] : v[3]);
        float s = (b2 ? k1 : k0) + dpp<0x141>(b2 ? k0 : k1);                     // row_half_mirror, lane ^ 7
        s += dpp<0xB1>(s);                                                       // lane ^ 1
        return s + dpp<0x4E>(s);                                                 // lane ^ 2
    }
};

template <bool ALIF, bool GRADED, bool POW2, int KQ>
__global__ __launch_bounds__(256 * KQ) void recurrent_reg_fwd_kernel(const RecurrentFwd p) {
    __shared__ float4 fired_s[2][16 * KQ];                    // values of the spikes of two steps
    const int C = p.C, T = p.T;
    const float w = p.w, inv_w = p.inv_w;
    const int c = threadIdx.x >> 2, q = threadIdx.x & 3;
    const bool live = c < C;
    const int64_t m = (int64_t)blockIdx.x * C + (live ? c : 0);
    const float* zrow = p.z + m * (int64_t)T;
    float* srow = p.spk + m * (int64_t)T;
    float* vrow = p.vol + m * (int64_t)T;
    float* trow = ALIF ? p.theta + m * (int64_t)T : nullptr;
    auto from = [&](int y) -> float { const float f = (float)y; return POW2 ? f * inv_w : f / w; };

    RegisterMatrix<KQ> mat;
    if (__syncthreads_or(!mat.load(p.rec_t, C))) return recurrent_fwd_gather<ALIF, GRADED, POW2, false>(p);
    for (int i = threadIdx.x; i < 32 * KQ; i += blockDim.x) fired_s[0][i] = make_float4(0.f, 0.f, 0.f, 0.f);

    int yc = 0, yv = 0, th = 0, r = 0, mi = 0, mv = 0, mt = 0, mr = 0;
    unsigned acc_lif = 0u, acc_th = 0u;                       // range of the states, see range_bits in tile.h
    if (live) {
        yc = trunc_i32(p.i_state[p.n_is == 1 ? 0 : m] * w);
        yv = trunc_i32(p.v_state[p.n_vs == 1 ? 0 : m] * w);
        mi = 4096 - trunc_i32(rintf(p.i_decay[param_index(m, C, p.n_id)]));
        mv = 4096 - trunc_i32(rintf(p.v_decay[param_index(m, C, p.n_vd)]));
        if (ALIF) {
            th = trunc_i32(p.th_state[p.n_ts == 1 ? 0 : m] * w);
            r = trunc_i32(p.ref_state[p.n_rs == 1 ? 0 : m] * w);
            mt = 4096 - trunc_i32(rintf(p.th_decay[param_index(m, C, p.n_td)]));
            mr = 4096 - trunc_i32(rintf(p.ref_decay[param_index(m, C, p.n_rd)]));
            check_multiplier(mt, p.range_flag); check_multiplier(mr, p.range_flag);
        }
        check_multiplier(mi, p.range_flag); check_multiplier(mv, p.range_flag);
        acc_lif = ((unsigned)yc + (1u << 30)) | ((unsigned)yv + (1u << 30));
        acc_th = ((unsigned)th + (1u << 28)) | ((unsigned)r + (1u << 28));
    }
    float cur = 0.f, vol = 0.f, thf = 0.f, rf = 0.f;
    float zq = (live && q < T) ? zrow[q] : 0.f, sq = 0.f, vq = 0.f, tq = 0.f;
    __syncthreads();

    auto step = [&](int t, int e, float z_now) {
        const float fb = t > 0 ? mat.times(fired_s[(t - 1) & 1]) : 0.f;
        const float dend = z_now + fb;
        // the neuron of recurrent_fwd_kernel, operation by operation
        yc = add_sat(rs0_12(yc, mi), trunc_i32(w * dend));
        cur = from(yc);
        yc = trunc_i32(w * cur);
        const int yn = add_sat(rs0_12(yv, mv), yc);
        acc_lif |= ((unsigned)yc + (1u << 30)) | ((unsigned)yn + (1u << 30));
        vol = from(yn);
        float theta = p.spike_thr;
        if (ALIF) {
            r = rs0_12(r, mr);
            th = rs0_12(th - p.base, mt) + p.base;
            acc_th |= ((unsigned)th + (1u << 28)) | ((unsigned)r + (1u << 28));
            thf = from(th);
            rf = from(r);
            theta = thf + rf;
        }
        const bool fired = live && vol >= theta;
        const float s = GRADED ? ((fired ? 1.0f : 0.0f) * vol) / p.spike_scale : (fired ? 1.0f : 0.0f);
        const bool spiked = live && s > 0.0f;
        // (a padding neuron's state is zero; its rows and columns of the matrix are, too)
        if (q == 0) reinterpret_cast<float*>(fired_s[t & 1])[c] = live ? s : 0.f;
        if (ALIF) {
            yv = trunc_i32(w * vol);
            r = trunc_i32((spiked ? rf + 2.0f * thf : rf) * w);
            th = trunc_i32((spiked ? thf + p.th_step_f : thf) * w);
        } else {
            yv = spiked ? 0 : trunc_i32(w * vol);
        }
        if (e == q) {
            sq = s;
            vq = vol;
            tq = theta;
        }
        __syncthreads();
    };
    for (int t = 0; t < T; t += 4) {
        const float znext = (live && t + 4 + q < T) ? zrow[t + 4 + q] : 0.f;
        step(t, 0, of_quad<0>(zq));
        if (t + 1 < T) step(t + 1, 1, of_quad<1>(zq));
        if (t + 2 < T) step(t + 2, 2, of_quad<2>(zq));
        if (t + 3 < T) step(t + 3, 3, of_quad<3>(zq));
        if (live && t + q < T) {
            srow[t + q] = sq;
            vrow[t + q] = vq;
            if (ALIF) trow[t + q] = tq;
        }
        zq = znext;
    }
    if (live && (range_exceeded(acc_lif, 30) || range_exceeded(acc_th, 28))) raise_range_flag(p.range_flag);
    if (live && q == 0) {
        p.cur_last[m] = cur;
        p.vol_last[m] = vol;
        if (ALIF) {
            p.th_last[m] = thf;
            p.ref_last[m] = rf;
        }
    }
}

// The surrogate of a step does not depend on the carried gradient: lane q of the quad evaluates it for time 4 i + q
// ahead of the four steps, and a step is left with the product, one addition and one multiplication.
template <bool THETA, bool GRADED, int KQ>
__global__ __launch_bounds__(256 * KQ) void recurrent_reg_bwd_kernel(
    float* __restrict__ grad_z, const float* __restrict__ grad_spikes, const float* __restrict__ voltage,
    const float* __restrict__ theta, const float* __restrict__ rec, float spike_thr, float tau, float rho, int C,
    int T) {
    __shared__ float4 grad_s[2][16 * KQ];
    const int c = threadIdx.x >> 2, q = threadIdx.x & 3;
    const bool live = c < C;
    const int64_t row = ((int64_t)blockIdx.x * C + (live ? c : 0)) * (int64_t)T;
    const float lead = (rho / 2.0f) / tau;
    const float inv_tau = 1.0f / tau;

    RegisterMatrix<KQ> mat;
    mat.load(rec, C);
    for (int i = threadIdx.x; i < 32 * KQ; i += blockDim.x) grad_s[0][i] = make_float4(0.f, 0.f, 0.f, 0.f);

    float gq = 0.f, vq = 0.f, tq = spike_thr;
    auto load = [&](int t, float& g, float& v, float& th) {
        const bool in = live && t >= 0 && t < T;
        g = in ? grad_spikes[row + t] : 0.f;
        v = in ? voltage[row + t] : 0.f;
        if (THETA) th = in ? theta[row + t] : 0.f;
    };
    const int last = (T - 1) & ~3;
    load(last + q, gq, vq, tq);
    float out = 0.f;
    __syncthreads();

    auto step = [&](int t, int e, float g, float factor) {
        const float carry = t + 1 < T ? mat.times(grad_s[(t + 1) & 1]) : 0.f;
        const float gs = carry + g;
        const float gd = live ? factor * gs : 0.f;
        if (q == 0) reinterpret_cast<float*>(grad_s[t & 1])[c] = gd;
        if (e == q) out = gd;
        __syncthreads();
    };
    for (int t = last; t >= 0; t -= 4) {
        float gn = 0.f, vn = 0.f, tn = spike_thr;
        load(t - 4 + q, gn, vn, tn);
        const float d = vq - tq;
        const float factor = GRADED ? rho * expf(fminf(d, 0.0f) * inv_tau) : lead * expf(-fabsf(d) * inv_tau);
        if (t + 3 < T) step(t + 3, 3, of_quad<3>(gq), of_quad<3>(factor));
        if (t + 2 < T) step(t + 2, 2, of_quad<2>(gq), of_quad<2>(factor));
        if (t + 1 < T) step(t + 1, 1, of_quad<1>(gq), of_quad<1>(factor));
        step(t, 0, of_quad<0>(gq), of_quad<0>(factor));
        if (live && t + q < T) grad_z[row + t + q] = out;
        gq = gn; vq = vn; tq = tn;
    }
}

}  // namespace slayer

using namespace slayer;

namespace {

int check_recurrent_sizes(int64_t N, int64_t C, int64_t T) {
    if (N < 0 || C < 0 || T < 0) return SLAYER_EINVAL;
    if (C > kMaxRecurrent || T > 0x7fffffffLL || N > 0x7fffffffLL) return SLAYER_ERANGE;
    return 0;
}

template <bool ALIF>
int launch_recurrent_fwd(RecurrentFwd p, int graded, int w_scale, int64_t N, hipStream_t st) {
    const bool pow2 = is_pow2(w_scale);
    // Register form, except where its sixteen waves a sample (one sample at a time on a CU) have so many samples to do that
    // the gathering form, which works on the firing neurons only, is no slower at usual rates: 250 neurons, 100 steps,
    // 0.4 / 3 / 7 / 16 % of the neurons firing in a step, gathering 314 / 480 / 497 / 522 us for 1024 samples against 487, 556 / 854 /
    // 916 / 974 for 2048 against 970; 512 samples 165 / 300 / 327 / 347 against 216.  Narrower layers: 192 neurons 204 / 267 /
    // 293 / 306 for 1024 samples against 276, 128 neurons 127 / 175 / 190 / 198 against 129, fewer samples 1.5 to 3 times the register
    // form's time.  (Backward the register form takes 0.2 to 0.8 of the other's time everywhere.)
    if (p.C <= kRegisterNeurons && (p.C <= 192 || N < 1024)) {
        const dim3 threads((unsigned)((p.C + 15) / 16 * 64));
#define SLAYER_REG(G, P, KQ) \
    hipLaunchKernelGGL((recurrent_reg_fwd_kernel<ALIF, G, P, KQ>), dim3((unsigned)N), threads, 0, st, p)
#define SLAYER_REG2(G, P)                                                                                     \
    do {                                                                                                      \
        if (p.C <= 64) SLAYER_REG(G, P, 1); else if (p.C <= 128) SLAYER_REG(G, P, 2);                         \
        else if (p.C <= 192) SLAYER_REG(G, P, 3); else SLAYER_REG(G, P, 4);                                   \
    } while (0)
        if (graded) { if (pow2) SLAYER_REG2(true, true); else SLAYER_REG2(true, false); }
        else { if (pow2) SLAYER_REG2(false, true); else SLAYER_REG2(false, false); }
#undef SLAYER_REG2
#undef SLAYER_REG
        return (int)hipGetLastError();
    }
    bool vec = (p.T % 4) == 0 && aligned16(p.z) && aligned16(p.spk) && aligned16(p.vol);
    if (ALIF) vec = vec && aligned16(p.theta);
    const dim3 grid((unsigned)N), block((unsigned)((p.C + kWave - 1) / kWave * kWave));
#define SLAYER_REC(G, P, V) hipLaunchKernelGGL((recurrent_fwd_kernel<ALIF, G, P, V>), grid, block, 0, st, p)
#define SLAYER_REC2(G)                                                                                        \
    do {                                                                                                      \
        if (pow2) { if (vec) SLAYER_REC(G, true, true); else SLAYER_REC(G, true, false); }                    \
        else { if (vec) SLAYER_REC(G, false, true); else SLAYER_REC(G, false, false); }                       \
    } while (0)
    if (graded) SLAYER_REC2(true); else SLAYER_REC2(false);
#undef SLAYER_REC2
#undef SLAYER_REC
    return (int)hipGetLastError();
}

}  // namespace

extern "C" int slayer_cuba_recurrent_fwd(float* spk_out, float* vol_out, float* cur_last_out, float* vol_last_out,
                                         const float* z, const float* rec_t,
                                         const float* i_decay, const float* v_decay,
                                         const float* i_state, const float* v_state,
                                         float spike_threshold, int graded, float spike_scale, int w_scale,
                                         int64_t N, int64_t C, int64_t num_i_decays, int64_t num_v_decays,
                                         int64_t num_i_states, int64_t num_v_states, int64_t T, void* stream) {
    if (int e = check_recurrent_sizes(N, C, T)) return e;
    if (N == 0 || C == 0 || T == 0) return 0;
    if (!spk_out || !vol_out || !cur_last_out || !vol_last_out || !z || !rec_t || !i_decay || !v_decay || !i_state ||
        !v_state)
        return SLAYER_ENULL;
    if (int e = check_params(N * C, C, num_i_decays)) return e;
    if (int e = check_params(N * C, C, num_v_decays)) return e;
    if (int e = check_states(N * C, num_i_states)) return e;
    if (int e = check_states(N * C, num_v_states)) return e;
    if (w_scale == 0 || (graded && spike_scale == 0.0f)) return SLAYER_EINVAL;
    RecurrentFwd p{};
    p.spk = spk_out; p.vol = vol_out; p.cur_last = cur_last_out; p.vol_last = vol_last_out;
    p.z = z; p.rec_t = rec_t; p.i_decay = i_decay; p.v_decay = v_decay; p.i_state = i_state; p.v_state = v_state;
    p.n_id = num_i_decays; p.n_vd = num_v_decays; p.n_is = num_i_states; p.n_vs = num_v_states;
    p.w = (float)w_scale; p.inv_w = 1.0f / p.w; p.spike_thr = spike_threshold; p.spike_scale = spike_scale;
    p.C = (int)C; p.T = (int)T;
    p.range_flag = range_flag_device();
    return launch_recurrent_fwd<false>(p, graded, w_scale, N, (hipStream_t)stream);
}

extern "C" int slayer_alif_recurrent_fwd(float* spk_out, float* vol_out, float* theta_out,
                                         float* cur_last_out, float* vol_last_out, float* th_last_out,
                                         float* ref_last_out, const float* z, const float* rec_t,
                                         const float* i_decay, const float* v_decay, const float* th_decay,
                                         const float* ref_decay, const float* i_state, const float* v_state,
                                         const float* th_state, const float* ref_state,
                                         float th_step, int64_t th0_scaled, int graded, float spike_scale, int w_scale,
                                         int64_t N, int64_t C,
                                         int64_t num_i_decays, int64_t num_v_decays, int64_t num_th_decays,
                                         int64_t num_ref_decays, int64_t num_i_states, int64_t num_v_states,
                                         int64_t num_th_states, int64_t num_ref_states, int64_t T, void* stream) {
    if (int e = check_recurrent_sizes(N, C, T)) return e;
    if (N == 0 || C == 0 || T == 0) return 0;
    if (!spk_out || !vol_out || !theta_out || !cur_last_out || !vol_last_out || !th_last_out || !ref_last_out || !z ||
        !rec_t || !i_decay || !v_decay || !th_decay || !ref_decay || !i_state || !v_state || !th_state || !ref_state)
        return SLAYER_ENULL;
    for (int64_t n : {num_i_decays, num_v_decays, num_th_decays, num_ref_decays})
        if (int e = check_params(N * C, C, n)) return e;
    for (int64_t n : {num_i_states, num_v_states, num_th_states, num_ref_states})
        if (int e = check_states(N * C, n)) return e;
    if (w_scale == 0 || (graded && spike_scale == 0.0f)) return SLAYER_EINVAL;
    if (th0_scaled > 0x7fffffffLL || th0_scaled < -0x7fffffffLL) return SLAYER_ERANGE;
    RecurrentFwd p{};
    p.spk = spk_out; p.vol = vol_out; p.theta = theta_out;
    p.cur_last = cur_last_out; p.vol_last = vol_last_out; p.th_last = th_last_out; p.ref_last = ref_last_out;
    p.z = z; p.rec_t = rec_t;
    p.i_decay = i_decay; p.v_decay = v_decay; p.th_decay = th_decay; p.ref_decay = ref_decay;
    p.i_state = i_state; p.v_state = v_state; p.th_state = th_state; p.ref_state = ref_state;
    p.n_id = num_i_decays; p.n_vd = num_v_decays; p.n_td = num_th_decays; p.n_rd = num_ref_decays;
    p.n_is = num_i_states; p.n_vs = num_v_states; p.n_ts = num_th_states; p.n_rs = num_ref_states;
    p.w = (float)w_scale; p.inv_w = 1.0f / p.w; p.spike_scale = spike_scale; p.th_step_f = th_step;
    p.base = (int)th0_scaled;
    p.C = (int)C; p.T = (int)T;
    p.range_flag = range_flag_for_threshold(0, th0_scaled);
    return launch_recurrent_fwd<true>(p, graded, w_scale, N, (hipStream_t)stream);
}

extern "C" int slayer_recurrent_bwd(float* grad_z, const float* grad_spikes, const float* voltage, const float* theta,
                                    const float* rec, float spike_threshold, float tau_rho, float scale_rho,
                                    int graded, int64_t N, int64_t C, int64_t T, void* stream) {
    if (int e = check_recurrent_sizes(N, C, T)) return e;
    if (N == 0 || C == 0 || T == 0) return 0;
    if (!grad_z || !grad_spikes || !voltage || !rec) return SLAYER_ENULL;
    if (C <= kRegisterNeurons) {
        const dim3 threads((unsigned)((C + 15) / 16 * 64));
#define SLAYER_REG(TH, G, KQ)                                                                                      \
    hipLaunchKernelGGL((recurrent_reg_bwd_kernel<TH, G, KQ>), dim3((unsigned)N), threads, 0, (hipStream_t)stream, \
                       grad_z, grad_spikes, voltage, theta, rec, spike_threshold, tau_rho, scale_rho, (int)C, (int)T)
#define SLAYER_REG2(TH, G)                                                                                         \
    do {                                                                                                           \
        if (C <= 64) SLAYER_REG(TH, G, 1); else if (C <= 128) SLAYER_REG(TH, G, 2);                                \
        else if (C <= 192) SLAYER_REG(TH, G, 3); else SLAYER_REG(TH, G, 4);                                        \
    } while (0)
        if (theta) { if (graded) SLAYER_REG2(true, true); else SLAYER_REG2(true, false); }
        else { if (graded) SLAYER_REG2(false, true); else SLAYER_REG2(false, false); }
#undef SLAYER_REG2
#undef SLAYER_REG
        return (int)hipGetLastError();
    }
    const bool vec = (T % 4) == 0 && aligned16(grad_z) && aligned16(grad_spikes) && aligned16(voltage) &&
                     (!theta || aligned16(theta));
    const dim3 grid((unsigned)N), block((unsigned)((C + kWave - 1) / kWave * kWave));
    hipStream_t st = (hipStream_t)stream;
#define SLAYER_RB(TH, G, V)                                                                                     \
    hipLaunchKernelGGL((recurrent_bwd_kernel<TH, G, V>), grid, block, 0, st, grad_z, grad_spikes, voltage, theta, \
                       rec, spike_threshold, tau_rho, scale_rho, (int)C, (int)T)
#define SLAYER_RB2(TH, G) do { if (vec) SLAYER_RB(TH, G, true); else SLAYER_RB(TH, G, false); } while (0)
    if (theta) { if (graded) SLAYER_RB2(true, true); else SLAYER_RB2(true, false); }
    else { if (graded) SLAYER_RB2(false, true); else SLAYER_RB2(false, false); }
#undef SLAYER_RB2
#undef SLAYER_RB
    return (int)hipGetLastError();
}
