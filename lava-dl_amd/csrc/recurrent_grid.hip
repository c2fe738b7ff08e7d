// Recurrent layer of CUBA or ALIF neurons, the whole time loop in one launch spread over the chip.
//
//   feedback[t] = R s[t-1];  s[t] = neuron(z[t] + feedback[t])          (utils/recurrent.py:45-112 in the reference)
//
// A launch per time step (recurrent_steps.hip) reads the [C x C] matrix from the caches and starts and drains the chip
// once a step: 7.6 us forward at [32, 2048, 300].  The registers of the chip hold the matrix (2048 neurons:
// 16.8 MB as float32, against 128 MB): a workgroup owns 16 neurons x 16 samples, keeps its rows of R in registers for all
// steps, and what a step hands to the next crosses the chip through the caches.
//
// Forward exchange: one 32-bit word per sample and tile of 16 neurons, the spikes in the low half, the step's number
// in the high half, in two sets used in turn.  A wave polls the words it multiplies until all carry the
// previous step's number, so the data is its own flag: one store and one load across the chip per step, no barrier, no
// counter.  Two sets are enough: a workgroup writes step t after it has read all words of step t-1, and whoever
// published t-1 had read all of t-2.
//
// The product runs on the bfloat16 matrix instruction: a spike is the bfloat16 number 2.0 (one bit, which a shift and a
// mask put in place), a weight is halved and cut into three parts of 8 bits -- its 24 bits, nothing is
// rounded -- and the parts beyond the first are skipped by a wave whose weights have none (8-bit quantisers).
//
// The workgroups wait for one another, so all of them must be on the chip at once: the launch is a cooperative one,
// which the runtime refuses beyond what the device holds, does not run beside another and grants to one process at a time
// (a refused call takes a launch per step).  Every wait is bounded all the same (kSpinLimit polls); a workgroup that
// gives up leaves a mark, and the kernel that is launched behind computes the layer again when it finds it: forward with the same
// bits, one workgroup per sample tile; backward one workgroup per sample, its sums in double and so equal to rounding.
//
// Measured against a launch per step, whole layer, forward and backward, weights of an 8-bit quantiser: CUBA [32, 2048, 300] 5 216
// -> 2 316 us (forward kernel 2 430 -> 492, backward 2 075 -> 1 016), [32, 256, 300] 2 543 -> 928, ALIF [32, 512, 300] 2 534 -> 1 129,
// [64, 2048, 100] 2 973 -> 2 193; ALIF [32, 1024, 100] forward alone 684 -> 229.  A forward step of 2048 neurons is 1.6 us:
// 0.9 of them the way of the words across the chip, 0.7 the product, the sum over the waves and the neuron, a chain of
// dependent instructions.
#include "recurrent_step.h"
#include "split.h"
#include <initializer_list>

namespace slayer {

constexpr int kGridWaves = 8;                        // waves of a workgroup: each takes an eighth of the sum over k
constexpr int kGridThreads = kGridWaves * kWave;
constexpr int kGridMaxC = 2048;                      // the parts of 16 rows in the registers of eight waves
constexpr int kGridMaxT = 1 << 26;                   // 32-bit byte offsets of four rows
constexpr int kGridChunk = 16;                       // steps of the tensors a wave stages in LDS at a time
constexpr int kGridPitch = kGridChunk + 1;
#ifndef SLAYER_GRID_POLLS
#define SLAYER_GRID_POLLS (1 << 18)                   // about a third of a second
#endif
constexpr int kSpinLimit = SLAYER_GRID_POLLS;        // polls before a wave gives up
constexpr int kSoloThreads = 1024;

__device__ __forceinline__ void wave_lds_order() {   // LDS written by some lanes of this wave, read by others
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ void lds_barrier() {      // orders LDS only: stores to memory stay in flight
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Which workgroup does what.  Workgroups go to the chip's eight XCDs round-robin by index; those of one sample group
// share what they exchange, so they are put on as few XCDs as hold them (`xcds`, a power of two), `per_xcd` on each:
// [32, 2048, 300] forward 645 us with both groups on all eight XCDs, 520 with four XCDs to a group.  Where they
// really run changes only the time.
struct GridMap {
    int xcds, per_xcd;
    __device__ __forceinline__ int tile(int id) const { return ((id >> 3) % per_xcd) * xcds + (id & 7) % xcds; }
    __device__ __forceinline__ int group(int id) const { return (id >> 3) / per_xcd * (8 / xcds) + (id & 7) / xcds; }
};

struct GridFwd {
    StepFwd p;                                       // its time-major tensors and packed operands are not used
    float *spk, *vol, *theta;                        // [N][C][T]
    const float *z, *rec;
    unsigned* words;                                 // [2][S][words_of(KB)]
    int* carried;                                    // [4][N][C], see recurrent_solo_fwd_kernel
    GridMap map;
    unsigned* gave_up;
};
// words of one sample tile, [KB][16 samples], whole units
__host__ __device__ inline int words_of(int KB) { return (KB + 7) / 8 * 8 * 16; }

__global__ __launch_bounds__(256) void grid_fill_kernel(unsigned* dst, int64_t n, unsigned* gave_up) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = 0u;
    if (i == 0) *gave_up = 0u;
}

// the upper 8 bits of the significand as a bfloat16 in the upper half of a word; v keeps the rest
__device__ __forceinline__ unsigned cut(float& v) {
    const unsigned u = __float_as_uint(v);
    if ((u & 0x7f800000u) == 0x7f800000u) {          // infinities and NaN have no rest
        v = 0.f;
        return (u & 0x007fffffu) ? 0x7fc00000u : (u & 0xffff0000u);
    }
    const unsigned h = u & 0xffff0000u;
    v -= __uint_as_float(h);
    return h;
}

// Unit u of 16 rows of R as A operands, halved, in three parts.  A unit is 8 neuron tiles = 128 presynaptic neurons = four
// products; lane (kk, j) has tiles 8u + 2kk and 8u + 2kk + 1 of row c, element 2i (2i + 1) of product a is neuron 4a + i of
// the first (second) tile, k0 its first neuron.  Returns whether a part beyond the first has a bit.
__device__ __forceinline__ bool weight_parts(const float* rec, int C, int c, int k0, uint4 (&wh)[4], uint4 (&wm)[4], uint4 (&wl)[4]) {
    float v[32];
    unsigned rest = 0u;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const bool ok = c < C && k0 + 4 * q < C;                         // C is a multiple of 4
        const float4 f = ok ? load_quad_dword_aligned(rec + (int64_t)c * C + k0 + 4 * q) : make_float4(0.f, 0.f, 0.f, 0.f);
        v[4 * q] = 0.5f * f.x; v[4 * q + 1] = 0.5f * f.y; v[4 * q + 2] = 0.5f * f.z; v[4 * q + 3] = 0.5f * f.w;
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        unsigned h[4], m[4], l[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float &x = v[4 * a + i], &y = v[16 + 4 * a + i];
            h[i] = cut(x) >> 16; h[i] |= cut(y);
            m[i] = cut(x) >> 16; m[i] |= cut(y);
            l[i] = cut(x) >> 16; l[i] |= cut(y);
            rest |= m[i] | l[i];
        }
        wh[a] = make_uint4(h[0], h[1], h[2], h[3]);
        wm[a] = make_uint4(m[0], m[1], m[2], m[3]);
        wl[a] = make_uint4(l[0], l[1], l[2], l[3]);
    }
    return rest != 0u;
}

// The B operand of product a: the spikes of two tiles, side by side in a word, as the numbers 2.0 and 0.
__device__ __forceinline__ uint4 spike_parts(unsigned both, int a) {
    unsigned b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int bit = 4 * a + i;                                       // neuron `bit` of both tiles, to bits 14 and 30
        b[i] = (bit <= 14 ? both << (14 - bit) : both >> 1) & 0x40004000u;
    }
    return make_uint4(b[0], b[1], b[2], b[3]);
}

// Thread (wave v, lane 16 i + nn) of the first four waves runs neuron nn of the tile for sample 4 v + i; the ballot of its
// wave then holds the 16 spikes of a sample in one 16-bit field.
template <bool ALIF, bool POW2, int U, int NT>
__global__ __launch_bounds__(kGridThreads) void recurrent_grid_fwd_kernel(const GridFwd g) {
    constexpr int kPlane = 68;                       // pitch of a plane of red: reads of a wave meet 64 banks
    __shared__ float red[2][kGridWaves][4][kPlane];
    __shared__ float zbuf[NT][4][kWave * kGridPitch], vbuf[NT][4][kWave * kGridPitch];
    __shared__ float tbuf[ALIF ? NT : 1][4][ALIF ? kWave * kGridPitch : 1];
    __shared__ unsigned sbits[4][kWave];
    __shared__ int dead[2];
    const StepFwd& p = g.p;
    const int C = p.C, N = p.N, T = p.T, KB = p.KB;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kk = lane >> 4, j = lane & 15;
    const int P = g.map.tile(blockIdx.x), c0 = P * 16, group = g.map.group(blockIdx.x);
    if (P >= KB || group * NT >= p.S) return;
    const int words = words_of(KB);
    const int64_t set = (int64_t)p.S * words;
    if (tid < 2) dead[tid] = 0;

    uint4 wh[U][4], wm[U][4], wl[U][4];              // rows c0 .. c0 + 15 of R
    bool rest = false;
#pragma unroll
    for (int u = 0; u < U; ++u)
        rest |= weight_parts(g.rec, C, c0 + j, 16 * (8 * (wave + kGridWaves * u) + 2 * kk), wh[u], wm[u], wl[u]);
    const bool lower = __any(rest);
    // where this lane finds the words of its units, and which of the two tiles there are (an address beyond them is moved
    // to the first tiles; its words are of no consequence, the weights there are zero)
    int word_at[U];
    unsigned need_lo[U], need_hi[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int first = 8 * (wave + kGridWaves * u) + 2 * kk;
        word_at[u] = 16 * (16 * first < words ? first : 0) + j;
        need_lo[u] = first < KB ? 0xffff0000u : 0u;
        need_hi[u] = first + 1 < KB ? 0xffff0000u : 0u;
    }

    // this thread's neuron, one sample of each of the workgroup's sample tiles
    const int nn = lane & 15, c = c0 + nn;
    StepNeuron<ALIF, false, POW2> nrn[NT];
    unsigned fired[NT];
    bool mine[NT];
#pragma unroll
    for (int s = 0; s < NT; ++s) {
        const int n = (group * NT + s) * 16 + 4 * wave + kk;
        mine[s] = wave < 4 && n < N && c < C;
        nrn[s] = StepNeuron<ALIF, false, POW2>{};
        if (mine[s]) {
            nrn[s].load_decays(p, c);
            nrn[s].load_states(p, (int64_t)n * C + c);
            nrn[s].check(p.range_flag);
        }
        nrn[s].decay(p);
    }
    // staging of a wave's 64 rows, 16 steps at a time: access q covers rows 4q .. 4q + 3, lane (kk, j) step j of row 4q + kk
    auto row_ok = [&](int s, int q) -> bool {
        return (group * NT + s) * 16 + 4 * wave + (q >> 2) < N && c0 + 4 * (q & 3) < C;
    };
    // The address is a scalar, one addition further for every access, and the lane's 32-bit offset; what the empty asm keeps
    // the compiler from is holding all of them in registers at once.
    const unsigned lane_at = (unsigned)kk * (unsigned)T + (unsigned)j;
    auto first_row = [&](int s, int t0) -> int64_t {
        return ((int64_t)((group * NT + s) * 16 + 4 * wave) * C + c0) * T + t0;
    };
    auto next_rows = [&](int64_t& at, int q) {
        at += (int64_t)((q & 3) == 3 ? C - 12 : 4) * T;
        asm volatile("" : "+s"(at));
    };
    float zn[NT][16];
    auto fetch = [&](int t0) {
#pragma unroll
        for (int s = 0; s < NT; ++s) {
            int64_t at = first_row(s, t0);
#pragma unroll
            for (int q = 0; q < 16; ++q, next_rows(at, q - 1))
                zn[s][q] = (row_ok(s, q) && t0 + j < T) ? (g.z + at)[lane_at] : 0.f;
        }
    };
    auto put = [&]() {
#pragma unroll
        for (int s = 0; s < NT; ++s)
#pragma unroll
            for (int q = 0; q < 16; ++q) zbuf[s][wave][(4 * q + kk) * kGridPitch + j] = zn[s][q];
        wave_lds_order();
    };
    if (wave < 4) { fetch(0); put(); }
    lds_barrier();

    bool stop = false;
    for (int t0 = 0; t0 < T && !stop; t0 += kGridChunk) {
        if (wave < 4 && t0 + kGridChunk < T) fetch(t0 + kGridChunk);
        const int steps = T - t0 < kGridChunk ? T - t0 : kGridChunk;
#pragma unroll
        for (int s = 0; s < NT; ++s) fired[s] = 0u;
        for (int e = 0; e < steps && !stop; ++e) {
            const int t = t0 + e;
#pragma unroll
            for (int s = 0; s < NT; ++s) {
                const int sel = NT == 1 ? (t & 1) : s & 1;
                const int tile = group * NT + s;
                float z = wave < 4 ? zbuf[s][wave][lane * kGridPitch + e] : 0.f;
                if (t > 0) {
                    const unsigned tag = (unsigned)t << 16;
                    const unsigned* src = g.words + ((t - 1) & 1) * set + (int64_t)tile * words;
                    unsigned W[U];
                    for (int spin = 0;; ++spin) {
                        unsigned late = 0u, lo[U], hi[U];
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            lo[u] = __hip_atomic_load(src + word_at[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            hi[u] = __hip_atomic_load(src + word_at[u] + 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            late |= ((lo[u] ^ tag) & need_lo[u]) | ((hi[u] ^ tag) & need_hi[u]);
                            W[u] = __builtin_amdgcn_perm(hi[u], lo[u], 0x05040100u); // the low halves side by side
                        }
                        if (!__any(late != 0u)) break;
                        if (spin == kSpinLimit ||
                            ((spin & 1023) == 1023 &&
                             __hip_atomic_load(g.gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
                            dead[sel] = 1;
                            break;
                        }
                    }
                    split_f4 acc[2] = {split_f4{0.f, 0.f, 0.f, 0.f}, split_f4{0.f, 0.f, 0.f, 0.f}};
                    split_f4 low = split_f4{0.f, 0.f, 0.f, 0.f};
                    if (!lower) {
#pragma unroll
                        for (int u = 0; u < U; ++u)
#pragma unroll
                            for (int a = 0; a < 4; ++a) acc[a & 1] = mfma_bf16(wh[u][a], spike_parts(W[u], a), acc[a & 1]);
                    } else {
#pragma unroll
                        for (int u = 0; u < U; ++u)
#pragma unroll
                            for (int a = 0; a < 4; ++a) {
                                const uint4 b = spike_parts(W[u], a);
                                acc[a & 1] = mfma_bf16(wh[u][a], b, acc[a & 1]);
                                low = mfma_bf16(wm[u][a], b, low);
                                low = mfma_bf16(wl[u][a], b, low);
                            }
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) red[sel][wave][i][lane] = acc[0][i] + acc[1][i] + low[i];
                }
                lds_barrier();
                if (wave < 4) {
                    if (t > 0) {
                        float fb = 0.f;
#pragma unroll
                        for (int v = 0; v < kGridWaves; ++v) fb += red[sel][v][nn & 3][(nn >> 2) * 16 + 4 * wave + kk];
                        z += fb;
                    }
                    const float spike = nrn[s].fire(z, p);
                    const bool spiked = mine[s] && spike > 0.0f;
                    const unsigned long long mask = __ballot(spiked);
                    if (lane < 4)                                              // sample 4 wave + lane
                        __hip_atomic_store(g.words + (t & 1) * set + (int64_t)tile * words +
                                               P * 16 + 4 * wave + lane,
                                           ((unsigned)(t + 1) << 16) | (unsigned)((mask >> (16 * lane)) & 0xffffull),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    fired[s] |= (spiked ? 1u : 0u) << e;
                    vbuf[s][wave][lane * kGridPitch + e] = nrn[s].vol;
                    if (ALIF) tbuf[s][wave][lane * kGridPitch + e] = nrn[s].theta;
                    if (mine[s] && t == T - 1) {
                        const int64_t m = (int64_t)(tile * 16 + 4 * wave + kk) * C + c;
                        p.cur_last[m] = nrn[s].cur;
                        p.vol_last[m] = nrn[s].vol;
                        if (ALIF) { p.th_last[m] = nrn[s].thf; p.ref_last[m] = nrn[s].rf; }
                    }
                    nrn[s].carry(spike, p);
                    if (t < T - 1) nrn[s].decay(p);
                }
                stop = stop || dead[sel] != 0;
                // The waves without neurons wait here for those with: polling early, they hold up the words on their
                // way (763 us without this barrier, 520 with it).
                lds_barrier();
            }
        }
        if (wave < 4) {
#pragma unroll
            for (int s = 0; s < NT; ++s) {
                sbits[wave][lane] = fired[s];
                wave_lds_order();
                int64_t at = first_row(s, t0);
#pragma unroll
                for (int q = 0; q < 16; ++q, next_rows(at, q - 1)) {
                    const int r = 4 * q + kk;
                    if (!row_ok(s, q) || j >= steps) continue;
                    (g.spk + at)[lane_at] = (sbits[wave][r] >> j) & 1u ? 1.0f : 0.0f;
                    (g.vol + at)[lane_at] = vbuf[s][wave][r * kGridPitch + j];
                    if (ALIF) (g.theta + at)[lane_at] = tbuf[s][wave][r * kGridPitch + j];
                }
                wave_lds_order();
            }
            if (t0 + kGridChunk < T) put();
        }
    }
    if (stop) {
        if (tid == 0) __hip_atomic_store(g.gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
#pragma unroll
    for (int s = 0; s < NT; ++s)
        if (mine[s] && (range_exceeded(nrn[s].acc_lif, 30) || range_exceeded(nrn[s].acc_th, 28))) raise_range_flag(p.range_flag);
}

// The same layer, one workgroup per sample tile, when a workgroup of the kernel above gave up waiting: every product and sum in the
// same order (a part that is zero adds nothing), so which of the two computed a layer cannot be told from its bits.  The carried
// states lie in memory between two steps, and a workgroup reads the whole matrix every step, which is what bounds it: 0.28 ms a step at
// 1300 neurons (one workgroup per sample and a thread per row: 0.70).
template <bool ALIF, bool POW2>
__global__ __launch_bounds__(kGridThreads) void recurrent_solo_fwd_kernel(const GridFwd g) {
    __shared__ unsigned bits[2][kGridMaxC / 16][16];     // the spikes of a neuron tile and sample
    __shared__ float red[kGridWaves][4][68];
    if (*g.gave_up == 0u) return;
    const StepFwd& p = g.p;
    const int C = p.C, N = p.N, T = p.T, KB = p.KB;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6, kk = lane >> 4, j = lane & 15;
    const int n = 16 * blockIdx.x + 4 * wave + kk;       // of the first four waves
    const int64_t nc = (int64_t)N * C;
    for (int i = tid; i < 2 * (kGridMaxC / 16) * 16; i += kGridThreads) (&bits[0][0][0])[i] = 0u;
    __syncthreads();
    unsigned acc_lif = 0u, acc_th = 0u;
    for (int t = 0; t < T; ++t) {
        for (int P = 0; P < KB; ++P) {
            if (t > 0) {
                split_f4 acc[2] = {split_f4{0.f, 0.f, 0.f, 0.f}, split_f4{0.f, 0.f, 0.f, 0.f}};
                split_f4 low = split_f4{0.f, 0.f, 0.f, 0.f};
                for (int u = wave; 8 * u < KB; u += kGridWaves) {
                    uint4 wh[4], wm[4], wl[4];
                    const int first = 8 * u + 2 * kk;
                    weight_parts(g.rec, C, 16 * P + j, 16 * first, wh, wm, wl);
                    const unsigned both = bits[(t - 1) & 1][first][j] | bits[(t - 1) & 1][first + 1][j] << 16;
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        const uint4 b = spike_parts(both, a);
                        acc[a & 1] = mfma_bf16(wh[a], b, acc[a & 1]);
                        low = mfma_bf16(wm[a], b, low);
                        low = mfma_bf16(wl[a], b, low);
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) red[wave][i][lane] = acc[0][i] + acc[1][i] + low[i];
            }
            __syncthreads();
            const int c = 16 * P + j;
            if (wave < 4) {
                const bool mine = n < N && c < C;
                bool spiked = false;
                if (mine) {
                    const int64_t m = (int64_t)n * C + c, at = m * T + t;
                    StepNeuron<ALIF, false, POW2> nrn{};
                    nrn.load_decays(p, c);
                    if (t == 0) {
                        nrn.load_states(p, m);
                        nrn.check(p.range_flag);
                    } else {
                        nrn.yc = g.carried[m];
                        nrn.yv = g.carried[nc + m];
                        if (ALIF) { nrn.th = g.carried[2 * nc + m]; nrn.r = g.carried[3 * nc + m]; }
                    }
                    float z = g.z[at];
                    if (t > 0) {
                        float fb = 0.f;
#pragma unroll
                        for (int v = 0; v < kGridWaves; ++v) fb += red[v][j & 3][(j >> 2) * 16 + 4 * wave + kk];
                        z += fb;
                    }
                    const StepValues o = nrn.step(z, p);
                    spiked = o.spike > 0.0f;
                    g.spk[at] = o.spike;
                    g.vol[at] = o.voltage;
                    if (ALIF) g.theta[at] = o.theta;
                    g.carried[m] = nrn.yc;
                    g.carried[nc + m] = nrn.yv;
                    if (ALIF) { g.carried[2 * nc + m] = nrn.th; g.carried[3 * nc + m] = nrn.r; }
                    if (t == T - 1) {
                        p.cur_last[m] = o.current;
                        p.vol_last[m] = o.voltage;
                        if (ALIF) { p.th_last[m] = o.threshold; p.ref_last[m] = o.refractory; }
                    }
                    acc_lif |= nrn.acc_lif;
                    acc_th |= nrn.acc_th;
                }
                const unsigned long long mask = __ballot(spiked);
                if (lane < 4) bits[t & 1][P][4 * wave + lane] = (unsigned)((mask >> (16 * lane)) & 0xffffull);
            }
            __syncthreads();
        }
    }
    if (range_exceeded(acc_lif, 30) || range_exceeded(acc_th, 28)) raise_range_flag(p.range_flag);
}

// ---- backward -----------------------------------------------------------------------------------------------------
//
//   grad_z[t] = surrogate(v[t], theta[t]) * (grad_s[t] + grad_z[t+1] R)     (the carried state is a constant)
//
// The same split of the work; the product of two real operands stays on the float32 matrix instruction.  What a step
// hands on are 16 x 16 floats per workgroup in the order the product's lanes load them (a contiguous kilobyte), in
// a ring of four sets.  A float is its own flag here: a set is filled with kUnwritten, a NaN pattern that is never
// published, before it is used again.  A workgroup clears its part of the set of step t+3 when it begins step t: it has
// read all of t+2, whose publishers had read all of t+3; the clearing store has arrived before it publishes t, and
// nobody looks at the set again, for step t-1, before having read t.
//   Bound at [32, 2048, 300] by the float32 matrix rate (1.7 us a step) and by the 128 KB each compute unit
// reads a step (1.1 us from the L2).
constexpr unsigned kUnwritten = 0xffffffffu;

struct GridBwd {
    float* gz;                                       // [N][C][T]
    const float *g, *v, *theta, *rec;                // theta: nullptr for one threshold
    unsigned* ring;                                  // [4][S][KB][256]
    unsigned* gave_up;
    GridMap map;
    int KB, S, N, C, T, graded;
    float spike_thr, tau, rho;
    // groups of four samples and workgroups of 64 neurons to a group (0: not for these sizes), see grid_bwd_local; what
    // the blocks of grid_bwd_fill_kernel found
    int groups4, tiles64;
    const unsigned* inexact;                         // [kFillBlocks]
};
constexpr int kFillBlocks = 256;
constexpr float kLocalScale = 0x1p24f;               // small gradients keep their bits
constexpr float kLocalLargest = 0x1p85f;             // beyond it a scaled sum could leave the range

// Clears the ring, and looks whether every weight is a bfloat16 number of a size that leaves room for the scale.
__global__ __launch_bounds__(1024) void grid_bwd_fill_kernel(unsigned* ring, int64_t n, unsigned* gave_up, const float* rec,
                                                             int64_t weights, unsigned* inexact) {
    const int64_t first = (int64_t)blockIdx.x * 1024 + threadIdx.x, stride = (int64_t)kFillBlocks * 1024;
    for (int64_t i = first; i < n; i += stride) ring[i] = kUnwritten;
    bool bad = false;
#pragma unroll 8
    for (int64_t i = first; i < weights; i += stride) {
        const float w = rec[i], size = fabsf(w);
        bad = bad || (__float_as_uint(w) & 0xffffu) != 0u || !(size <= 256.0f) || (size != 0.0f && size < 0x1p-40f);
    }
    const int any = __syncthreads_or(bad);
    if (threadIdx.x == 0) inexact[blockIdx.x] = any ? 1u : 0u;
    if (first == 0) *gave_up = 0u;
}

__device__ __forceinline__ float surrogate_factor(const GridBwd& p, float v, float th) {
    const float lead = (p.rho / 2.0f) / p.tau, inv_tau = 1.0f / p.tau;
    const float d = v - th;
    return p.graded ? p.rho * expf(fminf(d, 0.0f) * inv_tau) : lead * expf(-fabsf(d) * inv_tau);
}

__device__ __forceinline__ float quad_swapped(float x) {         // that of the other lane of the pair
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xb1, 0xf, 0xf, true));
}
__device__ __forceinline__ unsigned quad_swapped(unsigned x) { return (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0xb1, 0xf, 0xf, true); }
__device__ __forceinline__ float quad_third(float x) {           // that of the third lane of the quad
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xaa, 0xf, 0xf, true));
}

// Weights that are bfloat16 numbers (8-bit quantisers): half the bytes, so a workgroup holds 64 columns of R, and the
// 32 workgroups that cover 2048 neurons are one XCD -- a group of four samples stays on one XCD, whose L2 is all a step
// crosses.  The gradients travel as three bfloat16 parts of 8 bits (cut: 24 bits, nothing is rounded) and the parts are
// columns of the product: column 4 s + q of the B operand is part q of sample s, so one product per 16 rows of weights and
// 32 k does all three (column 4 s + 3 is never written and never looked at).  [32, 2048, 300] 1 751 -> 1 170 us, both timed in one
// run (1 016 on another card): of a step's 3.4 ... 3.9 us the way of the gradients across the XCD takes 2.3, the products 0.4, the
// sum over the waves, the neuron and the barriers the rest.
//   ring: [4][groups4][2 tiles64 blocks of 32 k][64 lanes][8 bfloat16]; thread (wave v, lane) of the first four waves has
// sample v of the group and neuron `lane` of the tile.
template <bool THETA, int U>
__device__ __forceinline__ void grid_bwd_local(const GridBwd& p, float (*red)[kGridWaves][4 * 68], float* gbuf, float* fbuf,
                                               float* obuf, int* dead) {
    const int C = p.C, N = p.N, T = p.T, W = p.tiles64, blocks = 2 * W;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kk = lane >> 4, j = lane & 15, part = j & 3;
    const int group = (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / W), P = (blockIdx.x >> 3) % W, c0 = 64 * P;
    if (group >= p.groups4) return;

    uint4 w[U][4];                                   // columns c0 + 16 r + j, rows 32 b + 8 kk .. + 7 of block b = wave + 8 u
#pragma unroll
    for (int u = 0; u < U; ++u) {
        asm volatile("" ::: "memory");               // a block's loads at a time: all of them at once would not fit the registers
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = c0 + 16 * r + j, k = 32 * (wave + kGridWaves * u) + 8 * kk;
            unsigned h[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) h[e] = (c < C && k + e < C) ? __float_as_uint(p.rec[(int64_t)(k + e) * C + c]) : 0u;
            w[u][r] = make_uint4(__builtin_amdgcn_perm(h[1], h[0], 0x07060302u), __builtin_amdgcn_perm(h[3], h[2], 0x07060302u),
                                 __builtin_amdgcn_perm(h[5], h[4], 0x07060302u), __builtin_amdgcn_perm(h[7], h[6], 0x07060302u));
        }
    }
    const __amdgpu_buffer_rsrc_t ring = make_rsrc(reinterpret_cast<const float*>(p.ring), 4u * p.groups4 * blocks * 1024u);
    const int64_t per_set = (int64_t)p.groups4 * blocks * 256;                        // words
    // this thread's word of part (lane & 1); that of the third part, which the even lanes write, is part 2
    unsigned* mine = p.ring + ((int64_t)group * blocks + 2 * P + (lane >> 5)) * 256 +
                     (((lane >> 3) & 3) * 16 + 4 * (wave & 3)) * 4 + ((lane & 7) >> 1);
    const int own = (lane & 1) * 4, third = 2 * 4;

    // staging: all eight waves, a sample and 32 of its rows each (sixteen rows more in registers would not fit beside the
    // weights); access q covers neurons first + 4 q .. first + 4 q + 3
    const int n = 4 * group + (wave & 3), first_row = 32 * (wave >> 2);
    const unsigned lane_at = (unsigned)kk * (unsigned)T + (unsigned)j;
    auto row_ok = [&](int q) -> bool { return n < N && c0 + first_row + 4 * q < C; };
    auto next_rows = [&](int64_t& at) {
        at += 4 * (int64_t)T;
        asm volatile("" : "+s"(at));
    };
    float gn[8], vn[8], tn[THETA ? 8 : 1];
    auto fetch = [&](int t0) {
        int64_t at = ((int64_t)n * C + c0 + first_row) * T + t0;
#pragma unroll
        for (int q = 0; q < 8; ++q, next_rows(at)) {
            const bool ok = row_ok(q) && t0 + j < T;
            gn[q] = ok ? (p.g + at)[lane_at] : 0.f;
            vn[q] = ok ? (p.v + at)[lane_at] : 0.f;
            if (THETA) tn[q] = ok ? (p.theta + at)[lane_at] : 0.f;
        }
    };
    const int rows_of = (wave & 3) * kWave * kGridPitch;         // this wave's sample in the buffers
    float *gb = gbuf + rows_of, *fb = fbuf + rows_of, *ob = obuf + rows_of;
    auto put = [&]() {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            gb[(first_row + 4 * q + kk) * kGridPitch + j] = gn[q];
            fb[(first_row + 4 * q + kk) * kGridPitch + j] =
                row_ok(q) ? surrogate_factor(p, vn[q], THETA ? tn[q] : p.spike_thr) : 0.f;
        }
    };
    const int t_last = (T - 1) / kGridChunk * kGridChunk;
    fetch(t_last);
    put();
    lds_barrier();

    bool stop = false;
    int patience = kSpinLimit;                       // polls of a wait; none once one of this wave's has run out
    for (int t0 = t_last; t0 >= 0 && !stop; t0 -= kGridChunk) {
        if (t0 > 0) fetch(t0 - kGridChunk);
        const int steps = T - t0 < kGridChunk ? T - t0 : kGridChunk;
        for (int e = steps - 1; e >= 0; --e) {
            const int t = t0 + e, sel = t & 1;
            float gs = 0.f, factor = 0.f;
            if (wave < 4) {
                gs = gb[lane * kGridPitch + e];
                factor = fb[lane * kGridPitch + e];
                if (t + 3 < T) {
                    unsigned* at = mine + ((t + 3) & 3) * per_set;
                    __hip_atomic_store(at + own, kUnwritten, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if ((lane & 1) == 0) __hip_atomic_store(at + third, kUnwritten, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            if (t + 1 < T) {
                const int base = (((t + 1) & 3) * p.groups4 + group) * blocks * 1024 + lane * 16;
                auto load = [&](int u) -> v4u {
                    return __builtin_amdgcn_raw_buffer_load_b128(ring, base + (wave + kGridWaves * u) * 1024, 0, 16);
                };
                auto late = [&](v4u q) -> bool {
                    const unsigned m = max(max(max(q.x, q.y), q.z), q.w);        // kUnwritten is the largest word
                    return __any(part != 3 && m == kUnwritten);
                };
                v4u a[U];
                int spin = patience;
                auto wait = [&](int u) {
                    while (late(a[u])) {
                        if (spin == 0 || ((spin & 1023) == 1 &&
                                          __hip_atomic_load(p.gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
                            dead[(t0 / kGridChunk) & 1] = 1;
                            patience = spin = 0;
                            break;
                        }
                        --spin;
                        asm volatile("" ::: "memory");
                        a[u] = load(u);
                    }
                };
                // Eight blocks are requested at once ([32, 2048, 300] 1 170 us, one polled first and the others behind it 1 250),
                // fewer behind the first ([64, 1024, 100], whole layer 674 us, all at once 754).
                if (U < 8 && wave < blocks) { a[0] = load(0); wait(0); }
#pragma unroll
                for (int u = U < 8 ? 1 : 0; u < U; ++u)
                    if (wave + kGridWaves * u < blocks) a[u] = load(u);
                split_f4 acc[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] = split_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (wave + kGridWaves * u >= blocks) continue;
                    if (U >= 8 || u > 0) wait(u);
                    const uint4 b = make_uint4(a[u].x, a[u].y, a[u].z, a[u].w);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[r] = mfma_bf16(w[u][r], b, acc[r]);
                }
                // the three parts added up in the first two lanes of a quad, which keep two of the four row tiles each
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float x = acc[r][i];
                        x = (x + quad_swapped(x)) + quad_third(x);
                        asm volatile("" : "+v"(x));              // not moved behind the branch, so that the lanes are part of the addition
                        acc[r][i] = x;
                    }
                if (part < 2) {
                    float* at = &red[sel][wave][(j >> 2) * 68 + part * 32 + 4 * kk];
                    const split_f4 first = part == 0 ? acc[0] : acc[2], second = part == 0 ? acc[1] : acc[3];
                    *reinterpret_cast<float4*>(at) = make_float4(first[0], first[1], first[2], first[3]);
                    *reinterpret_cast<float4*>(at + 16) = make_float4(second[0], second[1], second[2], second[3]);
                }
            }
            lds_barrier();
            if (wave < 4) {
                if (t + 1 < T) {
                    float from[kGridWaves], carry = 0.f;
#pragma unroll
                    for (int v = 0; v < kGridWaves; ++v) from[v] = red[sel][v][wave * 68 + lane];
                    __builtin_amdgcn_sched_barrier(0);           // all eight under way before the first is waited for
#pragma unroll
                    for (int v = 0; v < kGridWaves; ++v) carry += from[v];
                    gs = carry * (1.0f / kLocalScale) + gs;
                }
                const float gz = c0 + lane < C ? factor * gs : 0.f;      // nothing beyond the layer: 0 times an infinity is none
                if (t > 0) {
                    // this neuron's parts, those of the pair's other neuron, and the words of both
                    const float x = gz * kLocalScale, size = fabsf(gz);
                    const unsigned bits = __float_as_uint(x);
                    unsigned h = bits & 0xffff0000u;
                    const float left = x - __uint_as_float(h);
                    unsigned m = __float_as_uint(left) & 0xffff0000u, l = __float_as_uint(left - __uint_as_float(m));
                    if (!(fabsf(x) <= 3.402823466e38f)) {        // infinities and NaN have no rest
                        h = x != x ? 0x7fc00000u : h;
                        m = l = 0u;
                    }
                    const unsigned sent = (lane & 1) ? h : m, got = quad_swapped(sent), l_odd = quad_swapped(l);
                    const unsigned first = (lane & 1) ? __builtin_amdgcn_perm(m, got, 0x07060302u)
                                                      : __builtin_amdgcn_perm(got, h, 0x07060302u);
                    unsigned* at = mine + (t & 3) * per_set;
                    __builtin_amdgcn_s_waitcnt(0x0f70);          // vmcnt(0): the clearing stores have arrived
                    __hip_atomic_store(at + own, first, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if ((lane & 1) == 0)
                        __hip_atomic_store(at + third, __builtin_amdgcn_perm(l_odd, l, 0x07060302u), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                    if (size >= kLocalLargest && size <= 3.402823466e38f) dead[(t0 / kGridChunk) & 1] = 1;      // left to the kernel behind
                }
                ob[lane * kGridPitch + e] = gz;
            }
            lds_barrier();                                       // see the forward kernel
        }
        int64_t at = ((int64_t)n * C + c0 + first_row) * T + t0;
#pragma unroll
        for (int q = 0; q < 8; ++q, next_rows(at))
            if (row_ok(q) && j < steps) (p.gz + at)[lane_at] = ob[(first_row + 4 * q + kk) * kGridPitch + j];
        if (t0 > 0) put();
        lds_barrier();
        stop = dead[(t0 / kGridChunk) & 1] != 0;                 // looked at once a chunk: the next step does not wait for it
    }
    if (stop && tid == 0) __hip_atomic_store(p.gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Thread (wave v, lane 4 j + i) of the first four waves has neuron 4 v + i of the tile and sample j.
template <bool THETA, int U, int NT>
__global__ __launch_bounds__(kGridThreads) void recurrent_grid_bwd_kernel(const GridBwd p) {
    constexpr int kPlane = 80;                       // pitch of a plane of red: reads of a wave meet 64 banks
    __shared__ __attribute__((aligned(16))) float red[2][kGridWaves][4][kPlane];
    __shared__ float gbuf[NT][4][kWave * kGridPitch], fbuf[NT][4][kWave * kGridPitch], obuf[NT][4][kWave * kGridPitch];
    __shared__ int dead[2];
    const int C = p.C, N = p.N, T = p.T, KB = p.KB;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (tid < 2) dead[tid] = 0;
    if constexpr (NT == 1)
        if (p.tiles64 > 0 && !__syncthreads_or(tid < kFillBlocks && p.inexact[tid] != 0u)) {
            grid_bwd_local<THETA, U / 2>(p, reinterpret_cast<float (*)[kGridWaves][4 * 68]>(&red[0][0][0][0]), gbuf[0][0], fbuf[0][0],
                                         obuf[0][0], dead);
            return;
        }
    const int kk = lane >> 4, j = lane & 15;
    const int P = p.map.tile(blockIdx.x), c0 = P * 16, group = p.map.group(blockIdx.x);
    if (P >= KB || group * NT >= p.S) return;

    // columns c0 .. c0 + 15 of R as A operands: lane (kk, j) has rows 16 kb + 4 kk .. + 3 of column c0 + j
    float4 w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int k = 16 * (wave + kGridWaves * u) + 4 * kk;
        const bool ok = c0 + j < C && k < C;                     // C is a multiple of 4
        const float* at = p.rec + (ok ? (int64_t)k * C + c0 + j : 0);
        w[u] = make_float4(at[0], at[ok ? C : 0], at[ok ? 2 * (int64_t)C : 0], at[ok ? 3 * (int64_t)C : 0]);
        if (!ok) w[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    const __amdgpu_buffer_rsrc_t ring = make_rsrc(reinterpret_cast<const float*>(p.ring), 4u * p.S * KB * 1024u);

    // staging as in the forward kernel: access q covers the four rows of sample q, lane (kk, j) step j of neuron 4 wave + kk
    const unsigned lane_at = (unsigned)kk * (unsigned)T + (unsigned)j;
    auto row_ok = [&](int s, int q) -> bool { return (group * NT + s) * 16 + q < N && c0 + 4 * wave < C; };
    auto first_row = [&](int s, int t0) -> int64_t {
        return ((int64_t)((group * NT + s) * 16) * C + c0 + 4 * wave) * T + t0;
    };
    auto next_rows = [&](int64_t& at) {
        at += (int64_t)C * T;
        asm volatile("" : "+s"(at));
    };
    float gn[NT][16], vn[NT][16], tn[THETA ? NT : 1][16];
    auto fetch = [&](int t0) {
#pragma unroll
        for (int s = 0; s < NT; ++s) {
            int64_t at = first_row(s, t0);
#pragma unroll
            for (int q = 0; q < 16; ++q, next_rows(at)) {
                const bool ok = row_ok(s, q) && t0 + j < T;
                gn[s][q] = ok ? (p.g + at)[lane_at] : 0.f;
                vn[s][q] = ok ? (p.v + at)[lane_at] : 0.f;
                if (THETA) tn[s][q] = ok ? (p.theta + at)[lane_at] : 0.f;
            }
        }
    };
    auto put = [&]() {
#pragma unroll
        for (int s = 0; s < NT; ++s)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                gbuf[s][wave][(4 * q + kk) * kGridPitch + j] = gn[s][q];
                fbuf[s][wave][(4 * q + kk) * kGridPitch + j] =
                    row_ok(s, q) ? surrogate_factor(p, vn[s][q], THETA ? tn[s][q] : p.spike_thr) : 0.f;
            }
        wave_lds_order();
    };
    const int t_last = (T - 1) / kGridChunk * kGridChunk;
    if (wave < 4) { fetch(t_last); put(); }
    lds_barrier();

    bool stop = false;
    for (int t0 = t_last; t0 >= 0 && !stop; t0 -= kGridChunk) {
        if (wave < 4 && t0 > 0) fetch(t0 - kGridChunk);
        const int steps = T - t0 < kGridChunk ? T - t0 : kGridChunk;
        for (int e = steps - 1; e >= 0 && !stop; --e) {
            const int t = t0 + e;
#pragma unroll
            for (int s = 0; s < NT; ++s) {
                const int sel = NT == 1 ? (t & 1) : s & 1;
                const int tile = group * NT + s;
                auto set_at = [&](int step) -> int { return (((step & 3) * p.S + tile) * KB) * 1024; };   // bytes
                unsigned* mine = p.ring + set_at(0) / 4 + P * 256 + tid;                    // of set 0; tid < 256
                const int per_set = p.S * KB * 256;
                float gs = 0.f, factor = 0.f;
                if (wave < 4) {
                    gs = gbuf[s][wave][lane * kGridPitch + e];
                    factor = fbuf[s][wave][lane * kGridPitch + e];
                    if (t + 3 < T)
                        __hip_atomic_store(mine + (int64_t)((t + 3) & 3) * per_set, kUnwritten, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                if (t + 1 < T) {
                    const int base = set_at(t + 1) + lane * 16;
                    auto load = [&](int u) -> v4u {
                        const int kb = wave + kGridWaves * u;
                        return __builtin_amdgcn_raw_buffer_load_b128(ring, base + kb * 1024, 0, 16);     // agent scope
                    };
                    auto unwritten = [&](v4u q) -> bool {
                        return q.x == kUnwritten || q.y == kUnwritten || q.z == kUnwritten || q.w == kUnwritten;
                    };
                    v4u a[U];
                    int spin = 0;
                    auto wait = [&](int u) {                     // until block u of this wave is there
                        while (__any(unwritten(a[u]))) {
                            if (spin == kSpinLimit ||
                                ((spin & 1023) == 1023 &&
                                 __hip_atomic_load(p.gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
                                dead[sel] = 1;
                                spin = kSpinLimit;
                                break;
                            }
                            ++spin;
                            asm volatile("" ::: "memory");
                            a[u] = load(u);
                        }
                    };
                    // the first block is polled, the others are requested when it is there
                    if (wave < KB) { a[0] = load(0); wait(0); }
#pragma unroll
                    for (int u = 1; u < U; ++u)
                        if (wave + kGridWaves * u < KB) a[u] = load(u);
                    split_f4 acc[2] = {split_f4{0.f, 0.f, 0.f, 0.f}, split_f4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        if (wave + kGridWaves * u >= KB) continue;                        // the same for the whole wave
                        if (u > 0) wait(u);
                        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u].x, __uint_as_float(a[u].x), acc[0], 0, 0, 0);
                        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u].y, __uint_as_float(a[u].y), acc[1], 0, 0, 0);
                        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u].z, __uint_as_float(a[u].z), acc[0], 0, 0, 0);
                        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u].w, __uint_as_float(a[u].w), acc[1], 0, 0, 0);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) red[sel][wave][i][lane] = acc[0][i] + acc[1][i];
                }
                lds_barrier();
                if (wave < 4) {
                    if (t + 1 < T) {
                        float carry = 0.f;
#pragma unroll
                        for (int v = 0; v < kGridWaves; ++v) carry += red[sel][v][lane & 3][wave * 16 + (lane >> 2)];
                        gs = carry + gs;
                    }
                    const float gz = c0 + 4 * wave < C ? factor * gs : 0.f;      // nothing beyond the layer: 0 times an infinity is none
                    if (t > 0) {
                        const unsigned bits = __float_as_uint(gz);
                        __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): the clearing store has arrived
                        __hip_atomic_store(mine + (int64_t)(t & 3) * per_set, bits == kUnwritten ? 0x7fffffffu : bits,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                    obuf[s][wave][lane * kGridPitch + e] = gz;
                }
                stop = stop || dead[sel] != 0;
                lds_barrier();                                   // see the forward kernel
            }
        }
        if (wave < 4) {
#pragma unroll
            for (int s = 0; s < NT; ++s) {
                wave_lds_order();
                int64_t at = first_row(s, t0);
#pragma unroll
                for (int q = 0; q < 16; ++q, next_rows(at))
                    if (row_ok(s, q) && j < steps) (p.gz + at)[lane_at] = obuf[s][wave][(4 * q + kk) * kGridPitch + j];
            }
            wave_lds_order();
            if (t0 > 0) put();
        }
    }
    if (stop && tid == 0) __hip_atomic_store(p.gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(kSoloThreads) void recurrent_solo_bwd_kernel(const GridBwd p) {
    __shared__ float next[2][kGridMaxC];
    if (*p.gave_up == 0u) return;
    for (int t = p.T - 1; t >= 0; --t) {
        for (int c = threadIdx.x; c < p.C; c += kSoloThreads) {
            const int64_t at = ((int64_t)blockIdx.x * p.C + c) * p.T + t;
            double carry = 0.0;
            if (t + 1 < p.T)
                for (int k = 0; k < p.C; ++k) carry += (double)next[(t + 1) & 1][k] * (double)p.rec[(int64_t)k * p.C + c];
            const float gz = surrogate_factor(p, p.v[at], p.theta ? p.theta[at] : p.spike_thr) * ((float)carry + p.g[at]);
            next[t & 1][c] = gz;
            p.gz[at] = gz;
        }
        __syncthreads();
    }
}

namespace {

struct GridPlan {
    int KB, S, NT;
    GridMap map;
    unsigned grid;
    int compute_units;
};

// One workgroup per compute unit: 16 neurons by one or two sample tiles.  A handful of steps costs more as a
// cooperative launch (14 us more than a plain one) than as separate launches (7 us each).
bool grid_plan(int64_t N, int64_t C, int64_t T, hipStream_t st, GridPlan* plan) {
    if (C > kGridMaxC || T < 8 || T > kGridMaxT) return false;
    int dev = 0, units = 0, coop = 0;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess || !coop ||
        hipStreamIsCapturing(st, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return false;
    }
    const int64_t KB = (C + 15) / 16, tiles = (N + 15) / 16;
    for (int nt = 1; nt <= 2; ++nt) {
        const int64_t groups = (tiles + nt - 1) / nt;
        for (int xcds = 1; xcds <= 8; xcds *= 2) {
            const int64_t per_xcd = (KB + xcds - 1) / xcds, rounds = (groups + 8 / xcds - 1) / (8 / xcds);
            if (8 * per_xcd * rounds > units) continue;
            plan->KB = (int)KB; plan->S = (int)(groups * nt); plan->NT = nt;
            plan->map.xcds = xcds; plan->map.per_xcd = (int)per_xcd;
            plan->grid = (unsigned)(8 * per_xcd * rounds);
            plan->compute_units = units;
            return true;
        }
    }
    return false;
}

struct Floats { const float* at; int64_t n; };                    // at = nullptr: none
// Whether results lie over inputs.  The kernel behind computes a layer again from its inputs, so such a call takes a launch per step,
// which copies its inputs first.
bool overlap(std::initializer_list<Floats> results, std::initializer_list<Floats> inputs) {
    for (const Floats& a : results)
        for (const Floats& b : inputs) {
            const uintptr_t p = (uintptr_t)a.at, q = (uintptr_t)b.at;
            if (a.at && b.at && p < q + 4 * (uintptr_t)b.n && q < p + 4 * (uintptr_t)a.n) return true;
        }
    return false;
}

// false: the runtime does not take the grid as a cooperative one
bool launch_grid(const void* kernel, unsigned grid, void* args, hipStream_t st) {
    void* list[] = {args};
    if (hipLaunchCooperativeKernel(kernel, dim3(grid), dim3(kGridThreads), list, 0, st) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
}

template <bool ALIF, bool POW2>
bool launch_grid_fwd(const GridFwd& g, const GridPlan& plan, hipStream_t st) {
    const bool narrow = plan.KB <= 8 * kGridWaves;               // one unit a wave
    const void* k = plan.NT == 1
        ? (narrow ? (const void*)recurrent_grid_fwd_kernel<ALIF, POW2, 1, 1> : (const void*)recurrent_grid_fwd_kernel<ALIF, POW2, 2, 1>)
        : (narrow ? (const void*)recurrent_grid_fwd_kernel<ALIF, POW2, 1, 2> : (const void*)recurrent_grid_fwd_kernel<ALIF, POW2, 2, 2>);
    if (!launch_grid(k, plan.grid, (void*)&g, st)) return false;
    hipLaunchKernelGGL((recurrent_solo_fwd_kernel<ALIF, POW2>), dim3((unsigned)(g.p.N + 15) / 16), dim3(kGridThreads), 0, st, g);
    return true;
}

}  // namespace

bool grid_fwd(StepFwd p, bool alif, bool pow2, float* spk, float* vol, float* theta, const float* z, const float* rec,
              float* workspace, int64_t workspace_floats, hipStream_t st, int* error) {
    GridPlan plan;
    if (!grid_plan(p.N, p.C, p.T, st, &plan)) return false;
    const int64_t words = (int64_t)2 * plan.S * words_of(plan.KB);
    const int64_t nc = (int64_t)p.N * p.C, nct = nc * p.T;
    if (workspace_floats < 4 + words + 4 * nc) return false;
    if (overlap({{spk, nct}, {vol, nct}, {theta, nct}, {p.cur_last, nc}, {p.vol_last, nc}, {p.th_last, nc}, {p.ref_last, nc}},
                {{z, nct}, {rec, (int64_t)p.C * p.C}, {p.i_decay, p.n_id}, {p.v_decay, p.n_vd}, {p.th_decay, p.n_td},
                 {p.ref_decay, p.n_rd}, {p.i_state, p.n_is}, {p.v_state, p.n_vs}, {p.th_state, p.n_ts}, {p.ref_state, p.n_rs}}))
        return false;
    GridFwd g{};
    g.p = p;
    g.p.KB = plan.KB; g.p.S = plan.S;
    g.map = plan.map;
    g.spk = spk; g.vol = vol; g.theta = theta; g.z = z; g.rec = rec;
    g.gave_up = reinterpret_cast<unsigned*>(workspace);
    g.words = reinterpret_cast<unsigned*>(workspace) + 4;
    g.carried = reinterpret_cast<int*>(workspace) + 4 + words;
    hipLaunchKernelGGL(grid_fill_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, g.words, words, g.gave_up);
    const bool taken = alif ? (pow2 ? launch_grid_fwd<true, true>(g, plan, st) : launch_grid_fwd<true, false>(g, plan, st))
                            : (pow2 ? launch_grid_fwd<false, true>(g, plan, st) : launch_grid_fwd<false, false>(g, plan, st));
    if (taken) *error = (int)hipGetLastError();
    return taken;
}

namespace {
template <bool THETA, int NT>
const void* grid_bwd_kernel(int KB) {
    if (KB <= 4 * kGridWaves) return (const void*)recurrent_grid_bwd_kernel<THETA, 4, NT>;
    if (KB <= 8 * kGridWaves) return (const void*)recurrent_grid_bwd_kernel<THETA, 8, NT>;
    return (const void*)recurrent_grid_bwd_kernel<THETA, 16, NT>;
}
}  // namespace

bool grid_bwd(float* gz, const float* grad_spikes, const float* voltage, const float* theta, const float* rec,
              float spike_thr, float tau, float rho, int graded, int64_t N, int64_t C, int64_t T,
              float* workspace, int64_t workspace_floats, hipStream_t st, int* error) {
    GridPlan plan;
    if (!grid_plan(N, C, T, st, &plan)) return false;
    int64_t ring = (int64_t)4 * plan.S * plan.KB * 256;
    const int64_t head = 4 + kFillBlocks;
    if (workspace_floats < ring + head) return false;
    const int64_t nct = N * C * T;
    if (overlap({{gz, nct}}, {{grad_spikes, nct}, {voltage, nct}, {theta, nct}, {rec, C * C}})) return false;
    GridBwd p{};
    p.gz = gz; p.g = grad_spikes; p.v = voltage; p.theta = theta; p.rec = rec;
    p.gave_up = reinterpret_cast<unsigned*>(workspace);
    p.ring = reinterpret_cast<unsigned*>(workspace) + head;
    p.map = plan.map;
    // four samples to an XCD, as long as the chip holds them all
    const int64_t groups4 = (N + 3) / 4, tiles64 = (C + 63) / 64, rounds = (groups4 + 7) / 8;
    const int64_t local_ring = (int64_t)4 * groups4 * 2 * tiles64 * 256;
    unsigned grid = plan.grid;
    if (plan.NT == 1 && 8 * rounds * tiles64 <= plan.compute_units && workspace_floats >= local_ring + head) {
        p.groups4 = (int)groups4;
        p.tiles64 = (int)tiles64;
        if (grid < 8 * rounds * tiles64) grid = (unsigned)(8 * rounds * tiles64);
        if (ring < local_ring) ring = local_ring;
    }
    unsigned* inexact = reinterpret_cast<unsigned*>(workspace) + 4;
    p.inexact = inexact;
    p.KB = plan.KB; p.S = plan.S; p.N = (int)N; p.C = (int)C; p.T = (int)T; p.graded = graded;
    p.spike_thr = spike_thr; p.tau = tau; p.rho = rho;
    hipLaunchKernelGGL(grid_bwd_fill_kernel, dim3(kFillBlocks), dim3(1024), 0, st, p.ring, ring, p.gave_up, rec, C * C, inexact);
    const void* k = theta ? (plan.NT == 1 ? grid_bwd_kernel<true, 1>(plan.KB) : grid_bwd_kernel<true, 2>(plan.KB))
                          : (plan.NT == 1 ? grid_bwd_kernel<false, 1>(plan.KB) : grid_bwd_kernel<false, 2>(plan.KB));
    if (!launch_grid(k, grid, (void*)&p, st)) return false;
    hipLaunchKernelGGL(recurrent_solo_bwd_kernel, dim3((unsigned)N), dim3(kSoloThreads), 0, st, p);
    *error = (int)hipGetLastError();
    return true;
}

}  // namespace slayer
