// Weight gradient of the convolution synapse on time-innermost tensors, products on the bfloat16 matrix instruction, of every
// geometry with one to five taps along the axis that is walked.
//
// As in the convolution (synapse_walk.hip) one axis of the image is walked and the other one and time are one line of
// positions, which here is what the sums run over: a visit is 32 positions, the 128 bytes of a line of memory where the rows
// of the image are whole lines.  Rows of a product are 16 channels of the gradient, its columns 16 (input channel, line tap, row
// of the step) triples; a step brings one gradient row and its input rows, the gradient of the last KS rows stays in
// registers, so a visit and step costs 1 + NPT loads for KS NPT tiles of sums.  With tiles of one pixel's steps (the form before) a
// line was fetched by the two tiles that met in it (rows of 300 steps: 2.0 x the tensors read) and strided layers, among them
// every transposed one, had the float32 instruction.  [32,8,32,32,300] -> 16 channels 338 -> 243 us between the layer's other passes
// (400 -> 291 with the caches swept; it fetches 1.02 x the tensors now), [16,32,16,16,300] -> 64 336 -> 296, 4x4 stride 2 between
// [32,8,32,32,300] and 16 channels 327 -> 184; 220 layers (3x3, 5x5, strides 1 and 2, 4x4 transposed): 0.64 of the time before
// in the mean.
//
// Neighbouring lanes of the operand's layout lie in sixteen different rows, so a load of 1 KB would look up 64 lines: eight
// lanes read the 128 bytes of a row together, and the split values reach the operand's layout through LDS of the wave's own.
// Either operand is split into three parts (split.h) where its values are not bfloat16 numbers as they are, looked at once a
// visit and step: one product, three or six.
//
// The instruction rounds its sums down, not to nearest: a bias of some 2^-27 a product that a sum over 10^4 of them
// collects (relative error of the result 1e-6, float32 instruction 1.3e-7 .. 5.7e-7).  The products of a visit and step therefore
// start from zero, every other step with the input negated, and the vector units add or subtract them: the biases cancel,
// and the error against float64 is 0.5e-7 .. 1.0e-7.
//
// The sums of a workgroup's waves are added in double before they are written; where waves are few, these are four pieces of the
// rows.  What is not finite (or overflows when it is scaled or rounded) shows in a tile at the end: the wave then runs its
// share again with the float32 instruction (float_products).
#include "synapse.h"
#include "split.h"

namespace slayer {

constexpr int kWgPitch = 80;                   // bytes of LDS per row of 32 bfloat16: no two quarters of a read collide
constexpr int kWgSlot = 16 * kWgPitch;         // one part of one tile of 16 rows
constexpr int kWgQuads = 8;                    // quads of steps to a visit

template <int KS, int NPT>
struct WgradWave {
    const WgradWalk& p;
    static constexpr int kSlots = 3 + 3 * NPT; // three parts of the gradient and of every tile of the input
    char* lds;                                 // kSlots slots of this wave
    __amdgpu_buffer_rsrc_t src, grd;
    int co0, pair0, q_lo, q_hi, s_lo, s_hi, lane;
    syn_f4 acc[KS][NPT];

    struct Pair { int off, shift, row; };      // offset of its input row at step 0, line shift, row of the step; off none: no such pair
    __device__ __forceinline__ Pair pair(int r) const {
        const int pr = pair0 + r, ci = p.by_triples.of(pr), rem = pr - ci * (p.XP * p.ss), x = p.by_ss.of(rem), row = rem - x * p.ss;
        const int shift = p.shift0 + x * p.shift_step;
        if (pr >= p.pairs) return {kOutOfRange, 0, 0};
        return {ci * p.in_ch + shift * p.in_line + row * p.in_slide, shift, row};
    }
    __device__ __forceinline__ int channel(int r) const { return co0 + r < p.Co ? (co0 + r) * p.out_ch : kOutOfRange; }
    // Quad `quad` of the line: pixel m, steps t .. t + 3.  A pixel's last quad is its last four steps; `repeats` of them belong
    // to the quad before and count as zero.
    struct Place { bool on; int m, t, repeats; };
    __device__ __forceinline__ Place place(int quad) const {
        Place a;
        a.on = quad < q_hi;
        a.m = a.on ? p.by_quads.of(quad) : 0;
        a.t = 4 * (quad - a.m * p.quads);
        a.repeats = a.on && a.t > p.T - 4 ? a.t - (p.T - 4) : 0;
        a.t -= a.repeats;
        return a;
    }
    __device__ __forceinline__ static float4 once(float4 v, int repeats) {
        return make_float4(repeats > 0 ? 0.f : v.x, repeats > 1 ? 0.f : v.y, repeats > 2 ? 0.f : v.z, v.w);
    }
    __device__ __forceinline__ int grad_at(int off, int s) const {
        return (off != kOutOfRange && s >= s_lo && s < s_hi) ? off + s * p.out_slide : kOutOfRange;
    }
    __device__ __forceinline__ int input_at(int off, int row, int c) const {
        return (off != kOutOfRange && (unsigned)(c * p.ss + p.row0 + row) < (unsigned)p.Hs) ? off + (c * p.ss + p.row0) * p.in_slide
                                                                                            : kOutOfRange;
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int x = 0; x < KS; ++x)
#pragma unroll
            for (int pt = 0; pt < NPT; ++pt) acc[x][pt] = syn_f4{0.f, 0.f, 0.f, 0.f};
    }
    // the wave's own LDS: its instructions run in order, the fences keep the compiler to that order
    __device__ __forceinline__ static void settle() {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // Lane l holds quad l % 8 of row l / 8 (+ 8 in the second quad); the operand's lane (kk, j) takes positions
    // 8 kk .. 8 kk + 7 of row j.
    __device__ __forceinline__ void put(int slot, int half, uint2 v) const {
        *reinterpret_cast<uint2*>(lds + slot * kWgSlot + ((lane >> 3) + 8 * half) * kWgPitch + (lane & 7) * 8) = v;
    }
    __device__ __forceinline__ uint4 get(int slot) const {
        return *reinterpret_cast<const uint4*>(lds + slot * kWgSlot + (lane & 15) * kWgPitch + (lane >> 4) * 16);
    }
    __device__ __forceinline__ static float4 scaled(float4 v) {
        return make_float4(v.x * kSplitScale, v.y * kSplitScale, v.z * kSplitScale, v.w * kSplitScale);
    }
    __device__ __forceinline__ static unsigned low_bits(float4 v) {
        return __float_as_uint(v.x) | __float_as_uint(v.y) | __float_as_uint(v.z) | __float_as_uint(v.w);
    }
    __device__ __forceinline__ void put_parts(int slot, const float4 (&raw)[2], bool more) const {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float4 v = scaled(raw[h]);
            if (!more) {
                put(slot, h, make_uint2(bf16_pair(v.x, v.y), bf16_pair(v.z, v.w)));
            } else {
                uint2 part;
                part.x = round_pair(v.x, v.y); part.y = round_pair(v.z, v.w);
                put(slot, h, part);
                part.x = round_pair(v.x, v.y); part.y = round_pair(v.z, v.w);
                put(slot + 1, h, part);
                put(slot + 2, h, make_uint2(bf16_pair(v.x, v.y), bf16_pair(v.z, v.w)));
            }
        }
    }

    __device__ __forceinline__ void split_products() {
        clear();
        const int c_end = s_hi + KS - 1;
        const int c_lo = s_lo > p.c_lo ? s_lo : p.c_lo, c_hi = c_end < p.c_hi ? c_end : p.c_hi;
        if (c_lo >= c_hi) return;
        Pair prs[NPT][2];
        int chan[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            chan[h] = channel((lane >> 3) + 8 * h);
#pragma unroll
            for (int pt = 0; pt < NPT; ++pt) prs[pt][h] = pair(16 * pt + (lane >> 3) + 8 * h);
        }
        for (int quad0 = q_lo; quad0 < q_hi; quad0 += kWgQuads) {
            const Place at = place(quad0 + (lane & 7));
            const bool repeats = __any(at.repeats != 0);
            int g_off[2], q_off[NPT][2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                g_off[h] = at.on && chan[h] != kOutOfRange ? chan[h] + at.m * p.out_line + at.t * 4 : kOutOfRange;
#pragma unroll
                for (int pt = 0; pt < NPT; ++pt) {
                    const Pair& pr = prs[pt][h];
                    const bool in = at.on && pr.off != kOutOfRange && (unsigned)(at.m * p.ls + pr.shift) < (unsigned)p.Ws;
                    q_off[pt][h] = in ? pr.off + at.m * p.ls * p.in_line + at.t * 4 : kOutOfRange;
                }
            }
            float4 raw_g[2], raw_q[NPT][2];
            auto fetch = [&](int c) {
#pragma unroll
                for (int h = 0; h < 2; ++h) raw_g[h] = buf_load4<false>(grd, grad_at(g_off[h], c));
#pragma unroll
                for (int pt = 0; pt < NPT; ++pt)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        raw_q[pt][h] = buf_load4<false>(src, input_at(q_off[pt][h], prs[pt][h].row, c));
            };
            // gw[x]: the gradient of row c - x for the step c at hand; gw[0] arrives with the step.  split_g: bit x, whether it
            // has lower parts.
            uint4 gw[KS][3];
            unsigned split_g = 0u;
            float4 first[KS][2];
#pragma unroll
            for (int x = KS - 1; x >= 1; --x)
#pragma unroll
                for (int h = 0; h < 2; ++h) first[x][h] = buf_load4<false>(grd, grad_at(g_off[h], c_lo - x));
            fetch(c_lo);
#pragma unroll
            for (int x = KS - 1; x >= 1; --x) {
                if (repeats)
#pragma unroll
                    for (int h = 0; h < 2; ++h) first[x][h] = once(first[x][h], at.repeats);
                put_parts(0, first[x], true);
                settle();
#pragma unroll
                for (int t = 0; t < 3; ++t) gw[x][t] = get(t);
                settle();
                split_g |= __any(((low_bits(first[x][0]) | low_bits(first[x][1])) & 0xffffu) != 0u) ? 1u << (x - 1) : 0u;
            }
            for (int c = c_lo; c < c_hi; ++c) {
                const unsigned flip = (c & 1) ? 0x80008000u : 0u;
                const float back = (c & 1) ? -kSplitProductScale : kSplitProductScale;
                auto flipped = [&](uint4 v) { return make_uint4(v.x ^ flip, v.y ^ flip, v.z ^ flip, v.w ^ flip); };
                if (repeats) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        raw_g[h] = once(raw_g[h], at.repeats);
#pragma unroll
                        for (int pt = 0; pt < NPT; ++pt) raw_q[pt][h] = once(raw_q[pt][h], at.repeats);
                    }
                }
                unsigned low = 0u;
#pragma unroll
                for (int pt = 0; pt < NPT; ++pt)
#pragma unroll
                    for (int h = 0; h < 2; ++h) low |= low_bits(raw_q[pt][h]);
                const bool more = __any((low & 0xffffu) != 0u);          // more than bfloat16 holds
                const bool more_g = __any(((low_bits(raw_g[0]) | low_bits(raw_g[1])) & 0xffffu) != 0u);
                split_g = split_g << 1 | (more_g ? 1u : 0u);
                const bool any_g = (split_g & ((1u << KS) - 1u)) != 0u;
                put_parts(0, raw_g, more_g);
#pragma unroll
                for (int pt = 0; pt < NPT; ++pt) put_parts(3 + 3 * pt, raw_q[pt], more);
                settle();
                if (c + 1 < c_hi) fetch(c + 1);                          // on its way during the products
                gw[0][0] = get(0);
                gw[0][1] = gw[0][2] = make_uint4(0u, 0u, 0u, 0u);
                if (more_g) { gw[0][1] = get(1); gw[0][2] = get(2); }
#pragma unroll
                for (int pt = 0; pt < NPT; ++pt) {
                    const uint4 q = flipped(get(3 + 3 * pt));
                    syn_f4 d[KS];
#pragma unroll
                    for (int x = 0; x < KS; ++x) d[x] = syn_f4{0.f, 0.f, 0.f, 0.f};
                    if (any_g)
#pragma unroll
                        for (int x = 0; x < KS; ++x) d[x] = mfma_bf16(gw[x][2], q, d[x]);
                    if (more) {
                        const uint4 q1 = flipped(get(4 + 3 * pt)), q2 = flipped(get(5 + 3 * pt));
#pragma unroll
                        for (int x = 0; x < KS; ++x) d[x] = mfma_bf16(gw[x][0], q2, d[x]);
                        if (any_g)
#pragma unroll
                            for (int x = 0; x < KS; ++x) d[x] = mfma_bf16(gw[x][1], q1, d[x]);
#pragma unroll
                        for (int x = 0; x < KS; ++x) d[x] = mfma_bf16(gw[x][0], q1, d[x]);
                    }
                    if (any_g)
#pragma unroll
                        for (int x = 0; x < KS; ++x) d[x] = mfma_bf16(gw[x][1], q, d[x]);
#pragma unroll
                    for (int x = 0; x < KS; ++x) d[x] = mfma_bf16(gw[x][0], q, d[x]);
#pragma unroll
                    for (int x = 0; x < KS; ++x)
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[x][pt][i] = __fmaf_rn(back, d[x][i], acc[x][pt][i]);
                }
                settle();
#pragma unroll
                for (int x = KS - 1; x >= 1; --x)
#pragma unroll
                    for (int t = 0; t < 3; ++t) gw[x][t] = gw[x - 1][t];
            }
        }
    }
    // the same sums on the float32 instruction, 16 positions at a time
    __device__ __forceinline__ void float_products() {
        clear();
        const int chan = channel(lane & 15);
        Pair prs[NPT];
#pragma unroll
        for (int pt = 0; pt < NPT; ++pt) prs[pt] = pair(16 * pt + (lane & 15));
        const int c_end = s_hi + KS - 1;
        const int c_lo = s_lo > p.c_lo ? s_lo : p.c_lo, c_hi = c_end < p.c_hi ? c_end : p.c_hi;
        for (int quad0 = q_lo; quad0 < q_hi; quad0 += 4) {
            const Place at = place(quad0 + (lane >> 4));
            const int g_off = at.on && chan != kOutOfRange ? chan + at.m * p.out_line + at.t * 4 : kOutOfRange;
            for (int c = c_lo; c < c_hi; ++c) {
#pragma unroll
                for (int x = 0; x < KS; ++x) {
                    if (c - x < s_lo || c - x >= s_hi) continue;             // another piece's row, or none: no product with zero
                    const float4 g = once(buf_load4<false>(grd, grad_at(g_off, c - x)), at.repeats);
#pragma unroll
                    for (int pt = 0; pt < NPT; ++pt) {
                        const bool in = at.on && prs[pt].off != kOutOfRange &&
                                        (unsigned)(at.m * p.ls + prs[pt].shift) < (unsigned)p.Ws;
                        const int off = in ? prs[pt].off + at.m * p.ls * p.in_line + at.t * 4 : kOutOfRange;
                        const float4 q = once(buf_load4<false>(src, input_at(off, prs[pt].row, c)), at.repeats);
                        acc[x][pt] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.x, q.x, acc[x][pt], 0, 0, 0);
                        acc[x][pt] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.y, q.y, acc[x][pt], 0, 0, 0);
                        acc[x][pt] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.z, q.z, acc[x][pt], 0, 0, 0);
                        acc[x][pt] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.w, q.w, acc[x][pt], 0, 0, 0);
                    }
                }
            }
        }
    }
    __device__ __forceinline__ bool not_finite() const {
        bool bad = false;
#pragma unroll
        for (int x = 0; x < KS; ++x)
#pragma unroll
            for (int pt = 0; pt < NPT; ++pt)
#pragma unroll
                for (int i = 0; i < 4; ++i) bad = bad || !(fabsf(acc[x][pt][i]) < __builtin_inff());
        return __any(bad);
    }
};

template <int KS, int NPT>
__global__ __launch_bounds__(kSynWaves * kWave) __attribute__((amdgpu_waves_per_eu(KS <= 3 || NPT == 1 ? 3 : 2)))
void synapse_wgrad_walk_kernel(const WgradWalk p) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int cobs = (p.Co + 15) / 16;
    // The waves of a workgroup take neighbouring shares, or the pieces of one, and their sums are one set of tiles; or, with many
    // channel blocks and passes, these of one share: they read the same input rows and gradient rows at about the same time
    // and find them in the L1 and L2.
    const bool together = p.pieces > 1 || p.sets < p.shares;
    int b = xcd_contiguous(blockIdx.x, gridDim.x);
    if (!together) b = b * kSynWaves + wave;
    const int cob = p.by_cobs.rest(b); b = p.by_cobs.of(b);
    const int pass = p.by_passes.rest(b); b = p.by_passes.of(b);
    const int set = p.by_sets.rest(b), n = p.by_sets.of(b);
    if (n >= p.N) return;                               // (never together: those are whole workgroups)
    const int share = p.sets < p.shares ? set * kSynWaves + wave : set, piece = p.pieces > 1 ? wave : 0;
    const int per = (p.S + p.pieces - 1) / p.pieces;
    __shared__ __attribute__((aligned(16))) char lds[kSynWaves][WgradWave<KS, NPT>::kSlots * kWgSlot];
    WgradWave<KS, NPT> w{p};
    w.lds = lds[wave];
    w.src = make_rsrc(p.in + (int64_t)n * (p.in_plane / 4), (unsigned)p.in_plane);
    w.grd = make_rsrc(p.grad_out + (int64_t)n * (p.out_plane / 4), (unsigned)p.out_plane);
    w.lane = lane;
    w.co0 = cob * 16;
    w.pair0 = pass * NPT * 16;
    w.q_lo = share * p.share_quads;
    w.q_hi = w.q_lo + p.share_quads < p.line_quads ? w.q_lo + p.share_quads : p.line_quads;
    w.s_lo = piece * per;
    w.s_hi = w.s_lo + per < p.S ? w.s_lo + per : p.S;      // at or below s_lo: nothing to do
    w.split_products();
    if (w.not_finite()) w.float_products();
    // lane (q, j) of tile (x, pt): channels co0 + 4 q + i, pair 16 (pass NPT + pt) + j, tap x of the walk
    float4* dst = reinterpret_cast<float4*>(p.partial) +
                  ((((int64_t)(n * cobs + cob) * p.sets + set) * p.passes + pass) * (KS * NPT)) * kWave + lane;
    if (!together) {
#pragma unroll
        for (int x = 0; x < KS; ++x)
#pragma unroll
            for (int pt = 0; pt < NPT; ++pt)
                dst[(x * NPT + pt) * kWave] = make_float4(w.acc[x][pt][0], w.acc[x][pt][1], w.acc[x][pt][2], w.acc[x][pt][3]);
        return;
    }
    static_assert(sizeof(lds) >= kSynWaves * KS * NPT * kWave * sizeof(float4), "the waves' tiles fit their slots");
    float4* tiles = reinterpret_cast<float4*>(&lds[0][0]);
    __syncthreads();                                    // every wave is done with its slots
#pragma unroll
    for (int x = 0; x < KS; ++x)
#pragma unroll
        for (int pt = 0; pt < NPT; ++pt)
            tiles[(wave * KS * NPT + x * NPT + pt) * kWave + lane] =
                make_float4(w.acc[x][pt][0], w.acc[x][pt][1], w.acc[x][pt][2], w.acc[x][pt][3]);
    __syncthreads();
    for (int tl = wave; tl < KS * NPT; tl += kSynWaves) {
        double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int other = 0; other < kSynWaves; ++other) {
            const float4 v = tiles[(other * KS * NPT + tl) * kWave + lane];
            sum[0] += v.x; sum[1] += v.y; sum[2] += v.z; sum[3] += v.w;
        }
        dst[tl * kWave] = make_float4((float)sum[0], (float)sum[1], (float)sum[2], (float)sum[3]);
    }
}

int launch_synapse_wgrad_walk(WgradWalk& w, hipStream_t st) {
    w.by_cobs = (w.Co + 15) / 16; w.by_passes = w.passes; w.by_sets = w.sets; w.by_quads = w.quads; w.by_triples = w.XP * w.ss; w.by_ss = w.ss;
    const int64_t sets = (int64_t)w.N * ((w.Co + 15) / 16) * w.sets * w.passes;          // of tiles
    const int64_t blocks = w.pieces > 1 || w.sets < w.shares ? sets : (sets + kSynWaves - 1) / kSynWaves;
    if (blocks > 0x7fffffffLL / kSynWaves) return SLAYER_ERANGE;
    const dim3 grid((unsigned)blocks), block(kSynWaves * kWave);
#define SLAYER_WGRAD_WALK(KS)                                                                                   \
    do {                                                                                                          \
        if (w.npt == 1) hipLaunchKernelGGL((synapse_wgrad_walk_kernel<KS, 1>), grid, block, 0, st, w);             \
        else hipLaunchKernelGGL((synapse_wgrad_walk_kernel<KS, 2>), grid, block, 0, st, w);                        \
    } while (0)
    if (w.KS == 1) SLAYER_WGRAD_WALK(1);
    else if (w.KS == 2) SLAYER_WGRAD_WALK(2);
    else if (w.KS == 3) SLAYER_WGRAD_WALK(3);
    else SLAYER_WGRAD_WALK(5);
#undef SLAYER_WGRAD_WALK
    return (int)hipGetLastError();
}

}  // namespace slayer
