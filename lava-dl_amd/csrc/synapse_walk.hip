// Convolution synapse on time-innermost tensors, products on the bfloat16 matrix instruction: forward pass, input gradient and
// transposed convolution of every geometry with one to five taps along the axis that is walked.
//
// One axis of the image (the rows, where the filter allows) is walked, the other one and time are one "line" of positions: M
// pixels of T steps, in memory one piece.  A wave owns 64 positions of the line and 16 or 32 output channels and walks the rows: a
// step brings the input row (`ss` rows, the stride along the walk) at the line's XP taps, each loaded and split into bfloat16
// parts once for all KS taps along the walk, whose sums are KS sets of accumulators; an output row is stored when its last
// row has come.  Tiles are 64 positions of the line rather than of a pixel's row, so their stores fill whole 128-byte lines
// whatever T is, and no tile is half empty: [32,8,32,32,300] -> 16 channels 313 -> 247 us (64 steps of one pixel a tile: rows of
// 300 steps end inside a line, 20 of 320 positions idle), 31x30 pixels of 301 steps 283 -> 213.
//
// The terms of a product are (input channel, line tap, row of the step) triples, E to a lane and group (4 E to a group): as few loads
// as the layer has triples, 24 of them are one group of six.  The rows of a product are (channel, pixel) pairs: XS neighbouring
// pixels of the line of a layer with few channels share a position, and their taps, so that 8 channels of two pixels load four
// taps where one pixel each would load six, and no row of the product is empty (input gradient [20,8,31,30,324], 5x5, 8 -> 4
// channels 293 -> 126 us).  In a transposed convolution the pixels of a position are those of all residues modulo the stride,
// and the classes of the walked axis are one launch: one read of the source instead of one per class, and lines written once
// (4x4 stride 2, [32,16,16,16,300] -> 8 channels 245 -> 185 us, 13x11 pixels of 173 steps 139 -> 25).
//
// Steps that are not whole quads: a pixel's last quad is its last four steps, overlapping the one before; the steps they share are
// computed and stored twice, to the same bits (also beside results that are not finite, see below), instead of being moved into place ([16,8,24,24,250] -> 16 channels, 5x5: 204 -> 114 us).
//
// Operands are split into three parts (split.h) unless they are bfloat16 numbers as they are: the weights are looked at once
// per workgroup, the input once per group, and the products run to match: one for spikes and quantised weights, three for one
// split operand, six for two.  The instruction rounds every sum it leaves, so the products of the lower parts, 2^-8 of
// the whole at most, are added up from zero and join the sum in one addition: it is rounded twice for 32 terms, not up to
// six times (error against float64 1.0e-7 real x real over 96 terms, float32 instruction 2.9e-7; every product into the one sum
// 2.6e-7; over 8 to 24 terms 0.30e-7 .. 0.37e-7, float32 instruction 0.45e-7 .. 0.89e-7).  The last addition rounds down as well: the mean of
// the errors, with sign, is -1.1e-8 of the mean result over 8 terms, -0.3e-8 over 800, a third of their spread or less.
//
// The walk loads the rows that an output row meets one after another.  Short launches, which wait for their loads, take all of them in
// one step instead, as terms of one product (WalkCut::whole): [9,1,13,13,132] -> 2 channels, real values, 14.4 -> 5.8 us.
//
// What bounds it: with the products left out the forward pass of [32,8,32,32,300] -> 16 channels takes as long (254 us): a group
// of loads has to arrive before its step, and 12 waves hold 72 KB of a CU's loads in flight.  Two blocks of channels to a wave
// (MB) halve the loads and the splitting of wide layers: [16,32,16,16,300] -> 64 channels 259 -> 216 us, its input gradient 355 ->
// 260 (both 296 and 337 with the kernel before), though two waves stay on a SIMD instead of three.
//
// A value that is not finite, or overflows when it is scaled or rounded, leaves parts of either sign, and infinity times
// each of them is not infinity times their sum: a wave with a result that is not finite computes its piece again in
// float32 multiplications and additions, and so does every wave of a workgroup with such a weight.  Of the input's, the sums replace
// results that are not finite and no others: a finite one has met no such value, and the quad that shares its steps may be
// another wave's.  A weight that is not finite is met outside the image too, and by every wave that stores these channels.
//
// LDS: the parts of the weights in the operand's layout, [group][tap][part][block][lane]; per triple its byte offset, its line tap
// and row, its channel; what the waves' weights are; where lanes store that have no registers for it.
#include "synapse.h"
#include "split.h"

namespace slayer {

constexpr int kWalkQuads = 16;          // quads of steps to a tile

// Rows of the result that take the same taps along the walk: all of them, or, in a transposed convolution, a residue class.
struct WalkClass {
    int s0;                             // weights: slide tap i of the launch is row s0 + i * WalkConv::sstep of the filter
    int row0;                           // input row of step 0's first row
    int S, per;                         // output rows, of a piece
    int c_lo, c_hi;                     // the steps that meet a row inside the image
    int out0;                           // bytes to the first output row
};

struct WalkConv {
    float* out;
    const float* in;
    const float* weight;                // [Co][Ci][...]
    int N, Ci, Co, T;
    int in_plane, out_plane;            // bytes of one sample
    int in_ch, in_slide, in_line, out_ch, out_slide, out_line, out_rx;   // bytes
    int Hs, Ws;                         // input rows along the walk, pixels along the line
    int M, quads, line_quads;           // pixels along the line; quads of steps a pixel has, the line has
    int ss, ls;                         // strides along walk and line
    int rows;                           // input rows of a step: ss, or all that an output row meets (KS = 1)
    int XP, shift0, shift_step;         // line taps, the first one's shift, pixels from one to the next
    int XS, line_full;                  // outputs that share a line position, pixels of the output's line
    int pairs, groups;
    int wslide, wline, nslide, nline;   // weights: strides and sizes of the filter's axes
    int sstep, l0, lstep, lrx;          // filter row / column of a slide / line tap
    int tiles, pieces, items, blocks;   // per sample, class and channel block; blocks of 16 MB channels
    int MB;
    int classes;
    int waves;                          // of a workgroup
    Divisor by_cb, by_blocks, by_wgs, by_tiles, by_quads, by_XS, by_triples, by_rows;   // blocks * classes, blocks, workgroups of items,
                                                                                          // tiles, quads, XS, XP * rows, rows
    WalkClass cls[4];
    // weight of output channel v = co * XS + rx, line tap x, slide tap i (of cls), or -1 where the filter has none
    __device__ __forceinline__ int64_t weight_at(int co, int rx, int ci, int x, int i, int s0) const {
        const int y = s0 + i * sstep, l = l0 + x * lstep + rx * lrx;
        if ((unsigned)y >= (unsigned)nslide || (unsigned)l >= (unsigned)nline) return -1;
        return ((int64_t)co * Ci + ci) * (nslide * nline) + y * wslide + l * wline;
    }
};

// Whether a lane keeps in registers where it stores: three taps and eight loads leave none, and a register that comes back from
// memory waits for the loads of the next step (three channels of two pixels, [11,32,27,27,248] -> 2 channels 70 -> 81 us), so LDS has it
constexpr bool walk_keeps(int KS, int E, int MB) { return KS != 3 || E < 8 || MB > 1; }

// KS: taps along the walk; E: triples to a lane and group; MB: blocks of 16 rows of the product to a wave.  Three waves per SIMD where
// 168 registers do, else two.
template <int KS, int E, int MB>
__global__ __launch_bounds__(8 * kWave) __attribute__((amdgpu_waves_per_eu(KS <= 3 && MB == 1 ? 3 : 2)))
void synapse_walk_kernel(const WalkConv p) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int G = p.groups;                             // groups of 4 E pairs
    uint4* wt = reinterpret_cast<uint4*>(lds);          // [G][KS][3][MB][64]
    int* pair_off = reinterpret_cast<int*>(wt + G * KS * 3 * MB * kWave);     // [G][4][E] bytes
    int* pair_info = pair_off + G * 4 * E;              // line tap, row of the step << 8
    int* pair_ch = pair_info + G * 4 * E;               // input channel
    int* flags = pair_ch + G * 4 * E;                   // [8]: what a wave's weights are
    const int tid = threadIdx.x, lane = tid & (kWave - 1), waves = p.waves, threads = waves * kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int b = xcd_contiguous(blockIdx.x, gridDim.x);
    const int rest = p.by_cb.of(b), cb = b - rest * p.blocks * p.classes, which = p.by_blocks.of(cb);
    const int v0 = (cb - which * p.blocks) * 16 * MB;
    const WalkClass cls = p.cls[which];
    const int n = p.by_wgs.of(rest), ig = p.by_wgs.rest(rest);
    const int kk = lane >> 4, j = lane & 15;

    const int item = ig * waves + wave;
    const int piece = p.by_tiles.of(item), tile = item - piece * p.tiles;
    const int s_lo = piece * cls.per, s_hi = (s_lo + cls.per) < cls.S ? (s_lo + cls.per) : cls.S;
    const bool idle = item >= p.items || s_lo >= s_hi;

    // the lane's quad: pixel m of the line, steps t .. t + 3
    const int quad = tile * kWalkQuads + j;
    const bool on = quad < p.line_quads;
    const int m = on ? p.by_quads.of(quad) : 0;
    // where a pixel's steps are not whole quads its last quad is the last four steps: those that it shares with the one before
    // are computed, and stored, twice
    int t = 4 * (quad - m * p.quads);
    t = t < p.T - 4 ? t : p.T - 4;
    unsigned taps = 0u;                                 // line taps inside the image
    for (int x = 0; x < p.XP; ++x)
        taps |= (on && (unsigned)(m * p.ls + p.shift0 + x * p.shift_step) < (unsigned)p.Ws) ? 1u << x : 0u;
    const bool inner = __all(taps == (1u << p.XP) - 1u);   // no lane has a tap outside
    const int lane_in = m * p.ls * p.in_line + t * 4;
    const __amdgpu_buffer_rsrc_t src = make_rsrc(p.in + (int64_t)n * (p.in_plane / 4), (unsigned)p.in_plane);
    const __amdgpu_buffer_rsrc_t dst = make_rsrc(p.out + (int64_t)n * (p.out_plane / 4), (unsigned)p.out_plane);
    // step c brings rows c * ss + row0 .. + rows - 1: slide tap i of output row c - i
    const int c_end = s_hi + KS - 1;
    const int c_lo = s_lo > cls.c_lo ? s_lo : cls.c_lo;
    const int c_hi = c_end < cls.c_hi ? c_end : cls.c_hi;
    float4 raw[E];
    auto fetch = [&](int c, int g) {
        const int* off = pair_off + (4 * g + kk) * E;
        const int row = c * p.ss + cls.row0;
        const int at = lane_in + row * p.in_slide;
        int o[E];
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] = off[e] + at;
        if (!inner || row < 0 || row + p.rows > p.Hs) {
            const int* info = pair_info + (4 * g + kk) * E;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int what = info[e];
                const bool in = (taps >> (what & 31) & 1u) != 0u && (unsigned)(row + (what >> 8)) < (unsigned)p.Hs;
                o[e] = in ? o[e] : kOutOfRange;
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e) raw[e] = buf_load4<false>(src, o[e]);
    };
    for (int i = tid; i < G * 4 * E; i += threads) {
        const int e = i % E, q = (i / E) & 3, g = i / (4 * E);
        const int pr = 4 * E * g + 4 * e + q;
        const int ci = p.by_triples.of(pr), r = pr - ci * (p.XP * p.rows), x = p.by_rows.of(r), row = r - x * p.rows;
        const bool is = pr < p.pairs;
        pair_off[i] = is ? ci * p.in_ch + (p.shift0 + x * p.shift_step) * p.in_line + row * p.in_slide : kOutOfRange;
        pair_info[i] = is ? x | row << 8 : 31;          // tap 31 is outside in every lane
        pair_ch[i] = is ? ci : -1;
    }
    __syncthreads();
    if (!idle && c_lo < c_hi) fetch(c_lo, 0);           // on its way while the weights are set up
    unsigned low = 0u;
    bool odd = false;                                   // a weight that is not finite
    for (int i = tid; i < G * KS * MB * kWave; i += threads) {
        const int l = i & (kWave - 1), mb = (i >> 6) % MB, tap = (i >> 6) / MB % KS, g = (i >> 6) / (MB * KS);
        const int vc = v0 + 16 * mb + (l & 15), co = p.by_XS.of(vc), rx = vc - co * p.XS;
        float v[8];
        int64_t at[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (e >= E) { v[e] = 0.0f; at[e] = -1; continue; }
            const int pr = (4 * g + (l >> 4)) * E + e, ci = pair_ch[pr], what = pair_info[pr];
            at[e] = ci >= 0 && co < p.Co ? p.weight_at(co, rx, ci, what & 31, tap * p.rows + (what >> 8), cls.s0) : -1;
            v[e] = p.weight[at[e] < 0 ? 0 : at[e]];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = at[e] < 0 ? 0.0f : v[e];
            low |= __float_as_uint(v[e]);
            odd = odd || !(fabsf(v[e]) < __builtin_inff());
            v[e] *= kSplitScale;
        }
        uint4* to = wt + (((g * KS + tap) * 3) * MB + mb) * kWave + l;
        to[0] = round_eight(v);
        to[MB * kWave] = round_eight(v);
        to[2 * MB * kWave] = bf16_eight(v);
    }
    // bit 0: a weight has lower parts, bit 1: one is not finite
    const int mine = (__any((low & 0xffffu) != 0u) ? 1 : 0) | (__any(odd) ? 2 : 0);
    if (lane == 0) flags[wave] = mine;
    __syncthreads();
    if (idle) return;
    const int seen = lane < waves ? flags[lane] : 0;
    const bool split_w = __any((seen & 1) != 0), float_only = __any((seen & 2) != 0);
    int to[MB][4];                                      // where the lane's four channels go, row 0
#pragma unroll
    for (int i = 0; i < 4 * MB; ++i) {
        const int vc = v0 + 16 * (i >> 2) + 4 * kk + (i & 3), co = p.by_XS.of(vc), rx = vc - co * p.XS;
        to[i >> 2][i & 3] = (on && co < p.Co && m * p.XS + rx < p.line_full)
                                ? co * p.out_ch + rx * p.out_rx + m * p.out_line + t * 4 + cls.out0 : kOutOfRange;
    }
    constexpr bool kKept = walk_keeps(KS, E, MB);
    int4* kept = reinterpret_cast<int4*>(flags + 8) + wave * kWave + lane;
    if (!kKept) {
        *kept = make_int4(to[0][0], to[0][1], to[0][2], to[0][3]);
        asm volatile("" ::: "memory");
    }
    auto place = [&](int mb, int (&at)[4]) {
        at[0] = to[mb][0]; at[1] = to[mb][1]; at[2] = to[mb][2]; at[3] = to[mb][3];
        if (!kKept) { const int4 k = *kept; at[0] = k.x; at[1] = k.y; at[2] = k.z; at[3] = k.w; }
    };
    // lane (kk, j): output channels v0 + 16 mb + 4 kk + i, steps t .. t + 3
    auto store = [&](int s, int mb, const syn_f4 (&d)[4]) {
        int at[4];
        place(mb, at);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            buf_store4<false>(dst, at[i] != kOutOfRange ? at[i] + s * p.out_slide : kOutOfRange,
                              make_float4(d[0][i], d[1][i], d[2][i], d[3][i]));
    };
    float stored = 0.f;                                                  // not finite once a result is not
    syn_f4 acc[MB][KS][4];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int x = 0; x < KS; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[b][x][e] = syn_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int c = s_lo; c < c_end; ++c) {                                 // tap i of step c goes to row c - i: acc[i]
        if (c >= c_lo && c < c_hi) {
#pragma unroll 1
            for (int g = 0; g < G; ++g) {
                float v[4][8];                                           // [step of the quad][pair]
                unsigned bits = 0u;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (i >= E) { v[0][i] = v[1][i] = v[2][i] = v[3][i] = 0.f; continue; }
                    const float4 r = raw[i < E ? i : 0];
                    v[0][i] = r.x * kSplitScale; v[1][i] = r.y * kSplitScale;
                    v[2][i] = r.z * kSplitScale; v[3][i] = r.w * kSplitScale;
                    bits |= __float_as_uint(r.x) | __float_as_uint(r.y) | __float_as_uint(r.z) | __float_as_uint(r.w);
                }
                const bool split_x = __any((bits & 0xffffu) != 0u);
                int here = lane;
                if (!walk_keeps(KS, E, MB)) asm("" : "+v"(here));        // the address is worked out here, not kept
                const uint4* wg = wt + g * KS * 3 * MB * kWave + here;
                const bool last = g + 1 == G;                            // the next loads are on their way during the products
                if (!last || c + 1 < c_hi) fetch(last ? c + 1 : c, last ? 0 : g + 1);
                // kH steps of the quad at a time, so that a part of the weights is read once for them: all four where two waves stay on
                // a SIMD (gradient of [16,32,16,16,300] -> 64 channels 273 -> 260 us) or the accumulators leave room, two for
                // three taps and one block (four: [32,8,32,32,300] 312 -> 341 us, registers).  Branches around the products of the
                // lower parts only: around several copies of the whole they cost the compiler a second set of accumulators.
                constexpr int kH = KS == 3 && MB == 1 ? 2 : 4;
                const syn_f4 zero = syn_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int h = 0; h < 4; h += kH) {
                    uint4 q[kH][3];
#pragma unroll
                    for (int e = 0; e < kH; ++e) {
                        q[e][0] = bf16_eight(v[h + e]);
                        if (split_x) {
                            leave_eight(v[h + e], q[e][0]);
                            q[e][1] = round_eight(v[h + e]);
                            q[e][2] = bf16_eight(v[h + e]);
                        }
                    }
#pragma unroll
                    for (int xb = 0; xb < KS * MB; ++xb) {
                        const int x = xb / MB, mb = xb % MB;
                        const uint4* wx = wg + (x * 3 * MB + mb) * kWave;
                        const uint4 w0 = wx[0];
                        syn_f4 d[kH];
                        if (split_x) {
                            if (split_w) {
                                const uint4 w1 = wx[MB * kWave], w2 = wx[2 * MB * kWave];
#pragma unroll
                                for (int e = 0; e < kH; ++e) d[e] = mfma_bf16(w2, q[e][0], zero);
#pragma unroll
                                for (int e = 0; e < kH; ++e) d[e] = mfma_bf16(w1, q[e][1], d[e]);
#pragma unroll
                                for (int e = 0; e < kH; ++e) d[e] = mfma_bf16(w1, q[e][0], d[e]);
#pragma unroll
                                for (int e = 0; e < kH; ++e) d[e] = mfma_bf16(w0, q[e][2], d[e]);
                            } else {
#pragma unroll
                                for (int e = 0; e < kH; ++e) d[e] = mfma_bf16(w0, q[e][2], zero);
                            }
#pragma unroll
                            for (int e = 0; e < kH; ++e) acc[mb][x][h + e] += mfma_bf16(w0, q[e][1], d[e]);
                        } else if (split_w) {
                            const uint4 w1 = wx[MB * kWave], w2 = wx[2 * MB * kWave];
#pragma unroll
                            for (int e = 0; e < kH; ++e) d[e] = mfma_bf16(w2, q[e][0], zero);
#pragma unroll
                            for (int e = 0; e < kH; ++e) acc[mb][x][h + e] += mfma_bf16(w1, q[e][0], d[e]);
                        }
#pragma unroll
                        for (int e = 0; e < kH; ++e) acc[mb][x][h + e] = mfma_bf16(w0, q[e][0], acc[mb][x][h + e]);
                    }
                }
            }
        }
        const int s = c - (KS - 1);
        if (s >= s_lo) {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                syn_f4 d[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    d[e] = acc[mb][KS - 1][e];
                    stored += (d[e][0] + d[e][1]) + (d[e][2] + d[e][3]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) d[e][i] *= kSplitProductScale;
                }
                store(s, mb, d);
            }
        }
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int x = KS - 1; x >= 0; --x)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[b][x][e] = x > 0 ? acc[b][x - 1][e] : syn_f4{0.f, 0.f, 0.f, 0.f};
    }
    if (!float_only && !__any(!(fabsf(stored) < __builtin_inff()))) return;

    // Once more in float32 multiplications and additions, taps outside the image as products with zero, for the results that are
    // not finite, or all of them: a wave's own stores are in place when it loads them, and of steps that another wave stores as
    // well either one's result is what the other one would put there.
    int kq = kk;                                         // (nothing of this loop is kept in registers during the one before)
    asm("" : "+v"(kq));
#pragma unroll 1
    for (int sb = s_lo * MB; sb < s_hi * MB; ++sb) {
        const int s = sb / MB, mb = sb % MB;
        syn_f4 d[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = syn_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int pr = 0; pr < p.pairs; ++pr) {
            const int ci = p.by_triples.of(pr), r = pr - ci * (p.XP * p.rows), x = p.by_rows.of(r), sub = r - x * p.rows;
            const int off = ci * p.in_ch + (p.shift0 + x * p.shift_step) * p.in_line + lane_in;
#pragma unroll 1
            for (int tap = 0; tap < KS; ++tap) {
                const int row = (s + tap) * p.ss + cls.row0 + sub;
                const bool in = (taps >> x & 1u) != 0u && (unsigned)row < (unsigned)p.Hs;
                const float4 q = buf_load4<false>(src, in ? off + row * p.in_slide : kOutOfRange);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int vc = v0 + 16 * mb + 4 * kq + i, co = p.by_XS.of(vc), rx = vc - co * p.XS;
                    const int64_t at = co < p.Co ? p.weight_at(co, rx, ci, x, tap * p.rows + sub, cls.s0) : -1;
                    if (at < 0) continue;
                    const float w = p.weight[at];
                    d[0][i] = __fmaf_rn(w, q.x, d[0][i]);
                    d[1][i] = __fmaf_rn(w, q.y, d[1][i]);
                    d[2][i] = __fmaf_rn(w, q.z, d[2][i]);
                    d[3][i] = __fmaf_rn(w, q.w, d[3][i]);
                }
            }
        }
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            if (b != mb) continue;
            int at[4];
            place(b, at);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 was = buf_load4<false>(dst, at[i] != kOutOfRange ? at[i] + s * p.out_slide : kOutOfRange);
                d[0][i] = !float_only && fabsf(was.x) < __builtin_inff() ? was.x : d[0][i];
                d[1][i] = !float_only && fabsf(was.y) < __builtin_inff() ? was.y : d[1][i];
                d[2][i] = !float_only && fabsf(was.z) < __builtin_inff() ? was.z : d[2][i];
                d[3][i] = !float_only && fabsf(was.w) < __builtin_inff() ? was.w : d[3][i];
            }
            store(s, b, d);
        }
    }
}

namespace {

constexpr int kMaxLineTaps = 31;        // bits of a lane's mask, less one
constexpr size_t kWalkLds = 150 * 1024;

struct Axis { int in, out, k, stride, pad, dil, k0, kstep, kfull, o0, ostep, ofull, wstride; };

template <int KS, int MB>
void launch_walk(int E, const WalkConv& w, unsigned wgs, int waves, size_t bytes, hipStream_t st) {
    const dim3 grid(wgs), block((unsigned)(waves * kWave));
    if (E == 2) hipLaunchKernelGGL((synapse_walk_kernel<KS, 2, MB>), grid, block, bytes, st, w);
    else if (E == 4) hipLaunchKernelGGL((synapse_walk_kernel<KS, 4, MB>), grid, block, bytes, st, w);
    else if (E == 6) hipLaunchKernelGGL((synapse_walk_kernel<KS, 6, MB>), grid, block, bytes, st, w);
    else hipLaunchKernelGGL((synapse_walk_kernel<KS, 8, MB>), grid, block, bytes, st, w);
}

int slide_taps(int taps) { return taps == 4 ? 5 : taps; }              // those there are kernels for

// The loads of one walk step for `pairs` (channel, line tap, row) triples: E to a lane and group, groups.
struct Grouping { int E, groups; };
Grouping grouping(int pairs) {
    Grouping best = {8, (pairs + 31) / 32};
    for (int e : {6, 4, 2}) {
        const int g = (pairs + 4 * e - 1) / (4 * e);
        if (g * (e + 4) < best.groups * (best.E + 4)) best = {e, g};
    }
    return best;
}

// of a workgroup of four waves
size_t walk_lds(const Grouping& g, int KS, int MB) {
    return (size_t)g.groups * (KS * 3 * 1024 * MB + 4 * g.E * 3 * sizeof(int)) + 8 * sizeof(int) +
           (walk_keeps(KS, g.E, MB) ? 0 : 4 * kWave * sizeof(int4));
}
// Workgroups of four waves: the registers hold three of them on a CU (two with five taps or two blocks of channels), but one of eight.
// Eight where the LDS has room for one workgroup only and there are more than four waves to a CU.
int walk_waves(size_t lds, double waves) { return 2 * lds > 160 * 1024 && waves > 4 * 256 ? 8 : 4; }

// What the launches of one form (KS, MB, the groups) take, in us: a workgroup sets up its weights; a wave walks its piece, KS - 1 steps
// more than it has rows; a group of loads is a wait or, where a SIMD has several waves, its share of the instructions; of what the
// last, partly filled round of workgroups leaves idle, some is lost.  load: waves per SIMD.  (A layer has some hundred cuts: what
// is the same for all of a form is worked out once.)
struct WalkTime {
    bool wide;                          // LDS has room for one workgroup only
    float room, held;                   // workgroups of four waves that LDS, waves that the registers of a SIMD hold
    float start, busy, wait, slots;
    float short_start, short_busy, short_wait, part;

    WalkTime(int KS, int MB, const Grouping& g) {
        const size_t lds = walk_lds(g, KS, MB);
        const float terms = (float)(g.groups * g.E), taps = (float)(g.groups * KS * MB);
        wide = 2 * lds > 160 * 1024;
        room = (float)(160 * 1024 / lds);
        start = 0.4f * taps; busy = 0.38f * MB + 0.097f * terms; wait = 1.5f * g.groups; slots = KS > 3 || MB == 2 ? 2.f : 3.f;
        held = KS == 1 && MB == 1 && g.E <= 4 ? 4.f : (KS == 1 || (KS <= 3 && MB == 1) || (KS == 2 && g.E == 2) ? 3.f : 2.f);
        short_start = 0.443f + 0.182f * taps;
        short_busy = 0.306f * MB + 0.081f * terms + 0.024f * taps + (KS == 5 ? 0.025f : 0.f);
        short_wait = 0.426f + 1.308f * g.groups;
        part = g.groups > 1 ? 0.336f : 0.573f;
    }
    static float rounds(float load, float slots, float lost, float one, float left_over) {   // a full round; what is left over
        const float all = load / slots, full = (float)(int)all;
        return (1.f - lost) * all * one + lost * (full * one + (load - full * slots > 0.02f ? left_over : 0.f));
    }
    // Fitted to 814 layers (3x3 and 5x5, strides 1 and 2, 4x4 transposed and its gradient, 2 to 64 channels, 1 to 32 samples of 4x4 to
    // 34x34 pixels, 50 to 350 steps), each walked in all the ways below.
    float walk(float load, int steps) const {
        const float by_lds = room * (wide && load > 1.f ? 2.f : 1.f), most = by_lds < slots ? by_lds : slots;
        const auto round = [&](float l) { return start + steps * (l * busy > wait ? l * busy : wait); };
        return load <= most ? round(load) : rounds(load, most, 0.44f, round(most), round(load - (float)(int)(load / most) * most));
    }
    // Short launches of either form: also the start of a wave, the products, and that compute units with fewer workgroups than others
    // wait for these with 0.34 to 0.57 of what they have less.  Fitted to 3408 passes (forward and input gradient of 860 layers: 1x1 to
    // 5x5, strides 1 and 2, transposed, 1 to 64 channels, 1 to 32 samples of 4x4 to 34x34 pixels, 20 to 350 steps, spikes x 8-bit and
    // real x real), each cut in all the ways below.  What it decides for below kShort takes 0.87 times what walk() decides for, in the
    // mean (2.3 % of these passes: more than 1.03 times).  Above, the two differ by less than what either misses, and walk()
    // stays (0.90 in the mean between 20 and 60 us, but up to 1.39 times, 0.95 and up to 1.35 times beyond), unless the `whole` form
    // is estimated at less than 0.85 of it.
    float brief(float load, int steps) const {
        const float unit = wide && load > 1.f ? 2.f : 1.f, by_lds = room * unit, most = by_lds < held ? by_lds : held;
        const auto round = [&](float l) {
            const float units = l / unit, whole = (float)(int)units, full = (units - whole > 1e-6f ? whole + 1.f : whole) * unit;
            const float b = (l + part * (full - l)) * short_busy;
            return short_start + steps * (b > short_wait ? b : short_wait);
        };
        return load <= most ? round(load) : rounds(load, most, 0.5f, round(most), round(load - (float)(int)(load / most) * most));
    }
};
constexpr float kShort = 20.f;

bool beyond_cache(int64_t N, const WalkConv& w) { return N * ((int64_t)w.in_plane + w.out_plane) > 250000000; }

// The cut that takes least.  `step`: pixels come in whole multiples of it; taps(XS): the line taps they have together; count:
// samples and classes; Ci channels of the input, of which a step brings `stride` rows or all `k` that an output row meets; large:
// tensors beyond the last-level cache.
template <typename Taps>
WalkCut cut_launch(int64_t count, int Co, int width, int quads, int S, int taps_walked, int Ci, int stride, int k, int step, bool together,
                   bool large, Taps taps) {
    WalkCut best = {step, 1, 1, false}, best_short = best;
    constexpr float none = 1e30f;
    float least = none, least_short = none, kept = none;                  // kept: the short estimate of `best`
    for (int XS = step; XS == step || (together && Co * XS <= 16 && XS < width + step); XS += step) {
        const int XP = taps(XS);
        if (XS > step && XP > kMaxLineTaps) break;
        const int64_t tiles = ((int64_t)((width + XS - 1) / XS) * quads + kWalkQuads - 1) / kWalkQuads;
        const bool wide = Co * XS > 16;
        for (int form = 0; form < (wide ? 4 : 2); ++form) {
            const bool whole = (form & 1) != 0;
            const int MB = 1 + form / 2, KS = whole ? 1 : taps_walked;
            if (KS > 5 || (MB == 2 && KS > 3)) continue;
            const Grouping g = grouping(Ci * (whole ? k : stride) * XP);
            if (walk_lds(g, KS, MB) > kWalkLds) continue;
            const WalkTime time(KS, MB, g);
            const float loads = (float)(count * ((Co * XS + 16 * MB - 1) / (16 * MB)) * tiles) * (1.f / 1024.f);
            const float apart = large && XS > step ? 1.15f : 1.f;
            for (int cut = 1; cut <= 32 && (cut == 1 || cut < 2 * S); cut *= 2) {
                const int per = (S + cut - 1) / cut, pieces = (S + per - 1) / per;
                const float brief = time.brief(loads * pieces, per + KS - 1);
                if (brief < least_short) { least_short = brief; best_short = {XS, MB, pieces, whole}; }
                if (whole || cut > 16 || cut > S) continue;
                // large tensors: pieces of a line that does not lie in one piece cost more (8 of 274 passes, 0.99 times the time without)
                const float t = time.walk(loads * cut, per + KS - 1) * apart;
                if (t < least) { least = t; best = {XS, MB, cut, false}; kept = brief; }
            }
        }
    }
    if (least < kShort || least == none || (best_short.whole && least_short < 0.85f * kept)) return best_short;
    // ... and large tensors' pieces that leave less than a round and a half waves take longer than they should: 54 of 274 passes with
    // up to three taps, 0.98 times the time without, in the mean (0.74 to 1.20); with five taps it would be 1.1
    if (large && best.MB == 1 && taps_walked <= 3) {
        const int64_t tiles = ((int64_t)((width + best.XS - 1) / best.XS) * quads + kWalkQuads - 1) / kWalkQuads;
        const int64_t waves = count * ((Co * best.XS + 15) / 16) * tiles;
        while (waves * best.pieces < 4608 && S >= 16 * best.pieces) best.pieces *= 2;
    }
    return best;
}

// Whether a cut that was asked for is one there is
bool may_cut(const WalkCut& c, int step, bool together, int taps_walked) {
    const int KS = c.whole ? 1 : taps_walked;
    return KS <= 5 && c.XS >= step && c.XS % step == 0 && c.XS <= 64 && (c.XS == step || together) && (c.MB == 1 || (c.MB == 2 && KS <= 3)) &&
           c.pieces >= 1 && c.pieces <= 1024;
}

// The launch of a WalkConv whose geometry is filled in; KS taps along the walk.  false: not one that the kernel takes.
bool launch(WalkConv& w, int KS, hipStream_t st, int* code) {
    if (KS < 1 || KS > 5 || w.XP > kMaxLineTaps) return false;
    const int64_t pairs = (int64_t)w.Ci * w.XP * w.rows;
    if (pairs > 4096) return false;
    w.pairs = (int)pairs;
    const Grouping grp = grouping(w.pairs);
    const int E = grp.E;
    w.groups = grp.groups;
    size_t bytes = walk_lds(grp, KS, w.MB);
    if (bytes > kWalkLds) return false;
    w.quads = (w.T + 3) / 4;
    if ((int64_t)w.M * w.quads > 0x3fffffffLL) return false;
    w.line_quads = w.M * w.quads;
    w.tiles = (w.line_quads + kWalkQuads - 1) / kWalkQuads;
    w.blocks = (w.Co * w.XS + 16 * w.MB - 1) / (16 * w.MB);
    const int64_t base = (int64_t)w.N * w.blocks * w.classes * w.tiles;
    const int pieces = w.pieces;
    const int64_t items = (int64_t)w.tiles * pieces;
    const int waves = walk_waves(bytes, (double)(base * pieces));
    const int64_t wgs = (int64_t)w.N * w.blocks * w.classes * ((items + waves - 1) / waves);
    if (!walk_keeps(KS, E, w.MB)) bytes += (waves - 4) * kWave * sizeof(int4);
    if (items > 0x3fffffffLL || wgs > 0x7fffffffLL / 8) return false;
    w.items = (int)items;
    w.waves = waves;
    w.by_cb = w.blocks * w.classes; w.by_blocks = w.blocks; w.by_wgs = (w.items + waves - 1) / waves; w.by_tiles = w.tiles;
    w.by_quads = w.quads; w.by_XS = w.XS; w.by_triples = w.XP * w.rows; w.by_rows = w.rows;
    for (int i = 0; i < w.classes; ++i) w.cls[i].per = (w.cls[i].S + pieces - 1) / pieces;
#define SLAYER_WALK(KS, MB) launch_walk<KS, MB>(E, w, (unsigned)wgs, waves, bytes, st)
    if (w.MB == 2) { if (KS == 1) SLAYER_WALK(1, 2); else if (KS == 2) SLAYER_WALK(2, 2); else SLAYER_WALK(3, 2); }
    else if (KS == 1) SLAYER_WALK(1, 1);
    else if (KS == 2) SLAYER_WALK(2, 1);
    else if (KS == 3) SLAYER_WALK(3, 1);
    else SLAYER_WALK(5, 1);
#undef SLAYER_WALK
    *code = (int)hipGetLastError();
    return true;
}

void steps_inside(WalkClass& c, int ss, int rows, int Hs) {
    c.c_lo = c.row0 + rows - 1 >= 0 ? 0 : (-c.row0 - rows + 1 + ss - 1) / ss;
    c.c_hi = Hs - 1 - c.row0 < 0 ? 0 : (Hs - 1 - c.row0) / ss + 1;
}

}  // namespace

bool launch_synapse_walk(const SynapseConv& p, hipStream_t st, int* code) {
    if (p.kh < 1 || p.kw < 1) return false;
    const Axis h = {p.H, p.Ho, p.kh, p.sh, p.ph, p.dh, p.ky0, p.kys, p.kh_full, p.oy0, p.oys, p.Ho_full, p.kw_full};
    const Axis v = {p.W, p.Wo, p.kw, p.sw, p.pw, p.dw, p.kx0, p.kxs, p.kw_full, p.ox0, p.oxs, p.Wo_full, 1};
    auto taps = [](const Axis& a) { return a.k == 1 || a.dil == 1 ? (a.k + a.stride - 1) / a.stride : 0; };
    auto takes = [&](const Axis& a, const Axis& line) { return taps(a) >= 1 && taps(a) <= 5 && line.k <= kMaxLineTaps && a.stride <= 16; };
    // along the rows of the image, so that the line is one piece of memory, unless the filter has more taps the other way; along
    // the other axis where the weights do not fit LDS this way (9x2, stride 8 along the rows, 56 channels: 183 KB and 98)
    const bool down = takes(h, v), right = takes(v, h), rows_first = down && (!right || taps(h) >= taps(v));
    // filters of more rows than a line has taps (40x3) bring them all in one step
    const bool tall = !down && !right && h.dil == 1 && h.k > kMaxLineTaps && v.k <= 5;
    if (!down && !right && !tall) return false;
    const auto along = [&](bool use_h) {
        const Axis& s = use_h ? h : v;
        const Axis& l = use_h ? v : h;
        const int px = p.T * 4;
        WalkConv w;
        w.out = p.out; w.in = p.in; w.weight = p.weight;
        w.N = p.N; w.Ci = p.Ci; w.Co = p.Co; w.T = p.T;
        w.in_ch = p.H * p.W * px; w.in_plane = p.Ci * w.in_ch;
        w.out_ch = p.Ho_full * p.Wo_full * px; w.out_plane = p.Co * w.out_ch;
        w.in_slide = use_h ? p.W * px : px; w.in_line = use_h ? px : p.W * px;
        w.out_slide = s.ostep * (use_h ? p.Wo_full * px : px); w.out_line = l.ostep * (use_h ? px : p.Wo_full * px);
        w.out_rx = w.out_line;
        w.Hs = s.in; w.Ws = l.in;
        // pixels that lie together share their taps, unless these lie apart
        const auto line_taps = [&](int XS) { return (XS - 1) * l.stride + l.k; };
        const bool together = l.dil == 1 || l.k == 1;
        const int KS = slide_taps(taps(s));
        if (p.want && !may_cut(*p.want, 1, together, KS)) return false;
        const WalkCut cut = p.want ? *p.want
                                   : cut_launch(p.N, p.Co, l.out, (p.T + 3) / 4, s.out, KS, p.Ci, s.stride, s.k, 1, together,
                                                beyond_cache(p.N, w), [&](int XS) { return XS > 1 ? line_taps(XS) : l.k; });
        w.XS = cut.XS; w.pieces = cut.pieces; w.MB = cut.MB;
        w.rows = cut.whole ? s.k : s.stride;
        w.out_line *= w.XS;
        w.M = (l.out + w.XS - 1) / w.XS;
        w.ss = s.stride; w.ls = l.stride * w.XS;
        w.XP = w.XS > 1 ? line_taps(w.XS) : l.k; w.shift0 = -l.pad; w.shift_step = w.XS > 1 ? 1 : l.dil;
        w.line_full = l.out;
        w.wslide = s.wstride; w.wline = l.wstride; w.nslide = s.kfull; w.nline = l.kfull;
        w.sstep = s.kstep; w.l0 = l.k0; w.lstep = l.kstep; w.lrx = -l.stride * l.kstep;
        w.classes = 1;
        WalkClass& c = w.cls[0];
        c.s0 = s.k0; c.row0 = -s.pad; c.S = s.out;
        c.out0 = (p.oy0 * p.Wo_full + p.ox0) * px;
        steps_inside(c, w.ss, w.rows, w.Hs);
        return launch(w, cut.whole ? 1 : KS, st, code);
    };
    return along(rows_first || tall) || (down && right && along(!rows_first));
}

bool launch_synapse_walk_transposed(const SynapseConv& p, int kh, int kw, int sh, int sw, int ph, int pw, hipStream_t st, int* code) {
    const int H = p.Ho_full, W = p.Wo_full, px = p.T * 4;                // of the result
    if (sh > 4) return false;
    WalkConv w;
    w.out = p.out; w.in = p.in; w.weight = p.weight;
    w.N = p.N; w.Ci = p.Ci; w.Co = p.Co; w.T = p.T;
    w.in_ch = p.H * p.W * px; w.in_plane = p.Ci * w.in_ch;
    w.out_ch = H * W * px; w.out_plane = p.Co * w.out_ch;
    w.in_slide = p.W * px; w.in_line = px;
    int lo = 0, hi = 0;                                                  // shifts of the line taps, over the pixels together
    const auto line_taps = [&](int XS) {
        lo = 1 << 30; hi = -(1 << 30);
        for (int r = 0; r < XS; ++r)
            for (int x = 0; x < kw; ++x)
                if ((r + pw - x) % sw == 0) {
                    const int d = (r + pw - x) / sw;
                    lo = d < lo ? d : lo;
                    hi = d > hi ? d : hi;
                }
        return hi - lo + 1;
    };
    const int most = (kh + sh - 1) / sh, KS = slide_taps(most);              // taps of a class
    if (KS > 5) return false;
    if (p.want && !may_cut(*p.want, sw, true, KS)) return false;
    const WalkCut cut = p.want ? *p.want
                               : cut_launch((int64_t)p.N * (sh < H ? sh : H), p.Co, W, (p.T + 3) / 4, (H + sh - 1) / sh, KS, p.Ci, 1, most, sw, true,
                                            beyond_cache(p.N, w), line_taps);
    w.XS = cut.XS; w.pieces = cut.pieces; w.MB = cut.MB;
    w.XP = line_taps(w.XS); w.shift0 = lo; w.shift_step = 1;
    w.out_slide = sh * W * px; w.out_line = w.XS * px; w.out_rx = px;
    w.Hs = p.H; w.Ws = p.W; w.M = (W + w.XS - 1) / w.XS; w.line_full = W;
    w.ss = 1; w.ls = w.XS / sw; w.rows = cut.whole ? most : 1;
    w.wslide = kw; w.wline = 1; w.nslide = kh; w.nline = kw;
    w.sstep = -sh; w.l0 = pw - lo * sw; w.lstep = -sw; w.lrx = 1;
    w.classes = sh < H ? sh : H;
    for (int r = 0; r < w.classes; ++r) {
        WalkClass& c = w.cls[r];
        int count = 0, last = 0;
        for (int y = 0; y < kh; ++y)
            if ((r + ph - y) % sh == 0) { ++count; last = y; }
        c.S = (H - r + sh - 1) / sh;
        c.out0 = r * W * px;
        if (count) {
            c.s0 = last;
            c.row0 = (r + ph - last) / sh;
            steps_inside(c, 1, w.rows, w.Hs);
        } else {                                                         // rows that no tap reaches: zeros
            c.s0 = -1; c.row0 = 0; c.c_lo = c.c_hi = 0;
        }
    }
    return launch(w, cut.whole ? 1 : KS, st, code);
}

}  // namespace slayer
