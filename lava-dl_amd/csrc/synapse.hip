// Convolution synapse on time-innermost tensors.
//
// A SLAYER conv synapse is a spatial convolution applied at every time step (synapse/layer.py:297-323 in the
// reference: F.conv3d with a kernel of (kh, kw, 1) on [N, C, H, W, T]).  A library conv3d wants channels last: it
// transposes the tensor there and back around its kernel, three passes over tensors whose innermost axis is already
// the one the neuron kernels walk.  Here the tensors stay as they are: for an output pixel (n, h, w) and a tile of
// 64 time steps the [Co x 64] result is the [Co x K] weight matrix (K = Ci * kh * kw) times the [K x 64] matrix
// whose row k is the input row of tap k -- 64 consecutive floats of the input as it lies in memory.  One wavefront
// takes 16 output channels x 64 steps of one pixel at a time on the matrix cores (v_mfma_f32_16x16x4_f32: float32
// operands, float32 accumulation) and walks along the image row, so neighbouring pixels find their shared input
// rows in the cache; a wave-wide load is four input rows of 256 bytes, a wave-wide store four output rows.
//
// Lane (kk, j) = (lane / 16, lane % 16) loads steps 4j .. 4j+3 of tap 4g + kk for tap group g: element e of that
// quad is the B operand of the e-th of four matrix products, whose column j stands for step 4j + e; lane (q, j) of a
// result then holds output channels 4q .. 4q+3 of step 4j + e, i.e. over e a quad of consecutive steps per channel.
#include "common.h"
#include "split.h"
#include "tile.h"

namespace slayer {

int launch_zero_fill(float* p, int64_t n, hipStream_t stream);          // li.hip

typedef float syn_f4 __attribute__((ext_vector_type(4)));

// Rows of any length (T >= 4): a quad of steps is a 16-byte access at a dword-aligned address, and the last quad of
// a row may hold fewer than four steps (nv of them).  Such a quad is loaded four steps before the end of its row --
// never beyond it -- and moved into place: element e of the result is element e + 4 - nv of what was loaded, zero
// behind the row's end.  Stores leave the steps that do not exist out.
struct SynQuad {
    int t_load;                         // step the quad is loaded at
    int nv;                             // steps of the quad that exist (<= 0: none, the lane loads nothing)
    template <bool TAIL>
    __device__ __forceinline__ void set(int t, int t_end) {
        nv = t_end - t;
        t_load = (TAIL && nv > 0 && nv < 4) ? t_end - 4 : t;
    }
    __device__ __forceinline__ bool any() const { return nv > 0; }
    __device__ __forceinline__ bool partial() const { return nv > 0 && nv < 4; }
    // TAIL: the rows are not whole quads (decided on the host: a test per load would sit between the loads)
    template <bool TAIL>
    __device__ __forceinline__ float4 place(float4 q) const {
        if (!TAIL || !__any(partial())) return q;                        // only the tile that holds the end of the rows
        const int d = partial() ? 4 - nv : 0;
        const float a[4] = {q.x, q.y, q.z, q.w};
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = e + d;
            r[e] = i == 0 ? a[0] : (i == 1 ? a[1] : (i == 2 ? a[2] : (i == 3 ? a[3] : 0.f)));
        }
        return make_float4(r[0], r[1], r[2], r[3]);
    }
};
// the quad v at byte offset off, of which the first nv elements exist (nv <= 0: nothing is stored)
template <bool STREAM, bool TAIL>
__device__ __forceinline__ void syn_store_quad(__amdgpu_buffer_rsrc_t dst, bool on, int off, int nv, float4 v) {
    buf_store4<STREAM>(dst, (on && nv >= 4) ? off : kOutOfRange, v);
    if (TAIL && __any(on && nv > 0 && nv < 4)) {                                 // only the tile that holds the end of the rows
        const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 3; ++i) buf_store1<false>(dst, (on && nv < 4 && i < nv) ? off + 4 * i : kOutOfRange, e[i]);
    }
}

// Workgroups are handed to the chip's eight XCDs round-robin by their index, and each XCD has an L2 of its own.
// Neighbouring work items of the kernels below share most of what they read (an input row serves the output rows
// above and below it and the neighbouring time shares of the weight gradient), so taken in index order every XCD
// fetched nearly every row for itself: FETCH_SIZE read 5.0 x the input tensor for the forward kernel on
// [32,8,32,32,300] -> 16 channels, 1.4 x with the permuted index below, by which XCD x gets the x-th contiguous eighth
// of the work.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_contiguous(int b, int nb) {
    const int x = b % kXcds, slot = b / kXcds, q = nb / kXcds, r = nb % kXcds;
    return x * q + (x < r ? x : r) + slot;
}

constexpr int kSynTile = 64;            // time steps per tile
constexpr int kSynWaves = 4;            // waves per workgroup: same output channels, same image row, different tiles

constexpr int kSynChunk = 6;            // tap groups whose loads are in flight together (fewer for filters of a few taps)

struct SynapseConv {
    float* out;
    const float* in;
    const float* weight;                // [Co][Ci][kh_full][kw_full]
    int N, Ci, Co, H, W, Ho, Wo, T;
    int kh, kw, sh, sw, ph, pw, dh, dw; // ph, pw: may be negative (a window that begins inside the image)
    int K, KG;                          // taps, groups of four taps (a whole number of chunks, padded with null taps)
    int ttiles, wsplit;                 // tiles of 64 steps per row, pieces an image row is cut into
    int items;                          // (tile, piece, output row) triples of one (batch entry, channel block)
    // The taps may be a sub-lattice of a larger filter and the outputs a sub-lattice of a larger image (identity for
    // a plain convolution): row iy of the kh x kw taps is row ky0 + iy * kys of the weight tensor's kh_full rows,
    // output pixel (ho, wo) is pixel (oy0 + ho * oys, ox0 + wo * oxs) of a tensor [Co][Ho_full][Wo_full][T].
    int kh_full, kw_full, ky0, kys, kx0, kxs;
    int Ho_full, Wo_full, oy0, oys, ox0, oxs;
    __device__ __forceinline__ int weight_index(int ci, int iy, int ix) const {
        return (ci * kh_full + ky0 + iy * kys) * kw_full + kx0 + ix * kxs;
    }
    __device__ __forceinline__ int out_pixel(int ho, int wo) const {     // in pixels of the full output image
        return (oy0 + ho * oys) * Wo_full + ox0 + wo * oxs;
    }
};

// The gradient of the input of a convolution with strides (what conv_transpose3d computes, the ConvTranspose synapse
// of synapse/layer.py:513-560 in the reference) is one plain convolution per residue class of the output pixels: the
// pixels (ry + m sh, rx + m' sw) meet only the taps y with (ry + ph - y dh) divisible by sh (x likewise), and over
// m, m' those taps slide across the source with unit stride.  Each class is a launch of the kernels below on its
// sub-lattices of taps and of outputs (slayer_conv_synapse_input_grad), a fraction 1 / (sh sw) of the taps each.
//
// LDS: the weights of this workgroup's 16 output channels, tap-major (row k holds the 16 channels), and per tap the
// offset of its input row relative to the pixel's own position and its (row, column) displacement in the image.
// A workgroup's four waves take four consecutive items of one (batch entry, channel block): an item is one tile
// of 64 steps of a piece of one output row.
template <bool STREAM, bool TAIL, int CHUNK>
__global__ __launch_bounds__(kSynWaves * kWave) void synapse_conv_kernel(const SynapseConv p) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int Kp = p.KG * 4;
    float* wt = lds;                                    // [Kp][16]
    int* tap_off = reinterpret_cast<int*>(lds + Kp * 16);   // [Kp] bytes
    int* tap_dy = tap_off + Kp;                         // [Kp]
    int* tap_dx = tap_dy + Kp;                          // [Kp]

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup -> (batch entry, block of 16 output channels, four items)
    const int groups = (p.items + kSynWaves - 1) / kSynWaves;
    int b = xcd_contiguous(blockIdx.x, gridDim.x);
    const int ig = b % groups; b /= groups;
    const int cob = b % ((p.Co + 15) / 16);
    const int n = b / ((p.Co + 15) / 16);
    const int co0 = cob * 16;

    const int64_t k_full = (int64_t)p.Ci * p.kh_full * p.kw_full;
    for (int i = tid; i < Kp * 16; i += kSynWaves * kWave) {
        const int k = i >> 4, m = i & 15;
        const int ci = k / (p.kh * p.kw), r = k - ci * (p.kh * p.kw), y = r / p.kw, x = r - y * p.kw;
        wt[i] = (k < p.K && co0 + m < p.Co) ? p.weight[(int64_t)(co0 + m) * k_full + p.weight_index(ci, y, x)] : 0.0f;
    }
    for (int k = tid; k < Kp; k += kSynWaves * kWave) {
        const int ci = k / (p.kh * p.kw), r = k - ci * (p.kh * p.kw), y = r / p.kw, x = r - y * p.kw;
        const int dy = y * p.dh - p.ph;
        const int dx = x * p.dw - p.pw;
        tap_dy[k] = k < p.K ? dy : (1 << 28);                             // a tap that does not exist: always outside
        tap_dx[k] = dx;
        tap_off[k] = (((ci * p.H + dy) * p.W) + dx) * p.T * 4;
    }
    __syncthreads();

    const int item = ig * kSynWaves + wave;
    if (item >= p.items) return;
    const int tile = item % p.ttiles;
    const int piece = (item / p.ttiles) % p.wsplit;
    const int ho = item / (p.ttiles * p.wsplit);
    const int t0 = tile * kSynTile;
    const int kk = lane >> 4, j = lane & 15;
    SynQuad tq;
    tq.template set<TAIL>(t0 + 4 * j, p.T);
    const int nv = tq.nv;
    const bool t_ok = tq.any();
    const int hin = ho * p.sh;                                           // image row of tap (0, 0) before padding
    const int64_t in_plane = (int64_t)p.Ci * p.H * p.W * p.T;
    const __amdgpu_buffer_rsrc_t src = make_rsrc(p.in + (int64_t)n * in_plane, (unsigned)(in_plane * 4));
    const int64_t out_plane = (int64_t)p.Co * p.Ho_full * p.Wo_full * p.T;
    const __amdgpu_buffer_rsrc_t dst = make_rsrc(p.out + (int64_t)n * out_plane, (unsigned)(out_plane * 4));

    const int per = (p.Wo + p.wsplit - 1) / p.wsplit;
    const int w_lo = piece * per, w_hi = (w_lo + per) < p.Wo ? (w_lo + per) : p.Wo;
    for (int wo = w_lo; wo < w_hi; ++wo) {
        const int win = wo * p.sw;
        const int pix = ((hin * p.W) + win) * p.T * 4 + tq.t_load * 4;   // byte offset of tap (0,0,0)'s quad
        syn_f4 acc[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = syn_f4{0.f, 0.f, 0.f, 0.f};
        for (int g0 = 0; g0 < p.KG; g0 += CHUNK) {
            float4 q[CHUNK];
            float a[CHUNK];
#pragma unroll
            for (int u = 0; u < CHUNK; ++u) {
                const int k = 4 * (g0 + u) + kk;
                const int yy = hin + tap_dy[k], xx = win + tap_dx[k];
                const bool ok = t_ok && (unsigned)yy < (unsigned)p.H && (unsigned)xx < (unsigned)p.W;
                q[u] = tq.template place<TAIL>(buf_load4<false>(src, ok ? pix + tap_off[k] : kOutOfRange));
                a[u] = wt[k * 16 + j];
            }
#pragma unroll
            for (int u = 0; u < CHUNK; ++u) {
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], q[u].x, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], q[u].y, acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], q[u].z, acc[2], 0, 0, 0);
                acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], q[u].w, acc[3], 0, 0, 0);
            }
        }
        // lane (kk, j): output channels co0 + 4 kk + i, steps t0 + 4 j + e
        const int opix = p.out_pixel(ho, wo) * p.T * 4 + (t0 + 4 * j) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int co = co0 + 4 * kk + i;
            syn_store_quad<STREAM, TAIL>(dst, co < p.Co, co * (p.Ho_full * p.Wo_full * p.T * 4) + opix, nv,
                                   make_float4(acc[0][i], acc[1][i], acc[2][i], acc[3][i]));
        }
    }
}

// The common case -- unit stride and dilation along the image row, KW taps per row -- takes PIX neighbouring
// output pixels at a time: they share their input columns (PIX + KW - 1 of them instead of PIX * KW), so a group of
// four (input channel, kernel row) pairs costs PIX + KW - 1 loads for PIX * KW * 4 matrix products.  Measured on
// [32,8,32,32,300] -> 16 channels, 3x3: the one-pixel form is bound by what the caches deliver to the loads
// (18 KB per pixel and tile of 64 steps), not by the matrix cores.
// LDS: weights as above (tap k = pair * KW + x, pair = ci * kh + y), and per pair the byte offset of its input row
// relative to the pixel block's own position and its row displacement.
template <int KW, int PIX, bool STREAM, bool TAIL>
__device__ __forceinline__ void synapse_conv_row(const SynapseConv& p) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int PG = p.KG;                                // groups of four pairs
    const int Kp = PG * 4 * KW;
    float* wt = lds;                                    // [Kp][16]
    int* pair_off = reinterpret_cast<int*>(lds + Kp * 16);  // [4 PG] bytes
    int* pair_dy = pair_off + 4 * PG;                   // [4 PG]

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int groups = (p.items + kSynWaves - 1) / kSynWaves;
    int b = xcd_contiguous(blockIdx.x, gridDim.x);
    const int ig = b % groups; b /= groups;
    const int cob = b % ((p.Co + 15) / 16);
    const int n = b / ((p.Co + 15) / 16);
    const int co0 = cob * 16;

    const int64_t k_full = (int64_t)p.Ci * p.kh_full * p.kw_full;
    // eight loads of a thread in flight at a time (one after the other they were a fifth of a workgroup's life)
    for (int i0 = tid; i0 < Kp * 16; i0 += 8 * kSynWaves * kWave) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = i0 + u * kSynWaves * kWave;
            const int k = i >> 4, m = i & 15;
            const int pr = k / KW, x = k - pr * KW, ci = pr / p.kh, y = pr - ci * p.kh;
            v[u] = (k < p.K && co0 + m < p.Co) ? p.weight[(int64_t)(co0 + m) * k_full + p.weight_index(ci, y, x)] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = i0 + u * kSynWaves * kWave;
            if (i < Kp * 16) wt[i] = v[u];
        }
    }
    for (int pr = tid; pr < 4 * PG; pr += kSynWaves * kWave) {
        const int ci = pr / p.kh, y = pr - ci * p.kh;
        const int dy = y * p.dh - p.ph;
        pair_dy[pr] = pr < p.Ci * p.kh ? dy : (1 << 28);                 // a pair that does not exist: always outside
        pair_off[pr] = (((ci * p.H + dy) * p.W) - p.pw) * p.T * 4;
    }
    __syncthreads();

    const int item = ig * kSynWaves + wave;
    if (item >= p.items) return;
    const int tile = item % p.ttiles;
    const int piece = (item / p.ttiles) % p.wsplit;
    const int ho = item / (p.ttiles * p.wsplit);
    const int t0 = tile * kSynTile;
    const int kk = lane >> 4, j = lane & 15;
    SynQuad tq;
    tq.template set<TAIL>(t0 + 4 * j, p.T);
    const int nv = tq.nv;
    const bool t_ok = tq.any();
    const int hin = ho * p.sh;
    const int64_t in_plane = (int64_t)p.Ci * p.H * p.W * p.T;
    const __amdgpu_buffer_rsrc_t src = make_rsrc(p.in + (int64_t)n * in_plane, (unsigned)(in_plane * 4));
    const int64_t out_plane = (int64_t)p.Co * p.Ho_full * p.Wo_full * p.T;
    const __amdgpu_buffer_rsrc_t dst = make_rsrc(p.out + (int64_t)n * out_plane, (unsigned)(out_plane * 4));
    const int col = p.T * 4;                                             // bytes from a pixel to its right neighbour

    const int per = ((p.Wo + p.wsplit - 1) / p.wsplit + PIX - 1) / PIX * PIX;
    const int w_lo = piece * per, w_hi = (w_lo + per) < p.Wo ? (w_lo + per) : p.Wo;
    for (int wo0 = w_lo; wo0 < w_hi; wo0 += PIX) {
        const int pix = ((hin * p.W) + wo0) * col + tq.t_load * 4;
        syn_f4 acc[PIX][4];
#pragma unroll
        for (int i = 0; i < PIX; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][e] = syn_f4{0.f, 0.f, 0.f, 0.f};
        for (int g = 0; g < PG; ++g) {
            const int pr = 4 * g + kk;
            const bool row_ok = t_ok && (unsigned)(hin + pair_dy[pr]) < (unsigned)p.H;
            const int base = pix + pair_off[pr];
            float4 q[PIX + KW - 1];
#pragma unroll
            for (int c = 0; c < PIX + KW - 1; ++c) {
                const bool ok = row_ok && (unsigned)(wo0 + c - p.pw) < (unsigned)p.W;
                q[c] = tq.template place<TAIL>(buf_load4<false>(src, ok ? base + c * col : kOutOfRange));
            }
            float a[KW];
#pragma unroll
            for (int x = 0; x < KW; ++x) a[x] = wt[(pr * KW + x) * 16 + j];
#pragma unroll
            for (int x = 0; x < KW; ++x) {
#pragma unroll
                for (int i = 0; i < PIX; ++i) {
                    acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], q[i + x].x, acc[i][0], 0, 0, 0);
                    acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], q[i + x].y, acc[i][1], 0, 0, 0);
                    acc[i][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], q[i + x].z, acc[i][2], 0, 0, 0);
                    acc[i][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], q[i + x].w, acc[i][3], 0, 0, 0);
                }
            }
        }
        // lane (kk, j): output channels co0 + 4 kk + i, steps t0 + 4 j + e
#pragma unroll
        for (int px = 0; px < PIX; ++px) {
            const int opix = p.out_pixel(ho, wo0 + px) * col + (t0 + 4 * j) * 4;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int co = co0 + 4 * kk + i;
                syn_store_quad<STREAM, TAIL>(dst, co < p.Co && wo0 + px < w_hi, co * (p.Ho_full * p.Wo_full * col) + opix, nv,
                                       make_float4(acc[px][0][i], acc[px][1][i], acc[px][2][i], acc[px][3][i]));
            }
        }
    }
}

// Rows of whole quads at five waves per SIMD (88 registers, no spills; four waves otherwise: 2-3 % slower); the
// forms for rows that end inside a quad need a few registers more and keep the compiler's own choice.
template <int KW, int PIX, bool STREAM>
__global__ __launch_bounds__(kSynWaves * kWave) __attribute__((amdgpu_waves_per_eu(5)))
void synapse_conv_row_kernel(const SynapseConv p) { synapse_conv_row<KW, PIX, STREAM, false>(p); }
template <int KW, int PIX, bool STREAM>
__global__ __launch_bounds__(kSynWaves * kWave) void synapse_conv_row_tail_kernel(const SynapseConv p) {
    synapse_conv_row<KW, PIX, STREAM, true>(p);
}

// The row form on the bfloat16 matrix instruction, for layers with enough (input channel, kernel row) pairs to fill its 32
// terms.  The float32 instruction bounds wide layers: 32 -> 64 channels on [16,32,16,16,300] 398 us forward (72 % of its
// peak) and 429 us for the input gradient.  Operands are split into three parts (split.h) unless they are bfloat16
// numbers as they are: the weights are looked at once per workgroup (those of an 8-bit quantiser always are), the input
// once per column and group of 32 pairs (spikes are, gradients are not), and the products run to match: one for spikes
// and quantised weights, three for one split operand, six for two.
//
// A wave walks the columns of its image row: lane (kk, j) loads steps 4j .. 4j+3 of pairs 32 g + 8 kk + {0 .. 7} at the
// column, turns them into the operands of four products (one per step of the quad: eight pairs each), and uses these
// for the KW output pixels the column meets, whose accumulators it keeps -- every column is loaded and split once.  A
// pixel is complete, and stored, after its last column.  The next loads are on their way during the products.
// The instruction rounds every sum it leaves, so the products of the lower parts, 2^-8 of the whole at most, are added up
// from zero and join the sum in one addition: it is rounded twice for 32 terms, not up to six times.  The error against
// float64 is 0.3 to 0.6 times that of the float32 form, sparse (graded) inputs included (96 pairs: real x real 1.0e-7 and
// 2.9e-7, graded x real 0.7e-7 and 1.2e-7, real x quantised over 192 pairs 1.3e-7 and 4.2e-7; every product into the one sum:
// 2.6e-7, 2.1e-7, 2.4e-7).
// [16,32,16,16,300] -> 64 channels forward 402 -> 262 us, input gradient 418 -> 287 us with quantised weights, 357 without;
// [32,8,32,32,300] -> 16 channels 352 -> 297 and 415 -> 328 us (168 registers, three waves per SIMD; five taps 213, two waves).
// What bounds it now: the unaligned rows of the result (T = 300) for few channels, the vector instructions of the split
// for gradients.
//
// A value that is not finite, or overflows when it is scaled or rounded, leaves parts of either sign, and infinity times
// each of them is not infinity times their sum: a wave with a result that is not finite computes its row again from
// the operands as they are, and so does every wave of a workgroup with such a weight.
// LDS: the parts of the weights in the operand's layout, [group][tap][part][lane]; per wave the byte
// offset of every pair's input row (or kOutOfRange).
template <int KW, bool STREAM, bool TAIL>
__global__ __launch_bounds__(8 * kWave) __attribute__((amdgpu_waves_per_eu(KW <= 3 ? 3 : 2)))
void synapse_conv_split_kernel(const SynapseConv p) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int G = p.KG;                                 // groups of 32 pairs
    const int pairs = p.Ci * p.kh;
    uint4* wt = reinterpret_cast<uint4*>(lds);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), threads = blockDim.x, waves = threads / kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int* row_off = reinterpret_cast<int*>(wt + G * KW * 3 * kWave) + wave * G * 32;
    // neighbouring workgroups take the channel blocks of the same items: they share the input rows
    const int cobs = (p.Co + 15) / 16;
    const int groups = (p.items + waves - 1) / waves;
    int b = xcd_contiguous(blockIdx.x, gridDim.x);
    const int cob = b % cobs; b /= cobs;
    const int ig = b % groups;
    const int n = b / groups;
    const int co0 = cob * 16;
    const int kk = lane >> 4, j = lane & 15;

    const int64_t k_full = (int64_t)p.Ci * p.kh_full * p.kw_full;
    unsigned low = 0u;
    bool odd = false;                                   // a weight that is not finite
    for (int i = tid; i < G * KW * kWave; i += threads) {
        const int l = i & (kWave - 1), x = (i >> 6) % KW, g = (i >> 6) / KW;
        const int co = co0 + (l & 15);
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int pr = 32 * g + 8 * (l >> 4) + e, ci = pr / p.kh, y = pr - ci * p.kh;
            v[e] = (pr < pairs && co < p.Co) ? p.weight[(int64_t)co * k_full + p.weight_index(ci, y, x)] : 0.0f;
            low |= __float_as_uint(v[e]);
            odd = odd || !(fabsf(v[e]) < __builtin_inff());
            v[e] *= kSplitScale;
        }
        uint4* to = wt + (i >> 6) * 3 * kWave + l;
        to[0] = round_eight(v);
        to[kWave] = round_eight(v);
        to[2 * kWave] = bf16_eight(v);
    }
    const int item = ig * waves + wave;
    const bool on = item < p.items;
    const int tile = item % p.ttiles;
    const int piece = (item / p.ttiles) % p.wsplit;
    const int ho = item / (p.ttiles * p.wsplit);
    const int hin = ho * p.sh;
    const int col = p.T * 4;                                             // bytes from a pixel to its right neighbour
    for (int pr = lane; pr < 32 * G; pr += kWave) {
        const int ci = pr / p.kh, row = hin + (pr - ci * p.kh) * p.dh - p.ph;
        row_off[pr] = (pr < pairs && (unsigned)row < (unsigned)p.H) ? (ci * p.H + row) * p.W * col : kOutOfRange;
    }
    const bool split_w = __syncthreads_or((low & 0xffffu) != 0u);
    const bool float_only = __syncthreads_or(odd);
    if (!on) return;
    const int t0 = tile * kSynTile;
    SynQuad tq;
    tq.template set<TAIL>(t0 + 4 * j, p.T);
    const bool t_ok = tq.any();
    const int64_t in_plane = (int64_t)p.Ci * p.H * p.W * p.T;
    const __amdgpu_buffer_rsrc_t src = make_rsrc(p.in + (int64_t)n * in_plane, (unsigned)(in_plane * 4));
    const int64_t out_plane = (int64_t)p.Co * p.Ho_full * p.Wo_full * p.T;
    const __amdgpu_buffer_rsrc_t dst = make_rsrc(p.out + (int64_t)n * out_plane, (unsigned)(out_plane * 4));
    const int per = (p.Wo + p.wsplit - 1) / p.wsplit;
    const int w_lo = piece * per, w_hi = (w_lo + per) < p.Wo ? (w_lo + per) : p.Wo;
    if (w_lo >= w_hi) return;

    // column c (counted with the padding: tap x of output pixel wo lies at column wo + x) is image column c - pw
    const int c_end = w_hi + KW - 1;
    const int c_lo = w_lo > p.pw ? w_lo : p.pw;                          // the columns inside the image
    const int c_hi = c_end < p.W + p.pw ? c_end : p.W + p.pw;
    float4 raw[8];
    auto fetch = [&](int c, int g) {
        const int4* off = reinterpret_cast<const int4*>(row_off + 32 * g + 8 * kk);
        const int4 o[2] = {off[0], off[1]};
        const int at = (c - p.pw) * col + tq.t_load * 4;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            raw[4 * i] = buf_load4<false>(src, t_ok ? o[i].x + at : kOutOfRange);
            raw[4 * i + 1] = buf_load4<false>(src, t_ok ? o[i].y + at : kOutOfRange);
            raw[4 * i + 2] = buf_load4<false>(src, t_ok ? o[i].z + at : kOutOfRange);
            raw[4 * i + 3] = buf_load4<false>(src, t_ok ? o[i].w + at : kOutOfRange);
        }
    };
    // lane (kk, j): output channels co0 + 4 kk + i, steps t0 + 4 j + e
    auto store = [&](int wo, const syn_f4 (&d)[4]) {
        const int opix = p.out_pixel(ho, wo) * col + (t0 + 4 * j) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int co = co0 + 4 * kk + i;
            syn_store_quad<STREAM, TAIL>(dst, co < p.Co, co * (p.Ho_full * p.Wo_full * col) + opix, tq.nv,
                                         make_float4(d[0][i], d[1][i], d[2][i], d[3][i]));
        }
    };
    float stored = 0.f;                                                  // not finite once a result is not
    syn_f4 acc[KW][4];
    if (c_lo < c_hi) fetch(c_lo, 0);
#pragma unroll
    for (int x = 0; x < KW; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[x][e] = syn_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int c = w_lo; c < c_end; ++c) {                                 // tap x of column c goes to pixel c - x: acc[x]
        if (c >= c_lo && c < c_hi) {
#pragma unroll 1
            for (int g = 0; g < G; ++g) {
                float v[4][8];                                       // [step of the quad][pair]
                unsigned bits = 0u;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float4 r = tq.template place<TAIL>(raw[i]);
                    v[0][i] = r.x * kSplitScale; v[1][i] = r.y * kSplitScale;
                    v[2][i] = r.z * kSplitScale; v[3][i] = r.w * kSplitScale;
                    bits |= __float_as_uint(r.x) | __float_as_uint(r.y) | __float_as_uint(r.z) | __float_as_uint(r.w);
                }
                const bool split_x = __any((bits & 0xffffu) != 0u);
                const uint4* wg = wt + g * KW * 3 * kWave + lane;
                const bool last = g + 1 == G;                            // the next loads are on their way during the products
                if (!last || c + 1 < c_hi) fetch(last ? c + 1 : c, last ? 0 : g + 1);
                // kH steps of the quad at a time (the parts of all four do not fit beside the accumulators), and branches
                // around the products of the lower parts only: around several copies of the whole they cost the compiler a
                // second set of accumulators and spills.
                constexpr int kH = KW == 5 ? 4 : 2;
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
                    for (int x = 0; x < KW; ++x) {
                        const uint4 w0 = wg[x * 3 * kWave];
                        syn_f4 d[kH];
                        if (split_x) {
                            if (split_w) {
                                const uint4 w1 = wg[(x * 3 + 1) * kWave], w2 = wg[(x * 3 + 2) * kWave];
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
                            for (int e = 0; e < kH; ++e) acc[x][h + e] += mfma_bf16(w0, q[e][1], d[e]);
                        } else if (split_w) {
                            const uint4 w1 = wg[(x * 3 + 1) * kWave], w2 = wg[(x * 3 + 2) * kWave];
#pragma unroll
                            for (int e = 0; e < kH; ++e) d[e] = mfma_bf16(w2, q[e][0], zero);
#pragma unroll
                            for (int e = 0; e < kH; ++e) acc[x][h + e] += mfma_bf16(w1, q[e][0], d[e]);
                        }
#pragma unroll
                        for (int e = 0; e < kH; ++e) acc[x][h + e] = mfma_bf16(w0, q[e][0], acc[x][h + e]);
                    }
                }
            }
        }
        const int wo = c - (KW - 1);
        if (wo >= w_lo) {
            syn_f4 d[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                d[e] = acc[KW - 1][e];
                stored += (d[e][0] + d[e][1]) + (d[e][2] + d[e][3]);
#pragma unroll
                for (int i = 0; i < 4; ++i) d[e][i] *= kSplitProductScale;
            }
            store(wo, d);
        }
#pragma unroll
        for (int x = KW - 1; x >= 0; --x)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[x][e] = x > 0 ? acc[x - 1][e] : syn_f4{0.f, 0.f, 0.f, 0.f};
    }
    if (!float_only && !__any(!(fabsf(stored) < __builtin_inff()))) return;

    // once more in float32 multiplications and additions, taps outside the image as products with zero like the float32 form
#pragma unroll 1
    for (int wo = w_lo; wo < w_hi; ++wo) {
        syn_f4 d[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = syn_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int pr = 0; pr < pairs; ++pr) {
            const int ci = pr / p.kh, y = pr - ci * p.kh, row = row_off[pr];
#pragma unroll 1
            for (int x = 0; x < KW; ++x) {
                const int c = wo + x - p.pw;
                const bool in = t_ok && row != kOutOfRange && (unsigned)c < (unsigned)p.W;
                const float4 q = tq.template place<TAIL>(buf_load4<false>(src, in ? row + c * col + tq.t_load * 4 : kOutOfRange));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int co = co0 + 4 * kk + i;
                    const float w = co < p.Co ? p.weight[(int64_t)co * k_full + p.weight_index(ci, y, x)] : 0.f;
                    d[0][i] = __fmaf_rn(w, q.x, d[0][i]);
                    d[1][i] = __fmaf_rn(w, q.y, d[1][i]);
                    d[2][i] = __fmaf_rn(w, q.z, d[2][i]);
                    d[3][i] = __fmaf_rn(w, q.w, d[3][i]);
                }
            }
        }
        store(wo, d);
    }
}

// One input and one output channel (the pooling layers, which fold their channels into the image height,
// synapse/layer.py:438-508 and :770-838 in the reference): there is no contraction for the matrix cores, and a wave
// that owns 16 channels x 64 steps of one pixel would move 256 bytes per instruction.  One thread per quad of output
// steps on the vector units instead: a block row of the grid is ROWS image rows of the output, grid.z the batch.
// SPREAD: the gradient of the input (the unpooling layer's forward pass): output pixel (h, w) sums the taps (y, x)
// whose source coordinates (h + ph - y dh) / sh, (w + pw - x dw) / sw are exact.  Which taps those are depends on
// h mod sh alone: a table in LDS lists them per residue (at most ny per residue: tap_y, and quot_y = the quotient
// less h / sh; likewise nx, tap_x, quot_x), so that a pixel visits ny * nx slots -- one for a pooling window that is
// as large as its stride -- instead of all kh * kw taps.
constexpr int kPlaneThreads = 256;
#ifndef SLAYER_PLANE_ROWS_SUM
#define SLAYER_PLANE_ROWS_SUM 1
#endif
#ifndef SLAYER_PLANE_ROWS_SPREAD
#define SLAYER_PLANE_ROWS_SPREAD 8
#endif
constexpr int kPlaneRowsSum = SLAYER_PLANE_ROWS_SUM, kPlaneRowsSpread = SLAYER_PLANE_ROWS_SPREAD;
template <bool SPREAD, bool STREAM, bool TAIL, int ROWS>
__global__ __launch_bounds__(kPlaneThreads) void synapse_plane_kernel(const SynapseConv p, int quads, int ny, int nx) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* wt = lds;                                                      // [kh * kw]
    int* quot_y = reinterpret_cast<int*>(lds + p.kh * p.kw);              // SPREAD: [sh * ny]
    int* tap_y = quot_y + p.sh * ny;                                      //         [sh * ny], times kw
    int* quot_x = tap_y + p.sh * ny;                                      //         [sw * nx]
    int* tap_x = quot_x + p.sw * nx;                                      //         [sw * nx]
    const int none = 1 << 28;
    for (int i = threadIdx.x; i < p.kh * p.kw; i += kPlaneThreads) wt[i] = p.weight[i];
    if (SPREAD) {
        for (int r = threadIdx.x; r < p.sh + p.sw; r += kPlaneThreads) {
            const bool rows = r < p.sh;
            const int res = rows ? r : r - p.sh, k = rows ? p.kh : p.kw, stride = rows ? p.sh : p.sw;
            const int pad = rows ? p.ph : p.pw, dil = rows ? p.dh : p.dw, slots = rows ? ny : nx;
            int* quot = (rows ? quot_y : quot_x) + res * slots;
            int* tap = (rows ? tap_y : tap_x) + res * slots;
            int found = 0;
            for (int y = 0; y < k; ++y) {
                const int c = res + pad - y * dil;
                if (c % stride == 0) { quot[found] = c / stride; tap[found] = rows ? y * p.kw : y; ++found; }
            }
            for (; found < slots; ++found) { quot[found] = none; tap[found] = 0; }
        }
    }
    __syncthreads();
    const int n = blockIdx.z;
    const int idx = blockIdx.x * kPlaneThreads + threadIdx.x;
    const int wo = idx / quads, j = idx - wo * quads;
    const bool on = wo < p.Wo;
    SynQuad tq;
    tq.template set<TAIL>(4 * j, p.T);
    const bool lane_on = on && tq.any();
    const int64_t in_plane = (int64_t)p.H * p.W * p.T;
    const __amdgpu_buffer_rsrc_t src = make_rsrc(p.in + (int64_t)n * in_plane, (unsigned)(in_plane * 4));
    const int64_t out_plane = (int64_t)p.Ho * p.Wo * p.T;
    const __amdgpu_buffer_rsrc_t dst = make_rsrc(p.out + (int64_t)n * out_plane, (unsigned)(out_plane * 4));
    // SPREAD: the pixel as quotient and residue of the strides (the rows' are the same for the whole block)
    const int wq = SPREAD ? wo / p.sw : 0, rx = SPREAD ? (on ? wo - wq * p.sw : 0) : 0;
    // A block takes ROWS image rows at once: the tables above are set up once for all of them, and a slot is
    // loaded for all the rows before the first product waits for it.
    const int ho0 = blockIdx.y * ROWS;
    int hq[ROWS], ry[ROWS];
    float4 acc[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        hq[r] = SPREAD ? (ho0 + r) / p.sh : 0;
        ry[r] = SPREAD ? (ho0 + r < p.Ho ? ho0 + r - hq[r] * p.sh : 0) : 0;
        acc[r] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    for (int y = 0; y < (SPREAD ? ny : p.kh); ++y) {
        int row_off[ROWS], w_row[ROWS];                                   // source row of this slot or none, its weights
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const int yy = SPREAD ? hq[r] + quot_y[ry[r] * ny + y] : (ho0 + r) * p.sh + y * p.dh - p.ph;
            row_off[r] = (ho0 + r < p.Ho && (unsigned)yy < (unsigned)p.H) ? yy * p.W : -1;
            w_row[r] = SPREAD ? tap_y[ry[r] * ny + y] : y * p.kw;
        }
        for (int x = 0; x < (SPREAD ? nx : p.kw); ++x) {
            const int xx = SPREAD ? wq + quot_x[rx * nx + x] : wo * p.sw + x * p.dw - p.pw;
            const int w_col = SPREAD ? tap_x[rx * nx + x] : x;
            const bool ok = lane_on && (unsigned)xx < (unsigned)p.W;
            float4 q[ROWS];
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
                q[r] = buf_load4<false>(src, (ok && row_off[r] >= 0) ? ((row_off[r] + xx) * p.T + tq.t_load) * 4 : kOutOfRange);
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const float f = wt[w_row[r] + w_col];
                const float4 v = tq.template place<TAIL>(q[r]);
                acc[r].x = __fmaf_rn(f, v.x, acc[r].x); acc[r].y = __fmaf_rn(f, v.y, acc[r].y);
                acc[r].z = __fmaf_rn(f, v.z, acc[r].z); acc[r].w = __fmaf_rn(f, v.w, acc[r].w);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
        syn_store_quad<STREAM, TAIL>(dst, on && ho0 + r < p.Ho, (((ho0 + r) * p.Wo + wo) * p.T + 4 * j) * 4, tq.nv, acc[r]);
}

// Gradient of the weights: grad_w[co][k] = sum over batch, output pixels and time of grad_out[co][pixel][t] *
// (input row of tap k at that pixel)[t] -- a [Co x P] x [P x K] product with P = N * Ho * Wo * T positions, reduced
// along time on the matrix cores: lane (kk, j) loads steps 4 kk .. 4 kk + 3 of a 16-step group of the gradient row of
// channel co0 + j (the A operand of four products) and of the input row of tap 16 tt + j (the B operand), so that
// a group of 16 steps costs 1 + NTT loads and 4 NTT products and adds to NTT accumulator tiles [16 channels x 16
// taps].  A wave owns one output row of one batch entry and a share of the time axis, walks the row pixel by pixel
// and leaves its tiles in the workspace; synapse_wgrad_reduce_kernel adds the tiles of all waves in double, in a
// fixed order.  Filters of more than 16 NTT taps take several passes (grid dimension z).
struct SynapseWgrad {
    float* partial;                     // [items][passes][NTT][64] quads
    const float* grad_out;
    const float* in;
    int N, Ci, Co, H, W, Ho, Wo, T;
    int kh, kw, sh, sw, ph, pw, dh, dw;
    int K, passes;                      // taps, passes of 16 NTT taps
    int tparts, tlen;                   // shares of the time axis, steps per share (a multiple of 32)
    int items;                          // (share of time, output row) pairs of one (batch entry, channel block)
};

template <int NTT, bool TAIL>
__global__ __launch_bounds__(kSynWaves * kWave) void synapse_wgrad_kernel(const SynapseWgrad p) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int Kp = NTT * 16;
    int* tap_off = reinterpret_cast<int*>(lds);         // [Kp] bytes
    int* tap_dy = tap_off + Kp;                         // [Kp]
    int* tap_dx = tap_dy + Kp;                          // [Kp]

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int groups = (p.items + kSynWaves - 1) / kSynWaves;
    const int cobs = (p.Co + 15) / 16;
    int b = xcd_contiguous(blockIdx.x, gridDim.x);
    const int ig = b % groups; b /= groups;
    const int cob = b % cobs;
    const int n = b / cobs;
    const int co0 = cob * 16;
    const int pass = blockIdx.y;
    const int k0 = pass * Kp;

    for (int kl = tid; kl < Kp; kl += kSynWaves * kWave) {
        const int k = k0 + kl;
        const int ci = k / (p.kh * p.kw), r = k - ci * (p.kh * p.kw), y = r / p.kw, x = r - y * p.kw;
        const int dy = y * p.dh - p.ph, dx = x * p.dw - p.pw;
        tap_dy[kl] = k < p.K ? dy : (1 << 28);                           // a tap that does not exist: always outside
        tap_dx[kl] = dx;
        tap_off[kl] = (((ci * p.H + dy) * p.W) + dx) * p.T * 4;
    }
    __syncthreads();

    const int item = ig * kSynWaves + wave;
    if (item >= p.items) return;
    const int tpart = item % p.tparts;
    const int ho = item / p.tparts;
    const int kk = lane >> 4, j = lane & 15;
    const int hin = ho * p.sh;
    const int64_t in_plane = (int64_t)p.Ci * p.H * p.W * p.T;
    const __amdgpu_buffer_rsrc_t src = make_rsrc(p.in + (int64_t)n * in_plane, (unsigned)(in_plane * 4));
    const int64_t out_plane = (int64_t)p.Co * p.Ho * p.Wo * p.T;
    const __amdgpu_buffer_rsrc_t grd = make_rsrc(p.grad_out + (int64_t)n * out_plane, (unsigned)(out_plane * 4));
    const int col = p.T * 4;
    const bool co_ok = co0 + j < p.Co;
    const int g_row = (co0 + j) * (p.Ho * p.Wo * col) + ho * p.Wo * col;  // gradient row of this lane's channel
    // this lane's taps: offset of the input row relative to the pixel, and whether its image row exists
    int my_off[NTT], my_dx[NTT];
    bool my_row[NTT];
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt) {
        my_off[tt] = tap_off[16 * tt + j];
        my_dx[tt] = tap_dx[16 * tt + j];
        my_row[tt] = (unsigned)(hin + tap_dy[16 * tt + j]) < (unsigned)p.H;
    }
    syn_f4 acc[NTT][2];                                                  // two chains per tile: no product waits for the one before
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt) acc[tt][0] = acc[tt][1] = syn_f4{0.f, 0.f, 0.f, 0.f};

    const int t_lo = tpart * p.tlen, t_hi = (t_lo + p.tlen) < p.T ? (t_lo + p.tlen) : p.T;
    for (int t0 = t_lo; t0 < t_hi; t0 += 32) {                           // one 128-byte line of every row per visit
        for (int wo = 0; wo < p.Wo; ++wo) {
            const int win = wo * p.sw;
            const int pix = ((hin * p.W) + win) * col;
            float4 g[2], q[2][NTT];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = t0 + 16 * u + 4 * kk;
                SynQuad tq;                                              // the shares are whole quads; a row's last quad may not be
                tq.template set<TAIL>(t, t_hi);
                const bool t_ok = tq.any();
                g[u] = tq.template place<TAIL>(buf_load4<false>(grd, (t_ok && co_ok) ? g_row + wo * col + tq.t_load * 4 : kOutOfRange));
#pragma unroll
                for (int tt = 0; tt < NTT; ++tt) {
                    const bool ok = t_ok && my_row[tt] && (unsigned)(win + my_dx[tt]) < (unsigned)p.W;
                    q[u][tt] = tq.template place<TAIL>(buf_load4<false>(src, ok ? pix + my_off[tt] + tq.t_load * 4 : kOutOfRange));
                }
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int tt = 0; tt < NTT; ++tt) {
                    acc[tt][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(g[u].x, q[u][tt].x, acc[tt][0], 0, 0, 0);
                    acc[tt][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(g[u].y, q[u][tt].y, acc[tt][1], 0, 0, 0);
                }
#pragma unroll
                for (int tt = 0; tt < NTT; ++tt) {
                    acc[tt][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(g[u].z, q[u][tt].z, acc[tt][0], 0, 0, 0);
                    acc[tt][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(g[u].w, q[u][tt].w, acc[tt][1], 0, 0, 0);
                }
            }
        }
    }
    // lane (q, j) of tile tt: channels co0 + 4 q + i, tap k0 + 16 tt + j
    float4* dst = reinterpret_cast<float4*>(p.partial) +
                  ((((int64_t)(n * cobs + cob) * p.items + item) * p.passes + pass) * NTT) * kWave + lane;
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt)
        dst[tt * kWave] = make_float4(acc[tt][0][0] + acc[tt][1][0], acc[tt][0][1] + acc[tt][1][1],
                                      acc[tt][0][2] + acc[tt][1][2], acc[tt][0][3] + acc[tt][1][3]);
}

// The common case again (unit stride and dilation along the image row, KW taps per row): the taps of a tile are 16
// (input channel, kernel row) pairs at one input column, and that column meets KW output pixels, one per tap of the
// row -- so the wave walks the input columns of its image row, keeps the gradient of the last KW pixels in registers
// (one new visit per column), and a column costs 1 + NPT visits for KW * NPT tiles.
// Accumulator tile (x, pt): [16 channels x 16 pairs] for tap x.
//
// The float32 instruction (16 steps of time in 4 x 32 cycles) was one bound of wide layers: 32 -> 64 channels on
// [16,32,16,16,300] 539 us, 84 % of its peak.  Here the products run on the bfloat16
// instruction (32 steps in 16 cycles): the gradient split into three parts (split.h), the input as it is where its
// values are bfloat16 numbers -- spikes, and pooled spikes, always are; a visit that brings anything else splits it, too,
// and takes six products instead of three.  The parts of the gradient are formed once per visit and stay in the window.
// The other bound was the L1: in the operand's layout neighbouring lanes lie in sixteen different rows, so a load
// of 1 KB looks up 64 lines.  Eight lanes now read the 128-byte line of a row together, and the split values
// reach the operand's layout through LDS of the wave's own.
//
// The instruction rounds its sums down, not to nearest: a bias of some 2^-27 a product that a sum over 10^4 of them
// collects (relative error of the result 1e-6, float32 instruction 1.3e-7 .. 5.7e-7).  A visit's products therefore start
// from zero, every other column with the input negated, and the vector units add or subtract them: the biases cancel,
// and the error is 0.8e-7 .. 1.2e-7 over spikes, graded spikes and real values.
//   [16,32,16,16,300] -> 64 channels 539 -> 271 us, [32,8,32,32,300] -> 16 channels 374 -> 340 us (3 waves per SIMD; 64
// steps per visit leave 2: 335 and 368 us).  What bounds it now: lines of the unaligned rows (T = 300) that two visits
// share and fetch twice, and the vector instructions of the split.
//
// What is not finite (or overflows when it is scaled or rounded) shows in a tile at the end: the wave then runs its
// share again with the float32 instruction (float_products), whose results such inputs had before.
constexpr int kWgPitch = 80;                   // bytes of LDS per row of 32 bfloat16: no two quarters of a read collide
constexpr int kWgSlot = 16 * kWgPitch;         // one part of one tile of 16 rows

template <int KW, int NPT, bool TAIL>
struct WgradRow {
    const SynapseWgrad& p;
    static constexpr int kSlots = 3 + 3 * NPT; // three parts of the gradient and of every tile of the input
    char* lds;                                 // kSlots slots of this wave
    __amdgpu_buffer_rsrc_t src, grd;
    int col, co0, ho, hin, pair0, t_lo, t_hi, lane;
    syn_f4 acc[KW][NPT];

    // byte offset of the gradient row of channel co0 + r / of the input row of pair pair0 + r at column 0, or none
    __device__ __forceinline__ int grad_row(int r) const {
        return co0 + r < p.Co ? ((co0 + r) * p.Ho + ho) * p.Wo * col : kOutOfRange;
    }
    __device__ __forceinline__ int pair_row(int r) const {
        const int pr = pair0 + r, ci = pr / p.kh, row = hin + (pr - ci * p.kh) * p.dh - p.ph;
        return (pr < p.Ci * p.kh && (unsigned)row < (unsigned)p.H) ? (ci * p.H + row) * p.W * col : kOutOfRange;
    }
    // steps t .. t + 3 of the pixel (or column) x of such a row, to be moved into place (SynQuad) where they are used
    __device__ __forceinline__ float4 grad_at(int row, int wo, const SynQuad& tq) const {
        return buf_load4<false>(
            grd, (tq.any() && row != kOutOfRange && (unsigned)wo < (unsigned)p.Wo) ? row + wo * col + tq.t_load * 4 : kOutOfRange);
    }
    __device__ __forceinline__ float4 pair_at(int row, int c, const SynQuad& tq) const {
        return buf_load4<false>(src, (tq.any() && row != kOutOfRange) ? row + c * col + tq.t_load * 4 : kOutOfRange);
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int x = 0; x < KW; ++x)
#pragma unroll
            for (int pt = 0; pt < NPT; ++pt) acc[x][pt] = syn_f4{0.f, 0.f, 0.f, 0.f};
    }
    // the wave's own LDS: its instructions run in order, the fences keep the compiler to that order
    __device__ __forceinline__ static void settle() {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // Lane l holds a quad of steps 4 (l % 8) of row l / 8 (+ 8 in the second quad); the operand's lane (kk, j) takes
    // steps 8 kk .. 8 kk + 7 of row j.
    __device__ __forceinline__ void put(int slot, int half, uint2 v) const {
        *reinterpret_cast<uint2*>(lds + slot * kWgSlot + ((lane >> 3) + 8 * half) * kWgPitch + (lane & 7) * 8) = v;
    }
    __device__ __forceinline__ uint4 get(int slot) const {
        return *reinterpret_cast<const uint4*>(lds + slot * kWgSlot + (lane & 15) * kWgPitch + (lane >> 4) * 16);
    }
    __device__ __forceinline__ static float4 scaled(float4 v) {
        return make_float4(v.x * kSplitScale, v.y * kSplitScale, v.z * kSplitScale, v.w * kSplitScale);
    }
    __device__ __forceinline__ void put_parts(int slot, const float4 (&raw)[2], const SynQuad& tq) const {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float4 v = scaled(tq.template place<TAIL>(raw[h]));
            uint2 part;
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                part.x = t < 2 ? round_pair(v.x, v.y) : bf16_pair(v.x, v.y);
                part.y = t < 2 ? round_pair(v.z, v.w) : bf16_pair(v.z, v.w);
                put(slot + t, h, part);
            }
        }
    }

    __device__ __forceinline__ void split_products() {
        clear();
        int g_row[2], q_row[NPT][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            g_row[h] = grad_row((lane >> 3) + 8 * h);
#pragma unroll
            for (int pt = 0; pt < NPT; ++pt) q_row[pt][h] = pair_row(16 * pt + (lane >> 3) + 8 * h);
        }
        for (int t0 = t_lo; t0 < t_hi; t0 += 32) {
            SynQuad tq;
            tq.template set<TAIL>(t0 + 4 * (lane & 7), t_hi);
            float4 raw_g[2], raw_q[NPT][2];
            auto fetch = [&](int c) {
#pragma unroll
                for (int h = 0; h < 2; ++h) raw_g[h] = grad_at(g_row[h], c + p.pw, tq);
#pragma unroll
                for (int pt = 0; pt < NPT; ++pt)
#pragma unroll
                    for (int h = 0; h < 2; ++h) raw_q[pt][h] = pair_at(q_row[pt][h], c, tq);
            };
            // gw[x]: the gradient at pixel c + pw - x for the column c at hand; gw[0] arrives with the column
            uint4 gw[KW][3];
            float4 first[KW][2];
#pragma unroll
            for (int x = KW - 1; x >= 1; --x)
#pragma unroll
                for (int h = 0; h < 2; ++h) first[x][h] = grad_at(g_row[h], p.pw - x, tq);
#pragma unroll
            for (int x = KW - 1; x >= 1; --x) {
                put_parts(0, first[x], tq);
                settle();
#pragma unroll
                for (int t = 0; t < 3; ++t) gw[x][t] = get(t);
                settle();
            }
            fetch(0);
            for (int c = 0; c < p.W; ++c) {
                const unsigned flip = (c & 1) ? 0x80008000u : 0u;
                const float back = (c & 1) ? -kSplitProductScale : kSplitProductScale;
                auto flipped = [&](uint4 v) { return make_uint4(v.x ^ flip, v.y ^ flip, v.z ^ flip, v.w ^ flip); };
                put_parts(0, raw_g, tq);
                unsigned low = 0u;
#pragma unroll
                for (int pt = 0; pt < NPT; ++pt)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const float4 v = raw_q[pt][h] = tq.template place<TAIL>(raw_q[pt][h]);
                        low |= __float_as_uint(v.x) | __float_as_uint(v.y) | __float_as_uint(v.z) | __float_as_uint(v.w);
                    }
                const bool more = __any((low & 0xffffu) != 0u);          // more than bfloat16 holds
#pragma unroll
                for (int pt = 0; pt < NPT; ++pt)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        float4 v = scaled(raw_q[pt][h]);
                        if (!more) {
                            put(3 + 3 * pt, h, make_uint2(bf16_pair(v.x, v.y), bf16_pair(v.z, v.w)));
                        } else {
                            uint2 part;
                            part.x = round_pair(v.x, v.y); part.y = round_pair(v.z, v.w);
                            put(3 + 3 * pt, h, part);
                            part.x = round_pair(v.x, v.y); part.y = round_pair(v.z, v.w);
                            put(4 + 3 * pt, h, part);
                            put(5 + 3 * pt, h, make_uint2(bf16_pair(v.x, v.y), bf16_pair(v.z, v.w)));
                        }
                    }
                settle();
                if (c + 1 < p.W) fetch(c + 1);                           // on its way during the products
#pragma unroll
                for (int t = 0; t < 3; ++t) gw[0][t] = get(t);
#pragma unroll
                for (int pt = 0; pt < NPT; ++pt) {
                    const uint4 q = flipped(get(3 + 3 * pt));
                    syn_f4 d[KW];
#pragma unroll
                    for (int x = 0; x < KW; ++x) d[x] = mfma_bf16(gw[x][2], q, syn_f4{0.f, 0.f, 0.f, 0.f});
                    if (more) {
                        const uint4 q1 = flipped(get(4 + 3 * pt)), q2 = flipped(get(5 + 3 * pt));
#pragma unroll
                        for (int x = 0; x < KW; ++x) {
                            d[x] = mfma_bf16(gw[x][0], q2, d[x]);
                            d[x] = mfma_bf16(gw[x][1], q1, d[x]);
                            d[x] = mfma_bf16(gw[x][0], q1, d[x]);
                        }
                    }
#pragma unroll
                    for (int x = 0; x < KW; ++x) d[x] = mfma_bf16(gw[x][1], q, d[x]);
#pragma unroll
                    for (int x = 0; x < KW; ++x) d[x] = mfma_bf16(gw[x][0], q, d[x]);
#pragma unroll
                    for (int x = 0; x < KW; ++x)
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[x][pt][i] = __fmaf_rn(back, d[x][i], acc[x][pt][i]);
                }
                settle();
#pragma unroll
                for (int x = KW - 1; x >= 1; --x)
#pragma unroll
                    for (int t = 0; t < 3; ++t) gw[x][t] = gw[x - 1][t];
            }
        }
    }
    // the same sums on the float32 instruction, 16 steps at a time
    __device__ __forceinline__ void float_products() {
        clear();
        const int g_row = grad_row(lane & 15);
        int q_row[NPT];
#pragma unroll
        for (int pt = 0; pt < NPT; ++pt) q_row[pt] = pair_row(16 * pt + (lane & 15));
        for (int t0 = t_lo; t0 < t_hi; t0 += 16) {
            SynQuad tq;
            tq.template set<TAIL>(t0 + 4 * (lane >> 4), t_hi);
            for (int c = 0; c < p.W; ++c) {
#pragma unroll
                for (int x = 0; x < KW; ++x) {
                    const float4 g = tq.template place<TAIL>(grad_at(g_row, c + p.pw - x, tq));
#pragma unroll
                    for (int pt = 0; pt < NPT; ++pt) {
                        const float4 q = tq.template place<TAIL>(pair_at(q_row[pt], c, tq));
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
        for (int x = 0; x < KW; ++x)
#pragma unroll
            for (int pt = 0; pt < NPT; ++pt)
#pragma unroll
                for (int i = 0; i < 4; ++i) bad = bad || !(fabsf(acc[x][pt][i]) < __builtin_inff());
        return __any(bad);
    }
};

template <int KW, int NPT, bool TAIL>
__global__ __launch_bounds__(kSynWaves * kWave) __attribute__((amdgpu_waves_per_eu(KW == 3 || NPT == 1 ? 3 : 2)))
void synapse_wgrad_row_kernel(const SynapseWgrad p) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int cobs = (p.Co + 15) / 16;
    // The waves of a workgroup, and neighbouring workgroups, take the channel blocks and passes of one share: they read
    // the same input rows and gradient rows at about the same time and find them in the L1 and L2.
    int b = xcd_contiguous(blockIdx.x, gridDim.x) * kSynWaves + wave;
    const int cob = b % cobs; b /= cobs;
    const int pass = b % p.passes; b /= p.passes;
    const int item = b % p.items;
    const int n = b / p.items;
    if (n >= p.N) return;
    const int co0 = cob * 16;
    const int tpart = item % p.tparts;
    const int ho = item / p.tparts;
    __shared__ __attribute__((aligned(16))) char lds[kSynWaves][WgradRow<KW, NPT, TAIL>::kSlots * kWgSlot];
    const int64_t in_plane = (int64_t)p.Ci * p.H * p.W * p.T;
    const int64_t out_plane = (int64_t)p.Co * p.Ho * p.Wo * p.T;
    WgradRow<KW, NPT, TAIL> w{p};
    w.lds = lds[wave];
    w.src = make_rsrc(p.in + (int64_t)n * in_plane, (unsigned)(in_plane * 4));
    w.grd = make_rsrc(p.grad_out + (int64_t)n * out_plane, (unsigned)(out_plane * 4));
    w.col = p.T * 4;
    w.lane = lane;
    w.co0 = co0; w.ho = ho; w.hin = ho * p.sh;
    w.pair0 = pass * NPT * 16;
    w.t_lo = tpart * p.tlen;
    w.t_hi = (w.t_lo + p.tlen) < p.T ? (w.t_lo + p.tlen) : p.T;
    w.split_products();
    if (w.not_finite()) w.float_products();
    // lane (q, j) of tile (x, pt): channels co0 + 4 q + i, pair 16 (pass NPT + pt) + j, tap x of its row
    float4* dst = reinterpret_cast<float4*>(p.partial) +
                  ((((int64_t)(n * cobs + cob) * p.items + item) * p.passes + pass) * (KW * NPT)) * kWave + lane;
#pragma unroll
    for (int x = 0; x < KW; ++x)
#pragma unroll
        for (int pt = 0; pt < NPT; ++pt)
            dst[(x * NPT + pt) * kWave] = make_float4(w.acc[x][pt][0], w.acc[x][pt][1], w.acc[x][pt][2], w.acc[x][pt][3]);
}

// grad_w[co][k] = sum over batch entries and items of the waves' tiles, in double, in a fixed order, in two
// launches: block (tile, chunk) adds the tiles of its chunk of the (batch entry, item) pairs -- sixteen partial sums
// (every sixteenth pair each), then those in turn -- into stage[chunk][tile]; the second launch adds the chunks and
// writes the gradient.  `tiles` tiles per wave and pass; tile tl holds taps k = 16 (pass tiles + tl) + j
// (row_kw == 0) or, for the row kernel, pairs 16 (pass npt + tl % npt) + j at tap x = tl / npt of their row:
// k = pair * row_kw + x.
constexpr int kWgradParts = 16;
constexpr int kWgradChunks = 32;
__global__ __launch_bounds__(kWgradParts * kWave) void synapse_wgrad_reduce_kernel(
        double* __restrict__ stage, const float* __restrict__ partial, int N, int Co, int items, int passes, int tiles) {
    __shared__ double sums[kWgradParts][kWave][4];
    const int lane = threadIdx.x & (kWave - 1), part = threadIdx.x >> 6;
    const int tl = blockIdx.x % tiles;
    int b = blockIdx.x / tiles;
    const int pass = b % passes;
    const int cob = b / passes;
    const int cobs = (Co + 15) / 16;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    const float4* src = reinterpret_cast<const float4*>(partial);
    const int64_t total = (int64_t)N * items;
    const int64_t per = (total + kWgradChunks - 1) / kWgradChunks;
    const int64_t lo = blockIdx.y * per, hi = (lo + per) < total ? (lo + per) : total;
    for (int64_t at = lo + part; at < hi; at += kWgradParts) {
        const int64_t n = at / items, item = at - n * items;
        const float4 v = src[((((n * cobs + cob) * items + item) * passes + pass) * tiles + tl) * kWave + lane];
        s[0] += v.x; s[1] += v.y; s[2] += v.z; s[3] += v.w;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[part][lane][i] = s[i];
    __syncthreads();
    if (part != 0) return;
    double* dst = stage + (((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * kWave + lane) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        double tot = 0.0;
        for (int pp = 0; pp < kWgradParts; ++pp) tot += sums[pp][lane][i];
        dst[i] = tot;
    }
}

__global__ __launch_bounds__(kWave) void synapse_wgrad_final_kernel(float* __restrict__ grad_w,
                                                                     const double* __restrict__ stage, int Co, int K,
                                                                     int passes, int tiles, int row_kw, int npt) {
    const int lane = threadIdx.x, q = lane >> 4, j = lane & 15;
    const int tl = blockIdx.x % tiles;
    int b = blockIdx.x / tiles;
    const int pass = b % passes;
    const int cob = b / passes;
    int k;
    if (row_kw == 0) {
        k = (pass * tiles + tl) * 16 + j;
    } else {
        const int x = tl / npt, pt = tl - x * npt;
        const int pair = (pass * npt + pt) * 16 + j;
        k = pair * row_kw + x;
        if (pair * row_kw >= K) k = K;                                   // a pair that does not exist
    }
    double tot[4] = {0.0, 0.0, 0.0, 0.0};
    for (int c = 0; c < kWgradChunks; ++c) {
        const double* src = stage + (((int64_t)c * gridDim.x + blockIdx.x) * kWave + lane) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) tot[i] += src[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int co = cob * 16 + 4 * q + i;
        if (co < Co && k < K) grad_w[(int64_t)co * K + k] = (float)tot[i];
    }
}

}  // namespace slayer

using namespace slayer;

namespace {

#ifndef SLAYER_SYN_PIX
#define SLAYER_SYN_PIX 4
#endif

// What a launch of the row kernels takes, in us: every wave walks its piece of an image row -- the columns of the split
// form with 32 (input channel, kernel row) pairs to a group, the blocks of four pixels of the float32 form with four -- and a
// group costs a wait for its loads and its share of the SIMD, which all waves there divide up.  Fitted to 1900 layers
// (2, 3 and 5 taps, 17 to 192 pairs, 3 to 64 output channels, 1 to 64 samples of 8x8 to 34x34 pixels, 50 to 302 steps; real
// values times real weights) with an error of 12 to 15 % for the split and 13 to 22 % for the float32 form.
// Split form over float32 form for 500 layers of these ranges that it decides for the former, margins of the caller included,
// mean / 95 % of the layers / largest:
//            spikes x quantised     real x quantised       real x real
//   2 taps   0.60 / 0.84 / 0.97     0.76 / 1.01 / 1.12     0.85 / 1.18 / 1.27
//   3 taps   0.52 / 0.77 / 1.11     0.72 / 0.99 / 1.29     0.85 / 1.16 / 1.40
//   5 taps   0.42 / 0.68 / 0.74     0.60 / 0.90 / 1.05     0.75 / 1.11 / 1.28
// Taken always from 17 pairs on, the split form lost up to 2.8 times on single samples of small images, up to 1.7
// times with badly filled groups (5x5, 40 pairs, real x real 195 us against 141).
double row_form_time(bool split, const SynapseConv& p, int64_t row_tiles, int pieces) {
    struct Cost { double launch, step, wait, rate, tail; };               // tail: rows that end inside a quad
    static constexpr Cost costs[2][3] = {{{0.0, 2.0, 0.21, 0.645, 0.85}, {4.5, 0.0, 0.10, 0.96, 0.71}, {1.0, 3.25, 0.62, 1.26, 0.69}},
                                         {{1.7, 0.54, 0.03, 1.10, 0.70}, {0.0, 0.51, 0.30, 1.14, 0.63}, {0.0, 0.38, 0.71, 1.28, 0.92}}};
    const Cost& c = costs[split][p.kw == 5 ? 2 : p.kw - 2];
    const int pixels = (p.Wo + pieces - 1) / pieces, pairs = p.Ci * p.kh;
    const int steps = split ? pixels + p.kw - 1 : (pixels + 3) / 4;
    const int groups = split ? (pairs + 31) / 32 : (pairs + 3) / 4;
    const double load = (double)(row_tiles * pieces) / 1024;              // waves per SIMD
    return c.launch + steps * (c.step + groups * (c.wait + c.rate * (load > 1 ? load : 1))) * (p.T % 4 ? 1 + c.tail : 1);
}

// One launch of the convolution kernels for the geometry in p (tensors, sizes, taps and sub-lattices filled in by the
// caller): the row kernel for unit stride and dilation along the image row with 2, 3 or 5 taps per row, else the
// one-pixel kernel with as many tap groups in flight as the filter has, up to six.  A filter without taps (K = 0)
// clears its outputs.
int launch_synapse_conv(SynapseConv p, bool streaming, hipStream_t st) {
    // Non-temporal stores only for the classes of a transposed convolution, which leave every line they touch
    // unfinished for the next launch.  A plain convolution finishes the lines that two of its tiles share within
    // microseconds, and the L2 puts the pieces together if it is allowed to keep them: [32,8,32,32,300] -> 16 channels
    // forward 378 -> 329 us with cached stores (the transposed 4x4 stride-2 classes 251 -> 288 us).
    if (p.oys == 1 && p.oxs == 1) streaming = false;
    constexpr int kRowPix = SLAYER_SYN_PIX;
    const int64_t K = (int64_t)p.Ci * p.kh * p.kw;
    p.K = (int)K;
    p.ttiles = (p.T + kSynTile - 1) / kSynTile;
    // blocks of four neighbouring pixels that share their input columns: unit stride and dilation along the row
    const bool rows = p.sw == 1 && p.dw == 1 && (p.kw == 2 || p.kw == 3 || p.kw == 5) && p.Wo >= kRowPix;
    // enough waves for four rounds of the chip (16 waves on each of 256 compute units), so that the last, partly
    // filled round weighs little; image rows cut into as few pieces as that takes
    const int64_t cobs = (p.Co + 15) / 16;
    const int64_t base = (int64_t)p.N * cobs * p.Ho * p.ttiles;
    int wsplit = 1;
    while (base * wsplit < 16 * 1024 && wsplit * 2 * (rows ? kRowPix : 1) <= p.Wo) wsplit *= 2;
    p.wsplit = wsplit;
    const int64_t items = (int64_t)p.Ho * wsplit * p.ttiles;
    if (items > 0x7fffffffLL) return SLAYER_ERANGE;
    p.items = (int)items;
    const int64_t blocks = p.N * cobs * ((items + kSynWaves - 1) / kSynWaves);
    if (blocks > 0x7fffffffLL) return SLAYER_ERANGE;
    const bool tail = (p.T % 4) != 0;                                     // rows that end inside a quad
    const dim3 grid((unsigned)blocks), block(kSynWaves * kWave);
    // The split form where it is about as fast with both operands real, its worst case (row_form_time), from 17 pairs
    // on, and if the parts of 16 channels' weights fit LDS.  A piece of an image row visits kw - 1 columns more than it has
    // pixels: rows are cut while there are few waves, for five taps (two waves per SIMD) below 1024 only
    // ([4,16,16,16,300] -> 64 channels 182 us with 2560 waves, 140 with 1280).
    const int pairs = p.Ci * p.kh;
    const int g32 = (pairs + 31) / 32;
    const size_t split_lds = (size_t)g32 * p.kw * 3 * 1024;
    const size_t row_lds = (size_t)((pairs + 3) / 4) * 4 * (p.kw * 16 * sizeof(float) + 2 * sizeof(int));
    int pieces = 1;
    while (base * pieces < (p.kw == 5 ? 1024 : 6144) && p.Wo >= 16 * pieces) pieces *= 2;
    // In all but small launches a margin for what it gains with spikes and quantised weights, which the host cannot see:
    // layers estimated at 1.0 to 1.1 of the float32 form take 0.5 to 0.7 of it with both, 0.8 to 1.0 with one, 1.0 to 1.15 with
    // neither.
    const bool small = base * pieces < 640;
    const double margin = p.kw == 2 ? (small ? 1.1 : 1.2) : small ? 1.0 : p.kw == 3 ? 1.12 : 1.07;
    if (rows && pairs > 16 && split_lds <= 96 * 1024 &&
        (row_lds > 64 * 1024 || row_form_time(true, p, base, pieces) <= margin * row_form_time(false, p, base, wsplit))) {
        // Workgroups of four waves: the registers hold three of them on a CU (five taps: two), but one of eight.  Eight where the
        // LDS has room for one workgroup only and there are more than four waves to a CU.  Both operands real, us, float32
        // form / four / eight waves: 3x3 on [5,43,31,31,64] -> 40 channels 127 / 153 / 192, [2,43,32,32,300] -> 27 144 / 159 /
        // 215, 5x5 on [10,25,11,11,100] -> 2 97 / 98 / 128; with room for one, 5x5 on [1,33,35,35,300] -> 3 (700 waves)
        // 249 / 166 / 220, 3x3 on [3,86,23,23,159] -> 47 (1242 waves) 758 / 1006 / 553.
        const int waves = 2 * (split_lds + 4 * g32 * 32 * sizeof(int)) > 160 * 1024 && base * pieces > 4 * 256 ? 8 : 4;
        p.wsplit = pieces;
        p.KG = g32;
        const int64_t all = (int64_t)p.Ho * pieces * p.ttiles;
        const int64_t wgs = p.N * cobs * ((all + waves - 1) / waves);
        if (all > 0x7fffffffLL || wgs * waves > 0x3fffffffLL) return SLAYER_ERANGE;
        p.items = (int)all;
        const dim3 sgrid((unsigned)wgs), sblock((unsigned)(waves * kWave));
        const size_t bytes = split_lds + (size_t)waves * g32 * 32 * sizeof(int);
#define SLAYER_SYN_SPLIT(KW)                                                                                        \
        do {                                                                                                             \
            if (tail) { if (streaming) hipLaunchKernelGGL((synapse_conv_split_kernel<KW, true, true>), sgrid, sblock, bytes, st, p); \
                        else hipLaunchKernelGGL((synapse_conv_split_kernel<KW, false, true>), sgrid, sblock, bytes, st, p); } \
            else { if (streaming) hipLaunchKernelGGL((synapse_conv_split_kernel<KW, true, false>), sgrid, sblock, bytes, st, p); \
                   else hipLaunchKernelGGL((synapse_conv_split_kernel<KW, false, false>), sgrid, sblock, bytes, st, p); } \
        } while (0)
        if (p.kw == 2) SLAYER_SYN_SPLIT(2);
        else if (p.kw == 3) { SLAYER_SYN_SPLIT(3); }
        else SLAYER_SYN_SPLIT(5);
#undef SLAYER_SYN_SPLIT
        return (int)hipGetLastError();
    }
    if (rows) {
        p.KG = (pairs + 3) / 4;                                           // groups of four (channel, kernel row) pairs
        if (row_lds > 64 * 1024) return SLAYER_ERANGE;
#define SLAYER_SYN_ROW_T(KERNEL, KW)                                                                      \
        do {                                                                                             \
            if (streaming) hipLaunchKernelGGL((KERNEL<KW, kRowPix, true>), grid, block, row_lds, st, p);  \
            else hipLaunchKernelGGL((KERNEL<KW, kRowPix, false>), grid, block, row_lds, st, p);           \
        } while (0)
#define SLAYER_SYN_ROW(KW)                                                                                \
        do { if (tail) SLAYER_SYN_ROW_T(synapse_conv_row_tail_kernel, KW); else SLAYER_SYN_ROW_T(synapse_conv_row_kernel, KW); } while (0)
        if (p.kw == 2) SLAYER_SYN_ROW(2); else if (p.kw == 3) SLAYER_SYN_ROW(3); else SLAYER_SYN_ROW(5);
#undef SLAYER_SYN_ROW_T
#undef SLAYER_SYN_ROW
        return (int)hipGetLastError();
    }
    const int groups = (int)((K + 3) / 4);
    const int chunk = groups <= 1 ? 1 : (groups == 2 ? 2 : kSynChunk);
    p.KG = (groups + chunk - 1) / chunk * chunk;
    const size_t lds = (size_t)p.KG * 4 * (16 * sizeof(float) + 3 * sizeof(int));
    if (lds > 64 * 1024) return SLAYER_ERANGE;
#define SLAYER_SYN_ONE(S, TL, CH) hipLaunchKernelGGL((synapse_conv_kernel<S, TL, CH>), grid, block, lds, st, p)
#define SLAYER_SYN_CH(S, TL) \
    do { if (chunk == 1) SLAYER_SYN_ONE(S, TL, 1); else if (chunk == 2) SLAYER_SYN_ONE(S, TL, 2); else SLAYER_SYN_ONE(S, TL, kSynChunk); } while (0)
    if (streaming) { if (tail) SLAYER_SYN_CH(true, true); else SLAYER_SYN_CH(true, false); }
    else { if (tail) SLAYER_SYN_CH(false, true); else SLAYER_SYN_CH(false, false); }
#undef SLAYER_SYN_CH
#undef SLAYER_SYN_ONE
    return (int)hipGetLastError();
}

// the most taps of a filter row of k taps that pixels of one residue (mod stride) meet in a transposed convolution
int most_taps_per_residue(int k, int stride, int pad, int dil) {
    int most = 0;
    for (int r = 0; r < stride; ++r) {
        int found = 0;
        for (int y = 0; y < k; ++y) found += (r + pad - y * dil) % stride == 0;
        most = found > most ? found : most;
    }
    return most;
}

// The one-channel form (synapse_plane_kernel) for a plain convolution (spread = false: p as for
// launch_synapse_conv) or for the gradient of its input (spread = true: p.in the gradient of the output [H][W],
// p.out the gradient of the input [Ho][Wo], strides, padding and dilation those of the convolution).
// false: not a geometry it takes.
bool launch_synapse_plane(const SynapseConv& p, bool spread, bool streaming, hipStream_t st, int* code) {
    const int64_t quads = (p.T + 3) / 4;
    const int64_t blocks = ((int64_t)p.Wo * quads + kPlaneThreads - 1) / kPlaneThreads;
    if (p.Ci != 1 || p.Co != 1 || p.N > 65535 || blocks > 0x7fffffffLL || p.kh * p.kw > 1024) return false;
    const int ny = spread ? most_taps_per_residue(p.kh, p.sh, p.ph, p.dh) : 0;
    const int nx = spread ? most_taps_per_residue(p.kw, p.sw, p.pw, p.dw) : 0;
    const size_t lds = ((size_t)p.kh * p.kw + 2 * ((size_t)p.sh * ny + (size_t)p.sw * nx)) * 4;
    if (lds > 48 * 1024) return false;
    const int rows = spread ? kPlaneRowsSpread : kPlaneRowsSum;
    if ((p.Ho + rows - 1) / rows > 65535) return false;                   // grid.y
    const dim3 grid((unsigned)blocks, (unsigned)((p.Ho + rows - 1) / rows), (unsigned)p.N), block(kPlaneThreads);
    const bool tail = (p.T % 4) != 0;
#define SLAYER_SYN_PLANE(SP, S, TL)                                                                                      \
    hipLaunchKernelGGL((synapse_plane_kernel<SP, S, TL, (SP ? kPlaneRowsSpread : kPlaneRowsSum)>), grid, block, lds, st, p, \
                       (int)quads, ny, nx)
#define SLAYER_SYN_PLANE_T(SP, S) do { if (tail) SLAYER_SYN_PLANE(SP, S, true); else SLAYER_SYN_PLANE(SP, S, false); } while (0)
    if (spread) { if (streaming) SLAYER_SYN_PLANE_T(true, true); else SLAYER_SYN_PLANE_T(true, false); }
    else { if (streaming) SLAYER_SYN_PLANE_T(false, true); else SLAYER_SYN_PLANE_T(false, false); }
#undef SLAYER_SYN_PLANE_T
#undef SLAYER_SYN_PLANE
    *code = (int)hipGetLastError();
    return true;
}

// the taps y of a filter row that output pixels of residue r (mod stride) meet in a transposed convolution:
// (r + pad - y * dil) divisible by stride; they are y_last, y_last - step, ... (count of them), and the source
// coordinate of y_last for the first pixel of the class, (r + pad - y_last * dil) / stride, is `first`
struct TapClass { int count, y_last, step, first; };
TapClass tap_class(int r, int k, int stride, int pad, int dil) {
    TapClass c{0, 0, 1, 0};
    int y_first = -1;
    for (int y = 0; y < k; ++y) {
        if ((r + pad - y * dil) % stride != 0) continue;
        if (c.count == 0) y_first = y;
        else if (c.count == 1) c.step = y - y_first;
        c.y_last = y;
        ++c.count;
    }
    if (c.count) {
        const int num = r + pad - c.y_last * dil;                         // divisible by stride, of either sign
        c.first = num / stride;
    }
    return c;
}

}  // namespace

extern "C" int slayer_conv_synapse(float* out, const float* in, const float* weight,
                                   int64_t N, int64_t Ci, int64_t Co, int64_t H, int64_t W, int64_t T,
                                   int64_t kh, int64_t kw, int64_t stride_h, int64_t stride_w,
                                   int64_t pad_h, int64_t pad_w, int64_t dil_h, int64_t dil_w, void* stream) {
    if (N < 0 || Ci < 1 || Co < 1 || H < 1 || W < 1 || T < 0 || kh < 1 || kw < 1 || stride_h < 1 || stride_w < 1 ||
        pad_h < 0 || pad_w < 0 || dil_h < 1 || dil_w < 1)
        return SLAYER_EINVAL;
    const int64_t Ho = (H + 2 * pad_h - dil_h * (kh - 1) - 1) / stride_h + 1;
    const int64_t Wo = (W + 2 * pad_w - dil_w * (kw - 1) - 1) / stride_w + 1;
    if (Ho < 1 || Wo < 1) return SLAYER_EINVAL;
    if (N == 0 || T == 0) return 0;
    if (!out || !in || !weight) return SLAYER_ENULL;
    // 32-bit byte offsets inside one batch entry; rows of any length from four steps on (16-byte accesses at
    // dword-aligned addresses)
    if (T < 4) return SLAYER_ERANGE;
    const int64_t K = Ci * kh * kw, lim = (int64_t)1 << 31;
    if (Ci * H * W * T * 4 >= lim || Co * Ho * Wo * T * 4 >= lim || K > 4096 || pad_h > 4096 || pad_w > 4096 ||
        H * stride_h > (1 << 20) || W * stride_w > (1 << 20))
        return SLAYER_ERANGE;
    SynapseConv p;
    p.out = out; p.in = in; p.weight = weight;
    p.N = (int)N; p.Ci = (int)Ci; p.Co = (int)Co; p.H = (int)H; p.W = (int)W; p.Ho = (int)Ho; p.Wo = (int)Wo; p.T = (int)T;
    p.kh = (int)kh; p.kw = (int)kw; p.sh = (int)stride_h; p.sw = (int)stride_w; p.ph = (int)pad_h; p.pw = (int)pad_w;
    p.dh = (int)dil_h; p.dw = (int)dil_w;
    p.kh_full = p.kh; p.kw_full = p.kw; p.ky0 = p.kx0 = 0; p.kys = p.kxs = 1;
    p.Ho_full = p.Ho; p.Wo_full = p.Wo; p.oy0 = p.ox0 = 0; p.oys = p.oxs = 1;
    const bool streaming = N * Co * Ho * Wo * T * 4 > ((int64_t)64 << 20);
    int code = 0;
    if (launch_synapse_plane(p, false, streaming, (hipStream_t)stream, &code)) return code;
    return launch_synapse_conv(p, streaming, (hipStream_t)stream);
}

namespace {

// The form of the weight-gradient kernels for a geometry: the row kernel (tiles of 16 (channel, kernel row) pairs,
// row_kw taps each) for unit stride and dilation along the image row with 3 or 5 taps per row, else tiles of 16
// taps; `tiles` accumulator tiles per wave and pass; the shares the time axis is cut into.
struct WgradForm { int row_kw, npt, tiles; };
WgradForm wgrad_form(int64_t Ci, int64_t kh, int64_t kw, int64_t stride_w, int64_t dil_w) {
    WgradForm f;
    if (stride_w == 1 && dil_w == 1 && (kw == 3 || kw == 5)) {
        const int64_t pairs = Ci * kh;
        f.row_kw = (int)kw;
        f.npt = pairs <= 16 ? 1 : 2;
        f.tiles = f.row_kw * f.npt;
    } else {
        const int64_t K = Ci * kh * kw;
        f.row_kw = 0;
        f.npt = 0;
        f.tiles = K <= 16 ? 1 : (K <= 32 ? 2 : 5);
    }
    return f;
}
void wgrad_shape(int64_t N, int64_t Ci, int64_t Co, int64_t Ho, int64_t T, int64_t kh, int64_t kw, const WgradForm& f,
                 SynapseWgrad& p) {
    if (f.row_kw) p.passes = (int)((Ci * kh + 16 * f.npt - 1) / (16 * f.npt));
    else p.passes = (int)((Ci * kh * kw + 16 * f.tiles - 1) / (16 * f.tiles));
    // Shares of whole visits of 32 steps, about eight thousand waves: a wave's set-up (the gradient window) is paid once per
    // share ([16,32,16,16,300] -> 64 channels 310 us with 4096 waves, 285 with 8192).  A row of up to 16 pairs has few
    // products to a visit and is bound by its loads, and a line that two visits of one share have in common is gone
    // from the caches when the second one comes, while the waves of neighbouring shares find it there: one visit a
    // share, up to 32768 waves (float32 kernel before / 8192 / 32768 waves: [32,4,32,32,300] -> 16 channels 237 / 280 / 206 us,
    // [64,1,32,32,300] -> 16 383 / 445 / 313, [8,4,64,64,300] -> 64 904 / 1008 / 685, 5x5 [32,2,32,32,300] -> 16
    // 303 / 260 / 198, and where rows are whole lines [32,4,32,32,256] -> 16 147 / 147 / 146, [128,4,32,32,64] -> 16
    // 167 / 176 / 177).
    const int64_t waves = f.npt == 1 ? 32768 : 8192;
    const int64_t base = N * ((Co + 15) / 16) * Ho;
    const int64_t visits = (T + 31) / 32;
    int64_t parts = (waves + base - 1) / base;
    parts = parts > visits ? visits : (parts < 1 ? 1 : parts);
    const int64_t len = (visits + parts - 1) / parts * 32;
    p.tparts = (int)((T + len - 1) / len);
    p.tlen = (int)len;
    p.items = (int)(Ho * p.tparts);
}

}  // namespace

extern "C" int64_t slayer_conv_synapse_wgrad_workspace(int64_t N, int64_t Ci, int64_t Co, int64_t H, int64_t W,
                                                       int64_t T, int64_t kh, int64_t kw, int64_t stride_h,
                                                       int64_t pad_h, int64_t dil_h) {
    if (N < 0 || Ci < 1 || Co < 1 || H < 1 || W < 1 || T < 0 || kh < 1 || kw < 1 || stride_h < 1 || pad_h < 0 ||
        dil_h < 1)
        return SLAYER_EINVAL;
    const int64_t Ho = (H + 2 * pad_h - dil_h * (kh - 1) - 1) / stride_h + 1;
    if (Ho < 1) return SLAYER_EINVAL;
    const int64_t K = Ci * kh * kw;
    if (K > 4096 || Ho > (1 << 20) || T > (1 << 24)) return SLAYER_ERANGE;
    // enough for either form of the kernel (which one runs depends on stride and dilation along the image row)
    int64_t need = 0;
    for (int64_t stride_w : {1, 2}) {
        const WgradForm f = wgrad_form(Ci, kh, kw, stride_w, 1);
        SynapseWgrad p;
        wgrad_shape(N, Ci, Co, Ho, T, kh, kw, f, p);
        const int64_t floats = (N * p.items + 2 * kWgradChunks) * ((Co + 15) / 16) * p.passes * f.tiles * 256;
        need = floats > need ? floats : need;
    }
    return need;
}

extern "C" int slayer_conv_synapse_wgrad(float* grad_weight, const float* grad_out, const float* in,
                                         int64_t N, int64_t Ci, int64_t Co, int64_t H, int64_t W, int64_t T,
                                         int64_t kh, int64_t kw, int64_t stride_h, int64_t stride_w,
                                         int64_t pad_h, int64_t pad_w, int64_t dil_h, int64_t dil_w,
                                         float* workspace, int64_t workspace_floats, void* stream) {
    if (N < 0 || Ci < 1 || Co < 1 || H < 1 || W < 1 || T < 0 || kh < 1 || kw < 1 || stride_h < 1 || stride_w < 1 ||
        pad_h < 0 || pad_w < 0 || dil_h < 1 || dil_w < 1)
        return SLAYER_EINVAL;
    const int64_t Ho = (H + 2 * pad_h - dil_h * (kh - 1) - 1) / stride_h + 1;
    const int64_t Wo = (W + 2 * pad_w - dil_w * (kw - 1) - 1) / stride_w + 1;
    if (Ho < 1 || Wo < 1) return SLAYER_EINVAL;
    if (!grad_weight) return SLAYER_ENULL;
    const int64_t K = Ci * kh * kw, lim = (int64_t)1 << 31;
    hipStream_t st = (hipStream_t)stream;
    if (N == 0 || T == 0) return launch_zero_fill(grad_weight, Co * K, st);
    if (!grad_out || !in || !workspace) return SLAYER_ENULL;
    if (T < 4 || !aligned16(workspace)) return SLAYER_ERANGE;
    if (Ci * H * W * T * 4 >= lim || Co * Ho * Wo * T * 4 >= lim || K > 4096 || pad_h > 4096 || pad_w > 4096 ||
        H * stride_h > (1 << 20) || W * stride_w > (1 << 20) || Ho > (1 << 20) || T > (1 << 24))
        return SLAYER_ERANGE;
    SynapseWgrad p;
    p.partial = workspace; p.grad_out = grad_out; p.in = in;
    p.N = (int)N; p.Ci = (int)Ci; p.Co = (int)Co; p.H = (int)H; p.W = (int)W; p.Ho = (int)Ho; p.Wo = (int)Wo; p.T = (int)T;
    p.kh = (int)kh; p.kw = (int)kw; p.sh = (int)stride_h; p.sw = (int)stride_w; p.ph = (int)pad_h; p.pw = (int)pad_w;
    p.dh = (int)dil_h; p.dw = (int)dil_w;
    p.K = (int)K;
    const WgradForm f = wgrad_form(Ci, kh, kw, stride_w, dil_w);
    wgrad_shape(N, Ci, Co, Ho, T, kh, kw, f, p);
    const int64_t cobs = (Co + 15) / 16;
    // the waves' tiles, then the chunk sums of the first reduction launch (doubles)
    const int64_t tile_floats = N * cobs * p.items * p.passes * f.tiles * 256;
    const int64_t stage_floats = 2 * kWgradChunks * cobs * p.passes * f.tiles * 256;
    if (workspace_floats < tile_floats + stage_floats) return SLAYER_ERANGE;
    double* stage = reinterpret_cast<double*>(workspace + tile_floats);
    const int64_t blocks = N * cobs * ((p.items + kSynWaves - 1) / kSynWaves);
    if (blocks > 0x7fffffffLL || p.passes > 65535) return SLAYER_ERANGE;
    const int64_t row_blocks = (N * cobs * p.items * p.passes + kSynWaves - 1) / kSynWaves;
    if (row_blocks > 0x7fffffffLL / kSynWaves) return SLAYER_ERANGE;
    const dim3 grid((unsigned)blocks, (unsigned)p.passes), row_grid((unsigned)row_blocks), block(kSynWaves * kWave);
    const bool tail = (T % 4) != 0;                                       // rows that end inside a quad
#define SLAYER_WGRAD(NTT)                                                                                              \
    do {                                                                                                               \
        if (tail) hipLaunchKernelGGL((synapse_wgrad_kernel<NTT, true>), grid, block, NTT * 16 * 3 * sizeof(int), st, p); \
        else hipLaunchKernelGGL((synapse_wgrad_kernel<NTT, false>), grid, block, NTT * 16 * 3 * sizeof(int), st, p);    \
    } while (0)
#define SLAYER_WGRAD_ROW(KW, NPT)                                                                                      \
    do {                                                                                                               \
        if (tail) hipLaunchKernelGGL((synapse_wgrad_row_kernel<KW, NPT, true>), row_grid, block, 0, st, p);             \
        else hipLaunchKernelGGL((synapse_wgrad_row_kernel<KW, NPT, false>), row_grid, block, 0, st, p);                 \
    } while (0)
    if (f.row_kw == 3) { if (f.npt == 1) SLAYER_WGRAD_ROW(3, 1); else SLAYER_WGRAD_ROW(3, 2); }
    else if (f.row_kw == 5) { if (f.npt == 1) SLAYER_WGRAD_ROW(5, 1); else SLAYER_WGRAD_ROW(5, 2); }
    else if (f.tiles == 1) SLAYER_WGRAD(1);
    else if (f.tiles == 2) SLAYER_WGRAD(2);
    else SLAYER_WGRAD(5);
#undef SLAYER_WGRAD_ROW
#undef SLAYER_WGRAD
    const unsigned tile_blocks = (unsigned)(cobs * p.passes * f.tiles);
    hipLaunchKernelGGL(synapse_wgrad_reduce_kernel, dim3(tile_blocks, kWgradChunks), dim3(kWgradParts * kWave), 0, st,
                       stage, workspace, (int)N, (int)Co, p.items, p.passes, f.tiles);
    hipLaunchKernelGGL(synapse_wgrad_final_kernel, dim3(tile_blocks), dim3(kWave), 0, st, grad_weight, stage, (int)Co,
                       (int)K, p.passes, f.tiles, f.row_kw, f.npt);
    return (int)hipGetLastError();
}

// The gradient of the input of slayer_conv_synapse for any stride (and, read as a layer of its own, the transposed
// convolution): one plain convolution per residue class of the pixels of grad_in, see SynapseConv.
extern "C" int slayer_conv_synapse_input_grad(float* grad_in, const float* grad_out, const float* weight_t,
                                              int64_t N, int64_t Ci, int64_t Co, int64_t H, int64_t W, int64_t T,
                                              int64_t kh, int64_t kw, int64_t stride_h, int64_t stride_w,
                                              int64_t pad_h, int64_t pad_w, int64_t dil_h, int64_t dil_w, void* stream) {
    if (N < 0 || Ci < 1 || Co < 1 || H < 1 || W < 1 || T < 0 || kh < 1 || kw < 1 || stride_h < 1 || stride_w < 1 ||
        pad_h < 0 || pad_w < 0 || dil_h < 1 || dil_w < 1)
        return SLAYER_EINVAL;
    const int64_t Ho = (H + 2 * pad_h - dil_h * (kh - 1) - 1) / stride_h + 1;
    const int64_t Wo = (W + 2 * pad_w - dil_w * (kw - 1) - 1) / stride_w + 1;
    if (Ho < 1 || Wo < 1) return SLAYER_EINVAL;
    if (N == 0 || T == 0) return 0;
    if (!grad_in || !grad_out || !weight_t) return SLAYER_ENULL;
    if (T < 4) return SLAYER_ERANGE;
    const int64_t K = Co * kh * kw, lim = (int64_t)1 << 31;
    if (Ci * H * W * T * 4 >= lim || Co * Ho * Wo * T * 4 >= lim || K > 4096 || pad_h > 4096 || pad_w > 4096 ||
        dil_h > 4096 || dil_w > 4096 || H + pad_h >= (1 << 16) || W + pad_w >= (1 << 16) || stride_h > 16 || stride_w > 16)
        return SLAYER_ERANGE;
    SynapseConv p;
    p.out = grad_in; p.in = grad_out; p.weight = weight_t;
    // in the kernels' names: the source is the gradient of the output, the result the gradient of the input
    p.N = (int)N; p.Ci = (int)Co; p.Co = (int)Ci; p.H = (int)Ho; p.W = (int)Wo; p.T = (int)T;
    p.sh = p.sw = 1;
    p.kh_full = (int)kh; p.kw_full = (int)kw; p.Ho_full = (int)H; p.Wo_full = (int)W;
    p.oys = (int)stride_h; p.oxs = (int)stride_w;
    const bool streaming = N * Ci * H * W * T * 4 > ((int64_t)64 << 20);
    {
        SynapseConv q = p;                                                // one channel: every class in one launch
        q.Ho = (int)H; q.Wo = (int)W; q.kh = (int)kh; q.kw = (int)kw; q.sh = (int)stride_h; q.sw = (int)stride_w;
        q.ph = (int)pad_h; q.pw = (int)pad_w; q.dh = (int)dil_h; q.dw = (int)dil_w;
        int code = 0;
        if (launch_synapse_plane(q, true, streaming, (hipStream_t)stream, &code)) return code;
    }
    for (int ry = 0; ry < (int)stride_h && ry < (int)H; ++ry) {
        const TapClass cy = tap_class(ry, (int)kh, (int)stride_h, (int)pad_h, (int)dil_h);
        for (int rx = 0; rx < (int)stride_w && rx < (int)W; ++rx) {
            const TapClass cx = tap_class(rx, (int)kw, (int)stride_w, (int)pad_w, (int)dil_w);
            p.oy0 = ry; p.ox0 = rx;
            p.Ho = ((int)H - ry + (int)stride_h - 1) / (int)stride_h;
            p.Wo = ((int)W - rx + (int)stride_w - 1) / (int)stride_w;
            const bool none = cy.count == 0 || cx.count == 0;            // pixels no tap reaches: zeros
            // the taps in the order of rising source coordinate: from the last one down, a step of
            // step * dil / stride pixels of the source each
            p.kh = none ? 0 : cy.count; p.kw = none ? 0 : cx.count;
            p.ky0 = cy.y_last; p.kys = -cy.step; p.kx0 = cx.y_last; p.kxs = -cx.step;
            p.dh = cy.count > 1 ? cy.step * (int)dil_h / (int)stride_h : 1;
            p.dw = cx.count > 1 ? cx.step * (int)dil_w / (int)stride_w : 1;
            p.ph = -cy.first; p.pw = -cx.first;
            const int code = launch_synapse_conv(p, streaming, (hipStream_t)stream);
            if (code != 0) return code;
        }
    }
    return 0;
}
