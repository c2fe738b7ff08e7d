// Convolution synapse on time-innermost tensors.
//
// A SLAYER conv synapse is a spatial convolution applied at every time step (synapse/layer.py:297-323 in the
// reference: F.conv3d with a kernel of (kh, kw, 1) on [N, C, H, W, T]).  A library conv3d wants channels last: it
// transposes the tensor there and back around its kernel, three passes over tensors whose innermost axis is already
// the one the neuron kernels walk.  Here the tensors stay as they are.  Forward pass and input gradient run on the walking
// kernel (synapse_walk.hip); this file has the one-pixel kernel for the geometries that it does not take, the
// one-channel layers, the weight gradient and the entry points.
//
// One-pixel kernel: for an output pixel (n, h, w) and a tile of 64 time steps the [Co x 64] result is the [Co x K] weight matrix
// (K = Ci * kh * kw) times the [K x 64] matrix whose row k is the input row of tap k -- 64 consecutive floats of the input as it
// lies in memory.  One wavefront takes 16 output channels x 64 steps of one pixel at a time on the matrix cores
// (v_mfma_f32_16x16x4_f32: float32 operands, float32 accumulation) and walks along the image row, so neighbouring pixels find
// their shared input rows in the cache; a wave-wide load is four input rows of 256 bytes, a wave-wide store four output rows.
//
// Lane (kk, j) = (lane / 16, lane % 16) loads steps 4j .. 4j+3 of tap 4g + kk for tap group g: element e of that
// quad is the B operand of the e-th of four matrix products, whose column j stands for step 4j + e; lane (q, j) of a
// result then holds output channels 4q .. 4q+3 of step 4j + e, i.e. over e a quad of consecutive steps per channel.
#include "synapse.h"

namespace slayer {

int launch_zero_fill(float* p, int64_t n, hipStream_t stream);          // li.hip

constexpr int kSynChunk = 6;            // tap groups whose loads are in flight together (fewer for filters of a few taps)

// The gradient of the input of a convolution with strides (what conv_transpose3d computes, the ConvTranspose synapse
// of synapse/layer.py:513-560 in the reference) is one plain convolution per residue class of the output pixels: the
// pixels (ry + m sh, rx + m' sw) meet only the taps y with (ry + ph - y dh) divisible by sh (x likewise), and over
// m, m' those taps slide across the source with unit stride.  The walking kernel takes all classes in one launch where there
// is no dilation and up to four classes of rows; otherwise each class is a launch of its own on its sub-lattices of taps and of outputs,
// of the walking kernel or of the one below, a fraction 1 / (sh sw) of the taps each.
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

// grad_w[co][k] = sum over batch entries and items of the waves' tiles, in double, in a fixed order, in two
// launches: block (tile, chunk) adds the tiles of its chunk of the (batch entry, item) pairs -- sixteen partial sums
// (every sixteenth pair each), then those in turn -- into stage[chunk][tile]; the second launch adds the chunks and
// writes the gradient.  Up to kWgradFew pairs are one chunk, and its launch writes the gradient.  `tiles` tiles per wave and pass;
// tile tl holds taps k = 16 (pass tiles + tl) + j (map.npt == 0) or, for the walking kernel, triples (channel, line tap, row of the
// step) 16 (pass npt + tl % npt) + j at tap tl / npt of the walk.
struct WgradMap {
    int npt, pairs, XP, ss, kslide, wslide, wline;
    // tap of lane j of tile tl of a pass, or K where there is none
    __device__ __forceinline__ int tap(int K, int pass, int tiles, int tl, int j) const {
        if (npt == 0) return (pass * tiles + tl) * 16 + j;
        const int walked = tl / npt, pr = (pass * npt + tl - walked * npt) * 16 + j;
        const int ci = pr / (XP * ss), r = pr - ci * (XP * ss), x = r / ss;
        const int y = walked * ss + r - x * ss;
        return pr < pairs && y < kslide ? ci * XP * kslide + y * wslide + x * wline : K;
    }
    __device__ __forceinline__ void write(float* grad_w, const double (&tot)[4], int Co, int K, int cob, int pass, int tiles, int tl,
                                          int lane) const {
        const int k = tap(K, pass, tiles, tl, lane & 15);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int co = cob * 16 + 4 * (lane >> 4) + i;
            if (co < Co && k < K) grad_w[(int64_t)co * K + k] = (float)tot[i];
        }
    }
};
constexpr int kWgradParts = 16;
constexpr int kWgradChunks = 32;
// six a thread, a launch less ([1,3,8,5,201] -> 10 channels, 3x3: 14.2 -> 10.3 us with its shares); 16 a thread took up to 1.15 times
// as long as two launches
constexpr int kWgradFew = 96;
__global__ __launch_bounds__(kWgradParts * kWave) void synapse_wgrad_reduce_kernel(
        double* __restrict__ stage, float* __restrict__ grad_w, const float* __restrict__ partial, int N, int Co, int K, int items,
        int passes, int tiles, const WgradMap map) {
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
    const int64_t per = (total + gridDim.y - 1) / gridDim.y;
    const int64_t lo = blockIdx.y * per, hi = (lo + per) < total ? (lo + per) : total;
    for (int64_t at = lo + part; at < hi; at += kWgradParts) {
        // pair `at` of this block of channels: the blocks lie between the batch entries
        const int64_t row = cobs == 1 ? at : at + (at / items * (cobs - 1) + cob) * items;
        const float4 v = src[((row * passes + pass) * tiles + tl) * kWave + lane];
        s[0] += v.x; s[1] += v.y; s[2] += v.z; s[3] += v.w;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[part][lane][i] = s[i];
    __syncthreads();
    if (part != 0) return;
    double tot[4] = {0.0, 0.0, 0.0, 0.0};
    for (int pp = 0; pp < kWgradParts; ++pp)
#pragma unroll
        for (int i = 0; i < 4; ++i) tot[i] += sums[pp][lane][i];
    if (gridDim.y == 1) {
        map.write(grad_w, tot, Co, K, cob, pass, tiles, tl, lane);
        return;
    }
    double* dst = stage + (((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * kWave + lane) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[i] = tot[i];
}

__global__ __launch_bounds__(kWave) void synapse_wgrad_final_kernel(float* __restrict__ grad_w,
                                                                     const double* __restrict__ stage, int Co, int K,
                                                                     int passes, int tiles, const WgradMap map) {
    const int lane = threadIdx.x;
    const int tl = blockIdx.x % tiles;
    int b = blockIdx.x / tiles;
    const int pass = b % passes;
    const int cob = b / passes;
    double tot[4] = {0.0, 0.0, 0.0, 0.0};
    for (int c = 0; c < kWgradChunks; ++c) {
        const double* src = stage + (((int64_t)c * gridDim.x + blockIdx.x) * kWave + lane) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) tot[i] += src[i];
    }
    map.write(grad_w, tot, Co, K, cob, pass, tiles, tl, lane);
}

}  // namespace slayer

using namespace slayer;

namespace {

// Whether a filter is one of those taken, by its size alone: about 860 taps, 960 to 1024 of two, three or five columns without stride
// or dilation along the row.  The walking kernel takes 150 KB of LDS for them; the one-pixel kernel, where that does not take the
// geometry, at most 78 KB of a workgroup's 160.
bool filter_fits(const SynapseConv& p) {
    const int64_t pairs = (int64_t)p.Ci * p.kh, K = pairs * p.kw;
    if (p.sw == 1 && p.dw == 1 && (p.kw == 2 || p.kw == 3 || p.kw == 5) && p.Wo >= 4)
        return (pairs + 31) / 32 * p.kw * 3 <= 96 || (pairs + 3) / 4 * 4 * (p.kw * 64 + 8) <= 64 * 1024;
    const int64_t groups = (K + 3) / 4, chunk = groups <= 2 ? (groups < 1 ? 1 : groups) : kSynChunk;
    return (groups + chunk - 1) / chunk * chunk * 4 * 76 <= 64 * 1024;
}

// One launch of the convolution kernels for the geometry in p (tensors, sizes, taps and sub-lattices filled in by the
// caller): the walking kernel where it takes the geometry, else the one-pixel kernel with as many tap groups in flight as
// the filter has, up to six.  A filter without taps (K = 0) clears its outputs.
int launch_synapse_conv(SynapseConv p, bool streaming, hipStream_t st) {
    if (!filter_fits(p)) return SLAYER_ERANGE;
    int code = 0;
    if (launch_synapse_walk(p, st, &code)) return code;
    if (p.want && p.kh > 0 && p.kw > 0) return SLAYER_ERANGE;
    // Non-temporal stores only for the classes of a transposed convolution, which leave every line they touch
    // unfinished for the next launch.  A plain convolution finishes the lines that two of its tiles share within
    // microseconds, and the L2 puts the pieces together if it is allowed to keep them.
    if (p.oys == 1 && p.oxs == 1) streaming = false;
    const int64_t K = (int64_t)p.Ci * p.kh * p.kw;
    p.K = (int)K;
    p.ttiles = (p.T + kSynTile - 1) / kSynTile;
    // enough waves for four rounds of the chip (16 waves on each of 256 compute units), so that the last, partly
    // filled round weighs little; image rows cut into as few pieces as that takes
    const int64_t cobs = (p.Co + 15) / 16;
    const int64_t base = (int64_t)p.N * cobs * p.Ho * p.ttiles;
    int wsplit = 1;
    while (base * wsplit < 16 * 1024 && wsplit * 2 <= p.Wo) wsplit *= 2;
    p.wsplit = wsplit;
    const int64_t items = (int64_t)p.Ho * wsplit * p.ttiles;
    if (items > 0x7fffffffLL) return SLAYER_ERANGE;
    p.items = (int)items;
    const int64_t blocks = p.N * cobs * ((items + kSynWaves - 1) / kSynWaves);
    if (blocks > 0x7fffffffLL) return SLAYER_ERANGE;
    const bool tail = (p.T % 4) != 0;                                     // rows that end inside a quad
    const dim3 grid((unsigned)blocks), block(kSynWaves * kWave);
    const int groups = (int)((K + 3) / 4);
    const int chunk = groups <= 1 ? 1 : (groups == 2 ? 2 : kSynChunk);
    p.KG = (groups + chunk - 1) / chunk * chunk;
    const size_t lds = (size_t)p.KG * 4 * (16 * sizeof(float) + 3 * sizeof(int));
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
// coordinate of y_last for the first pixel of the class, (r + pad - y_last * dil) / stride, is `first`.  `step` is what
// lies between any two of them, also for a class of one: a step beyond either end of a class is outside the filter, by
// which the walking kernel tells the taps that a pixel does not have
struct TapClass { int count, y_last, step, first; };
TapClass tap_class(int r, int k, int stride, int pad, int dil) {
    int both = stride, rest = dil;                                        // their greatest common divisor
    while (rest) { const int next = both % rest; both = rest; rest = next; }
    TapClass c{0, 0, stride / both, 0};
    for (int y = 0; y < k; ++y) {
        if ((r + pad - y * dil) % stride != 0) continue;
        c.y_last = y;
        ++c.count;
    }
    if (c.count) {
        const int num = r + pad - c.y_last * dil;                         // divisible by stride, of either sign
        c.first = num / stride;
    }
    return c;
}

int conv_synapse(float* out, const float* in, const float* weight, int64_t N, int64_t Ci, int64_t Co, int64_t H, int64_t W, int64_t T,
                 int64_t kh, int64_t kw, int64_t stride_h, int64_t stride_w, int64_t pad_h, int64_t pad_w, int64_t dil_h, int64_t dil_w,
                 const WalkCut* want, void* stream) {
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
    p.want = want;
    const bool streaming = N * Co * Ho * Wo * T * 4 > ((int64_t)64 << 20);
    int code = 0;
    if (!want && launch_synapse_plane(p, false, streaming, (hipStream_t)stream, &code)) return code;
    return launch_synapse_conv(p, streaming, (hipStream_t)stream);
}

// The gradient of the input of slayer_conv_synapse for any stride (and, read as a layer of its own, the transposed
// convolution): one launch, or one plain convolution per residue class of the pixels of grad_in, see SynapseConv.
int conv_synapse_input_grad(float* grad_in, const float* grad_out, const float* weight_t, int64_t N, int64_t Ci, int64_t Co, int64_t H,
                            int64_t W, int64_t T, int64_t kh, int64_t kw, int64_t stride_h, int64_t stride_w, int64_t pad_h, int64_t pad_w,
                            int64_t dil_h, int64_t dil_w, const WalkCut* want, bool by_class, void* stream) {
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
    p.want = want;
    const bool streaming = N * Ci * H * W * T * 4 > ((int64_t)64 << 20);
    if (!want) {
        SynapseConv q = p;                                                // one channel: every class in one launch
        q.Ho = (int)H; q.Wo = (int)W; q.kh = (int)kh; q.kw = (int)kw; q.sh = (int)stride_h; q.sw = (int)stride_w;
        q.ph = (int)pad_h; q.pw = (int)pad_w; q.dh = (int)dil_h; q.dw = (int)dil_w;
        int code = 0;
        if (launch_synapse_plane(q, true, streaming, (hipStream_t)stream, &code)) return code;
    }
    // the plain convolution of one residue class
    auto one_class = [&](int ry, int rx) {
        const TapClass cy = tap_class(ry, (int)kh, (int)stride_h, (int)pad_h, (int)dil_h);
        const TapClass cx = tap_class(rx, (int)kw, (int)stride_w, (int)pad_w, (int)dil_w);
        p.oy0 = ry; p.ox0 = rx;
        p.Ho = ((int)H - ry + (int)stride_h - 1) / (int)stride_h;
        p.Wo = ((int)W - rx + (int)stride_w - 1) / (int)stride_w;
        const bool none = cy.count == 0 || cx.count == 0;                // pixels no tap reaches: zeros
        // the taps in the order of rising source coordinate: from the last one down, a step of
        // step * dil / stride pixels of the source each
        p.kh = none ? 0 : cy.count; p.kw = none ? 0 : cx.count;
        p.ky0 = cy.y_last; p.kys = -cy.step; p.kx0 = cx.y_last; p.kxs = -cx.step;
        p.dh = cy.count > 1 ? cy.step * (int)dil_h / (int)stride_h : 1;
        p.dw = cx.count > 1 ? cx.step * (int)dil_w / (int)stride_w : 1;
        p.ph = -cy.first; p.pw = -cx.first;
    };
    const int classes_h = (int)(stride_h < H ? stride_h : H), classes_w = (int)(stride_w < W ? stride_w : W);
    bool fits = true;
    for (int r = 0; r < classes_h * classes_w; ++r) { one_class(r / classes_w, r % classes_w); fits = fits && filter_fits(p); }
    if (!fits) return SLAYER_ERANGE;
    int code = 0;
    if (!by_class && dil_h == 1 && dil_w == 1 &&
        launch_synapse_walk_transposed(p, (int)kh, (int)kw, (int)stride_h, (int)stride_w, (int)pad_h, (int)pad_w, (hipStream_t)stream, &code))
        return code;
    for (int r = 0; r < classes_h * classes_w; ++r) {
        one_class(r / classes_w, r % classes_w);
        code = launch_synapse_conv(p, streaming, (hipStream_t)stream);
        if (code != 0) return code;
    }
    return 0;
}


// What a workspace holds at least, so that the sizes of layers that fill the chip stay what they were: `tiles` of sums per wave and
// pass and the shares of the time axis, of the one-pixel kernel (row_kw 0; these it runs with) or, for 3 or 5 taps along the image
// row without stride or dilation, of tiles of 16 (channel, kernel row) pairs, which no kernel has: the walking kernel cuts its line
// to what there is room for.
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
    // Shares of whole visits of 32 steps, about eight thousand waves, since a wave's start is paid once per share; layers of up to
    // 16 pairs, which have few products to a visit and are bound by their loads, one visit a share up to 32768 waves.
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

// The walking form of a geometry ([0]: rows, [1]: columns) in a workspace of `floats`, or false.  w: tensors, N, Co and T filled in.
bool wgrad_walk(WgradWalk& w, int Ci, const int (&k)[2], const int (&stride)[2], const int (&pad)[2], const int (&dil)[2],
                const int (&in)[2], const int (&out)[2], int64_t floats) {
    const int px = w.T * 4;
    auto taps = [&](int a) { return (k[a] == 1 || dil[a] == 1) && stride[a] <= 16 ? (k[a] + stride[a] - 1) / stride[a] : 0; };
    const bool down = taps(0) >= 1 && taps(0) <= 5, right = taps(1) >= 1 && taps(1) <= 5;
    if (!down && !right) return false;
    const int s = down && (!right || taps(0) >= taps(1)) ? 0 : 1, l = 1 - s;
    w.KS = taps(s) == 4 ? 5 : taps(s);
    w.in_ch = in[0] * in[1] * px; w.in_plane = Ci * w.in_ch;
    w.out_ch = out[0] * out[1] * px; w.out_plane = w.Co * w.out_ch;
    w.in_slide = s == 0 ? in[1] * px : px; w.in_line = s == 0 ? px : in[1] * px;
    w.out_slide = s == 0 ? out[1] * px : px; w.out_line = s == 0 ? px : out[1] * px;
    w.Hs = in[s]; w.Ws = in[l];
    w.quads = (w.T + 3) / 4;
    if ((int64_t)out[l] * w.quads > 0x3fffffffLL) return false;
    w.line_quads = out[l] * w.quads;
    w.ss = stride[s]; w.ls = stride[l];
    w.row0 = -pad[s]; w.S = out[s];
    w.c_lo = w.row0 + w.ss - 1 >= 0 ? 0 : -w.row0 / w.ss;
    w.c_hi = w.Hs - 1 - w.row0 < 0 ? 0 : (w.Hs - 1 - w.row0) / w.ss + 1;
    w.XP = k[l]; w.shift0 = -pad[l]; w.shift_step = dil[l];
    w.kslide = k[s]; w.kline = k[l];
    w.wslide = s == 0 ? k[1] : 1; w.wline = s == 0 ? 1 : k[1];
    w.pairs = Ci * w.XP * w.ss;
    w.npt = w.pairs <= 16 ? 1 : 2;
    w.passes = (w.pairs + 16 * w.npt - 1) / (16 * w.npt);
    // as many waves as the workspace has room for, and no more than the line has visits; few waves: pieces of the rows
    const int64_t cobs = (w.Co + 15) / 16, visits = (w.line_quads + 7) / 8;
    // The waves of a workgroup take neighbouring shares and leave one set of tiles: a quarter of the tiles to write and add, and
    // room for shares of one visit, which leaves no line to two visits of one wave.  [32,8,32,32,300] -> 16 channels 330 -> 290 us
    // (cold caches), 4x4 stride 2 194 -> 184, [16,16,20,18,128] -> 32 97 -> 86, 5x5 [16,32,12,12,150] -> 64 280 -> 252.  With many
    // blocks of channels and passes, and visits enough for all of them, these are what the waves of a workgroup had better share:
    // [16,32,16,16,300] -> 64, twelve of them, 268 us with the same operands in a workgroup, 274 without (cold caches 294, 307).  154
    // passes of nine blocks and passes or more: 1.00 of the time in the mean from 720 visits on (0.94 to 1.06), 1.03 to 1.32 with
    // fewer; up to eight 1.01 to 1.04 and five taps, which have enough products a load, 1.04 to 1.23 in all sizes.
    const int merged = cobs * w.passes <= 8 || w.KS == 5 || w.N * visits < 640 ? kSynWaves : 1;
    const int64_t room = (floats / (256 * cobs * w.passes * w.KS * w.npt) - 2 * kWgradChunks) / w.N;   // sets of tiles
    if (room < 1) return false;
    // The rows in pieces where that is fewer steps for the chip, which two waves to a SIMD fill: a piece has KS - 1 steps more than
    // it has rows, its start is worth about three, and every set of tiles is written and added.  800 layers like those of short_walk_time, spikes
    // and real values: what it decides for takes 1.02 times the better of the two in the mean.
    double least = 1e30;
    for (int pieces : {1, kSynWaves}) {
        const int64_t most = pieces == 1 ? room * merged : room, each = (visits + most - 1) / most, shares = (visits + each - 1) / each;
        const double load = (double)(w.N * cobs * w.passes * shares * pieces) / 2250;
        const int64_t sets = pieces == 1 ? (shares + merged - 1) / merged : shares;
        const double steps = (double)each * ((w.S + pieces - 1) / pieces + w.KS + 2) * (load > 1 ? load : 1) +
                             0.0003 * w.N * sets * cobs * w.passes * w.KS * w.npt;
        if (steps >= least) continue;
        least = steps;
        w.share_quads = (int)(8 * each);
        w.shares = (int)shares;
        w.pieces = pieces;
        w.sets = (int)sets;
    }
    return true;
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
    // enough for either form (stride and dilation along the image row are not known here)
    int64_t need = 0;
    for (int64_t stride_w : {1, 2}) {
        const WgradForm f = wgrad_form(Ci, kh, kw, stride_w, 1);
        SynapseWgrad p;
        wgrad_shape(N, Ci, Co, Ho, T, kh, kw, f, p);
        const int64_t floats = (N * p.items + 2 * kWgradChunks) * ((Co + 15) / 16) * p.passes * f.tiles * 256;
        need = floats > need ? floats : need;
    }
    // ... and for the walking form of few waves, a set of its tiles for every visit of the line, or 4096 of them in all: small layers have
    // more of these than the forms above have waves, and longer shares are a longer way for each wave ([1,1,16,15,168] -> 32 channels,
    // 2x2: 38 us with the shares that fit these forms, the kernel before the walk 15)
    const auto walked = [&](int64_t KS, int64_t pairs, int64_t pixels) {
        if (KS < 1 || KS > 5) return;
        KS = KS == 4 ? 5 : KS;
        const int64_t npt = pairs <= 16 ? 1 : 2, passes = (pairs + 16 * npt - 1) / (16 * npt), cobs = (Co + 15) / 16;
        const int64_t visits = (pixels * ((T + 3) / 4) + 7) / 8, waves = N * cobs * passes, most = (4096 + waves - 1) / (waves < 1 ? 1 : waves);
        const int64_t floats = (N * (visits < most ? visits : most) + 2 * kWgradChunks) * cobs * passes * KS * npt * 256;
        need = floats > need ? floats : need;
    };
    if (kh == 1 || dil_h == 1) walked((kh + stride_h - 1) / stride_h, Ci * kw * stride_h, W);   // the rows walked, the line of about W pixels
    walked(kw, Ci * kh, Ho);                                                                    // the columns, with stride 1
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
    const int64_t cobs = (Co + 15) / 16;
    const int64_t floats = slayer_conv_synapse_wgrad_workspace(N, Ci, Co, H, W, T, kh, kw, stride_h, pad_h, dil_h);
    auto reduce = [&](int items, int passes, int tiles, const WgradMap& map) {
        double* stage = reinterpret_cast<double*>(workspace + N * cobs * items * passes * tiles * 256);
        const unsigned tile_blocks = (unsigned)(cobs * passes * tiles);
        const bool few = N * items <= kWgradFew;
        hipLaunchKernelGGL(synapse_wgrad_reduce_kernel, dim3(tile_blocks, few ? 1 : kWgradChunks), dim3(kWgradParts * kWave), 0, st, stage,
                           grad_weight, workspace, (int)N, (int)Co, (int)K, items, passes, tiles, map);
        if (few) return (int)hipGetLastError();
        hipLaunchKernelGGL(synapse_wgrad_final_kernel, dim3(tile_blocks), dim3(kWave), 0, st, grad_weight, stage, (int)Co, (int)K,
                           passes, tiles, map);
        return (int)hipGetLastError();
    };
    WgradWalk w;
    w.partial = workspace; w.grad_out = grad_out; w.in = in;
    w.N = (int)N; w.Co = (int)Co; w.T = (int)T;
    const int ker[2] = {(int)kh, (int)kw}, str[2] = {(int)stride_h, (int)stride_w}, pad[2] = {(int)pad_h, (int)pad_w};
    const int dil[2] = {(int)dil_h, (int)dil_w}, size[2] = {(int)H, (int)W}, size_out[2] = {(int)Ho, (int)Wo};
    // (a workspace of fewer floats than are asked for now is cut to as far as it goes)
    if (wgrad_walk(w, (int)Ci, ker, str, pad, dil, size, size_out, workspace_floats < floats ? workspace_floats : floats)) {
        if (workspace_floats < (N * w.sets + 2 * kWgradChunks) * cobs * w.passes * w.KS * w.npt * 256) return SLAYER_ERANGE;
        const int code = launch_synapse_wgrad_walk(w, st);
        if (code != 0) return code;
        return reduce(w.sets, w.passes, w.KS * w.npt, {w.npt, w.pairs, w.XP, w.ss, w.kslide, w.wslide, w.wline});
    }
    SynapseWgrad p;
    p.partial = workspace; p.grad_out = grad_out; p.in = in;
    p.N = (int)N; p.Ci = (int)Ci; p.Co = (int)Co; p.H = (int)H; p.W = (int)W; p.Ho = (int)Ho; p.Wo = (int)Wo; p.T = (int)T;
    p.kh = (int)kh; p.kw = (int)kw; p.sh = (int)stride_h; p.sw = (int)stride_w; p.ph = (int)pad_h; p.pw = (int)pad_w;
    p.dh = (int)dil_h; p.dw = (int)dil_w;
    p.K = (int)K;
    const WgradForm f = wgrad_form(Ci, kh, kw, 2, 1);                     // tiles of 16 taps
    wgrad_shape(N, Ci, Co, Ho, T, kh, kw, f, p);
    // the waves' tiles, then the chunk sums of the first reduction launch (doubles)
    if (workspace_floats < (N * p.items + 2 * kWgradChunks) * cobs * p.passes * f.tiles * 256) return SLAYER_ERANGE;
    const int64_t blocks = N * cobs * ((p.items + kSynWaves - 1) / kSynWaves);
    if (blocks > 0x7fffffffLL || p.passes > 65535) return SLAYER_ERANGE;
    const dim3 grid((unsigned)blocks, (unsigned)p.passes), block(kSynWaves * kWave);
    const bool tail = (T % 4) != 0;                                       // rows that end inside a quad
#define SLAYER_WGRAD(NTT)                                                                                              \
    do {                                                                                                               \
        if (tail) hipLaunchKernelGGL((synapse_wgrad_kernel<NTT, true>), grid, block, NTT * 16 * 3 * sizeof(int), st, p); \
        else hipLaunchKernelGGL((synapse_wgrad_kernel<NTT, false>), grid, block, NTT * 16 * 3 * sizeof(int), st, p);    \
    } while (0)
    if (f.tiles == 1) SLAYER_WGRAD(1);
    else if (f.tiles == 2) SLAYER_WGRAD(2);
    else SLAYER_WGRAD(5);
#undef SLAYER_WGRAD
    return reduce(p.items, p.passes, f.tiles, {0, 0, 1, 1, 0, 0, 0});
}

extern "C" int slayer_conv_synapse(float* out, const float* in, const float* weight,
                                   int64_t N, int64_t Ci, int64_t Co, int64_t H, int64_t W, int64_t T,
                                   int64_t kh, int64_t kw, int64_t stride_h, int64_t stride_w,
                                   int64_t pad_h, int64_t pad_w, int64_t dil_h, int64_t dil_w, void* stream) {
    return conv_synapse(out, in, weight, N, Ci, Co, H, W, T, kh, kw, stride_h, stride_w, pad_h, pad_w, dil_h, dil_w, nullptr, stream);
}

extern "C" int slayer_conv_synapse_input_grad(float* grad_in, const float* grad_out, const float* weight_t,
                                              int64_t N, int64_t Ci, int64_t Co, int64_t H, int64_t W, int64_t T,
                                              int64_t kh, int64_t kw, int64_t stride_h, int64_t stride_w,
                                              int64_t pad_h, int64_t pad_w, int64_t dil_h, int64_t dil_w, void* stream) {
    return conv_synapse_input_grad(grad_in, grad_out, weight_t, N, Ci, Co, H, W, T, kh, kw, stride_h, stride_w, pad_h, pad_w, dil_h, dil_w,
                                   nullptr, false, stream);
}

extern "C" int slayer_conv_synapse_cut(float* out, const float* in, const float* weight,
                                       int64_t N, int64_t Ci, int64_t Co, int64_t H, int64_t W, int64_t T,
                                       int64_t kh, int64_t kw, int64_t stride_h, int64_t stride_w,
                                       int64_t pad_h, int64_t pad_w, int64_t dil_h, int64_t dil_w,
                                       int input_grad, int by_class, int64_t pixels, int64_t blocks, int64_t pieces, int whole,
                                       void* stream) {
    if (pixels < 1 || blocks < 1 || pieces < 1) return SLAYER_EINVAL;
    if (pixels > 64 || blocks > 2 || pieces > 1024) return SLAYER_ERANGE;
    const WalkCut want = {(int)pixels, (int)blocks, (int)pieces, whole != 0};
    if (!input_grad) return conv_synapse(out, in, weight, N, Ci, Co, H, W, T, kh, kw, stride_h, stride_w, pad_h, pad_w, dil_h, dil_w, &want, stream);
    return conv_synapse_input_grad(out, in, weight, N, Ci, Co, H, W, T, kh, kw, stride_h, stride_w, pad_h, pad_w, dil_h, dil_w, &want,
                                   by_class != 0, stream);
}
