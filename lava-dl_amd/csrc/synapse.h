// What the kernels of the convolution synapse share (synapse.hip, synapse_walk.hip): quads of steps, the order of the
// workgroups, the geometry of a launch.
#pragma once
#include "common.h"
#include "tile.h"

namespace slayer {

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

// Division of a number below 2^31 by one that the host knows, as a multiplication (a division of integers is some thirty
// instructions, a chain of them in front of a kernel's first load): with 2^shift >= d, n / d = (n + n mul / 2^32) / 2^shift for
// mul = 2^32 (2^shift - d) / d + 1, rounded down.
struct Divisor {
    unsigned d, mul;
    int shift;
    Divisor() = default;
    Divisor(int by) : d((unsigned)by), shift(0) {
        while ((1ull << shift) < d) ++shift;
        mul = (unsigned)((1ull << 32) * ((1ull << shift) - d) / d + 1);
    }
    __device__ __forceinline__ int of(int n) const { return (int)((__umulhi((unsigned)n, mul) + (unsigned)n) >> shift); }
    __device__ __forceinline__ int rest(int n) const { return n - of(n) * (int)d; }
};

constexpr int kSynTile = 64;            // time steps per tile
constexpr int kSynWaves = 4;            // waves per workgroup: same output channels, same image row, different tiles

// How a launch of the walking kernel is cut: XS neighbouring pixels of the line share a position, their channels being the rows of a
// product, MB blocks of 16 rows to a wave, and the rows of the image are walked in pieces.  whole: a step brings all the input rows that
// its output row meets, as terms of one product, instead of `stride` rows that several output rows meet.
struct WalkCut { int XS, MB, pieces; bool whole; };

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
    const WalkCut* want;                // the cut of the walking kernel and no other kernel, or null: what takes least
    __device__ __forceinline__ int weight_index(int ci, int iy, int ix) const {
        return (ci * kh_full + ky0 + iy * kys) * kw_full + kx0 + ix * kxs;
    }
    __device__ __forceinline__ int out_pixel(int ho, int wo) const {     // in pixels of the full output image
        return (oy0 + ho * oys) * Wo_full + ox0 + wo * oxs;
    }
};

// synapse_walk.hip: true if the launch is one that it takes; *code is the launch's
bool launch_synapse_walk(const SynapseConv& p, hipStream_t stream, int* code);
// ... the gradient of the input of a convolution without dilation, all residue classes in one launch (p.in, p.H, p.W, p.Ci:
// the gradient of its output; p.out, p.Ho_full, p.Wo_full, p.Co: of its input)
bool launch_synapse_walk_transposed(const SynapseConv& p, int kh, int kw, int sh, int sw, int ph, int pw, hipStream_t stream,
                                    int* code);

// The weight gradient on the walking kernel (synapse_wgrad_walk.hip): the geometry as for the convolution, in bytes, the line
// cut into shares of whole visits of eight quads, the rows into kSynWaves pieces or one.
struct WgradWalk {
    float* partial;                     // [N][blocks of 16 channels][sets][passes][KS npt][64] quads
    const float* grad_out;
    const float* in;
    int N, Co, T;
    int in_plane, out_plane;            // bytes of one sample
    int in_ch, in_slide, in_line, out_ch, out_slide, out_line;           // bytes
    int Hs, Ws;                         // input rows along the walk, pixels along the line
    int quads, line_quads;              // quads of steps a pixel of the gradient has, its line has
    int ss, ls;                         // strides along walk and line
    int row0, S, c_lo, c_hi;            // input row of step 0, gradient rows, the steps that meet a row inside the image
    int XP, shift0, shift_step;         // line taps, the first one's shift, pixels from one to the next
    int pairs, npt, passes, KS;         // (channel, line tap, row of a step) triples, tiles of 16 of them a pass, taps along the walk
    int shares, share_quads, pieces, sets;   // sets of tiles: one a share, or one for the shares of a workgroup
    int kslide, kline, wslide, wline;   // the filter's axes: sizes and strides
    Divisor by_cobs, by_passes, by_sets, by_quads, by_triples, by_ss;    // blocks of channels, passes, sets, quads, XP * ss, ss
};
int launch_synapse_wgrad_walk(WgradWalk& w, hipStream_t stream);

}  // namespace slayer
