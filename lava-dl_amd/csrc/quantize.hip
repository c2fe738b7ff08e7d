// Weight quantiser of the synapse layers (utils/quantize.py:84-115 in the reference): round to a multiple of `step`, limit to
// [lo, hi], scale; backward the gradient of the weights inside the limits.  One launch each way for what the element-wise
// operators take four and five for (some 4 us apiece on weights of any usual size: nothing but the launches), operation by
// operation the same: the division is the multiplication by the reciprocal the operator makes of it.
#include "common.h"

namespace slayer {

__global__ __launch_bounds__(256) void quantize_kernel(float* __restrict__ out, unsigned char* __restrict__ inside,
                                                       const float* __restrict__ in, float inv_step, float step, float lo,
                                                       float hi, float scale, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const float q = rintf(in[i] * inv_step) * step;
        if (inside) inside[i] = q >= lo && q <= hi;
        out[i] = (q != q ? q : fminf(fmaxf(q, lo), hi)) * scale;
    }
}

__global__ __launch_bounds__(256) void quantize_bwd_kernel(float* __restrict__ grad_in, const float* __restrict__ grad_out,
                                                           const unsigned char* __restrict__ inside, float scale, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        grad_in[i] = inside[i] ? grad_out[i] * scale : 0.f;
}

// The rotation parameters of a resonate-and-fire neuron, in place: gain limited to `gain_max`, sin at least 1, cos at least 0
// (neuron/rf.py:136-257 in the reference) -- nine element-wise operators otherwise, on one value per channel, at the head of
// every forward pass of a neuron that learns.  The same operations in the same order, so the same bits.
__global__ __launch_bounds__(256) void rf_limit_kernel(float* __restrict__ sin_decay, float* __restrict__ cos_decay, float gain_max,
                                                       int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        float s = sin_decay[i], c = cos_decay[i];
        const float gain = sqrtf(s * s + c * c);
        const float ratio = (gain != gain ? gain : fminf(fmaxf(gain, 0.f), gain_max)) / gain;
        s *= ratio;
        c *= ratio;
        sin_decay[i] = s != s ? s : fmaxf(s, 1.f);
        cos_decay[i] = c != c ? c : fmaxf(c, 0.f);
    }
}

}  // namespace slayer

using namespace slayer;

namespace {
int check_count(int64_t n) { return n < 0 ? SLAYER_EINVAL : (n > ((int64_t)1 << 38) ? SLAYER_ERANGE : 0); }
// A launch takes fewer than 2^32 threads in all: beyond 2^31 entries a thread has several.
dim3 grid_of(int64_t n) { return dim3((unsigned)((n < ((int64_t)1 << 31) ? n + 255 : (int64_t)1 << 31) / 256)); }
}  // namespace

extern "C" int slayer_quantize(float* out, unsigned char* inside, const float* in, float step, float lo, float hi, float scale,
                               int64_t n, void* stream) {
    if (int e = check_count(n)) return e;
    if (step == 0.0f) return SLAYER_EINVAL;
    if (n == 0) return 0;
    if (!out || !in) return SLAYER_ENULL;
    hipLaunchKernelGGL(quantize_kernel, grid_of(n), dim3(256), 0, (hipStream_t)stream, out, inside, in,
                       1.0f / step, step, lo, hi, scale, n);
    return (int)hipGetLastError();
}

extern "C" int slayer_quantize_bwd(float* grad_in, const float* grad_out, const unsigned char* inside, float scale, int64_t n,
                                   void* stream) {
    if (int e = check_count(n)) return e;
    if (n == 0) return 0;
    if (!grad_in || !grad_out || !inside) return SLAYER_ENULL;
    hipLaunchKernelGGL(quantize_bwd_kernel, grid_of(n), dim3(256), 0, (hipStream_t)stream, grad_in,
                       grad_out, inside, scale, n);
    return (int)hipGetLastError();
}

extern "C" int slayer_rf_limit(float* sin_decay, float* cos_decay, float gain_max, int64_t n, void* stream) {
    if (int e = check_count(n)) return e;
    if (n == 0) return 0;
    if (!sin_decay || !cos_decay) return SLAYER_ENULL;
    hipLaunchKernelGGL(rf_limit_kernel, grid_of(n), dim3(256), 0, (hipStream_t)stream, sin_decay, cos_decay,
                       gain_max, n);
    return (int)hipGetLastError();
}
