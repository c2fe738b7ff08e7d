// Operands of the recurrent weight gradient (utils/recurrent.py:85-112 in the reference: grad R = sum over samples and time
// of the gradient of step t times the spikes of step t - 1): the product over (sample, step) is the library's, and wants
// rows of either operand in one piece.
#include "common.h"

namespace slayer {

// A workgroup takes 64 neurons x 64 steps of one sample: the gradient's rows move one step to the left, the spikes are turned
// over by way of LDS, so that reads and writes of both are pieces of 256 bytes.  Bound: memory.  [32,2048,300]: 121 us as two
// element-wise copies (the turned one 87, its writes scattered), 64 us (4.9 TB/s) in this one.
constexpr int kTurn = 64;
__global__ __launch_bounds__(256) void recurrent_operands_kernel(float* __restrict__ grad_rows, float* __restrict__ spike_rows,
                                                                 const float* __restrict__ grad, const float* __restrict__ spikes,
                                                                 int N, int C, int T, int c_tiles, int t_tiles) {
    __shared__ float tile[kTurn][kTurn + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int b = blockIdx.x;
    const int t0 = b % t_tiles * kTurn; b /= t_tiles;
    const int c0 = b % c_tiles * kTurn;
    const int n = b / c_tiles;
    const int t = t0 + lane;
    float g[16], s[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int c = c0 + 4 * i + wave;
        const int64_t at = ((int64_t)n * C + c) * T + t;
        const bool on = c < C && t < T;
        g[i] = on ? grad[at] : 0.f;
        s[i] = on ? spikes[at] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int c = c0 + 4 * i + wave;
        tile[4 * i + wave][lane] = s[i];
        if (c < C && t < T && t >= 1) grad_rows[((int64_t)c * N + n) * (T - 1) + t - 1] = g[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int step = t0 + 4 * i + wave;
        if (step < T - 1 && c0 + lane < C) spike_rows[((int64_t)n * (T - 1) + step) * C + c0 + lane] = tile[lane][4 * i + wave];
    }
}

}  // namespace slayer

using namespace slayer;

extern "C" int slayer_recurrent_operands(float* grad_rows, float* spike_rows, const float* grad, const float* spikes, int64_t N,
                                         int64_t C, int64_t T, void* stream) {
    if (N < 0 || C < 0 || T < 0) return SLAYER_EINVAL;
    if (N == 0 || C == 0 || T < 2) return 0;
    if (!grad_rows || !spike_rows || !grad || !spikes) return SLAYER_ENULL;
    if (N > (1 << 30) || C > (1 << 30) || T > (1 << 30)) return SLAYER_ERANGE;
    const int64_t c_tiles = (C + kTurn - 1) / kTurn, t_tiles = (T + kTurn - 1) / kTurn;
    if (c_tiles * t_tiles > (1 << 23) / N) return SLAYER_ERANGE;          // fewer than 2^32 threads in a launch
    hipLaunchKernelGGL(recurrent_operands_kernel, dim3((unsigned)(N * c_tiles * t_tiles)), dim3(256), 0, (hipStream_t)stream, grad_rows,
                       spike_rows, grad, spikes, (int)N, (int)C, (int)T, (int)c_tiles, (int)t_tiles);
    return (int)hipGetLastError();
}
