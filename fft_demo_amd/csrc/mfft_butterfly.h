// Short DFTs in fp32 registers, shared by the kernels that run a radix on the vector ALUs.
#pragma once
#include "mfft_common.h"

namespace mfft {

// Odd R: y_k = x_0 + sum_j S_j c_jk + i sum_j D_j t_jk and y_{R-k} = x_0 + sum_j S_j c_jk -
// i sum_j D_j t_jk (j, k = 1..(R-1)/2), with S_j = x_j + x_{R-j}, D_j = x_j - x_{R-j} and
// w[m] = W_R^m = c_m + i t_m (FP64-generated table, carries the transform's sign):
// (R-1)^2 real multiply-adds per line instead of 4 (R-1)^2.
template <int R>
__device__ __forceinline__ void dft_odd_w(float2 *v, const float2 *w)
{
    constexpr int H = (R - 1) / 2;
    float2 S[H + 1], D[H + 1];
#pragma unroll
    for (int j = 1; j <= H; ++j) {
        S[j] = make_float2(v[j].x + v[R - j].x, v[j].y + v[R - j].y);
        D[j] = make_float2(v[j].x - v[R - j].x, v[j].y - v[R - j].y);
    }
    float2 y0 = v[0];
#pragma unroll
    for (int j = 1; j <= H; ++j) y0 = make_float2(y0.x + S[j].x, y0.y + S[j].y);
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        float2 a = v[0], b = make_float2(0.f, 0.f);
#pragma unroll
        for (int j = 1; j <= H; ++j) {
            const float2 t = w[(j * k) % R];
            a.x += S[j].x * t.x;
            a.y += S[j].y * t.x;
            b.x += D[j].x * t.y;
            b.y += D[j].y * t.y;
        }
        // i * b = (-b.y, b.x)
        v[k] = make_float2(a.x - b.y, a.y + b.x);
        v[R - k] = make_float2(a.x + b.y, a.y - b.x);
    }
    v[0] = y0;
}

}  // namespace mfft
