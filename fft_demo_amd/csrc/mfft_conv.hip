// Elementwise kernels of the FFT convolution operator (pack/pad, pointwise multiply-
// accumulate, crop/unpack). The transforms themselves are mfft 2D plans.
//
// Reference steps these replace (tensorcore_fft_conv2d_kernel.cu): filter rotation
// (fft_conv2d_inverse_filter :1234-1253), real->complex padding with digit reversal
// (fft_conv2d_bit_rev_real_pad_to_cpx_double2half :1222-1232), the channel sum
// (fft_cpx_point_wise_mul_add :1033-1056), the per-filter power-of-10 quantisation
// (quant_p1/p2/p3 :1058-1098; only the reference-method mode uses it -- otherwise spectra
// stay fp32 or the transforms are scaled per stage), the dequantisation
// (fft_cpx_point_wise_dequant :1129-1139) and the crop/scale readout
// (read_out_scale_double2double_kernel :1390-1397).
#include "mfft_common.h"

#include <type_traits>

namespace mfft {

// Image and product spectra are complex fp32 (FMT_C32) or fp16 (FMT_C16) per operator.
template <int FMT>
__device__ __forceinline__ float2 spec_ld(const void *p, long long i)
{
    if constexpr (FMT == FMT_C32) {
        return reinterpret_cast<const float2 *>(p)[i];
    } else {
        const uint32_t w = reinterpret_cast<const uint32_t *>(p)[i];
        return make_float2((float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xffffu)),
                           (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)));
    }
}

template <int FMT>
__device__ __forceinline__ void spec_st(void *p, long long i, float2 v)
{
    if constexpr (FMT == FMT_C32)
        reinterpret_cast<float2 *>(p)[i] = v;
    else
        reinterpret_cast<uint32_t *>(p)[i] = pack_c16(v.x, v.y);
}

// Row kernels: the elements of a launch are rows of `width` elements, V consecutive ones per
// thread. A block of tx x ty threads covers ty rows, tx * V columns of each (xb blocks side by
// side). Where tx is 64 or more, a wave stays in one row, which it decodes once, in scalar
// registers; narrow rows share a wave (1024 planes of 64 x 64 packed in 10.9 us, with a wave for 32
// pairs of columns 13.7). Bound by memory: 64 planes of 256 x 256 packed in 14.5 us, 3.3 TB/s (one
// element per thread, its index divided down in 64 bits: 19.7 us).
struct RowGrid {
    unsigned xb;
    dim3 grid, block;
    bool ok;
};

static RowGrid row_grid(long long rows, int width, int V)
{
    RowGrid g;
    const int per = (width + V - 1) / V;
    unsigned tx = 16;
    while (tx < 256 && tx < (unsigned)per) tx *= 2;
    const unsigned ty = 256 / tx;
    g.xb = (per + tx - 1) / tx;
    const long long blocks = (rows + ty - 1) / ty * g.xb;
    g.grid = dim3((unsigned)blocks);
    g.block = dim3(tx, ty);
    g.ok = blocks <= 0x7fffffffLL && rows <= 0x7fffffffLL;
    return g;
}

// wave, narrow: the kernel for blocks whose rows are whole waves, and for others.
template <typename... A, typename... B>
static void launch_rows(void (*wave)(A...), void (*narrow)(A...), const RowGrid &g, hipStream_t s, B... args)
{
    hipLaunchKernelGGL(g.block.x >= 64 ? wave : narrow, g.grid, g.block, 0, s, static_cast<A>(args)...);
}

struct RowAt {
    unsigned row;
    int x;
};

template <int V, bool WAVE>
__device__ __forceinline__ RowAt row_at(unsigned xb)
{
    const unsigned q = blockIdx.x / xb;
    const unsigned ty = WAVE ? (unsigned)__builtin_amdgcn_readfirstlane((int)threadIdx.y) : threadIdx.y;  // WAVE: the wave's row
    return {q * blockDim.y + ty, (int)(((blockIdx.x - q * xb) * blockDim.x + threadIdx.x) * V)};
}

// Two adjacent spectrum elements (vec: i is even and the buffer aligned to the pair).
template <int FMT>
__device__ __forceinline__ void spec_st2(void *p, long long i, float2 a, float2 b)
{
    if constexpr (FMT == FMT_C32)
        *reinterpret_cast<float4 *>(reinterpret_cast<float2 *>(p) + i) = make_float4(a.x, a.y, b.x, b.y);
    else
        *reinterpret_cast<uint2 *>(reinterpret_cast<uint32_t *>(p) + i) = make_uint2(pack_c16(a.x, a.y), pack_c16(b.x, b.y));
}

// Two real images (batch items 2k and 2k+1, same channel) become the real and imaginary
// parts of one complex image, zero-padded to Ph x Pw at the origin.
// src: real [B][C][h][w] (fp32 or fp64); dst: complex [pairs][C][Ph][Pw] (FMT). V = 2: Pw even.
template <typename T, int FMT, int V, bool WAVE>
__global__ void pack_pairs_kernel(const T *src, void *dst, int B, int C, int h, int w, int Ph, int Pw, unsigned rows,
                                  unsigned xb)
{
    const RowAt at = row_at<V, WAVE>(xb);
    if (at.row >= rows || at.x >= Pw) return;
    const unsigned plane = at.row / (unsigned)Ph, y = at.row - plane * (unsigned)Ph;
    const unsigned k = plane / (unsigned)C, c = plane - k * (unsigned)C;
    float2 v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = make_float2(0.f, 0.f);
    if (y < (unsigned)h) {
        const long long hw = (long long)h * w, b0 = 2LL * k;
        const T *s0 = src + (b0 * C + c) * hw + (long long)y * w, *s1 = s0 + C * hw;
        const bool second = b0 + 1 < B;
#pragma unroll
        for (int j = 0; j < V; ++j)
            if (at.x + j < w) {
                v[j].x = (float)s0[at.x + j];
                if (second) v[j].y = (float)s1[at.x + j];
            }
    }
    const long long i = (long long)at.row * Pw + at.x;
    if constexpr (V == 2)
        spec_st2<FMT>(dst, i, v[0], v[1]);
    else
        spec_st<FMT>(dst, i, v[0]);
}

// Filter [F][C][fh][fw] real -> complex fp32 [F][C][Ph][Pw], optionally rotated by 180
// degrees (convolution by the rotated filter = cross-correlation). V = 2: Pw even.
template <typename T, int V, bool WAVE>
__global__ void pack_filters_kernel(const T *src, float2 *dst, int fh, int fw, int Ph, int Pw, int rotate, unsigned rows,
                                    unsigned xb)
{
    const RowAt at = row_at<V, WAVE>(xb);
    if (at.row >= rows || at.x >= Pw) return;
    const unsigned fc = at.row / (unsigned)Ph;
    const int y = (int)(at.row - fc * (unsigned)Ph);
    float2 v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int x = at.x + j;
        v[j] = make_float2(0.f, 0.f);
        if (y < fh && x < fw) {
            const int sy = rotate ? fh - 1 - y : y, sx = rotate ? fw - 1 - x : x;
            v[j].x = (float)src[((long long)fc * fh + sy) * fw + sx];
        }
    }
    const long long i = (long long)at.row * Pw + at.x;
    if constexpr (V == 2)
        spec_st2<FMT_C32>(dst, i, v[0], v[1]);
    else
        dst[i] = v[0];
}

// Blocks of the pointwise kernels: 256 points of a plane times a tile of output maps, the tiles
// of the same points next to each other, so that what they share comes from the caches.
constexpr int kMapTile = 4;
// Filters of at most this many taps a side go through the short-filter kernels.
constexpr int kShortTaps = 32;

struct MapAt {
    long long p;
    int a0, b0;  // first map of the tile along each of the two map axes
};

// Tiles of one map (TA = TB = 1): the threads walk all planes without gaps, so that small planes
// leave no lanes idle (p = P past the last one); na nb P < 2^31.
template <int TA, int TB, int PTS = 256>
__device__ __forceinline__ MapAt map_at(int na, int nb, long long P)
{
    if constexpr (TA * TB == 1) {
        const unsigned i = blockIdx.x * 256 + threadIdx.x, n = (unsigned)P, t = i / n, a = t / (unsigned)nb;
        return {a < (unsigned)na ? (long long)(i - t * n) : P, (int)a, (int)(t - a * (unsigned)nb)};
    }
    const unsigned ta = (na + TA - 1) / TA, tb = (nb + TB - 1) / TB;
    unsigned r = blockIdx.x;
    const unsigned pb = r / (ta * tb);
    r -= pb * (ta * tb);
    const unsigned ia = r / tb;
    return {(long long)pb * PTS + threadIdx.x % PTS, (int)ia * TA, (int)(r - ia * tb) * TB};
}

static long long map_blocks(long long P, long long na, long long nb, int ta = kMapTile, int tb = kMapTile, int pts = 256)
{
    if (ta * tb == 1) return (P * na * nb + 255) / 256;
    return (P + pts - 1) / pts * ((na + ta - 1) / ta) * ((nb + tb - 1) / tb);
}

// Y[k][f][p] = sum_c X[k][c][p] * H[f][c][p]   (X, Y: FMT; H: fp32). A thread sums a tile of T
// pairs x T filters at its point: an X or H value is read once per tile instead of once per
// output map (4 pairs, 3 channels, 16 filters of 256 x 256: 19.7 us with one map a thread, 15.9
// with 4 x 4; memory-bound, 3.9 TB/s).
template <int XFMT, int YFMT, int T>
__global__ void __launch_bounds__(256) pointwise_mac_kernel(const void *X, const float2 *H, void *Y, int pairs, int C, int F,
                                                            long long P)
{
    const MapAt m = map_at<T, T>(pairs, F, P);
    if (m.p >= P) return;
    const int nk = min(T, pairs - m.a0), nf = min(T, F - m.b0);
    float2 acc[T][T];
#pragma unroll
    for (int k = 0; k < T; ++k)
#pragma unroll
        for (int f = 0; f < T; ++f) acc[k][f] = make_float2(0.f, 0.f);
    constexpr int U = T > 1 ? 2 : 1;
#pragma unroll U
    for (int c = 0; c < C; ++c) {
        // maps past the last one repeat it: the loads of a step stay in one block and in flight together
        float2 a[T], b[T];
#pragma unroll
        for (int k = 0; k < T; ++k) a[k] = spec_ld<XFMT>(X, ((long long)(T > 1 ? min(m.a0 + k, pairs - 1) : m.a0) * C + c) * P + m.p);
#pragma unroll
        for (int f = 0; f < T; ++f) b[f] = H[((long long)(T > 1 ? min(m.b0 + f, F - 1) : m.b0) * C + c) * P + m.p];
#pragma unroll
        for (int k = 0; k < T; ++k)
#pragma unroll
            for (int f = 0; f < T; ++f) {
                // which product is fused is fixed here, as the kernel of one output a thread had
                // it per format: 16-bit words further on show a change of it
                acc[k][f].x += __builtin_fmaf(a[k].x, b[f].x, -(a[k].y * b[f].y));
                acc[k][f].y += XFMT == FMT_C16 ? __builtin_fmaf(a[k].x, b[f].y, a[k].y * b[f].x)
                                               : __builtin_fmaf(a[k].y, b[f].x, a[k].x * b[f].y);
            }
    }
#pragma unroll
    for (int k = 0; k < T; ++k)
#pragma unroll
        for (int f = 0; f < T; ++f)
            if (k < nk && f < nf) spec_st<YFMT>(Y, ((long long)(m.a0 + k) * F + m.b0 + f) * P + m.p, acc[k][f]);
}

// The reference method's quantisation of the product spectra (quant_p1/p2/p3,
// tensorcore_fft_conv2d_kernel.cu:1058-1098): per output map (pair, filter) the largest
// |re| or |im| m over its P values sets the scale s = 1 if m <= 1000, else 10^(trunc(log10 m)
// - 1), and the map is stored as fp16(R / s) for the fp16 inverse transform. Step 1: each
// workgroup takes a chunk of one map and writes the chunk's maximum.
__global__ void quant_max_kernel(const float2 *R, float *partial, long long P, int nchunk)
{
    __shared__ float red[256];
    const long long map = blockIdx.x / nchunk;
    const int chunk = (int)(blockIdx.x - map * nchunk);
    const long long per = (P + nchunk - 1) / nchunk;
    const long long b = chunk * per, e = b + per < P ? b + per : P;
    float m = 0.f;
    for (long long i = b + threadIdx.x; i < e; i += 256) {
        const float2 v = R[map * P + i];
        m = fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y)));
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// The quantisation scale of a map from its largest magnitude (quant_p2's rule; the power of
// ten by repeated products in fp32, exact up to 10^10). A map whose forward overflowed (an
// infinite or NaN maximum) keeps scale 1, so the overflow shows in its output as it does in
// the reference's; the loop is bounded by the largest finite maximum (k <= 37).
__device__ __forceinline__ float quant_scale(float m)
{
    if (!(m > 1000.f) || !(m <= 3.4e38f)) return 1.f;
    const int k = (int)log10f(m) - 1;
    float s = 1.f;
    for (int j = 0; j < k; ++j) s *= 10.f;
    return s;
}

// Step 2: each workgroup reduces its map's chunk maxima, takes the scale (chunk 0 records
// it for the dequantisation) and stores its chunk as fp16(R / s).
__global__ void quant_apply_kernel(const float2 *R, uint32_t *Q, const float *partial, float *scale, long long P,
                                   int nchunk)
{
    const long long map = blockIdx.x / nchunk;
    const int chunk = (int)(blockIdx.x - map * nchunk);
    float m = 0.f;
    for (int c = 0; c < nchunk; ++c) m = fmaxf(m, partial[map * nchunk + c]);
    const float s = quant_scale(m), inv = 1.f / s;
    if (chunk == 0 && threadIdx.x == 0) scale[map] = s;
    const long long per = (P + nchunk - 1) / nchunk;
    const long long b = chunk * per, e = b + per < P ? b + per : P;
    for (long long i = b + threadIdx.x; i < e; i += 256) {
        const float2 v = R[map * P + i];
        Q[map * P + i] = pack_c16(v.x * inv, v.y * inv);
    }
}

// out[2k][f][y][x] = scale * Re Y[k][f][y + oy][x + ox], out[2k+1][f][y][x] = scale * Im ...
// (each spectrum value is read once for both images; rows: pairs x F x oh). A thread takes V
// consecutive columns (V = 4: one 16-byte store per image, for fp32 output rows whose width is a
// multiple of 4 on a 16-byte aligned buffer).
template <typename T, int FMT, int V, bool WAVE>
__global__ void crop_unpack_kernel(const void *Y, T *out, int B, int F, int oh, int ow, int Ph, int Pw, int oy,
                                   int ox, float scale, unsigned rows, unsigned xb, const float *map_scale)
{
    const RowAt at = row_at<V, WAVE>(xb);
    if (at.row >= rows || at.x >= ow) return;
    const int x = at.x;
    const unsigned kf = at.row / (unsigned)oh;
    const int y = (int)(at.row - kf * (unsigned)oh);
    const long long k = kf / (unsigned)F;
    const int f = (int)(kf - (unsigned)k * (unsigned)F);
    const long long src = ((k * F + f) * Ph + (y + oy)) * (long long)Pw + (x + ox);
    const long long plane = (long long)F * oh * ow, off = ((long long)f * oh + y) * ow + x;
    const bool second = 2 * k + 1 < B;
    if (map_scale) scale *= map_scale[k * F + f];  // the reference method's dequantisation
    if constexpr (V == 1) {
        const float2 v = spec_ld<FMT>(Y, src);
        out[2 * k * plane + off] = (T)(v.x * scale);
        if (second) out[(2 * k + 1) * plane + off] = (T)(v.y * scale);
    } else {
        static_assert(V == 4, "4 columns per thread");
        float re[4], im[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float2 v = spec_ld<FMT>(Y, src + j);
            re[j] = v.x * scale;
            im[j] = v.y * scale;
        }
        *reinterpret_cast<float4 *>(out + 2 * k * plane + off) = make_float4(re[0], re[1], re[2], re[3]);
        if (second)
            *reinterpret_cast<float4 *>(out + (2 * k + 1) * plane + off) = make_float4(im[0], im[1], im[2], im[3]);
    }
}

// Two real images a, b (separate buffers, [h][w]) -> one complex image a + i b, zero-padded.
template <typename T, int FMT>
__global__ void pack_two_kernel(const T *a, const T *b, void *dst, int h, int w, int Ph, int Pw, long long total)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    int x = (int)(i % Pw), y = (int)(i / Pw);
    float2 v = make_float2(0.f, 0.f);
    if (y < h && x < w) {
        long long off = (long long)y * w + x;
        v = make_float2((float)a[off], (float)b[off]);
    }
    spec_st<FMT>(dst, i, v);
}

// Spectrum X of a + i b (a, b real): A = (X(k) + conj X(-k)) / 2 and B = (X(k) - conj X(-k))
// / 2i are the spectra of a and b, so Y = A H0 + i B H1 = ((X + X*)/2) H0 + ((X - X*)/2) H1
// (X* = conj X(-k)) transforms back to (a conv h0) + i (b conv h1): two convolutions with
// different filters from one forward and one inverse transform.
template <int FMT>
__global__ void pointwise_two_kernel(const void *X, const float2 *H0, const float2 *H1, void *Y, int Ph, int Pw)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)Ph * Pw) return;
    int v = (int)(i % Pw), u = (int)(i / Pw);
    int uq = u ? Ph - u : 0, vq = v ? Pw - v : 0;
    float2 xp = spec_ld<FMT>(X, i), xq = spec_ld<FMT>(X, (long long)uq * Pw + vq);
    xq.y = -xq.y;
    float2 s = make_float2(0.5f * (xp.x + xq.x), 0.5f * (xp.y + xq.y));
    float2 d = make_float2(0.5f * (xp.x - xq.x), 0.5f * (xp.y - xq.y));
    float2 h0 = H0[i], h1 = H1[i];
    spec_st<FMT>(Y, i,
                 make_float2(s.x * h0.x - s.y * h0.y + d.x * h1.x - d.y * h1.y,
                             s.x * h0.y + s.y * h0.x + d.x * h1.y + d.y * h1.x));
}

// out0 = Re Y, out1 = Im Y over the output window at (oy, ox).
template <typename T, int FMT>
__global__ void crop_two_kernel(const void *Y, T *out0, T *out1, int oh, int ow, int Pw, int oy, int ox, long long total)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    int x = (int)(i % ow), y = (int)(i / ow);
    float2 v = spec_ld<FMT>(Y, (long long)(y + oy) * Pw + (x + ox));
    out0[i] = (T)v.x;
    out1[i] = (T)v.y;
}

// ---------------------------------------------------------------- backward
// Filter gradient spectrum: G[f][c][p] = sum_k A_k[c] conj(DA_k[f]) + B_k[c] conj(DB_k[f]),
// where X_k = spectrum of the image pair (a + i b) and D_k of the delta pair (da + i db),
// separated per frequency with X(-p): A = (X + X*)/2, B = (X - X*)/2i (X* = conj X(-p)).
// Its inverse is sum_b in[b][c] (correlated with) delta[b][f], which is real: G(-p) = conj G(p),
// so a thread computes a tile of TF filters x TC channels at one point of the upper half plane
// and stores both. Per-map threads over the whole plane re-read X and D for every map (4
// pairs, 3 channels, 16 filters of 256 x 256: 27.3 us, 2 x 4 tiles 17.3).
template <int TF, int TC>
__global__ void __launch_bounds__(256) pointwise_gw_kernel(const float2 *X, const float2 *D, float2 *G, int pairs, int C, int F,
                                                           int Ph, int Pw)
{
    const MapAt m = map_at<TF, TC>(F, C, (long long)(Ph / 2 + 1) * Pw);
    if (m.p >= (long long)(Ph / 2 + 1) * Pw) return;
    const long long P = (long long)Ph * Pw;
    const unsigned u = (unsigned)m.p / (unsigned)Pw, v = (unsigned)m.p - u * (unsigned)Pw;
    const long long q = (long long)(u ? Ph - u : 0) * Pw + (v ? Pw - v : 0);
    const int nf = min(TF, F - m.a0), nc = min(TC, C - m.b0);
    float2 g[TF][TC];
#pragma unroll
    for (int f = 0; f < TF; ++f)
#pragma unroll
        for (int c = 0; c < TC; ++c) g[f][c] = make_float2(0.f, 0.f);
    constexpr int U = TF * TC > 4 ? 1 : 2;
#pragma unroll U
    for (int k = 0; k < pairs; ++k) {
        // maps past the last one repeat it, as in pointwise_mac_kernel
        float2 A[TC], B[TC];
#pragma unroll
        for (int c = 0; c < TC; ++c) {
            const float2 *x = X + ((long long)k * C + (TC > 1 ? min(m.b0 + c, C - 1) : m.b0)) * P;
            const float2 xp = x[m.p], xq = x[q];
            // A = (xp + conj xq)/2, B = (xp - conj xq)/(2i)
            A[c] = make_float2(0.5f * (xp.x + xq.x), 0.5f * (xp.y - xq.y));
            B[c] = make_float2(0.5f * (xp.y + xq.y), -0.5f * (xp.x - xq.x));
        }
#pragma unroll
        for (int f = 0; f < TF; ++f) {
            const float2 *d = D + ((long long)k * F + (TF > 1 ? min(m.a0 + f, F - 1) : m.a0)) * P;
            const float2 dp = d[m.p], dq = d[q];
            const float2 DA = make_float2(0.5f * (dp.x + dq.x), 0.5f * (dp.y - dq.y));
            const float2 DB = make_float2(0.5f * (dp.y + dq.y), -0.5f * (dp.x - dq.x));
            // A conj(DA) + B conj(DB)
#pragma unroll
            for (int c = 0; c < TC; ++c) {
                g[f][c].x += A[c].x * DA.x + A[c].y * DA.y + B[c].x * DB.x + B[c].y * DB.y;
                g[f][c].y += A[c].y * DA.x - A[c].x * DA.y + B[c].y * DB.x - B[c].x * DB.y;
            }
        }
    }
    // the rows that mirror into themselves (0 and, when Ph is even, Ph / 2) store their own points
    const bool both = u != 0 && 2 * u != (unsigned)Ph;
#pragma unroll
    for (int f = 0; f < TF; ++f)
#pragma unroll
        for (int c = 0; c < TC; ++c)
            if (f < nf && c < nc) {
                float2 *o = G + ((long long)(m.a0 + f) * C + m.b0 + c) * P;
                o[m.p] = g[f][c];
                if (both) o[q] = make_float2(g[f][c].x, -g[f][c].y);
            }
}

// Input gradient spectrum: R[k][c][p] = sum_f D_k[f][p] conj(H[f][c][p]) with H the spectrum
// of the 180-degree rotated filter; conj(H) is the spectrum of a real signal, so the image
// pair stays separable in the inverse. Tiles of T pairs x T channels, as pointwise_mac_kernel.
// NS: the waves of a block share 256 / NS points and each sums every NS-th filter: a layer has
// few input maps, so one thread per point leaves most of the device idle (4 pairs, 3 channels, 16
// filters of 256 x 256, 256 blocks of one point per thread: 17.4 us, split four ways 12.2).
template <int NS, int T>
__global__ void __launch_bounds__(256) pointwise_gi_kernel(const float2 *D, const float2 *H, float2 *R, int pairs, int C, int F,
                                                           long long P)
{
    constexpr int PTS = 256 / NS;
    __shared__ float2 red[NS > 1 ? NS : 1][T * T][NS > 1 ? PTS : 1];
    const MapAt m = map_at<T, T, PTS>(pairs, C, P);
    const int part = NS > 1 ? (int)threadIdx.x / PTS : 0, lane = threadIdx.x % PTS;
    const bool in = m.p < P;
    const int nk = min(T, pairs - m.a0), nc = min(T, C - m.b0);
    float2 acc[T][T];
#pragma unroll
    for (int k = 0; k < T; ++k)
#pragma unroll
        for (int c = 0; c < T; ++c) acc[k][c] = make_float2(0.f, 0.f);
    auto step = [&](int f, auto whole) {
        constexpr bool W = decltype(whole)::value;
        float2 d[T], h[T];
#pragma unroll
        for (int k = 0; k < T; ++k)
            if (W || k < nk) d[k] = D[((long long)(m.a0 + k) * F + f) * P + m.p];
#pragma unroll
        for (int c = 0; c < T; ++c)
            if (W || c < nc) h[c] = H[((long long)f * C + m.b0 + c) * P + m.p];
#pragma unroll
        for (int k = 0; k < T; ++k)
#pragma unroll
            for (int c = 0; c < T; ++c)
                if (W || (k < nk && c < nc)) {
                    acc[k][c].x += d[k].x * h[c].x + d[k].y * h[c].y;
                    acc[k][c].y += d[k].y * h[c].x - d[k].x * h[c].y;
                }
    };
    // whole tiles without a branch between the loads of a step, which then are in flight together
    if (T == 1 || (nk == T && nc == T)) {
        constexpr int U = T > 1 ? 2 : 1;
#pragma unroll U
        for (int f = part; f < F && in; f += NS) step(f, std::true_type{});
    } else {
        for (int f = part; f < F && in; f += NS) step(f, std::false_type{});
    }
    if constexpr (NS > 1) {
        // wave w finishes the tile's pair w (NS = T)
        static_assert(NS == T, "one pair per part");
#pragma unroll
        for (int k = 0; k < T; ++k)
#pragma unroll
            for (int c = 0; c < T; ++c) red[part][k * T + c][lane] = acc[k][c];
        __syncthreads();
        if (!in || part >= nk) return;
#pragma unroll
        for (int c = 0; c < T; ++c)
            if (c < nc) {
                float2 s = make_float2(0.f, 0.f);
#pragma unroll
                for (int w = 0; w < NS; ++w) {
                    const float2 t = red[w][part * T + c][lane];
                    s.x += t.x;
                    s.y += t.y;
                }
                R[((long long)(m.a0 + part) * C + m.b0 + c) * P + m.p] = s;
            }
    } else {
        if (!in) return;
#pragma unroll
        for (int k = 0; k < T; ++k)
#pragma unroll
            for (int c = 0; c < T; ++c)
                if (k < nk && c < nc) R[((long long)(m.a0 + k) * C + m.b0 + c) * P + m.p] = acc[k][c];
    }
}

// ---------------------------------------------------------------- short filters
// A filter of fh x fw taps, fh far below Ph: its Ph x Pw spectrum is a product of two small DFT
// matrices, H = Ey w Ex, which one kernel computes straight from the taps instead of a padded
// plane going through a whole 2D transform. 48 filters of 13 x 13 on 256 x 256: 12.8 us, 2 TB/s of
// spectra written (packing, rows and columns took 30.6 us). Up to 32 taps the 2 x 32 products a
// point stay below the transform's passes over memory. The matrices are tables: ty[ky][y] = W_Ph^(ky y) (rows
// of NR entries, ky <= Ph / 2) and tx[x][kx] = W_Pw^(x kx), evaluated in FP64 and rounded once.

// One block: 64 columns kx and a strip of rows ky of one filter's spectrum. The waves transform
// the taps' rows along x into LDS; then a lane keeps its column's NR sums in registers, and a wave
// takes one row ky at a time, the row's factors in scalar registers. The filter is real: row Ph -
// ky is stored from row ky's sums. Both sums go in parts (four taps of a row, a quarter of the rows),
// added up last: 31 x 31 positive taps sum up 3.4e-8 off (rms), in one chain a row and then one of the
// rows 7.7e-8, which showed in the outputs.
template <typename T, int NR>
__global__ void __launch_bounds__(256) filter_spectrum_kernel(const T *__restrict__ src, float2 *__restrict__ H,
                                                              const float2 *__restrict__ ty, const float2 *__restrict__ tx,
                                                              int fh, int fw, int Ph, int Pw, int rotate, int nkx, int nstrip)
{
    __shared__ float2 r[NR][64];
    __shared__ float taps[kShortTaps][NR];  // the rotation undone
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const unsigned fk = blockIdx.x / (unsigned)nstrip;
    const int strip = (int)(blockIdx.x - fk * (unsigned)nstrip);
    const unsigned fc = fk / (unsigned)nkx;
    const int kx = (int)(fk - fc * (unsigned)nkx) * 64 + lane, kxc = min(kx, Pw - 1);
    const T *w = src + (long long)fc * fh * fw;
    for (int i = threadIdx.x; i < fw * NR; i += 256) {
        const int x = i / NR, y = i - x * NR;
        const int sy = rotate ? fh - 1 - y : y, sx = rotate ? fw - 1 - x : x;
        taps[x][y] = y < fh ? (float)w[sy * fw + sx] : 0.f;
    }
    __syncthreads();
    {
        float2 a[NR / 4];
#pragma unroll
        for (int j = 0; j < NR / 4; ++j) a[j] = make_float2(0.f, 0.f);
        auto tap = [&](int x, float2 *p) {
            const float2 t = tx[(long long)x * Pw + kxc];
#pragma unroll
            for (int j = 0; j < NR / 4; ++j) {
                const float v = taps[x][wave + 4 * j];
                p[j].x += v * t.x;
                p[j].y += v * t.y;
            }
        };
        for (int x0 = 0; x0 < fw; x0 += 4) {
            float2 p[NR / 4];
#pragma unroll
            for (int j = 0; j < NR / 4; ++j) p[j] = make_float2(0.f, 0.f);
            if (x0 + 4 <= fw) {
#pragma unroll
                for (int x = 0; x < 4; ++x) tap(x0 + x, p);
            } else {
                for (int x = x0; x < fw; ++x) tap(x, p);
            }
#pragma unroll
            for (int j = 0; j < NR / 4; ++j) a[j] = make_float2(a[j].x + p[j].x, a[j].y + p[j].y);
        }
#pragma unroll
        for (int j = 0; j < NR / 4; ++j) r[wave + 4 * j][lane] = a[j];
    }
    __syncthreads();
    float2 v[NR];
#pragma unroll
    for (int y = 0; y < NR; ++y) v[y] = r[y][lane];
    const int rows = Ph / 2 + 1, per = (rows + nstrip - 1) / nstrip;
    const int end = min(rows, (strip + 1) * per);
    float2 *h = H + (long long)fc * Ph * Pw;
    const int mx = kx ? Pw - kx : 0;
    typedef __attribute__((address_space(4))) const float cf;
    for (int ky = strip * per + wave; ky < end; ky += 4) {
        const cf *t = (const cf *)(ty + (long long)ky * NR);
        float2 p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j] = make_float2(0.f, 0.f);
#pragma unroll
        for (int y = 0; y < NR; ++y) {
            p[y / (NR / 4)].x += v[y].x * t[2 * y] - v[y].y * t[2 * y + 1];
            p[y / (NR / 4)].y += v[y].x * t[2 * y + 1] + v[y].y * t[2 * y];
        }
        const float2 a = make_float2((p[0].x + p[1].x) + (p[2].x + p[3].x), (p[0].y + p[1].y) + (p[2].y + p[3].y));
        if (kx < Pw) {
            h[(long long)ky * Pw + kx] = a;
            if (ky != 0 && 2 * ky != Ph) h[(long long)(Ph - ky) * Pw + mx] = make_float2(a.x, -a.y);
        }
    }
}

// ty and tx of the short-filter kernels (tx: entry i = x * Pw + kx).
__global__ void gen_dft_rows_kernel(float2 *out, int n, int pitch, long long count)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const long long a = i / pitch, b = i - a * pitch;
    const long long e = a * b % n;
    double sn, cs;
    sincospi(2.0 * (double)e / (double)n, &sn, &cs);
    out[i] = make_float2((float)cs, (float)-sn);
}

// out[b][c][y][x] = scale * (Re or Im) Y[b/2][c][(y + oy) mod Ph][(x + ox) mod Pw], oy < Ph and
// ox < Pw; both images of a pair from one read (rows: pairs x C x oh).
template <typename T, bool WAVE>
__global__ void crop_cyclic_kernel(const float2 *Y, T *out, int B, int C, int oh, int ow, int Ph, int Pw, int oy, int ox,
                                   float scale, unsigned rows, unsigned xb)
{
    const RowAt at = row_at<1, WAVE>(xb);
    if (at.row >= rows || at.x >= ow) return;
    const unsigned plane = at.row / (unsigned)oh, y = at.row - plane * (unsigned)oh;
    const unsigned k = plane / (unsigned)C, c = plane - k * (unsigned)C;
    int yy = (int)y + oy, xx = at.x + ox;
    yy -= yy >= Ph ? Ph : 0;
    xx -= xx >= Pw ? Pw : 0;
    const float2 v = Y[((long long)plane * Ph + yy) * Pw + xx];
    const long long n = (long long)C * oh * ow, i = 2LL * k * n + ((long long)c * oh + y) * ow + at.x;
    out[i] = (T)(v.x * scale);
    if (2 * (int)k + 1 < B) out[i + n] = (T)(v.y * scale);
}

// out[n][y][x] = scale * Re Y[n][y][x] for the top-left oh x ow window of each of N planes
template <typename T>
__global__ void crop_real_kernel(const float2 *Y, T *out, int oh, int ow, int Ph, int Pw, float scale, long long total)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    int x = (int)(i % ow);
    long long r = i / ow;
    int y = (int)(r % oh);
    long long n = r / oh;
    out[i] = (T)(Y[(n * Ph + y) * (long long)Pw + x].x * scale);
}

static inline unsigned nblocks(long long n) { return (unsigned)((n + 255) / 256); }

template <typename T, int FMT>
static hipError_t launch_pack_pairs(const T *src, void *dst, int B, int C, int h, int w, int Ph, int Pw, hipStream_t s)
{
    const long long rows = (long long)((B + 1) / 2) * C * Ph;
    const int V = Pw % 2 ? 1 : 2;
    const RowGrid g = row_grid(rows, Pw, V);
    if (!g.ok) return hipErrorInvalidValue;
    if (V == 2)
        launch_rows(pack_pairs_kernel<T, FMT, 2, true>, pack_pairs_kernel<T, FMT, 2, false>, g, s, src, dst, B, C, h, w, Ph, Pw, (unsigned)rows, g.xb);
    else
        launch_rows(pack_pairs_kernel<T, FMT, 1, true>, pack_pairs_kernel<T, FMT, 1, false>, g, s, src, dst, B, C, h, w, Ph, Pw, (unsigned)rows, g.xb);
    return hipGetLastError();
}

hipError_t conv_pack_pairs(const void *src, int f64, void *dst, int fmt, int B, int C, int h, int w, int Ph, int Pw,
                           hipStream_t s)
{
    if (fmt == FMT_C16)
        return f64 ? launch_pack_pairs<double, FMT_C16>((const double *)src, dst, B, C, h, w, Ph, Pw, s)
                   : launch_pack_pairs<float, FMT_C16>((const float *)src, dst, B, C, h, w, Ph, Pw, s);
    return f64 ? launch_pack_pairs<double, FMT_C32>((const double *)src, dst, B, C, h, w, Ph, Pw, s)
               : launch_pack_pairs<float, FMT_C32>((const float *)src, dst, B, C, h, w, Ph, Pw, s);
}

template <typename T>
static hipError_t launch_pack_filters(const T *src, float2 *dst, int FC, int fh, int fw, int Ph, int Pw, int rotate, hipStream_t s)
{
    const long long rows = (long long)FC * Ph;
    const int V = Pw % 2 ? 1 : 2;
    const RowGrid g = row_grid(rows, Pw, V);
    if (!g.ok) return hipErrorInvalidValue;
    if (V == 2)
        launch_rows(pack_filters_kernel<T, 2, true>, pack_filters_kernel<T, 2, false>, g, s, src, dst, fh, fw, Ph, Pw, rotate, (unsigned)rows, g.xb);
    else
        launch_rows(pack_filters_kernel<T, 1, true>, pack_filters_kernel<T, 1, false>, g, s, src, dst, fh, fw, Ph, Pw, rotate, (unsigned)rows, g.xb);
    return hipGetLastError();
}

hipError_t conv_pack_filters(const void *src, int f64, float2 *dst, int FC, int fh, int fw, int Ph, int Pw, int rotate,
                             hipStream_t s)
{
    return f64 ? launch_pack_filters((const double *)src, dst, FC, fh, fw, Ph, Pw, rotate, s)
               : launch_pack_filters((const float *)src, dst, FC, fh, fw, Ph, Pw, rotate, s);
}

// Blocks below which a launch of 256-thread blocks leaves compute units idle.
constexpr long long kFillBlocks = 1024;

// Whether tiles of one map may be used: their threads are numbered in 32 bits.
static bool flat_fits(long long P, long long na, long long nb) { return map_blocks(P, na, nb, 1, 1) <= 0x7fffff; }

template <int XFMT, int YFMT>
static hipError_t launch_pointwise(const void *X, const float2 *H, void *Y, int pairs, int C, int F, long long P, hipStream_t s)
{
    // Tiles where both map axes have something to share (one filter shares its spectrum, but with more
    // than one channel to wait for that is not enough) and the launch fills the device; a tile's thread
    // waits as long for each channel's loads, so with fewer blocks one map a thread is faster
    // (us, tiles / one map: 1 pair, 128 channels, 16 filters of 64 x 64 59 / 37; 8 x 64 x 64 of 16 x 16,
    // 32 blocks, 22 / 11; 2 x 8 x 8 of 192 x 192, 288 blocks, 7.9 / 7.0; 4 x 8 x 16 of 160 x 160, 400
    // blocks, 12 / 17).
    const int T = flat_fits(P, pairs, F) && (map_blocks(P, pairs, F) < 300 || pairs == 1 || (F == 1 && C > 1)) ? 1 : kMapTile;
    const long long blocks = map_blocks(P, pairs, F, T, T);
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)blocks), block(256);
    if (T == 1)
        hipLaunchKernelGGL((pointwise_mac_kernel<XFMT, YFMT, 1>), grid, block, 0, s, X, H, Y, pairs, C, F, P);
    else
        hipLaunchKernelGGL((pointwise_mac_kernel<XFMT, YFMT, kMapTile>), grid, block, 0, s, X, H, Y, pairs, C, F, P);
    return hipGetLastError();
}

hipError_t conv_pointwise(const void *X, const float2 *H, void *Y, int fmt, long long pairs, int C, int F, long long P,
                          hipStream_t s, int yfmt)
{
    if (pairs > 0x7fffffffLL) return hipErrorInvalidValue;
    if (fmt != FMT_C16) return launch_pointwise<FMT_C32, FMT_C32>(X, H, Y, (int)pairs, C, F, P, s);
    return yfmt < 0 || yfmt == FMT_C16 ? launch_pointwise<FMT_C16, FMT_C16>(X, H, Y, (int)pairs, C, F, P, s)
                                       : launch_pointwise<FMT_C16, FMT_C32>(X, H, Y, (int)pairs, C, F, P, s);
}

hipError_t conv_quantise(const float2 *R, void *Q, float *partial, float *scale, long long maps, long long P,
                         int nchunk, hipStream_t s)
{
    const long long blocks = maps * nchunk;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(quant_max_kernel, dim3((unsigned)blocks), dim3(256), 0, s, R, partial, P, nchunk);
    hipLaunchKernelGGL(quant_apply_kernel, dim3((unsigned)blocks), dim3(256), 0, s, R, (uint32_t *)Q, partial, scale, P,
                       nchunk);
    return hipGetLastError();
}

template <int FMT>
static hipError_t launch_crop(const void *Y, void *out, int f64, int B, int F, int oh, int ow, int Ph, int Pw, int oy,
                              int ox, float scale, hipStream_t s, const float *map_scale)
{
    const bool vec = !f64 && ow % 4 == 0 && ((uintptr_t)out & 15) == 0;
    const long long rows = (long long)((B + 1) / 2) * F * oh;
    if (rows == 0) return hipSuccess;
    const RowGrid g = row_grid(rows, ow, vec ? 4 : 1);
    if (!g.ok) return hipErrorInvalidValue;
    if (f64)
        launch_rows(crop_unpack_kernel<double, FMT, 1, true>, crop_unpack_kernel<double, FMT, 1, false>, g, s, Y, (double *)out, B, F, oh, ow, Ph, Pw,
                           oy, ox, scale, (unsigned)rows, g.xb, map_scale);
    else if (vec)
        launch_rows(crop_unpack_kernel<float, FMT, 4, true>, crop_unpack_kernel<float, FMT, 4, false>, g, s, Y, (float *)out, B, F, oh, ow, Ph, Pw,
                           oy, ox, scale, (unsigned)rows, g.xb, map_scale);
    else
        launch_rows(crop_unpack_kernel<float, FMT, 1, true>, crop_unpack_kernel<float, FMT, 1, false>, g, s, Y, (float *)out, B, F, oh, ow, Ph, Pw,
                           oy, ox, scale, (unsigned)rows, g.xb, map_scale);
    return hipGetLastError();
}

hipError_t conv_crop(const void *Y, int fmt, void *out, int f64, int B, int F, int oh, int ow, int Ph, int Pw, int oy,
                     int ox, float scale, hipStream_t s, const float *map_scale)
{
    if (fmt == FMT_C16) return launch_crop<FMT_C16>(Y, out, f64, B, F, oh, ow, Ph, Pw, oy, ox, scale, s, map_scale);
    return launch_crop<FMT_C32>(Y, out, f64, B, F, oh, ow, Ph, Pw, oy, ox, scale, s, map_scale);
}

hipError_t conv_pointwise_gw(const float2 *X, const float2 *D, float2 *G, int pairs, int C, int F, int Ph, int Pw,
                             hipStream_t s)
{
    const long long P = (long long)(Ph / 2 + 1) * Pw;
    if ((long long)Ph * Pw > 0x7fffffffLL) return hipErrorInvalidValue;
    // Tiles by the blocks that the largest would give; a tile's thread walks the pairs one after the
    // other, so a launch of few blocks takes the time of one thread's walk (us, 4 x 4 / 2 x 4 / 2 x 2 /
    // 1 x 1: 64 pairs, 3 channels, 8 filters of 16 x 16, 2 blocks, 80 / 57 / 17 / 11; 16 x 16 x 32 of 40 x
    // 40, 128 blocks, 39 / 28 / 12 / 20; of 96 x 96, 608 blocks, 53 / 43 / 52 / 134; of 128 x 128, 1056
    // blocks, 62 / 80 / 84 / 211). Tiles of four repeat loads along an axis of one map (32 x 1 x 64 of 128 x
    // 128: 121 / 98 / 54 / 62).
    const long long full = map_blocks(P, F, C);
    const int tf = full < 128 && flat_fits(P, F, C) ? 1 : full < kFillBlocks || F == 1 || C == 1 ? 2 : kMapTile;
    const int tc = tf == 2 && full >= kFillBlocks / 2 && C >= 3 && F > 1 ? kMapTile : tf;
    const long long blocks = map_blocks(P, F, C, tf, tc);
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)blocks), block(256);
    if (tf == 1)
        hipLaunchKernelGGL((pointwise_gw_kernel<1, 1>), grid, block, 0, s, X, D, G, pairs, C, F, Ph, Pw);
    else if (tc == 2)
        hipLaunchKernelGGL((pointwise_gw_kernel<2, 2>), grid, block, 0, s, X, D, G, pairs, C, F, Ph, Pw);
    else if (tf == 2)
        hipLaunchKernelGGL((pointwise_gw_kernel<2, kMapTile>), grid, block, 0, s, X, D, G, pairs, C, F, Ph, Pw);
    else
        hipLaunchKernelGGL((pointwise_gw_kernel<kMapTile, kMapTile>), grid, block, 0, s, X, D, G, pairs, C, F, Ph, Pw);
    return hipGetLastError();
}

hipError_t conv_pointwise_gi(const float2 *D, const float2 *H, float2 *R, long long pairs, int C, int F, long long P,
                             hipStream_t s)
{
    const long long full = map_blocks(P, pairs, C);
    // One map a thread where tiles would leave the device idle or share nothing along an axis (us,
    // one map / tiles: 64 pairs, 3 channels, 8 filters of 16 x 16, 16 blocks, 3.1 / 4.1; 1 x 32 x 32 of
    // 128 x 128 21 / 26; 16 x 16 x 32 of 64 x 64, 256 blocks, 34 / 18); many filters gain from the split.
    if (flat_fits(P, pairs, C) && F <= 32 && (full < 32 || ((pairs == 1 || (C == 1 && F > 1)) && full < kFillBlocks))) {
        const dim3 flat((unsigned)map_blocks(P, pairs, C, 1, 1));
        hipLaunchKernelGGL((pointwise_gi_kernel<1, 1>), flat, dim3(256), 0, s, D, H, R, (int)pairs, C, F, P);
        return hipGetLastError();
    }
    const bool split = F >= kMapTile && full < kFillBlocks;
    const long long blocks = map_blocks(P, pairs, C, kMapTile, kMapTile, split ? 256 / kMapTile : 256);
    if (blocks > 0x7fffffffLL || pairs > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)blocks), block(256);
    if (split)
        hipLaunchKernelGGL((pointwise_gi_kernel<kMapTile, kMapTile>), grid, block, 0, s, D, H, R, (int)pairs, C, F, P);
    else
        hipLaunchKernelGGL((pointwise_gi_kernel<1, kMapTile>), grid, block, 0, s, D, H, R, (int)pairs, C, F, P);
    return hipGetLastError();
}

// ---------------------------------------------------------------- short filters, host side
int conv_short_rows(int fh, int fw)
{
    if (fw > kShortTaps || fh > kShortTaps) return 0;
    for (int nr : {4, 8, 12, 16, 24})
        if (fh <= nr) return nr;
    return kShortTaps;
}

hipError_t conv_short_tables(float2 *ty, float2 *tx, int nr, int fw, int Ph, int Pw, hipStream_t s)
{
    const long long ny = (long long)(Ph / 2 + 1) * nr, nx = (long long)fw * Pw;
    hipLaunchKernelGGL(gen_dft_rows_kernel, dim3((unsigned)((ny + 255) / 256)), dim3(256), 0, s, ty, Ph, nr, ny);
    hipLaunchKernelGGL(gen_dft_rows_kernel, dim3((unsigned)((nx + 255) / 256)), dim3(256), 0, s, tx, Pw, Pw, nx);
    return hipGetLastError();
}

// Strips of rows per (filter, 64 columns): enough blocks to fill the device, at least 8 rows each.
static int short_strips(long long planes, int Ph, int nkx)
{
    const long long want = (kFillBlocks + planes * nkx - 1) / (planes * nkx), most = (Ph / 2 + 1 + 7) / 8;
    return (int)(want < most ? want : most);
}

template <typename T, int NR>
static void launch_filter_spectrum(const T *src, float2 *H, const float2 *ty, const float2 *tx, unsigned grid, int fh, int fw,
                                   int Ph, int Pw, int rotate, int nkx, int nstrip, hipStream_t s)
{
    hipLaunchKernelGGL((filter_spectrum_kernel<T, NR>), dim3(grid), dim3(256), 0, s, src, H, ty, tx, fh, fw, Ph, Pw, rotate, nkx,
                       nstrip);
}

hipError_t conv_filter_spectrum(const void *src, int f64, float2 *H, const float2 *ty, const float2 *tx, int nr, int FC, int fh,
                                int fw, int Ph, int Pw, int rotate, hipStream_t s)
{
    const int nkx = (Pw + 63) / 64, ns = short_strips(FC, Ph, nkx);
    const long long blocks = (long long)FC * nkx * ns;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
#define MFFT_SHORT_CASE(n)                                                                                                      \
    case n:                                                                                                                     \
        if (f64)                                                                                                                \
            launch_filter_spectrum<double, n>((const double *)src, H, ty, tx, (unsigned)blocks, fh, fw, Ph, Pw, rotate, nkx,    \
                                              ns, s);                                                                           \
        else                                                                                                                    \
            launch_filter_spectrum<float, n>((const float *)src, H, ty, tx, (unsigned)blocks, fh, fw, Ph, Pw, rotate, nkx, ns,  \
                                             s);                                                                                \
        break
    switch (nr) {
    MFFT_SHORT_CASE(4);
    MFFT_SHORT_CASE(8);
    MFFT_SHORT_CASE(12);
    MFFT_SHORT_CASE(16);
    MFFT_SHORT_CASE(24);
    MFFT_SHORT_CASE(kShortTaps);
    default: return hipErrorInvalidValue;
    }
#undef MFFT_SHORT_CASE
    return hipGetLastError();
}

hipError_t conv_crop_cyclic(const float2 *Y, void *out, int f64, int B, int C, int oh, int ow, int Ph, int Pw, int oy,
                            int ox, float scale, hipStream_t s)
{
    const long long rows = (long long)((B + 1) / 2) * C * oh;
    const RowGrid g = row_grid(rows, ow, 1);
    if (!g.ok) return hipErrorInvalidValue;
    oy %= Ph;
    ox %= Pw;
    if (f64)
        launch_rows(crop_cyclic_kernel<double, true>, crop_cyclic_kernel<double, false>, g, s, Y, (double *)out, B, C, oh, ow, Ph, Pw, oy, ox,
                           scale, (unsigned)rows, g.xb);
    else
        launch_rows(crop_cyclic_kernel<float, true>, crop_cyclic_kernel<float, false>, g, s, Y, (float *)out, B, C, oh, ow, Ph, Pw, oy, ox,
                           scale, (unsigned)rows, g.xb);
    return hipGetLastError();
}

hipError_t conv_crop_real(const float2 *Y, void *out, int f64, long long planes, int oh, int ow, int Ph, int Pw,
                          float scale, hipStream_t s)
{
    long long total = planes * oh * ow;
    if (f64)
        hipLaunchKernelGGL(crop_real_kernel<double>, dim3(nblocks(total)), dim3(256), 0, s, Y, (double *)out, oh, ow,
                           Ph, Pw, scale, total);
    else
        hipLaunchKernelGGL(crop_real_kernel<float>, dim3(nblocks(total)), dim3(256), 0, s, Y, (float *)out, oh, ow,
                           Ph, Pw, scale, total);
    return hipGetLastError();
}

template <int FMT>
static void launch_pack_two(const void *a, const void *b, int f64, void *dst, int h, int w, int Ph, int Pw,
                            long long total, hipStream_t s)
{
    if (f64)
        hipLaunchKernelGGL((pack_two_kernel<double, FMT>), dim3(nblocks(total)), dim3(256), 0, s, (const double *)a,
                           (const double *)b, dst, h, w, Ph, Pw, total);
    else
        hipLaunchKernelGGL((pack_two_kernel<float, FMT>), dim3(nblocks(total)), dim3(256), 0, s, (const float *)a,
                           (const float *)b, dst, h, w, Ph, Pw, total);
}

hipError_t conv_pack_two(const void *a, const void *b, int f64, void *dst, int fmt, int h, int w, int Ph, int Pw,
                         hipStream_t s)
{
    long long total = (long long)Ph * Pw;
    if (fmt == FMT_C16)
        launch_pack_two<FMT_C16>(a, b, f64, dst, h, w, Ph, Pw, total, s);
    else
        launch_pack_two<FMT_C32>(a, b, f64, dst, h, w, Ph, Pw, total, s);
    return hipGetLastError();
}

hipError_t conv_pointwise_two(const void *X, const float2 *H0, const float2 *H1, void *Y, int fmt, int Ph, int Pw,
                              hipStream_t s)
{
    if (fmt == FMT_C16)
        hipLaunchKernelGGL(pointwise_two_kernel<FMT_C16>, dim3(nblocks((long long)Ph * Pw)), dim3(256), 0, s, X, H0, H1,
                           Y, Ph, Pw);
    else
        hipLaunchKernelGGL(pointwise_two_kernel<FMT_C32>, dim3(nblocks((long long)Ph * Pw)), dim3(256), 0, s, X, H0, H1,
                           Y, Ph, Pw);
    return hipGetLastError();
}

template <int FMT>
static void launch_crop_two(const void *Y, void *out0, void *out1, int f64, int oh, int ow, int Pw, int oy, int ox,
                            long long total, hipStream_t s)
{
    if (f64)
        hipLaunchKernelGGL((crop_two_kernel<double, FMT>), dim3(nblocks(total)), dim3(256), 0, s, Y, (double *)out0,
                           (double *)out1, oh, ow, Pw, oy, ox, total);
    else
        hipLaunchKernelGGL((crop_two_kernel<float, FMT>), dim3(nblocks(total)), dim3(256), 0, s, Y, (float *)out0,
                           (float *)out1, oh, ow, Pw, oy, ox, total);
}

hipError_t conv_crop_two(const void *Y, int fmt, void *out0, void *out1, int f64, int oh, int ow, int Pw, int oy,
                         int ox, hipStream_t s)
{
    long long total = (long long)oh * ow;
    if (fmt == FMT_C16)
        launch_crop_two<FMT_C16>(Y, out0, out1, f64, oh, ow, Pw, oy, ox, total, s);
    else
        launch_crop_two<FMT_C32>(Y, out0, out1, f64, oh, ow, Pw, oy, ox, total, s);
    return hipGetLastError();
}

}  // namespace mfft
