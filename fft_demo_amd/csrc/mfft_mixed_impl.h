// Mixed-radix tile kernels: contiguous lines of 2^a 3^b 5^c 17^d <= 4096 points, any number of
// them, natural order in and out (included by mfft_mixed.hip, once per precision).
//
// Method: the tile kernel's Stockham schedule (radix-16 stages as DFT-matrix products on the
// matrix cores, the other radices in fp32 on the vector ALUs), with the first stage reading
// global memory and the last one writing it, so LDS carries only what lies between stages.
//
// Bound: instruction issue (about 100 vector instructions a point over three stages) and, for a
// launch of one tile per compute unit, the latency of that tile. 512 threads hold 8 points each
// between the barriers of a stage (81-100 registers, 2-4 workgroups per compute unit by LDS);
// the geometry is runtime, so every index is a product with a reciprocal instead of a division,
// and a stage's item decodes its line and column once for all of its points. 1200 points x 3001
// (16 x 15 x 5, split fp16, 16-bit words): 14.2 us, 2.0 TB/s; the tile kernel with integer
// divisions per element, copies in and out of LDS and radices 3 and 5 apart took 87.3 us.
#pragma once
#include "mfft_butterfly.h"
#include "mfft_fast_impl.h"
#include "mfft_mixed.h"

namespace mfft {
namespace mixed {

using fast::cmulf;
using fast::Elem;
using fast::f4;
using fast::h8;
using fast::b8;
using fast::u4;

enum Role { FIRST = 0, MID = 1, LAST = 2 };
constexpr int NT = kMixThreads;

// What the stages of one tile share. data: nl lines of R points (dense); tw: the stage
// twiddles, both in LDS; gtw: the same table in global memory (uniform reads: the constants
// of the odd butterflies, which then sit in scalar registers).
struct Ctx {
    float2 *data;
    const float2 *tw;
    const float2 *gtw;
    const void *in;
    void *out;
    int R, nl, sign;
    const float *w16;
    int tid;
};

// x / d for 0 <= x < 2^20 with inv = 1.0f / d: x + 0.5 is at least 0.5 / d away from the next
// integer multiple, more than the product's rounding.
__device__ __forceinline__ int fdiv(int x, float inv) { return (int)(((float)x + 0.5f) * inv); }

// W_N^m, m < N, from the table of W_R (N divides R): one scalar load each.
template <int N>
__device__ __forceinline__ void root_table(const Ctx &c, float2 *w)
{
    typedef __attribute__((address_space(4))) const float cf;
    const cf *t = (const cf *)c.gtw;
    const int step = __builtin_amdgcn_readfirstlane(2 * (c.R / N));
#pragma unroll
    for (int m = 1; m < N; ++m) w[m] = make_float2(t[m * step], t[m * step + 1]);
    w[0] = make_float2(1.f, 0.f);
}

template <int N>
__device__ __forceinline__ void dft_n(float2 *v, const float2 *w, int sign, const float *w16)
{
    if constexpr (N == 16)
        fast::dft16v(v, sign, w16);
    else if constexpr (N == 2 || N == 4 || N == 8)
        fast::dft_tail<N>(v, sign, w16);
    else
        dft_odd_w<N>(v, w);
}

constexpr int inv_mod(int a, int m)
{
    for (int x = 1; x < m; ++x)
        if (a * x % m == 1) return x;
    return 1;
}

// N1 x N2 points, N1 and N2 coprime (Good's index maps: no twiddles between the two).
template <int N1, int N2>
__device__ __forceinline__ void dft_pfa(float2 *v, const float2 *w1, const float2 *w2, int sign, const float *w16)
{
    constexpr int N = N1 * N2;
    float2 a[N1][N2];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) {
#pragma unroll
        for (int n2 = 0; n2 < N2; ++n2) a[n1][n2] = v[(N2 * n1 + N1 * n2) % N];
        dft_n<N2>(a[n1], w2, sign, w16);
    }
    constexpr int e1 = N2 * inv_mod(N2 % N1, N1), e2 = N1 * inv_mod(N1 % N2, N2);
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) {
        float2 u[N1];
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) u[n1] = a[n1][k2];
        dft_n<N1>(u, w1, sign, w16);
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) v[(k1 * e1 + k2 * e2) % N] = u[k1];
    }
}

template <int r>
struct Split {
    static constexpr int A = r == 6 || r == 10 ? 2 : r == 12 ? 4 : r == 15 ? 3 : 1;
    static constexpr int B = r / A;
};

// One radix-r stage on the vector ALUs. An item is one r-point butterfly: line t, column col.
template <int r, int ROLE, int INF, int OUTF>
__device__ __forceinline__ void vstage(const Ctx &c, int cols, int s, float inv_cols, float inv_s, float mul)
{
    typedef typename Elem<INF>::raw iraw;
    typedef typename Elem<OUTF>::raw oraw;
    constexpr int MAXI = (kMaxTile + r * NT - 1) / (r * NT);
    constexpr int A = Split<r>::A, B = Split<r>::B;
    const int items = c.nl * cols;
    float2 w1[A > 1 ? A : 1], w2[B];
    if constexpr (r > 1) {
        if constexpr (A == 3) root_table<A>(c, w1);
        if constexpr (B & 1) root_table<B>(c, w2);
    }
    iraw rw[ROLE == FIRST ? MAXI : 1][r];
    float2 v[MAXI][r];
    int at[MAXI], p[MAXI];  // element of the item's first point, line * R + col; column
#pragma unroll
    for (int k = 0; k < MAXI; ++k) {
        const int I = c.tid + k * NT;
        const int t = fdiv(I, inv_cols);
        p[k] = I - t * cols;
        at[k] = t * c.R + p[k];
        if (I < items) {
            if constexpr (ROLE == FIRST) {
#pragma unroll
                for (int j = 0; j < r; ++j) rw[k][j] = reinterpret_cast<const iraw *>(c.in)[(unsigned)(at[k] + j * cols)];
            } else {
#pragma unroll
                for (int j = 0; j < r; ++j) v[k][j] = c.data[at[k] + j * cols];
            }
        }
    }
    if constexpr (ROLE == MID) __syncthreads();  // every read of the tile precedes its writes
#pragma unroll
    for (int k = 0; k < MAXI; ++k) {
        const int I = c.tid + k * NT;
        if (I >= items) continue;
        if constexpr (ROLE == FIRST) {
#pragma unroll
            for (int j = 0; j < r; ++j) v[k][j] = Elem<INF>::f(rw[k][j]);
        }
        if constexpr (r > 1) {
            if constexpr (A > 1)
                dft_pfa<A, B>(v[k], w1, w2, c.sign, c.w16);
            else
                dft_n<r>(v[k], w2, c.sign, c.w16);
        }
        if constexpr (ROLE == LAST) {
            oraw *dst = reinterpret_cast<oraw *>(c.out);
#pragma unroll
            for (int j = 0; j < r; ++j)
                dst[(unsigned)(at[k] + j * cols)] = Elem<OUTF>::pack(make_float2(v[k][j].x * mul, v[k][j].y * mul));
        } else {
            // output j of column q + s p goes to q + s (r p + j), times W_R^(s p j)
            int ps, base, step;
            if constexpr (ROLE == FIRST) {
                ps = p[k];
                base = at[k] + p[k] * (r - 1);
                step = 1;
            } else {
                ps = fdiv(p[k], inv_s) * s;
                base = at[k] + ps * (r - 1);
                step = s;
            }
            if constexpr (ROLE == FIRST) {
#pragma unroll
                for (int j = 0; j < r; ++j) v[k][j] = make_float2(v[k][j].x * mul, v[k][j].y * mul);
            }
#pragma unroll
            for (int j = 1; j < r; ++j) v[k][j] = cmulf(v[k][j], c.tw[j * ps]);
            if constexpr (ROLE == FIRST && r % 2 == 0) {
                // r consecutive words per lane: 16-byte writes (8-byte ones at this stride share banks)
#pragma unroll
                for (int j = 0; j < r; j += 2)
                    *reinterpret_cast<f4 *>(c.data + base + j) = f4{v[k][j].x, v[k][j].y, v[k][j + 1].x, v[k][j + 1].y};
            } else {
#pragma unroll
                for (int j = 0; j < r; ++j) c.data[base + j * step] = v[k][j];
            }
        }
    }
    if constexpr (ROLE != LAST) __syncthreads();
}

// One radix-16 stage on the matrix cores: 16 columns per group, lane (g, col) feeds points
// 4g..4g+3 of its column and receives outputs 4g..4g+3 of it.
template <int PREC, int ROLE, int INF, int OUTF>
__device__ __forceinline__ void mstage(const Ctx &c, const fast::Ops<PREC> &op, int cols, int s, float inv_cols,
                                       float inv_s, float mul)
{
    typedef typename Elem<INF>::raw iraw;
    typedef typename Elem<OUTF>::raw oraw;
    constexpr int NW = NT / 64;
    constexpr int MAXP = kMaxTile / 256 / NW;
    constexpr bool EXACT =
        ROLE == FIRST && ((INF == FMT_C16 && PREC != PREC_BF16) || (INF == FMT_CBF16 && PREC == PREC_BF16));
    const int lane = c.tid & 63, wave = c.tid >> 6;
    const int g = lane >> 4;
    const int slots = c.nl * cols;
    f4 yr[MAXP], yi[MAXP];
    int at[MAXP], col[MAXP];
    iraw rw[ROLE == FIRST ? MAXP : 1][4];
    float2 x[MAXP][4];
#pragma unroll
    for (int u = 0; u < MAXP; ++u) {
        // lanes past the last column repeat it (their outputs are dropped): the matrix
        // instruction takes all 64 lanes
        const int slot = min((wave + u * NW) * 16 + (lane & 15), slots - 1);
        const int t = fdiv(slot, inv_cols);
        col[u] = slot - t * cols;
        at[u] = t * c.R + col[u];
        if ((wave + u * NW) * 16 < slots) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (ROLE == FIRST)
                    rw[u][i] = reinterpret_cast<const iraw *>(c.in)[(unsigned)(at[u] + (4 * g + i) * cols)];
                else
                    x[u][i] = c.data[at[u] + (4 * g + i) * cols];
            }
        }
    }
#pragma unroll
    for (int u = 0; u < MAXP; ++u) {
        if ((wave + u * NW) * 16 >= slots) continue;  // the same for the whole wave
        h8 r16;
        b8 rb;
        if constexpr (ROLE == FIRST) {
            if constexpr (EXACT) {
                const u4 v = {rw[u][0], rw[u][1], rw[u][2], rw[u][3]};
                r16 = __builtin_bit_cast(h8, v);
                rb = __builtin_bit_cast(b8, v);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) x[u][i] = Elem<INF>::f(rw[u][i]);
            }
        }
        fast::dft16<PREC, EXACT>(x[u], r16, rb, op, yr[u], yi[u]);
    }
    if constexpr (ROLE == MID) __syncthreads();
#pragma unroll
    for (int u = 0; u < MAXP; ++u) {
        if ((wave + u * NW) * 16 + (lane & 15) >= slots) continue;
        if constexpr (ROLE == LAST) {
            oraw *dst = reinterpret_cast<oraw *>(c.out);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                dst[(unsigned)(at[u] + (4 * g + i) * cols)] = Elem<OUTF>::pack(make_float2(yr[u][i] * mul, yi[u][i] * mul));
        } else {
            const int ps = ROLE == FIRST ? col[u] : fdiv(col[u], inv_s) * s;
            float2 y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                y[i] = cmulf(make_float2(yr[u][i] * mul, yi[u][i] * mul), c.tw[(4 * g + i) * ps]);
            float2 *d = c.data + at[u] + ps * 15;
            if constexpr (ROLE == FIRST) {
                *reinterpret_cast<f4 *>(d + 4 * g) = f4{y[0].x, y[0].y, y[1].x, y[1].y};
                *reinterpret_cast<f4 *>(d + 4 * g + 2) = f4{y[2].x, y[2].y, y[3].x, y[3].y};
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) d[(4 * g + i) * s] = y[i];
            }
        }
    }
    if constexpr (ROLE != LAST) __syncthreads();
}

template <int PREC, int ROLE, int INF, int OUTF>
__device__ __forceinline__ void stage(const Ctx &c, const fast::Ops<PREC> &op, const MixSched &sc, int st)
{
    const int cols = sc.cols[st], s = sc.s[st];
    const float ic = sc.inv_cols[st], is = sc.inv_s[st], mul = sc.mul[st];
#define MFFT_MIX_CASE(r) \
    case r: vstage<r, ROLE, INF, OUTF>(c, cols, s, ic, is, mul); break
    switch (sc.radix[st]) {
    case 16:
        if constexpr (PREC == PREC_FP32)
            vstage<16, ROLE, INF, OUTF>(c, cols, s, ic, is, mul);
        else
            mstage<PREC, ROLE, INF, OUTF>(c, op, cols, s, ic, is, mul);
        break;
    MFFT_MIX_CASE(3);
    MFFT_MIX_CASE(5);
    MFFT_MIX_CASE(6);
    MFFT_MIX_CASE(9);
    MFFT_MIX_CASE(10);
    MFFT_MIX_CASE(12);
    MFFT_MIX_CASE(15);
    MFFT_MIX_CASE(17);
    default:
        if constexpr (ROLE == FIRST) {
            vstage<1, ROLE, INF, OUTF>(c, cols, s, ic, is, mul);  // a length of one stage: a copy first
        } else {
            switch (sc.radix[st]) {
            MFFT_MIX_CASE(2);
            MFFT_MIX_CASE(4);
            default: vstage<8, ROLE, INF, OUTF>(c, cols, s, ic, is, mul); break;
            }
        }
        break;
    }
#undef MFFT_MIX_CASE
}

template <int PREC, int INF, int OUTF>
__device__ __forceinline__ void tile(const Ctx &c, const fast::Ops<PREC> &op, const MixSched &sc)
{
    stage<PREC, FIRST, INF, OUTF>(c, op, sc, 0);
    for (int st = 1; st < sc.nst - 1; ++st) stage<PREC, MID, INF, OUTF>(c, op, sc, st);
    stage<PREC, LAST, INF, OUTF>(c, op, sc, sc.nst - 1);
}

__device__ __forceinline__ void load_table(float2 *dst, const float2 *src, int R)
{
    for (int i = threadIdx.x; i < R; i += NT) dst[i] = src[i];
}

// One workgroup per tile: in a loop over tiles the lane addresses of every stage are loop
// invariants, which the compiler keeps in registers until they spill.
template <int PREC, int INF, int OUTF>
__global__ void __launch_bounds__(kMixThreads, 4) fft_mixed(MixArgs a)
{
    extern __shared__ __attribute__((aligned(16))) float2 sm[];
    const int R = a.sc.R;
    fast::Ops<PREC> op;
    if constexpr (PREC != PREC_FP32) op.load(reinterpret_cast<const DftOps *>(a.dft_ops), threadIdx.x & 63);
    float2 *tw = sm + a.T * R;
    load_table(tw, a.tw, R);
    __syncthreads();
    const long long l0 = (long long)blockIdx.x * a.T, left = a.nlines - l0;
    const Ctx c{sm, tw, a.tw, reinterpret_cast<const typename Elem<INF>::raw *>(a.in) + l0 * R,
                reinterpret_cast<typename Elem<OUTF>::raw *>(a.out) + l0 * R, R, (int)(left < a.T ? left : a.T), a.sign,
                a.w16, (int)threadIdx.x};
    tile<PREC, INF, OUTF>(c, op, a.sc);
}

// Many transforms of uneven length and count in one launch: workgroup b takes tile b, then
// further tiles from the device-side counter until every tile is handed out. The last
// workgroup to finish leaves the counter at zero for the next launch. 48 items of 16..4096
// points (0.33 M points): 9.1 us per call, one launch; copying the job records, resetting the
// counter and 4096-point tiles on the tile kernel took 58 us.
template <int PREC, int INF, int OUTF>
__global__ void __launch_bounds__(kMixThreads, 4) fft_mixed_queue(MixQueueArgs a)
{
    extern __shared__ __attribute__((aligned(16))) float2 sm[];
    __shared__ unsigned s_next;
    const int lane = threadIdx.x & 63;
    fast::Ops<PREC> op;
    if constexpr (PREC != PREC_FP32) op.load(reinterpret_cast<const DftOps *>(a.dft_ops), lane);
    int t = blockIdx.x, have = -1;  // have: the length whose table is in LDS
    float2 *tw = sm + a.tw_at;
    while (t < a.total) {
        // the last item whose first tile is <= t; 64 items per step
        int j = -1;
        for (int i0 = 0; i0 < a.nitems; i0 += 64) {
            const int i = i0 + lane;
            const int f = i >= a.nitems ? 0x7fffffff : a.first ? a.first[i] : a.first_in[i];
            const int n = __popcll(__ballot(f <= t));
            j += n;
            if (n < 64) break;
        }
        j = __builtin_amdgcn_readfirstlane(j);
        const MixItem it = a.items ? a.items[j] : a.item_in[j];
        const int first = a.first ? a.first[j] : a.first_in[j];
        const int li = __builtin_amdgcn_readfirstlane(it.len);
        const MixLen &len = a.lens[li];
        const int R = len.sc.R;
        if (have != li) {
            load_table(tw, len.tw, R);
            have = li;
        }
        __syncthreads();
        int tid = threadIdx.x;
        __asm__("" : "+v"(tid));  // not a loop invariant: see fft_mixed
        const long long l0 = (long long)(t - first) * it.T, left = it.nlines - l0;
        const Ctx c{sm, tw, len.tw, reinterpret_cast<const typename Elem<INF>::raw *>(it.in) + l0 * R,
                    reinterpret_cast<typename Elem<OUTF>::raw *>(it.out) + l0 * R, R, (int)(left < it.T ? left : it.T),
                    a.sign, a.w16, tid};
        tile<PREC, INF, OUTF>(c, op, len.sc);
        if (a.total <= (int)gridDim.x) return;  // one tile per workgroup: no queue
        if (threadIdx.x == 0) s_next = gridDim.x + atomicAdd(a.counter, 1u);
        __syncthreads();
        t = (int)s_next;
        __syncthreads();
    }
    if (threadIdx.x == 0 && atomicAdd(a.counter + 1, 1u) == gridDim.x - 1) {
        // every workgroup has taken its last number: both counters back to zero
        atomicExch(a.counter, 0u);
        atomicExch(a.counter + 1, 0u);
    }
}

}  // namespace mixed
}  // namespace mfft
