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
// (16 x 15 x 5, split fp16, 16-bit words; a call on new inputs): 13.9 us, 2.1 TB/s; the tile kernel with
// integer divisions per element, copies in and out of LDS and radices 3 and 5 apart took 87.5 us.
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

// Geometry of a kernel: threads per workgroup and the points its tiles hold at most.
// Contiguous lines lie one after the other in LDS. Strided lines (columns) lie interleaved,
// point by point: the tile is then one Stockham array whose innermost factor is the line.
template <bool COLS_, int NT_, int CAP_>
struct Geo {
    static constexpr bool COLS = COLS_;
    static constexpr int NT = NT_, CAP = CAP_;
};

// What the stages of one tile share. data: nl lines of R points; tw: the stage twiddles, both
// in LDS; gtw: the same table in global memory (uniform reads: the constants of the odd
// butterflies, which then sit in scalar registers). in, out: the tile's first element;
// ps_in, ps_out: bytes between a strided line's points.
struct Ctx {
    float2 *data;
    const float2 *tw;
    const float2 *gtw;
    const void *dft_ops;
    const char *in;
    char *out;
    int R, nl, sign;
    unsigned ps_in, ps_out;
    const float *w16;
    int tid;
};

// x / d for 0 <= x < 2^17 with inv = 1 / d to an ulp or two: x + 0.5 is at least 0.5 / d away
// from the next multiple, more than the product's error.
__device__ __forceinline__ int fdiv(int x, float inv) { return (int)(((float)x + 0.5f) * inv); }
__device__ __forceinline__ float recip(int d) { return __builtin_amdgcn_rcpf((float)d); }

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

// Where the columns of a stage lie. A column is r points, the stage's butterfly; item I is a
// (line, column) pair, columns fastest for contiguous lines, lines fastest for strided ones.
// In LDS point j of item I is at lds(I) + j * pitch.
template <class G>
struct Cols {
    int n, pitch, mul;   // items; elements between a column's points; elements per point step
    int cols;
    float inv;
    __device__ __forceinline__ Cols(const Ctx &c, int cols_)
    {
        cols = cols_;
        n = c.nl * cols;
        mul = G::COLS ? c.nl : 1;
        pitch = cols * mul;
        inv = recip(G::COLS ? c.nl : cols);
    }
    // item -> first point's LDS element and column
    __device__ __forceinline__ void at(const Ctx &c, int I, int &e, int &col, int &t) const
    {
        if constexpr (G::COLS) {
            col = fdiv(I, inv);
            t = I - col * c.nl;
            e = I;
        } else {
            t = fdiv(I, inv);
            col = I - t * cols;
            e = t * c.R + col;
        }
    }
    // byte offset of an item's point 0 on the input or output side, and the step between points
    template <int EB>
    __device__ __forceinline__ unsigned goff(int e, int col, int t, unsigned ps) const
    {
        return G::COLS ? (unsigned)t * EB + (unsigned)col * ps : (unsigned)e * EB;
    }
    template <int EB>
    __device__ __forceinline__ unsigned gstep(unsigned ps) const
    {
        return G::COLS ? (unsigned)cols * ps : (unsigned)cols * EB;
    }
};

// One radix-r stage on the vector ALUs.
template <class G, int r, int ROLE, int INF, int OUTF>
__device__ __forceinline__ void vstage(const Ctx &c, int ncols, int s, float mul)
{
    typedef typename Elem<INF>::raw iraw;
    typedef typename Elem<OUTF>::raw oraw;
    constexpr int NT = G::NT, MAXI = (G::CAP + r * NT - 1) / (r * NT);
    constexpr int A = Split<r>::A, B = Split<r>::B;
    const Cols<G> K(c, ncols);
    float2 w1[A > 1 ? A : 1], w2[B];
    if constexpr (r > 1) {
        if constexpr (A == 3) root_table<A>(c, w1);
        if constexpr (B & 1) root_table<B>(c, w2);
    }
    iraw rw[ROLE == FIRST ? MAXI : 1][r];
    float2 v[MAXI][r];
    int e[MAXI], col[MAXI], t[MAXI];
#pragma unroll
    for (int k = 0; k < MAXI; ++k) {
        const int I = c.tid + k * NT;
        K.at(c, I, e[k], col[k], t[k]);
        if (I < K.n) {
            if constexpr (ROLE == FIRST) {
                const unsigned o = K.template goff<sizeof(iraw)>(e[k], col[k], t[k], c.ps_in);
                const unsigned st = K.template gstep<sizeof(iraw)>(c.ps_in);
#pragma unroll
                for (int j = 0; j < r; ++j) rw[k][j] = *reinterpret_cast<const iraw *>(c.in + (o + j * st));
            } else {
#pragma unroll
                for (int j = 0; j < r; ++j) v[k][j] = c.data[e[k] + j * K.pitch];
            }
        }
    }
    if constexpr (ROLE == MID) __syncthreads();  // every read of the tile precedes its writes
    const int sm = s * K.mul;
    const float inv_s = ROLE == MID ? recip(sm) : 0.f;
#pragma unroll
    for (int k = 0; k < MAXI; ++k) {
        if (c.tid + k * NT >= K.n) continue;
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
            const unsigned o = K.template goff<sizeof(oraw)>(e[k], col[k], t[k], c.ps_out);
            const unsigned st = K.template gstep<sizeof(oraw)>(c.ps_out);
#pragma unroll
            for (int j = 0; j < r; ++j)
                *reinterpret_cast<oraw *>(c.out + (o + j * st)) =
                    Elem<OUTF>::pack(make_float2(v[k][j].x * mul, v[k][j].y * mul));
        } else {
            // output j of column q + s p goes to q + s (r p + j), times W_R^(s p j)
            const int p = ROLE == FIRST ? col[k] : fdiv(G::COLS ? e[k] : col[k], inv_s);
            const int ps = p * s, base = e[k] + p * sm * (r - 1);
            if constexpr (ROLE == FIRST) {
#pragma unroll
                for (int j = 0; j < r; ++j) v[k][j] = make_float2(v[k][j].x * mul, v[k][j].y * mul);
            }
#pragma unroll
            for (int j = 1; j < r; ++j) v[k][j] = cmulf(v[k][j], c.tw[j * ps]);
            if constexpr (ROLE == FIRST && !G::COLS && r % 2 == 0) {
                // r consecutive words per lane: 16-byte writes (8-byte ones at this stride share banks)
#pragma unroll
                for (int j = 0; j < r; j += 2)
                    *reinterpret_cast<f4 *>(c.data + base + j) = f4{v[k][j].x, v[k][j].y, v[k][j + 1].x, v[k][j + 1].y};
            } else {
#pragma unroll
                for (int j = 0; j < r; ++j) c.data[base + j * sm] = v[k][j];
            }
        }
    }
    if constexpr (ROLE != LAST) __syncthreads();
}

// One radix-16 stage on the matrix cores: 16 columns per group, lane (g, column) feeds points
// 4g..4g+3 of its column and receives outputs 4g..4g+3 of it.
template <class G, int PREC, int ROLE, int INF, int OUTF>
__device__ __forceinline__ void mstage(const Ctx &c, int ncols, int s, float mul)
{
    typedef typename Elem<INF>::raw iraw;
    typedef typename Elem<OUTF>::raw oraw;
    constexpr int NW = G::NT / 64;
    constexpr int MAXP = (G::CAP / 16 + 16 * NW - 1) / (16 * NW);
    constexpr bool EXACT =
        ROLE == FIRST && ((INF == FMT_C16 && PREC != PREC_BF16) || (INF == FMT_CBF16 && PREC == PREC_BF16));
    // the operands are loaded by the stage that needs them: held through the vector-ALU stages
    // they would cost the kernel a wave per SIMD
    fast::Ops<PREC> op;
    op.load(reinterpret_cast<const DftOps *>(c.dft_ops), c.tid & 63);
    const Cols<G> K(c, ncols);
    const int wave = c.tid >> 6, l15 = c.tid & 15;
    const int g = (c.tid & 63) >> 4;
    f4 yr[MAXP], yi[MAXP];
    int e[MAXP], col[MAXP], t[MAXP];
    iraw rw[ROLE == FIRST ? MAXP : 1][4];
    float2 x[MAXP][4];
#pragma unroll
    for (int u = 0; u < MAXP; ++u) {
        // lanes past the last column repeat it (their outputs are dropped): the matrix
        // instruction takes all 64 lanes
        K.at(c, min((wave + u * NW) * 16 + l15, K.n - 1), e[u], col[u], t[u]);
        if ((wave + u * NW) * 16 < K.n) {
            if constexpr (ROLE == FIRST) {
                const unsigned st = K.template gstep<sizeof(iraw)>(c.ps_in);
                const unsigned o = K.template goff<sizeof(iraw)>(e[u], col[u], t[u], c.ps_in) + 4 * g * st;
#pragma unroll
                for (int i = 0; i < 4; ++i) rw[u][i] = *reinterpret_cast<const iraw *>(c.in + (o + i * st));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) x[u][i] = c.data[e[u] + (4 * g + i) * K.pitch];
            }
        }
    }
#pragma unroll
    for (int u = 0; u < MAXP; ++u) {
        if ((wave + u * NW) * 16 >= K.n) continue;  // the same for the whole wave
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
    const int sm = s * K.mul;
    const float inv_s = ROLE == MID ? recip(sm) : 0.f;
#pragma unroll
    for (int u = 0; u < MAXP; ++u) {
        if ((wave + u * NW) * 16 + l15 >= K.n) continue;
        if constexpr (ROLE == LAST) {
            const unsigned st = K.template gstep<sizeof(oraw)>(c.ps_out);
            const unsigned o = K.template goff<sizeof(oraw)>(e[u], col[u], t[u], c.ps_out) + 4 * g * st;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<oraw *>(c.out + (o + i * st)) =
                    Elem<OUTF>::pack(make_float2(yr[u][i] * mul, yi[u][i] * mul));
        } else {
            const int p = ROLE == FIRST ? col[u] : fdiv(G::COLS ? e[u] : col[u], inv_s);
            const int ps = p * s;
            float2 y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                y[i] = cmulf(make_float2(yr[u][i] * mul, yi[u][i] * mul), c.tw[(4 * g + i) * ps]);
            float2 *d = c.data + e[u] + p * sm * 15;
            if constexpr (ROLE == FIRST && !G::COLS) {
                *reinterpret_cast<f4 *>(d + 4 * g) = f4{y[0].x, y[0].y, y[1].x, y[1].y};
                *reinterpret_cast<f4 *>(d + 4 * g + 2) = f4{y[2].x, y[2].y, y[3].x, y[3].y};
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) d[(4 * g + i) * sm] = y[i];
            }
        }
    }
    if constexpr (ROLE != LAST) __syncthreads();
}

template <class G, int PREC, int ROLE, int INF, int OUTF>
__device__ __forceinline__ void stage(const Ctx &c, const MixSched &sc, int st)
{
    const int cols = sc.cols[st], s = sc.s[st];
    const float mul = sc.mul[st];
#define MFFT_MIX_CASE(r) \
    case r: vstage<G, r, ROLE, INF, OUTF>(c, cols, s, mul); break
    switch (sc.radix[st]) {
    case 16:
        if constexpr (PREC == PREC_FP32)
            vstage<G, 16, ROLE, INF, OUTF>(c, cols, s, mul);
        else
            mstage<G, PREC, ROLE, INF, OUTF>(c, cols, s, mul);
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
            vstage<G, 1, ROLE, INF, OUTF>(c, cols, s, mul);  // a length of one stage: a copy first
        } else {
            switch (sc.radix[st]) {
            MFFT_MIX_CASE(2);
            MFFT_MIX_CASE(4);
            default: vstage<G, 8, ROLE, INF, OUTF>(c, cols, s, mul); break;
            }
        }
        break;
    }
#undef MFFT_MIX_CASE
}

template <class G, int PREC, int INF, int OUTF>
__device__ __forceinline__ void tile(const Ctx &c, const MixSched &sc)
{
    stage<G, PREC, FIRST, INF, OUTF>(c, sc, 0);
    for (int st = 1; st < sc.nst - 1; ++st) stage<G, PREC, MID, INF, OUTF>(c, sc, st);
    stage<G, PREC, LAST, INF, OUTF>(c, sc, sc.nst - 1);
}

template <int NT>
__device__ __forceinline__ void load_table(float2 *dst, const float2 *src, int R)
{
    for (int i = threadIdx.x; i < R; i += NT) dst[i] = src[i];
}

// Waves per SIMD the registers are held to. Contiguous lines, 1200 x 3001 in us at 4 / 5 / 6 / 8:
// fp32 15.5 / 15.6 / 14.8 / 13.2; split fp16 spills from 6 on.
template <int PREC>
constexpr int row_waves() { return PREC == PREC_FP32 ? 8 : PREC == PREC_SPLIT ? 5 : 6; }

// One workgroup per tile: in a loop over tiles the lane addresses of every stage are loop
// invariants, which the compiler keeps in registers until they spill.
template <int PREC, int INF, int OUTF>
__global__ void __launch_bounds__(kMixThreads, row_waves<PREC>()) fft_mixed(MixArgs a)
{
    typedef Geo<false, kMixThreads, kMaxTile> G;
    extern __shared__ __attribute__((aligned(16))) float2 sm[];
    const int R = a.sc.R;
    float2 *tw = sm + a.T * R;
    load_table<G::NT>(tw, a.tw, R);
    __syncthreads();
    const long long l0 = (long long)blockIdx.x * a.T, left = a.nlines - l0;
    const Ctx c{sm, tw, a.tw, a.dft_ops,
                reinterpret_cast<const char *>(a.in) + l0 * R * (long long)sizeof(typename Elem<INF>::raw),
                reinterpret_cast<char *>(a.out) + l0 * R * (long long)sizeof(typename Elem<OUTF>::raw),
                R, (int)(left < a.T ? left : a.T), a.sign, 0u, 0u, a.w16, (int)threadIdx.x};
    tile<G, PREC, INF, OUTF>(c, a.sc);
}

// Strided lines: the lines of a transform are adjacent (a point of T lines is one segment of
// memory), c0 of them, transforms in_dist / out_dist elements apart. CAP: points per tile.
// Bound: instruction issue, and segment length (16 lines of 16-bit words are 64 bytes). Tiles
// of up to 8192 points run 512 threads at 16 points each, two workgroups per compute unit (480
// x 640 x 18 2D split fp16 39.9 us; 256 threads 44.4, 1024 threads 42.1); longer lines fill the
// LDS with one workgroup of 1024, and tiles of up to 2048 points (narrow transforms, short lines) run
// 256 threads, more of which are busy (2D, 16-bit intermediates, in us, 512 / 256 threads: 5461 x 48 x
// 16 54 / 41, in two passes of columns 46; 1000 x 24 x 24 11.1 / 9.2; 5461 x 1000 x 2 104 / 47; 500 x 96
// x 16 11.2 / 11.0, with 128 threads 11.6). 2D execs with both axes on the mixed-radix kernels against an
// odd pass and a power-of-two pass per axis (us), execs repeated on the same buffers: 480 x 640 x 18
// fp32 89 -> 40, split fp16 86 -> 40, 960 x 960 x 16 fp32 164 -> 96, 96 x 96 x 100 split fp16 90 ->
// 14. On new inputs at every call, which come from memory: 480 x 640 x 18 fp32 95.6 -> 47.4.
template <int CAP, int PREC, int INF, int OUTF>
__global__ void __launch_bounds__(mix_col_threads(CAP), 4) fft_mixed_cols(MixColArgs a)
{
    typedef Geo<true, mix_col_threads(CAP), CAP> G;
    typedef typename Elem<INF>::raw iraw;
    typedef typename Elem<OUTF>::raw oraw;
    extern __shared__ __attribute__((aligned(16))) float2 sm[];
    const int R = a.sc.R;
    float2 *tw = sm + a.T * R;
    load_table<G::NT>(tw, a.tw, R);
    __syncthreads();
    // each XCD (workgroups are dealt to the 8 of them in turn) takes a run of tiles, so that
    // neighbouring tiles, which share cache lines, meet in one L2
    unsigned b = blockIdx.x;
    const unsigned nb = gridDim.x;
    if ((nb & 7) == 0) b = (b & 7) * (nb >> 3) + (b >> 3);
    const unsigned tr = b / (unsigned)a.tiles0, t0 = b - tr * (unsigned)a.tiles0;
    const int l0 = (int)t0 * a.T;
    const Ctx c{sm, tw, a.tw, a.dft_ops, reinterpret_cast<const char *>(reinterpret_cast<const iraw *>(a.in) + tr * a.in_dist + l0),
                reinterpret_cast<char *>(reinterpret_cast<oraw *>(a.out) + tr * a.out_dist + l0),
                R, min(a.c0 - l0, a.T), a.sign, (unsigned)(a.ps_in * (int)sizeof(iraw)), (unsigned)(a.ps_out * (int)sizeof(oraw)),
                a.w16, (int)threadIdx.x};
    tile<G, PREC, INF, OUTF>(c, a.sc);
}

// Many transforms of uneven length and count in one launch: workgroup b takes tile b, then
// further tiles from the device-side counter until every tile is handed out. The last
// workgroup to finish leaves the counter at zero for the next launch. 48 items of 16..4096
// points (0.33 M points): 9.5 us per call, one launch; copying the job records, resetting the
// counter and 4096-point tiles on the tile kernel took 58 us.
template <int PREC, int INF, int OUTF>
__global__ void __launch_bounds__(kMixThreads, 4) fft_mixed_queue(MixQueueArgs a)
{
    typedef Geo<false, kMixThreads, kMaxTile> G;
    extern __shared__ __attribute__((aligned(16))) float2 sm[];
    __shared__ unsigned s_next;
    const int lane = threadIdx.x & 63;
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
            load_table<G::NT>(tw, len.tw, R);
            have = li;
        }
        __syncthreads();
        int tid = threadIdx.x;
        __asm__("" : "+v"(tid));  // not a loop invariant: see fft_mixed
        const long long l0 = (long long)(t - first) * it.T, left = it.nlines - l0;
        const Ctx c{sm, tw, len.tw, a.dft_ops,
                    reinterpret_cast<const char *>(it.in) + l0 * R * (long long)sizeof(typename Elem<INF>::raw),
                    reinterpret_cast<char *>(it.out) + l0 * R * (long long)sizeof(typename Elem<OUTF>::raw),
                    R, (int)(left < it.T ? left : it.T), a.sign, 0u, 0u, a.w16, tid};
        tile<G, PREC, INF, OUTF>(c, len.sc);
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
