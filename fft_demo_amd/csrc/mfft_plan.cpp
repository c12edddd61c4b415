// Host side of the matrix-core FFT: planner, device tables, exec and the C ABI.
//
// The reference plans a fixed radix/"merging" table per size (tcfftCreate,
// tcfft_half.cu:1235-1345; tcfftCreate_2d, tcfft_half_2d.cu:1151-1221) and launches one
// in-block pass plus strided merge passes (tcfftExec, tcfft_half.cu:1177-1233). This
// planner decomposes any supported axis length with the four-step method instead:
//   L = L1 * L2 :  pass A = L2 strided DFT_L1 (stride L2) times the twiddle W_L^(n2*k1),
//                  then DFT_L2 on each row k1, written to k1 + L1*k2 (recursively).
// Every pass is one launch of the tile kernel; intermediates live in a per-plan
// workspace, processed in batch chunks small enough to stay in the 256 MB Infinity Cache.
#include "../../include/mfft.h"
#include "mfft_common.h"
#include "mfft_fast.h"
#include "mfft_internal.h"
#include "mfft_mixed.h"
#include "mfft_onchip.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

namespace mfft {
hipError_t gen_twiddle(float2 *out, long long n, long long count, long long mult, int sign, hipStream_t s,
                       double scale = 1.0);
hipError_t gen_dft_ops(DftOps *ops, int sign, hipStream_t s);
hipError_t gen_w16(float *host3);
typedef void (*tile_fn)(TileArgs);
tile_fn find_tile_kernel(int prec, int R, int TL, bool generic);
tile_fn find_merged_tile_kernel(int prec, int R, bool small);
int pow2_tile_lines(int R, int TL);
hipError_t launch_tile(const void *fn, const TileArgs &a, long long ntiles, hipStream_t stream, hipEvent_t start = nullptr,
                       hipEvent_t stop = nullptr);
const void *find_small_kernel(int R, int inf, int outf);
hipError_t launch_queue(int prec, const TileArgs *jobs, const long long *first_tile, int njobs, long long total,
                        unsigned long long *counter, int grid, hipStream_t s);
int queue_grid(int prec);
hipError_t stage_convert(const void *src, int sfmt, void *dst, int dfmt, long long n_inner, long long batch,
                         const int *perm_x, int nx, const int *perm_y, int ny, double scale, hipStream_t s);
}  // namespace mfft

using namespace mfft;

// ------------------------------------------------------------------ errors
static thread_local std::string g_err;

static int fail(int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

#define HIP_TRY(expr)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess) return fail(MFFT_ERR_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

// ------------------------------------------------------------------ factorisation
static bool is_pow2(long long n) { return n > 0 && (n & (n - 1)) == 0; }

// Stage radices of one in-tile line length, tail stage first (matches fft_tile_pow2).
static bool line_radices(int R, std::vector<int> &out)
{
    out.clear();
    if (R < 2) return false;
    int n = R, e2 = 0;
    while (n % 2 == 0) { n /= 2; ++e2; }
    int tail2 = 1 << (e2 % 4);
    int n16 = e2 / 4;
    if (tail2 > 1) out.push_back(tail2);
    // odd factors
    const int odd[] = {17, 5, 3};
    for (int p : odd)
        while (n % p == 0) { out.push_back(p); n /= p; }
    if (n != 1) return false;
    for (int i = 0; i < n16; ++i) out.push_back(16);
    return true;
}

// The radix list that defines the digit-reversed input order of a length-n axis.
// The sizes tcfftCreate knows get the reference's own lists (tcfft_half.cu:1250-1330:
// the tail after every second radix-16 digit, where its 512/1024-point passes put it);
// every other length: radix-16 digits first, then the 2/4/8 tail, then odd factors.
static void rev_radices(int n, std::vector<int> &out)
{
    out.clear();
    switch (n) {
    case 1 << 17: out = {16, 16, 2, 16, 16}; return;
    case 1 << 18: out = {16, 16, 2, 16, 16, 2}; return;
    case 1 << 19: out = {16, 16, 4, 16, 16, 2}; return;
    case 1 << 24: out = {16, 16, 16, 16, 16, 16}; return;
    case 1 << 25: out = {16, 16, 2, 16, 16, 16, 16}; return;
    case 1 << 26: out = {16, 16, 2, 16, 16, 2, 16, 16}; return;
    case 1 << 27: out = {16, 16, 2, 16, 16, 2, 16, 16, 2}; return;
    default: break;
    }
    int m = n, e2 = 0;
    while (m % 2 == 0) { m /= 2; ++e2; }
    for (int i = 0; i < e2 / 4; ++i) out.push_back(16);
    if (e2 % 4) out.push_back(1 << (e2 % 4));
    const int odd[] = {17, 5, 3};
    for (int p : odd)
        while (m % p == 0) { out.push_back(p); m /= p; }
}

static void gen_rev(int n, const std::vector<int> &radices, std::vector<int> &rev)
{
    // restates gen_rev (tcfft_half.cu:1351-1374)
    std::vector<int> a(n), b(n);
    for (int i = 0; i < n; ++i) a[i] = i;
    int now = n;
    for (int i = (int)radices.size() - 1; i >= 0; --i) {
        int r = radices[i], sub = now / r;
        for (int j = 0; j < n; j += now)
            for (int k = 0; k < r; ++k)
                for (int l = 0; l < sub; ++l) b[j + l + k * sub] = a[j + l * r + k];
        now = sub;
        std::swap(a, b);
    }
    rev = a;
}

// DigitRev of an index whose digits, least significant first, have the radices `digits`
// (powers of two, at most four digits): the result holds the digits in reverse order.
static bool make_digit_rev(const std::vector<int> &digits, DigitRev &d)
{
    memset(&d, 0, sizeof d);
    if (digits.size() > 4) return false;
    int total = 0;
    for (int r : digits) {
        if (!is_pow2(r)) return false;
        total += __builtin_ctz(r);
    }
    int sh = 0;
    d.n = (int)digits.size();
    for (size_t i = 0; i < digits.size(); ++i) {
        const int w = __builtin_ctz(digits[i]);
        d.sh[i] = sh;
        d.mask[i] = digits[i] - 1;
        d.out[i] = total - sh - w;
        sh += w;
    }
    return true;
}

// Lines of length R stored in the digit-reversed order of `list` (position p holds natural
// point gen_rev(list)[p]) can be read by the fast kernels' first stage when the list starts
// with 16 and the rest reverses with a DigitRev q: natural point col + (R/16) j is then at
// position j + 16 q(col). Fills q and checks that identity on every point.
static bool fast_rev_spec(int R, const std::vector<int> &list, DigitRev &q)
{
    if (R < 64 || !is_pow2(R) || list.empty() || list[0] != 16) return false;
    long long prod = 1;
    for (int r : list) prod *= r;
    if (prod != R) return false;
    std::vector<int> col_digits(list.rbegin(), list.rend() - 1);  // r_{m-1}, ..., r_1
    if (!make_digit_rev(col_digits, q)) return false;
    std::vector<int> rev;
    gen_rev(R, list, rev);
    const int R16 = R / 16;
    for (int pos = 0; pos < R; ++pos) {
        const int n = rev[pos];
        if (pos != n / R16 + 16 * digit_rev(n % R16, q)) return false;
    }
    return true;
}

// ------------------------------------------------------------------ plan structures
struct Level {
    long long count, in_stride, out_stride;
    bool batch;  // the batch level (chunked at exec time)
};

enum Buf { BUF_IN = 0, BUF_OUT = 1, BUF_WORK = 2 };

struct PassSpec {
    int R;
    long long ps_in, ps_out;
    std::vector<Level> lines;
    int tw_N = 0;
    int tw_level = -1;  // index into lines
    int src = BUF_IN, dst = BUF_OUT;
    int perm_axis = -1; // axis whose digit-reversal is fused into this pass's loads
    // the pass's input lines are stored in the digit-reversed order of this radix list
    // (gen_rev, tcfft_half.cu:1351-1374); empty = natural order
    std::vector<int> rev_list;
    DigitRev rev_tw{};  // four-step twiddle line factor of a digit-reversed first pass
    long long work_stride = 0;  // workspace elements per transform when padded (0 = dense)
    // derived
    std::vector<int> radix;
    bool generic = false;
    int fast_kind = -1;   // KIND_* of the fast kernel, -1 = tile kernel
    bool small = false;   // streaming short-DFT kernel (R <= 16, one thread per line)
    float2 *stage_tw_s = nullptr, *tw_lo_s = nullptr;
    float last_mul = 1.f, tail_mul = 1.f;
    long long max_grid = 0;  // persistent grid of the fast kernel; tiles the mixed one wants
    int TL = 1, T = 1;
    int l0 = 0, l1 = -1, l2 = -1;  // indices into lines
    const void *fn = nullptr;
    float2 *tw_lo = nullptr, *tw_hi = nullptr;
    int tw_bits = 0;
    float2 *stage_tw = nullptr;
    int *perm = nullptr;
    bool rev_fast = false;  // the fast kernel reads the digit-reversed lines (rev_q)
    DigitRev rev_q{};
    bool onchip = false;    // the whole 65536-point line in one pass (fft_onchip)
    bool onchip_cols = false;  // 2048-point lines, 32 per workgroup (fft_onchip_cols)
    bool onchip_rows = false;  // ... contiguous lines stored transposed (its rows kind)
    bool mixed = false;     // lines on the mixed-radix kernels (fft_mixed, fft_mixed_cols)
    bool col_axis = false;  // a pass of a 2D plan's column axis
    int mixed_cap = 0;      // strided lines: points per tile at most; 0 = dense contiguous lines
    MixSched mix{};
};

struct mfft_plan_s {
    int kind = 1;
    int n = 0, nx = 0, ny = 0;
    long long batch = 0;
    mfft_desc d{};
    long long total = 0;      // complex elements per transform
    int mid_fmt = FMT_C32;
    std::vector<PassSpec> passes;
    DftOps *ops = nullptr;
    void *work = nullptr;
    long long work_bytes = 0;
    long long chunk = 1;
    double out_scale = 1.0;
    long long cus = 256;      // compute units, asked for once (at every pass: 2 us of a 16 x 16 conv's 23)
    std::vector<void *> allocs;
    std::vector<int> rev_axis[2];
    std::vector<int> rev_list_axis[2];  // the radix lists rev_axis was generated from
    std::mutex exec_mu;       // the workspace is per plan
    StreamOrder ws_order;     // streams that used the plan's own workspace
    // A plan whose passes include an on-chip kernel (one workgroup per line, or per 32
    // columns) keeps the plan of the same transform without it for execs of fewer than
    // small_below transforms, which would leave most of the device idle on the on-chip pass.
    mfft_plan_s *small = nullptr;
    long long small_below = 0;
    // A 1D plan of odd * 2^a points whose one pass writes elements of another size than it reads keeps
    // the plan of an odd pass and a power-of-two pass, which meet in a workspace, for execs in place:
    // in one pass, tiles would overwrite lines that others have not read.
    mfft_plan_s *aliased = nullptr;
    // A transform of the conv operator: no mixed-radix kernels. Their stages round in another order
    // than the passes its filters and images have always gone through; with 16-bit words on the way
    // the difference grows to whole fp16 steps (1e-4 of the fp32 result), and the filter gradient's
    // inverse, whose values are near fp16's smallest, changes in its third digit.
    bool conv = false;
    // Intermediates that a pass stores in the output buffer are kept in mid_fmt (the last
    // pass writes out_fmt there): with 16-bit intermediates and 32-bit output, every pass
    // boundary then moves 16-bit words. Execs must not alias a pass's source and destination
    // across a format change (checked at exec).
    bool out_mid = false;
};

// Element formats a pass reads and writes.
static int src_fmt(const mfft_plan_s *p, const PassSpec &ps)
{
    if (ps.src == BUF_IN) return p->d.in_fmt;
    if (ps.src == BUF_OUT) return p->out_mid ? p->mid_fmt : p->d.out_fmt;
    return p->mid_fmt;
}
static int dst_fmt(const mfft_plan_s *p, const PassSpec &ps)
{
    if (ps.dst == BUF_OUT) return p->out_mid && &ps != &p->passes.back() ? p->mid_fmt : p->d.out_fmt;
    if (ps.dst == BUF_IN) return p->d.in_fmt;
    return p->mid_fmt;
}

// Transforms (lines, or images of 2048-row 2D plans) an on-chip pass needs to occupy the
// device enough to beat the multi-pass plan: a workgroup per 65536-point line, 2/3 of the
// compute units (65536 x 256 on 256 CUs: 36 us against 53 us; at 128 lines the two-pass plan is
// faster); a workgroup per 32 columns of 2048 points, 3/4 of them (2048 x 2048: one image
// 49 us against 38 us, eight 129 us against 149 us).
static long long device_cus()
{
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) !=
                                                 hipSuccess || ncu < 1)
        ncu = 256;
    return ncu;
}
static long long onchip_min_lines() { return (2 * device_cus() + 2) / 3; }
static long long onchip_rows_min_lines(int l1)
{
    const long long blocks = std::max(1, l1 / kOnchipColsLines);
    return std::max(1LL, (3 * device_cus() / 4 + blocks - 1) / blocks);
}
static long long onchip_cols_min_images(int ny)
{
    const long long blocks = std::max(1, ny / kOnchipColsLines);
    return std::max(1LL, (3 * device_cus() / 4 + blocks - 1) / blocks);
}

static int fmt_bytes(int fmt) { return fmt == FMT_C32 ? 8 : 4; }

// ------------------------------------------------------------------ axis planning
// fast_cols: the pass may run on the strided matrix-core kernel (natural-order input), which
// holds 8192 / R lines of up to kColsMaxR points per tile; the tile kernels hold at most
// kMaxTile points, so a strided single pass there needs R <= kMaxTile / 16 for 16 lines.
static bool single_pass_ok(int R, long long ps_in, const std::vector<Level> &lines, bool fast_cols)
{
    if (R < 2 || R > kMaxTile) return false;
    std::vector<int> rad;
    if (!line_radices(R, rad)) return false;
    if (ps_in == 1) return true;
    bool has_unit = false;
    for (auto &l : lines)
        if (l.in_stride == 1) has_unit = true;
    if (!has_unit) return true;
    return R * 16 <= kMaxTile || (fast_cols && is_pow2(R) && R >= 64 && R <= kColsMaxR);
}

static bool factorable(long long n)
{
    std::vector<int> r;
    return n <= kMaxTile && line_radices((int)n, r);
}

static long long odd_part(long long L)
{
    while (L > 0 && L % 2 == 0) L /= 2;
    return L;
}

// Odd factors the streaming kernel takes as a pass of its own.
static bool small_odd(long long o) { return o == 3 || o == 5 || o == 9 || o == 15 || o == 17; }

// Lines per tile of the strided mixed-radix kernels at most: 32 up to 256 points (a point of a
// tile is then a segment of 128 bytes of 16-bit words), 16 up to 1088, 8 up to 2176.
static int mixed_col_lines(long long R)
{
    return R * 32 <= kMixColSmall ? 32 : R * 16 <= kMixColLarge ? 16 : R * 8 <= kMixColLarge ? 8 : 0;
}

// An axis with odd factors that runs in one pass of the mixed-radix kernels instead of an odd
// pass and a power-of-two pass. Where the two passes stay (us, two passes / one): contiguous
// lines above 2048 points with a factor 17 on the matrix cores, one line a tile, whose radix-17
// stage then keeps a quarter of the threads busy (2176 x 4000 split fp16: 39 / 43, with 16-bit
// intermediates 31 / 43; plain fp32 45 / 36, 3072 x 4000 split fp16 60 / 42); strided lines
// above 1088 points with 16-bit words, 8 lines a tile, segments of 32 bytes (2176 x 2176 x 4
// split fp16 110 / 151, plain fp32 209 / 185; 1088 x 1088 x 16 split fp16 129 / 119).
static bool mixed_one_pass(int prec, long long L, long long ps_in, long long ps_out, const std::vector<Level> &lines)
{
    std::vector<int> r;
    if (is_pow2(L) || L > kMaxTile || !mix_radices((int)L, r)) return false;
    if (ps_in == 1 && ps_out == 1) return prec == PREC_FP32 || L <= kMaxTile / 2 || L % 17 || !small_odd(odd_part(L));
    const long long T = mixed_col_lines(L);
    if (ps_in == 1 || T < (prec == PREC_FP32 ? 8 : 16) || std::max(ps_in, ps_out) * L >= (1LL << 29)) return false;
    for (auto &l : lines)
        if (l.in_stride == 1 && l.out_stride == 1 && !l.batch) return lines.size() <= 2;
    return false;
}

// Whether a plan's intermediates between passes are 16-bit (the rule finalize_plan applies).
static bool narrow_mid(const mfft_desc *d)
{
    if (d->mid_fmt >= 0) return d->mid_fmt != MFFT_FMT_C32;
    return d->precision == MFFT_PREC_FP16 || d->precision == MFFT_PREC_BF16;
}

// Append the passes of a length-L DFT along an axis. Input element (line, j) is at
// line_in + j*ps_in, output element (line, k) at line_out + k*ps_out.
// narrow: the intermediates between passes are 16-bit (an extra pass costs 8 bytes a point)
// rev_cols: a digit-reversed strided axis may still run in one pass of the strided
// matrix-core kernel (it reads the reversed order itself)
// mixed: the precision whose mixed-radix kernels exist for the axis's formats, -1 = none
static int plan_axis(std::vector<PassSpec> &out, long long L, long long ps_in, long long ps_out,
                     std::vector<Level> lines, int src, int dst, int perm_axis, int split_hint, bool narrow,
                     bool rev_cols = false, int mixed = -1)
{
    // odd * 2^a (2176 = 17 x 128): the odd factor in a streaming pass, the power of two on
    // the matrix-core kernels, instead of one generic mixed-radix tile pass.
    // split_hint = 1 keeps the single pass.
    const long long odd = odd_part(L);
    const bool odd_split = perm_axis < 0 && split_hint != 1 && odd > 1 && small_odd(odd) && L / odd >= 16 &&
                           L / odd <= kMaxTile;
    const bool fast_cols = (perm_axis < 0 || rev_cols) && split_hint <= 1;  // no split asked for
    // 1088 = 17 * 64 columns of 16-bit words at a wide pitch keep their two passes, for any batch (14
    // transforms of 1088 x 2048, 3072 and 4096 with 16-bit intermediates: 133, 282 and 254 us, in one
    // pass 142, 300 and 273; one and two of 1088 x 2048 30 and 37, in one 24 and 31; 3 of 1088 x 1024
    // 37, in one 33)
    const bool wide = narrow && odd_split && L > 1024 && ps_in >= 2048;
    const bool one_mixed =
        mixed >= 0 && perm_axis < 0 && split_hint <= 1 && !wide && mixed_one_pass(mixed, L, ps_in, ps_out, lines);
    if (one_mixed || (!odd_split && single_pass_ok((int)std::min<long long>(L, 1 << 30), ps_in, lines, fast_cols))) {
        PassSpec p;
        p.R = (int)L;
        p.ps_in = ps_in;
        p.ps_out = ps_out;
        p.lines = lines;
        p.src = src;
        p.dst = dst;
        p.perm_axis = perm_axis;
        out.push_back(p);
        return MFFT_OK;
    }
    // pass A's destination: the workspace, or -- when this axis must end in the workspace
    // (rows of a 2D transform) -- the output buffer, which is free until the last axis
    int a_dst = BUF_WORK;
    if (dst == BUF_WORK) {
        if (!odd_split || src != BUF_IN)
            return fail(MFFT_ERR_UNSUPPORTED, "an inner axis longer than %d points is not supported", kMaxTile);
        a_dst = BUF_OUT;
    }
    if (perm_axis >= 0)
        return fail(MFFT_ERR_UNSUPPORTED,
                    "digit-reversed input is supported for axes done in one pass (length <= %d)", kMaxTile);
    // choose L1 (strided pass, <= 256) and L2 = L / L1
    long long L1 = 0;
    if (odd_split) {
        L1 = odd;
    } else if (split_hint > 1 && L % split_hint == 0 && factorable(split_hint) &&
               (split_hint <= 256 || (is_pow2(split_hint) && split_hint <= kColsMaxR))) {
        L1 = split_hint;
    } else if (is_pow2(L) && ps_in != 1 && L >= 512 && L <= 4096) {
        // strided axis (2D columns) of 512..4096 points: both passes are strided; the first
        // on the matrix-core kernel (L / 16 points, at least 64), the rest (16 or fewer) on
        // the streaming kernel (2048 x 2048: 1.1x the 16 + 128 split, measured)
        L1 = std::max<long long>(64, L / 16);
    } else if (is_pow2(L) && ps_in != 1 && L % 256 == 0 && L / 256 <= 256) {
        // longer strided axes: give the second pass the 256-point matrix-core kernel and the
        // small remainder to the first
        L1 = L / 256;
    } else if (is_pow2(L)) {
        int m = 0;
        while ((1LL << m) < L) ++m;
        int m1 = (m + 1) / 2;
        if (m1 > 8) m1 = 8;
        if (m - m1 > 12 && m1 < 8) m1 = std::min(8, m - 12);
        // 2^17..2^19 (contiguous lines): a long strided first pass -- 1024 points at 8 lines
        // per tile with 16-bit intermediates, 512 at 16 lines with 32-bit ones -- and the
        // rest (128..1024 points) in one pass; the autotuner's pick on MI355X for split fp16
        // and fp32, 1.02-1.18x the 256-point first pass (and the three passes below)
        if (ps_in == 1 && m >= 17 && m <= 19) {
            m1 = narrow ? 10 : 9;
        } else if (narrow && m >= 19 && m <= 21) {
            // 2^20..2^21 with 16-bit intermediates: a second pass of 2048 or 4096 points
            // would hold one or two lines per tile and store them transposed in 4- or
            // 8-byte pieces; three passes instead, the rest (8192 = 128 x 64) split again
            // below (split fp16: 1.05-1.3x faster; with fp32 intermediates the third pass
            // costs more than it saves)
            m1 = m - 13;
        }
        L1 = 1LL << m1;
    } else {
        for (long long c = 256; c >= 2; --c)
            if (L % c == 0 && factorable(c) && (L / c <= kMaxTile ? factorable(L / c) : true)) {
                L1 = c;
                break;
            }
    }
    if (L1 < 2 || L % L1 != 0) return fail(MFFT_ERR_UNSUPPORTED, "cannot factor axis length %lld", L);
    long long L2 = L / L1;
    // pass A: DFT_L1 over n1 (stride L2*ps_in) for each (line, n2); in-place layout
    PassSpec a;
    a.R = (int)L1;
    a.ps_in = L2 * ps_in;
    a.ps_out = L2 * ps_in;
    a.lines = lines;
    for (auto &l : a.lines) l.out_stride = l.in_stride;  // pass A keeps the input layout
    a.lines.push_back(Level{L2, ps_in, ps_in, false});
    a.tw_N = (int)L;
    a.tw_level = (int)a.lines.size() - 1;
    a.src = src;
    a.dst = a_dst;
    out.push_back(a);
    // remaining: DFT_L2 over n2 for each (line, k1); output at k1 + L1*k2
    // input side of the sub-problem reads pass A's output, laid out like the input
    std::vector<Level> sub2;
    for (auto &l : lines) sub2.push_back(Level{l.count, l.in_stride, l.out_stride, l.batch});
    sub2.push_back(Level{L1, L2 * ps_in, ps_out, false});
    return plan_axis(out, L2, ps_in, L1 * ps_out, sub2, a_dst, dst, -1, 1, narrow);
}

// 65536-point lines with 16-bit words in, out and between the two 256-point halves, in
// natural order or in the digit-reversed order of the radix list {16, 16, 16, 16}: one pass
// of the on-chip kernel (the line is read and written once) instead of the four-step pair,
// unless a split is asked for (split_hint > 1). The halves are the same four-step
// decomposition (tcfft_half.cu:266-390 then 69-161 for the reference's long lines).
static bool plan_onchip(mfft_plan_s *p, const mfft_desc *d)
{
    if (p->n != kOnchipN || d->split_hint > 1) return false;
    const bool rev = d->in_order == MFFT_ORDER_DIGIT_REVERSED;
    if (rev && p->rev_list_axis[0] != std::vector<int>{16, 16, 16, 16}) return false;
    const int fmt = d->precision == MFFT_PREC_BF16 ? MFFT_FMT_CBF16 : MFFT_FMT_C16;
    const int mid = d->mid_fmt >= 0                         ? d->mid_fmt
                    : d->precision == MFFT_PREC_FP16 ? MFFT_FMT_C16
                    : d->precision == MFFT_PREC_BF16 ? MFFT_FMT_CBF16
                                                     : MFFT_FMT_C32;
    if (d->in_fmt != fmt || d->out_fmt != fmt || mid != fmt) return false;
    if (!find_onchip_kernel(d->precision, fmt, rev)) return false;
    PassSpec ps;
    ps.R = kOnchipN;
    ps.ps_in = ps.ps_out = 1;
    ps.lines = {Level{p->batch, kOnchipN, kOnchipN, true}};
    ps.tw_N = kOnchipN;  // the four-step tables between the halves
    ps.tw_level = 0;
    ps.src = BUF_IN;
    ps.dst = BUF_OUT;
    ps.onchip = true;
    if (rev) ps.rev_list = p->rev_list_axis[0];
    p->passes.push_back(ps);
    return true;
}

// N = L1 x 2048 (2^19, 2^20) with 16-bit words in, out and between the passes: the four-step
// split with the 2048-point half on the on-chip line kernel -- pass A: DFT_L1 over n1 (stride
// 2048, the strided matrix-core kernel) times W_N^(n2 k1); pass B: DFT_2048 of each row k1, 32
// rows per workgroup read whole and stored transposed at k1 + L1 k2. Split fp16 on MI355X:
// 2^20 x 16 / 64 in 72 / 303 us against 78 / 316 us for the three-pass plan, 2^19 x 32 / 64 in
// 63 / 131 us against 68 / 172 us for 1024 + 512; at 2^17 and 2^18 (L1 = 64, 128) it was no
// faster than the 1024-point first pass, which those lengths keep.
static bool plan_onchip_rows(mfft_plan_s *p, const mfft_desc *d)
{
    const long long N = p->n;
    if (N < (1LL << 19) || N > (1LL << 20) || !is_pow2(N) || d->in_order != MFFT_ORDER_NATURAL || d->split_hint > 1)
        return false;
    const int L1 = (int)(N / kOnchipColsN);
    const int fmt = d->precision == MFFT_PREC_BF16 ? MFFT_FMT_CBF16 : MFFT_FMT_C16;
    const int mid = d->mid_fmt >= 0                         ? d->mid_fmt
                    : d->precision == MFFT_PREC_FP16 ? MFFT_FMT_C16
                    : d->precision == MFFT_PREC_BF16 ? MFFT_FMT_CBF16
                                                     : MFFT_FMT_C32;
    if (d->in_fmt != fmt || d->out_fmt != fmt || mid != fmt) return false;
    if (!find_onchip_cols_kernel(d->precision, fmt, true) || !find_fast_kernel(d->precision, L1, KIND_COLS, fmt, fmt))
        return false;
    PassSpec a;
    a.R = L1;
    a.ps_in = a.ps_out = kOnchipColsN;
    a.lines = {Level{p->batch, N, N, true}, Level{kOnchipColsN, 1, 1, false}};
    a.tw_N = (int)N;
    a.tw_level = 1;
    a.src = BUF_IN;
    a.dst = BUF_WORK;
    PassSpec b;
    b.R = kOnchipColsN;
    b.ps_in = 1;
    b.ps_out = L1;
    b.lines = {Level{L1, kOnchipColsN, 1, false}, Level{p->batch, N, N, true}};
    b.src = BUF_WORK;
    b.dst = BUF_OUT;
    b.onchip_cols = b.onchip_rows = true;
    p->passes.push_back(a);
    p->passes.push_back(b);
    return true;
}

// Digit-reversed input (tcfftExec's order, tcfft_half.cu:1177-1233) of a 1D length longer
// than one tile: N = L1 L2, split after the first m radices of the list. Position
// p = p_lo + L1 p_hi holds natural element n2 + L2 n1 with n1 = gen_rev(list[:m])[p_lo] and
// n2 = gen_rev(list[m:])[p_hi], so
//   pass A: each contiguous block p_hi is a digit-reversed line of list[:m]: DFT_L1 over n1,
//           times W_N^(n2 k1) (n2 = the digit reversal of p_hi), stored transposed at
//           k1 L2 + p_hi;
//   pass B: row k1 of the workspace is a digit-reversed line of list[m:] (position p_hi holds
//           n2): DFT_L2, stored transposed at k1 + L1 k2, natural order.
// Both passes read contiguous lines. The halves must start with a radix-16 digit and run
// on the fast kernels, and L1, L2 are kept to 256..1024 points (longer lines hold too few
// per tile for the transposed stores).
static int plan_reversed_1d(mfft_plan_s *p)
{
    const std::vector<int> &list = p->rev_list_axis[0];
    const long long N = p->n;
    int best = -1;
    double bestd = 1e9;
    long long L1 = 1;
    for (size_t m = 1; m < list.size(); ++m) {
        L1 *= list[m - 1];
        const long long L2 = N / L1;
        if (list[0] != 16 || list[m] != 16 || L1 < 256 || L1 > 1024 || L2 < 256 || L2 > 1024) continue;
        const double dd = std::fabs(std::log2((double)L1) - std::log2((double)L2));
        if (dd < bestd) {
            bestd = dd;
            best = (int)m;
        }
    }
    if (best < 0) return fail(MFFT_ERR_UNSUPPORTED, "digit-reversed input of length %lld in two passes", N);
    std::vector<int> lo(list.begin(), list.begin() + best), hi(list.begin() + best, list.end());
    L1 = 1;
    for (int r : lo) L1 *= r;
    const long long L2 = N / L1;
    PassSpec a;
    a.R = (int)L1;
    a.ps_in = 1;
    a.ps_out = L2;
    a.lines = {Level{L2, L1, 1, false}, Level{p->batch, N, N, true}};
    a.tw_N = (int)N;
    a.tw_level = 0;
    a.src = BUF_IN;
    a.dst = BUF_WORK;
    a.rev_list = lo;
    if (!make_digit_rev(hi, a.rev_tw)) return fail(MFFT_ERR_UNSUPPORTED, "twiddle line reversal");
    {
        std::vector<int> rh;
        gen_rev((int)L2, hi, rh);
        for (int ph = 0; ph < (int)L2; ++ph)
            if (rh[ph] != digit_rev(ph, a.rev_tw)) return fail(MFFT_ERR_UNSUPPORTED, "twiddle line reversal");
    }
    PassSpec b;
    b.R = (int)L2;
    b.ps_in = 1;
    b.ps_out = L1;
    b.lines = {Level{L1, L2, 1, false}, Level{p->batch, N, N, true}};
    b.src = BUF_WORK;
    b.dst = BUF_OUT;
    b.rev_list = hi;
    p->passes.push_back(a);
    p->passes.push_back(b);
    return MFFT_OK;
}

// Whether a pass reads and writes whole contiguous lines that follow each other without gaps
// (a level's stride is the extent of the levels below it), on both sides alike; the batch is
// the outermost level, so that holds for any number of transforms.
static bool dense_rows(const PassSpec &ps)
{
    if (ps.ps_in != 1 || ps.ps_out != 1) return false;
    std::vector<Level> v = ps.lines;
    std::sort(v.begin(), v.end(), [](const Level &a, const Level &b) { return a.in_stride < b.in_stride; });
    long long stride = ps.R;
    for (size_t i = 0; i < v.size(); ++i) {
        if (v[i].in_stride != stride || v[i].out_stride != stride || (v[i].batch && i + 1 != v.size())) return false;
        stride *= v[i].count;
    }
    return true;
}

// Lines per tile of the mixed-radix kernel: as many as kMaxTile points hold, fewer when the
// launch would otherwise make fewer than `tiles` of them (two per compute unit).
static int mixed_tile_lines(int R, long long nlines, long long tiles)
{
    const long long most = std::max(1, kMaxTile / R), want = nlines / tiles;
    return (int)std::max(1LL, std::min(most, want));
}

// Order of a pass's stages on the mixed-radix kernels: none in which a 16-bit operand has less range
// or precision than in the passes of the same axis in two, a streaming pass of the odd factor in fp32,
// then the power of two, from 64 points on 16 before the even rest. (Strided lines of odd * 16 points
// are two streaming passes: 272 x 64 bf16 3.0e-3 off, with a matrix-core stage 3.2e-3. 320 points, split
// fp16 with 32-bit ends: unscaled inputs above 65504 / 5 overflow, with 16 last above 65504 / 20;
// scaled ones of 2^-8 are 1.7e-5 off, with 16 last 3.5e-5.) Results of split fp16 in 16-bit words are
// coarser than either; there 16 comes last, which rows of 64 and 128 times an odd factor run up to 5%
// faster.
static MixOrder mixed_order(const mfft_desc &d, int in_fmt, int R, bool cols)
{
    const int odd = (int)odd_part(R);
    if (!small_odd(odd) || (d.precision == PREC_SPLIT && d.out_fmt != FMT_C32)) return MIX_16_LAST;
    if (cols && R / odd == 16) return MIX_NO16;
    if (R / odd < 64) return MIX_16_LAST;
    return d.scale == MFFT_SCALE_STAGE || in_fmt != FMT_C32 ? MIX_16_EARLY : MIX_16_AFTER_ODD;
}

// Choose tile geometry and kernel for every pass.
static int finish_passes(mfft_plan_s *p)
{
    p->cus = device_cus();
    for (auto &ps : p->passes) {
        if (ps.onchip_cols) {
            ps.radix = {16, 16, 8};
            ps.fast_kind = KIND_ONCHIP_COLS;
            ps.fn = find_onchip_cols_kernel(p->d.precision, p->mid_fmt, ps.onchip_rows);
            ps.l0 = 0;
            ps.T = kOnchipColsLines;
            ps.TL = 1;
            if (!ps.fn) return fail(MFFT_ERR_UNSUPPORTED, "no on-chip column kernel for the formats");
            continue;
        }
        if (ps.onchip) {
            ps.radix = {16, 16, 16, 16};
            ps.fast_kind = KIND_ONCHIP;
            ps.fn = find_onchip_kernel(p->d.precision, p->d.in_fmt, !ps.rev_list.empty());
            ps.rev_fast = !ps.rev_list.empty();  // the kernel reads the stored order itself
            ps.l0 = 0;
            ps.T = 1;
            ps.TL = 1;
            if (!ps.fn) return fail(MFFT_ERR_UNSUPPORTED, "no on-chip kernel for the formats");
            continue;
        }
        if (!line_radices(ps.R, ps.radix)) return fail(MFFT_ERR_UNSUPPORTED, "line length %d", ps.R);
        if (ps.perm_axis >= 0 && ps.rev_list.empty()) ps.rev_list = p->rev_list_axis[ps.perm_axis];
        const bool rev = !ps.rev_list.empty();
        // merge adjacent levels that are contiguous on both sides (never the batch level)
        // choose l0
        int unit_in = -1, unit_out = -1;
        for (int i = 0; i < (int)ps.lines.size(); ++i) {
            if (ps.lines[i].in_stride == 1 && unit_in < 0) unit_in = i;
            if (ps.lines[i].out_stride == 1 && unit_out < 0) unit_out = i;
        }
        bool strided = ps.ps_in != 1;
        bool pow2 = is_pow2(ps.R) && ps.R >= 16;
        const int in_fmt = src_fmt(p, ps);
        const int out_fmt = dst_fmt(p, ps);
        if (p->out_mid && ps.src == ps.dst && in_fmt != out_fmt)
            return fail(MFFT_ERR_UNSUPPORTED, "in-place pass changes the element format");
        // digit-reversed lines on the fast kernels: the list starts with 16 and the rest
        // reverses digit by digit (every reference list does)
        ps.rev_fast = rev && fast_rev_ok(p->d.precision, in_fmt) && fast_rev_spec(ps.R, ps.rev_list, ps.rev_q);
        // strided lines longer than a 16-line tile kernel holds: the strided matrix-core
        // kernel when it exists for the formats (8192 / R lines of up to kColsMaxR points)
        const bool cols_long = strided && unit_in >= 0 && ps.R * 16 > kMaxTile && pow2 && ps.R <= kColsMaxR &&
                               (!rev || ps.rev_fast) && ps.lines[unit_in].out_stride == 1 &&
                               find_fast_kernel(p->d.precision, ps.R, KIND_COLS, in_fmt, out_fmt) != nullptr;
        if (strided && unit_in >= 0 && (ps.R * 16 <= kMaxTile || cols_long)) {
            ps.l0 = unit_in;
            ps.TL = 16;
        } else if (!strided) {
            ps.TL = 1;
            if (ps.ps_out != 1 && unit_out >= 0)
                ps.l0 = unit_out;
            else {
                // the level with the smallest input stride
                int best = 0;
                for (int i = 1; i < (int)ps.lines.size(); ++i)
                    if (ps.lines[i].in_stride < ps.lines[best].in_stride) best = i;
                ps.l0 = best;
            }
        } else {
            ps.l0 = 0;
            ps.TL = 1;
            pow2 = false;
        }
        ps.generic = !pow2;
        // short strided DFTs: streaming kernel, one thread per line
        if (!rev && ps.ps_in != 1 &&
            (ps.R == 2 || ps.R == 4 || ps.R == 8 || ps.R == 16 || small_odd(ps.R))) {
            const void *fn = find_small_kernel(ps.R, in_fmt, out_fmt);
            if (fn) {
                ps.small = true;
                ps.fn = fn;
                ps.l0 = unit_in >= 0 ? unit_in : 0;
                ps.T = 1;
                ps.TL = 1;
                ps.radix.assign(1, ps.R);
            }
        }
        // fast kernel: power of two 64..4096, natural order or digit-reversed lines it reads
        if (!ps.small && pow2 && ps.R >= 64 && ps.R <= kMaxTile && (!rev || ps.rev_fast)) {
            int kind = -1, l0 = -1;
            if (ps.ps_in == 1 && ps.ps_out == 1) {
                kind = KIND_ROWS;
                l0 = 0;
                for (int i = 1; i < (int)ps.lines.size(); ++i)
                    if (ps.lines[i].in_stride < ps.lines[l0].in_stride) l0 = i;
            } else if (ps.ps_in == 1 && unit_out >= 0) {
                kind = KIND_ROWS_TR;
                l0 = unit_out;
            } else if (ps.ps_in != 1 && ps.R <= kColsMaxR) {
                for (int i = 0; i < (int)ps.lines.size(); ++i)
                    if (ps.lines[i].in_stride == 1 && ps.lines[i].out_stride == 1) { l0 = i; break; }
                if (l0 >= 0) kind = KIND_COLS;
            }
            const void *fn = kind >= 0 ? (const void *)find_fast_kernel(p->d.precision, ps.R, kind, in_fmt, out_fmt) : nullptr;
            if (fn) {
                ps.fast_kind = kind;
                ps.l0 = l0;
                ps.T = fast_tile_lines(ps.R, kind);
                ps.TL = kind == KIND_COLS ? cols_lines(ps.R) : 1;
                ps.fn = fn;
                int dev = 0, ncu = 0, nb = 0;
                HIP_TRY(hipGetDevice(&dev));
                HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
                HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, fast_threads(p->d.precision, ps.R, kind), 0));
                ps.max_grid = (long long)std::max(1, nb) * std::max(1, ncu);
                ps.max_grid -= ps.max_grid % 8;
                if (ps.max_grid < 8) ps.max_grid = 8;
                // radix order of the fast schedule: 16, tail, 16, ...
                std::vector<int> r2;
                int tail = 1;
                for (int r : ps.radix) if (r != 16) tail = r;
                r2.push_back(16);
                if (tail > 1) r2.push_back(tail);
                for (size_t i = 1; i < ps.radix.size() - (tail > 1 ? 1 : 0); ++i) r2.push_back(16);
                ps.radix = r2;
            }
        }
        if (ps.fast_kind < 0) ps.rev_fast = false;
        const bool mixed_cols = !is_pow2(ps.R) && ps.ps_in != 1 && mixed_one_pass(p->d.precision, ps.R, ps.ps_in, ps.ps_out, ps.lines);
        if (!p->conv && !ps.small && ps.fast_kind < 0 && !rev && !ps.tw_N && (mixed_cols || (ps.generic && dense_rows(ps)))) {
            const int T = mixed_cols ? mixed_col_lines(ps.R) : 0;
            long long most = T;  // lines a tile has: a narrow transform has fewer
            if (mixed_cols)
                for (auto &l : ps.lines)
                    if (l.in_stride == 1 && l.out_stride == 1 && !l.batch) most = std::min<long long>(T, l.count);
            ps.mixed_cap = !mixed_cols ? 0 : ps.R * most <= kMixColTiny ? kMixColTiny : ps.R * T <= kMixColSmall ? kMixColSmall : kMixColLarge;
            const void *fn = find_mixed_kernel(p->d.precision, in_fmt, out_fmt, ps.mixed_cap);
            if (fn && mix_schedule(ps.R, p->d.precision, p->d.scale == MFFT_SCALE_STAGE, mixed_order(p->d, in_fmt, ps.R, mixed_cols), ps.mix)) {
                ps.mixed = true;
                ps.fn = fn;
                ps.radix.assign(ps.mix.radix, ps.mix.radix + ps.mix.nst);
                long long nl = 1;
                for (auto &l : ps.lines) nl *= l.count;
                ps.max_grid = 2 * p->cus;
                ps.TL = 1;
                ps.l0 = 0;
                if (mixed_cols) {
                    for (int i = 0; i < (int)ps.lines.size(); ++i)
                        if (ps.lines[i].in_stride == 1 && ps.lines[i].out_stride == 1 && !ps.lines[i].batch) ps.l0 = i;
                    ps.T = (int)std::min<long long>(T, ps.lines[ps.l0].count);
                } else {
                    ps.T = mixed_tile_lines(ps.R, nl, ps.max_grid);
                }
                // every plan of the kernel sets its largest: plans share the function
                HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, mix_lds_max(ps.mixed_cap)));
            }
        }
        if (rev && !ps.rev_fast && ps.perm_axis < 0)
            return fail(MFFT_ERR_UNSUPPORTED, "digit-reversed %d-point lines need the matrix-core kernels", ps.R);
        if (ps.fast_kind >= 0 || ps.small || ps.mixed) {
            // l0 chosen above
        } else if (!ps.generic) {
            ps.T = pow2_tile_lines(ps.R, ps.TL);
        } else {
            int t = kMaxTile / ps.R;
            if (ps.TL == 16 && t < 16) ps.TL = 1;
            ps.T = std::max(1, t);
            if (ps.TL > ps.T) ps.TL = 1;
            if (ps.T % ps.TL) ps.T = ps.TL;
        }
        // remaining levels -> l1, l2 (at most two besides l0)
        std::vector<int> rest;
        if (ps.tw_N && ps.tw_level != ps.l0) rest.push_back(ps.tw_level);
        for (int i = 0; i < (int)ps.lines.size(); ++i)
            if (i != ps.l0 && !(ps.tw_N && i == ps.tw_level)) rest.push_back(i);
        if (rest.size() > 2) return fail(MFFT_ERR_UNSUPPORTED, "too many line levels");
        ps.l1 = rest.size() > 0 ? rest[0] : -1;
        ps.l2 = rest.size() > 1 ? rest[1] : -1;
        if (ps.tw_N && ps.tw_level != ps.l0 && ps.tw_level != ps.l1)
            return fail(MFFT_ERR_UNSUPPORTED, "twiddle level layout");
        if (ps.fast_kind < 0 && !ps.small && !ps.mixed) {
            ps.fn = (const void *)find_tile_kernel(p->d.precision, ps.R, ps.TL, ps.generic);
            if (!ps.fn) return fail(MFFT_ERR_UNSUPPORTED, "no kernel for R=%d TL=%d", ps.R, ps.TL);
        }
    }
    return MFFT_OK;
}

// The VALU butterflies' constants (TileArgs::w16), generated on the GPU once per process by
// the first plan or batcher.
static float g_w16[3];
static std::once_flag g_w16_once;
static hipError_t g_w16_err = hipSuccess;

static int ensure_w16()
{
    std::call_once(g_w16_once, [] { g_w16_err = gen_w16(g_w16); });
    if (g_w16_err != hipSuccess) return fail(MFFT_ERR_HIP, "generating the butterfly constants: %s", hipGetErrorString(g_w16_err));
    return MFFT_OK;
}

static int alloc_dev(mfft_plan_s *p, void **ptr, size_t bytes)
{
    hipError_t e = hipMalloc(ptr, bytes ? bytes : 16);
    if (e != hipSuccess) return fail(MFFT_ERR_NOMEM, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
    p->allocs.push_back(*ptr);
    return MFFT_OK;
}

static int build_tables(mfft_plan_s *p)
{
    if (ensure_w16()) return MFFT_ERR_HIP;
    int sign = p->d.direction;
    if (alloc_dev(p, (void **)&p->ops, sizeof(DftOps))) return MFFT_ERR_NOMEM;
    HIP_TRY(gen_dft_ops(p->ops, sign, 0));
    for (auto &ps : p->passes) {
        // the on-chip kernel's stages are 256-point halves; the column kernel's second half
        // is 128 points (its 2048-point twiddle table is built below)
        const int Rst = ps.onchip ? 256 : ps.onchip_cols ? 128 : ps.R;
        if (alloc_dev(p, (void **)&ps.stage_tw, sizeof(float2) * Rst)) return MFFT_ERR_NOMEM;
        HIP_TRY(gen_twiddle(ps.stage_tw, Rst, Rst, 1, sign, 0));
        if (ps.tw_N) {
            int bits = 0;
            while ((1LL << (2 * bits)) < ps.tw_N) ++bits;
            long long nlo = 1LL << bits, nhi = (ps.tw_N + nlo - 1) / nlo;
            ps.tw_bits = bits;
            if (alloc_dev(p, (void **)&ps.tw_lo, sizeof(float2) * nlo)) return MFFT_ERR_NOMEM;
            if (alloc_dev(p, (void **)&ps.tw_hi, sizeof(float2) * nhi)) return MFFT_ERR_NOMEM;
            HIP_TRY(gen_twiddle(ps.tw_lo, ps.tw_N, nlo, 1, sign, 0));
            HIP_TRY(gen_twiddle(ps.tw_hi, ps.tw_N, nhi, nlo, sign, 0));
        }
        if (ps.fast_kind >= 0) {
            // radix-16 stage scale (1/16 per stage when scaling), divided by the factor 16
            // carried by the matrix-core operands; the fp32 path has no such factor
            double fac = (p->d.scale == MFFT_SCALE_STAGE ? 1.0 / 16 : 1.0) /
                         (p->d.precision == MFFT_PREC_FP32 ? 1.0 : 16.0);
            ps.last_mul = (float)fac;
            int tail = 1;
            for (int r : ps.radix) if (r != 16) tail = r;
            ps.tail_mul = (p->d.scale == MFFT_SCALE_STAGE) ? 1.0f / tail : 1.0f;
            if (alloc_dev(p, (void **)&ps.stage_tw_s, sizeof(float2) * Rst)) return MFFT_ERR_NOMEM;
            HIP_TRY(gen_twiddle(ps.stage_tw_s, Rst, Rst, 1, sign, 0, fac));
            if (ps.tw_N) {
                long long nlo = 1LL << ps.tw_bits;
                if (alloc_dev(p, (void **)&ps.tw_lo_s, sizeof(float2) * nlo)) return MFFT_ERR_NOMEM;
                HIP_TRY(gen_twiddle(ps.tw_lo_s, ps.tw_N, nlo, 1, sign, 0, fac));
            }
        }
        if (ps.onchip_cols) {
            // W_2048^e with the radix-16 stage scale, e in [0, 2048)
            if (alloc_dev(p, (void **)&ps.tw_lo_s, sizeof(float2) * kOnchipColsN)) return MFFT_ERR_NOMEM;
            HIP_TRY(gen_twiddle(ps.tw_lo_s, kOnchipColsN, kOnchipColsN, 1, sign, 0, ps.last_mul));
        }
        if (ps.small) ps.last_mul = p->d.scale == MFFT_SCALE_STAGE ? 1.0f / ps.R : 1.0f;
        if (ps.perm_axis >= 0 && p->d.in_order == MFFT_ORDER_DIGIT_REVERSED && !ps.rev_fast) {
            const std::vector<int> &rev = p->rev_axis[ps.perm_axis];
            if ((int)rev.size() != ps.R) return fail(MFFT_ERR_INVALID, "permutation size");
            if (alloc_dev(p, (void **)&ps.perm, sizeof(int) * ps.R)) return MFFT_ERR_NOMEM;
            HIP_TRY(hipMemcpy(ps.perm, rev.data(), sizeof(int) * ps.R, hipMemcpyHostToDevice));
        }
    }
    HIP_TRY(hipDeviceSynchronize());
    return MFFT_OK;
}

static int finalize_plan(mfft_plan_s *p)
{
    p->mid_fmt = (p->d.precision == MFFT_PREC_FP16) ? FMT_C16
                 : (p->d.precision == MFFT_PREC_BF16) ? FMT_CBF16
                                                      : FMT_C32;
    if (p->d.mid_fmt >= 0) p->mid_fmt = p->d.mid_fmt;
    int rc = finish_passes(p);
    if (rc) return rc;
    // scale bookkeeping
    double sc = 1.0;
    for (auto &ps : p->passes)
        for (int r : ps.radix) sc /= (p->d.scale == MFFT_SCALE_STAGE ? r : 1);
    p->out_scale = sc;
    // workspace and batch chunking
    bool need_work = false;
    for (auto &ps : p->passes)
        if (ps.src == BUF_WORK || ps.dst == BUF_WORK) need_work = true;
    long long wper = p->total;
    for (auto &ps : p->passes) wper = std::max(wper, ps.work_stride);
    long long per = wper * fmt_bytes(p->mid_fmt);
    long long limit = p->d.workspace_limit > 0 ? p->d.workspace_limit : (128LL << 20);
    p->chunk = p->batch;
    if (need_work) {
        long long c = std::max(1LL, limit / std::max(1LL, per));
        // as many chunks as the limit needs, of equal size (8 transforms under a limit of 7:
        // 4 + 4, not 7 + 1, whose one-transform launch would leave most of the device idle)
        const long long nch = (p->batch + c - 1) / c;
        p->chunk = std::min(p->batch, (p->batch + nch - 1) / nch);
        p->work_bytes = p->chunk * per;
        if (!p->d.external_workspace && alloc_dev(p, &p->work, (size_t)p->work_bytes)) return MFFT_ERR_NOMEM;
    }
    return build_tables(p);
}

// Lines per tile of a strided mixed-radix pass, of c0 lines per transform: fewer when the launch would
// leave compute units without a tile.
static int mixed_col_tile(const PassSpec &ps, long long c0, long long transforms)
{
    int T = ps.T;
    while (T > 8 && (c0 + T - 1) / T * transforms < ps.max_grid / 2) T /= 2;
    return T;
}

static int check_desc(const mfft_desc *d)
{
    if (d->precision < 0 || d->precision > 3) return fail(MFFT_ERR_INVALID, "precision %d", d->precision);
    if (d->direction != -1 && d->direction != 1) return fail(MFFT_ERR_INVALID, "direction %d", d->direction);
    if (d->scale != 0 && d->scale != 1) return fail(MFFT_ERR_INVALID, "scale %d", d->scale);
    if (d->in_fmt < 0 || d->in_fmt > 2 || d->out_fmt < 0 || d->out_fmt > 2)
        return fail(MFFT_ERR_INVALID, "format");
    if (d->in_order != 0 && d->in_order != 1) return fail(MFFT_ERR_INVALID, "in_order");
    if (d->mid_fmt < -1 || d->mid_fmt > 2) return fail(MFFT_ERR_INVALID, "mid_fmt");
    if (d->split_hint < 0) return fail(MFFT_ERR_INVALID, "split_hint %d", d->split_hint);
    return MFFT_OK;
}

// ------------------------------------------------------------------ exec
static void *buf_ptr(int which, const void *in, void *out, void *work)
{
    return which == BUF_IN ? const_cast<void *>(in) : which == BUF_OUT ? out : work;
}

// Launch-trace record of one pass launch: kernel family, line length and formats, and the
// algorithmic bytes (every element read and written once; a fused real-image input reads
// the images' pixels, a fused multiplier its table once).
static void trace_pass(const mfft_plan_s *p, const PassSpec &ps, const TileArgs &a, long long nb, long long b0,
                       hipStream_t s)
{
    const char *fam = ps.small ? "stream"
                      : ps.mixed ? (ps.mixed_cap ? "mixed_cols" : "mixed_rows")
                      : ps.fast_kind == KIND_ROWS ? "fast_rows"
                      : ps.fast_kind == KIND_ROWS_TR ? "fast_rows_tr"
                      : ps.fast_kind == KIND_COLS ? "fast_cols"
                      : ps.fast_kind == KIND_ONCHIP ? "onchip"
                      : ps.fast_kind == KIND_ONCHIP_COLS ? "onchip_cols"
                      : ps.generic ? "tile_generic" : "tile";
    const long long pts = (long long)a.c0 * a.c1 * a.c2 * ps.R;
    long long rd = pts * fmt_bytes(a.in_fmt);
    char src[16];
    snprintf(src, sizeof src, "%s", fmt_name(a.in_fmt));
    if (a.real_src) {
        // transforms b0 .. b0 + nb - 1: transform t holds channel t % C of images 2k and 2k + 1
        // (k = t / C; the second from real_src2 when given, absent past the batch)
        long long planes = 0;
        for (long long t = b0; t < b0 + nb; ++t) {
            const long long k = t / std::max(1, a.real_c);
            planes += (2 * k < a.real_b) + (a.real_src2 ? 1 : (2 * k + 1 < a.real_b));
        }
        rd = planes * a.real_h * a.real_w * (a.real_f64 ? 8 : 4);
        snprintf(src, sizeof src, "%s", a.real_f64 ? "real64" : "real32");
    }
    if (a.in_mul) rd += std::min(pts, a.in_mul_period) * 8;
    char name[64];
    snprintf(name, sizeof name, "%s R%d %s%s>%s%s", fam, ps.R, src, a.in_mul ? "*H" : "",
             a.crop_out ? "real32" : fmt_name(a.out_fmt), a.merge ? " merged" : "");
    (void)p;
    long long wr = pts * fmt_bytes(a.out_fmt);
    if (a.crop_out)  // the planes of the chunk's transforms (2 per transform, or 1)
        wr = (a.crop_b ? std::min(2 * nb, (long long)a.crop_b * a.crop_c) : nb) * a.crop_h * a.crop_w * 4;
    trace_launch(s, name, rd, wr);
}

// The second pass of a contiguous axis odd * 2^a has groups of `odd` lines: adjacent in the output,
// and on the input the lines of all groups follow each other. Where a group does not fill whole
// tiles, tiles take lines across groups (TileArgs::merge): 17 x 128 points otherwise fill 17 of a
// fast tile's 32 lines, 15 x 32 15 of a tile kernel's 128 (2176 points x 8704 lines, 16-bit words:
// 39.2 -> 32.1 us; 480 x 15360, fp32: 113 -> 37.6). Not where the groups' own tiles all run at once:
// fewer, fuller tiles then leave compute units idle (conv 183 x 657 x 2, 240 groups of 3 lines: 36
// us, merged into 45 tiles 42), nor up to four tiles a compute unit of the tile kernel's longer lines,
// which has no small tiles for them, or where those are over 60% full: a merged store walks the output
// value by value (whole set_filters calls of an fp16 operator, groups of 3 lines of 64 points: 768 of
// them 27.9 us, merged into 36 tiles 31.6; 2048 of them 33.6, merged 29.8; 2048 groups of 3 x 1024
// points 86 and 93).
static void merge_line_groups(const PassSpec &ps, long long cus, TileArgs &a)
{
    const bool fast = ps.fast_kind == KIND_ROWS_TR;
    const bool tile = ps.fast_kind < 0 && !ps.small && !ps.mixed && !ps.generic && ps.TL == 1 && ps.R <= 512 && ps.ps_in == 1 && ps.ps_out != 1;
    if ((!fast && !tile) || ps.tw_N || !ps.rev_list.empty() || a.in_perm || a.c0 % a.T == 0 || a.out_s0 != 1 ||
        a.c1 * (long long)a.c2 == 1)
        return;
    const long long m = a.c0, groups = (long long)a.c1 * a.c2;
    const long long own = (m + a.T - 1) / a.T * groups;
    if (own <= (fast ? ps.max_grid : (a.R > 32 ? 4 : 2) * cus)) return;
    if (tile && a.R > 32 && 5 * m * groups > 3 * own * a.T) return;
    const bool flat = a.c2 == 1 || (a.in_s2 == a.c1 * a.in_s1 && a.out_s2 == a.c1 * a.out_s1);
    if (a.in_s1 != m * a.in_s0 || (a.c2 > 1 && !flat) || m * groups >= (1LL << 31)) return;
    const unsigned mul = (65536u + (unsigned)m - 1) / (unsigned)m;
    if ((m + a.T) * (mul * m - 65536) >= 65536 || (a.T + 2 * m) * a.R >= (1 << 17)) return;
    a.merge = (int)m;
    a.merge_mul = mul;
    a.merge_out = a.out_s1;
    a.c0 = (int)(m * groups);
    a.c1 = a.c2 = 1;
    a.out_s0 = 0;
}

// The runtime takes fewer than 2^32 threads a launch. A workgroup of the mixed-radix kernels has few
// points where lines are few (columns of a narrow 2D transform), so a large batch goes in several
// launches; kstart and kstop are then those of the first and the last.
constexpr long long kMaxGridThreads = 0xffffffffLL;
static hipError_t launch_mixed(const void *fn, void *arg, long long blocks, int threads, size_t lds, hipStream_t s,
                               hipEvent_t kstart, hipEvent_t kstop)
{
    void *args[] = {arg};
    const dim3 grid((unsigned)blocks), block(threads);
    if (kstart || kstop) return hipExtLaunchKernel(fn, grid, block, args, lds, s, kstart, kstop, 0);
    return hipLaunchKernel(fn, grid, block, args, lds, s);
}

// only >= 0: run that pass alone; kstart/kstop: events the runtime records around that
// pass's kernel (its own execution window; one launch per exec).
static int exec_chunk(mfft_plan_s *p, const char *in, char *out, long long nb, hipStream_t s, hipEvent_t *ev,
                      int &evi, void *work, const mfft::ExecFuse *fz = nullptr, long long b0 = 0, int only = -1,
                      hipEvent_t kstart = nullptr, hipEvent_t kstop = nullptr)
{
    int k = -1;
    for (auto &ps : p->passes) {
        if (++k != only && only >= 0) continue;
        TileArgs a;
        memset(&a, 0, sizeof a);
        if (fz && &ps == &p->passes.front()) {
            a.in_mul = fz->in_mul;
            a.in_mul_period = fz->in_mul_period;
            a.real_src = fz->real_src;
            a.real_src2 = fz->real_src2;
            a.real_f64 = fz->real_f64;
            a.real_b = fz->real_b;
            a.real_c = fz->real_c;
            a.real_h = fz->real_h;
            a.real_w = fz->real_w;
            a.real_pw = p->kind == 2 ? p->ny : p->n;
            a.real_p = p->total;
            a.real_span = fz->real_f64 ? 0u : (unsigned)std::min<long long>(4LL * a.real_b * a.real_c * a.real_h * a.real_w, 0x7fffffff);
            a.batch_base = b0;
        }
        const void *fn = ps.fn;
        if (a.real_src && ps.fast_kind == KIND_ROWS) fn = (const void *)find_fast_ends(ps.R, ENDS_REAL, FMT_C32);
        if (fz && fz->crop_out && &ps == &p->passes.back()) {
            a.crop_out = fz->crop_out;
            a.crop_b = fz->crop_b;
            a.crop_c = fz->crop_c;
            a.crop_h = fz->crop_h;
            a.crop_w = fz->crop_w;
            a.crop_y = fz->crop_y;
            a.crop_x = fz->crop_x;
            a.crop_mul = fz->crop_mul;
            const long long planes = a.crop_b ? (long long)a.crop_b * a.crop_c : p->batch;
            a.crop_span = (unsigned)(4 * planes * a.crop_h * a.crop_w);
            a.batch_base = b0;
            a.crop_rows = p->nx;
            a.crop_sp = (int)(ps.ps_out / p->ny);
            a.crop_s2 = ps.l2 >= 0 ? (int)(ps.lines[ps.l2].out_stride / p->ny) : 0;
            fn = (const void *)find_fast_ends(ps.R, ENDS_CROP, dst_fmt(p, ps));
        }
        a.in = buf_ptr(ps.src, in, out, work);
        a.out = buf_ptr(ps.dst, in, out, work);
        a.in_fmt = src_fmt(p, ps);
        a.out_fmt = dst_fmt(p, ps);
        a.R = ps.R;
        a.nstages = (int)ps.radix.size();
        for (int i = 0; i < a.nstages; ++i) {
            a.radix[i] = ps.radix[i];
            a.stage_mul[i] = p->d.scale == MFFT_SCALE_STAGE ? 1.0f / ps.radix[i] : 1.0f;
        }
        a.T = ps.T;
        a.TL = ps.TL;
        auto cnt = [&](int li) -> long long {
            if (li < 0) return 1;
            // a pass of the column axis: the level of the columns
            if (fz && fz->cols && ps.col_axis && ps.lines[li].in_stride == 1 && !ps.lines[li].batch)
                return std::min<long long>(ps.lines[li].count, fz->cols);
            return ps.lines[li].batch ? nb : ps.lines[li].count;
        };
        a.c0 = (int)cnt(ps.l0);
        a.c1 = (int)cnt(ps.l1);
        a.c2 = (int)cnt(ps.l2);
        a.in_s0 = ps.lines[ps.l0].in_stride;
        a.out_s0 = ps.lines[ps.l0].out_stride;
        a.in_s1 = ps.l1 >= 0 ? ps.lines[ps.l1].in_stride : 0;
        a.out_s1 = ps.l1 >= 0 ? ps.lines[ps.l1].out_stride : 0;
        a.in_s2 = ps.l2 >= 0 ? ps.lines[ps.l2].in_stride : 0;
        a.out_s2 = ps.l2 >= 0 ? ps.lines[ps.l2].out_stride : 0;
        a.in_ps = ps.ps_in;
        a.out_ps = ps.ps_out;
        a.in_perm = ps.perm;
        a.stage_tw = ps.stage_tw;
        a.dft_ops = p->ops;
        a.tw_N = ps.tw_N;
        a.tw_level = ps.tw_level == ps.l0 ? 0 : 1;
        a.tw_bits = ps.tw_bits;
        a.tw_lo = ps.tw_lo;
        a.tw_hi = ps.tw_hi;
        a.out_mul = 1.0f;
        a.sign = p->d.direction;
        a.in_vec = ((uintptr_t)a.in & 15) == 0;
        a.out_vec = ((uintptr_t)a.out & 15) == 0;
        a.stage_tw_s = ps.stage_tw_s;
        a.tw_lo_s = ps.tw_lo_s;
        a.last_mul = ps.last_mul;
        a.tail_mul = ps.tail_mul;
        a.rev_input = ps.rev_fast ? 1 : 0;
        a.in_rev = ps.rev_q;
        a.tw_rev = ps.rev_tw;
        memcpy(a.w16, g_w16, sizeof a.w16);
        merge_line_groups(ps, p->cus, a);
        long long ntiles = ((a.c0 + a.T - 1) / a.T) * (long long)a.c1 * a.c2;
        if (a.merge && ps.fast_kind < 0) {
            // a full tile takes this kernel 11 us whatever the launch, a small one 6 (48 x 1680):
            // small ones until every compute unit has four full ones
            const void *small = ntiles < 4 * p->cus ? (const void *)find_merged_tile_kernel(p->d.precision, ps.R, true) : nullptr;
            fn = small ? small : (const void *)find_merged_tile_kernel(p->d.precision, ps.R, false);
            if (small) {
                a.T = kSmallTile / ps.R;
                ntiles = ((a.c0 + a.T - 1) / a.T) * (long long)a.c1 * a.c2;
            }
        }
        if (ntiles <= 0) continue;
        if (ntiles >= (1LL << 31)) return fail(MFFT_ERR_UNSUPPORTED, "grid too large");
        if (trace_active()) trace_pass(p, ps, a, nb, b0, s);
        if (ev) HIP_TRY(hipEventRecord(ev[evi++], s));
        auto launch = [&](dim3 grid, dim3 block) -> hipError_t {
            void *args[] = {&a};
            if (kstart || kstop) return hipExtLaunchKernel(fn, grid, block, args, 0, s, kstart, kstop, 0);
            return hipLaunchKernel(fn, grid, block, args, 0, s);
        };
        if (ps.fast_kind == KIND_ONCHIP_COLS) {
            // one workgroup per 32 adjacent columns of one image
            OnchipColsArgs oa;
            memset(&oa, 0, sizeof oa);
            oa.in = a.in;
            oa.out = a.out;
            oa.col_blocks = (int)(ps.lines[0].count / kOnchipColsLines);
            oa.blocks = (long long)oa.col_blocks * nb;
            oa.ps = (int)ps.ps_in;
            oa.ps_out = (int)ps.ps_out;
            oa.in_dist = ps.lines[1].in_stride;
            oa.out_dist = ps.lines[1].out_stride;
            oa.dft_ops = p->ops;
            oa.tw_s = ps.tw_lo_s;
            oa.stw_s = ps.stage_tw_s;
            oa.tail_mul = ps.tail_mul;
            oa.sign = p->d.direction;
            memcpy(oa.w16, g_w16, sizeof oa.w16);
            void *oargs[] = {&oa};
            if (oa.blocks >= (1LL << 31)) return fail(MFFT_ERR_UNSUPPORTED, "grid too large");
            const dim3 grid((unsigned)oa.blocks), block(kOnchipThreads);
            if (kstart || kstop)
                HIP_TRY(hipExtLaunchKernel(ps.fn, grid, block, oargs, 0, s, kstart, kstop, 0));
            else
                HIP_TRY(hipLaunchKernel(ps.fn, grid, block, oargs, 0, s));
            continue;
        }
        if (ps.fast_kind == KIND_ONCHIP) {
            // one workgroup per line; a digit-reversed line is read in 16-byte pieces
            if (!ps.rev_list.empty() && ((uintptr_t)a.in & 15))
                return fail(MFFT_ERR_INVALID, "digit-reversed 65536-point input must be 16-byte aligned");
            OnchipArgs oa;
            oa.in = a.in;
            oa.out = a.out;
            oa.batch = nb;
            oa.in_dist = ps.lines[0].in_stride;
            oa.out_dist = ps.lines[0].out_stride;
            oa.dft_ops = p->ops;
            oa.stage_tw_s = ps.stage_tw_s;
            oa.tw_lo_s = ps.tw_lo_s;
            oa.tw_hi = ps.tw_hi;
            oa.fac = ps.last_mul;
            void *oargs[] = {&oa};
            const dim3 grid((unsigned)nb), block(kOnchipThreads);
            if (kstart || kstop)
                HIP_TRY(hipExtLaunchKernel(ps.fn, grid, block, oargs, 0, s, kstart, kstop, 0));
            else
                HIP_TRY(hipLaunchKernel(ps.fn, grid, block, oargs, 0, s));
            continue;
        }
        if (ps.mixed && ps.mixed_cap) {
            MixColArgs m;
            m.in = a.in;
            m.out = a.out;
            m.tw = ps.stage_tw;
            m.dft_ops = p->ops;
            m.sign = p->d.direction;
            m.c0 = a.c0;
            m.T = mixed_col_tile(ps, a.c0, a.c1);
            m.tiles0 = (a.c0 + m.T - 1) / m.T;
            m.ps_in = (int)a.in_ps;
            m.ps_out = (int)a.out_ps;
            m.in_dist = a.in_s1;
            m.out_dist = a.out_s1;
            memcpy(m.w16, g_w16, sizeof m.w16);
            m.sc = ps.mix;
            const int threads = mix_col_threads(ps.mixed_cap);
            const long long step = std::max(1LL, kMaxGridThreads / threads / m.tiles0);
            for (long long t0 = 0; t0 < a.c1; t0 += step) {
                const long long nt = std::min<long long>(step, a.c1 - t0);
                m.in = (const char *)a.in + t0 * m.in_dist * fmt_bytes(a.in_fmt);
                m.out = (char *)a.out + t0 * m.out_dist * fmt_bytes(a.out_fmt);
                HIP_TRY(launch_mixed(ps.fn, &m, nt * m.tiles0, threads, mix_lds_bytes(m.T * ps.R, ps.R), s, t0 ? nullptr : kstart,
                                     t0 + nt < a.c1 ? nullptr : kstop));
            }
            continue;
        }
        if (ps.mixed) {
            MixArgs m;
            m.in = a.in;
            m.out = a.out;
            m.nlines = (long long)a.c0 * a.c1 * a.c2;
            m.tw = ps.stage_tw;
            m.dft_ops = p->ops;
            m.T = mixed_tile_lines(ps.R, m.nlines, ps.max_grid);
            m.sign = p->d.direction;
            memcpy(m.w16, g_w16, sizeof m.w16);
            m.sc = ps.mix;
            const long long lines = m.nlines, step = kMaxGridThreads / kMixThreads * m.T;
            for (long long l0 = 0; l0 < lines; l0 += step) {
                m.nlines = std::min(step, lines - l0);
                m.in = (const char *)a.in + l0 * ps.R * fmt_bytes(a.in_fmt);
                m.out = (char *)a.out + l0 * ps.R * fmt_bytes(a.out_fmt);
                HIP_TRY(launch_mixed(ps.fn, &m, (m.nlines + m.T - 1) / m.T, kMixThreads, mix_lds_bytes(m.T * ps.R, ps.R), s,
                                     l0 ? nullptr : kstart, l0 + m.nlines < lines ? nullptr : kstop));
            }
            continue;
        }
        if (ps.small) {
            long long nl = (long long)a.c0 * a.c1 * a.c2;
            if (a.in_mul) nl = in_mul_threads((long long)a.c0 * a.c1, a.c2);
            // largest byte offset a line's point reaches, per side (strides are >= 0)
            auto span = [&](long long s0, long long s1, long long s2, long long sp, int fmt) -> long long {
                if (s0 < 0 || s1 < 0 || s2 < 0 || sp < 0) return -1;
                return ((a.c0 - 1) * s0 + (a.c1 - 1) * s1 + (a.c2 - 1) * s2 + (a.R - 1) * sp) * fmt_bytes(fmt);
            };
            const long long si = span(a.in_s0, a.in_s1, a.in_s2, a.in_ps, a.in_fmt);
            const long long so = span(a.out_s0, a.out_s1, a.out_s2, a.out_ps, a.out_fmt);
            a.off32 = (si >= 0 && si < (1LL << 32) - 8 ? 1 : 0) | (so >= 0 && so < (1LL << 32) - 8 ? 2 : 0);
            a.in_span = (a.off32 & 1) ? (unsigned)(si + fmt_bytes(a.in_fmt)) : 0u;
            a.out_span = (a.off32 & 2) ? (unsigned)(so + fmt_bytes(a.out_fmt)) : 0u;
            HIP_TRY(launch(dim3((unsigned)((nl + 255) / 256)), dim3(256)));
            continue;
        }
        if (ps.fast_kind >= 0) {
            const int twc = ps.fast_kind == KIND_COLS ? kFastTwCols : kFastTw;
            a.tw_lds = ps.tw_N && (1 << ps.tw_bits) <= twc && ((ps.tw_N + (1 << ps.tw_bits) - 1) >> ps.tw_bits) <= twc;
            long long grid = std::min(ntiles, ps.max_grid);
            if (grid > 8) grid -= grid % 8;
            HIP_TRY(launch(dim3((unsigned)grid), dim3(fast_threads(p->d.precision, ps.R, ps.fast_kind))));
        } else {
            HIP_TRY(launch_tile(fn, a, ntiles, s, kstart, kstop));
        }
    }
    return MFFT_OK;
}

// ------------------------------------------------------------------ C ABI
namespace mfft {
void mfft_trace_reset(hipEvent_t *events, mfft_launch_record *rec, int cap);
hipError_t mfft_trace_stop(int *n, bool *overflow, hipEvent_t *last);
}  // namespace mfft

extern "C" {

int mfft_desc_default(mfft_desc *d)
{
    if (!d) return fail(MFFT_ERR_INVALID, "null desc");
    memset(d, 0, sizeof *d);
    d->precision = MFFT_PREC_SPLIT_FP16;
    d->direction = MFFT_FORWARD;
    d->scale = MFFT_SCALE_STAGE;
    d->in_fmt = MFFT_FMT_C16;
    d->out_fmt = MFFT_FMT_C16;
    d->in_order = MFFT_ORDER_NATURAL;
    d->mid_fmt = -1;
    return MFFT_OK;
}

// Plan creation is the set-up of mfft_exec_noalloc too: the address of its workspace array
// on the current device is resolved here, so an exec under graph capture or in a serving
// loop finds it cached (a failure is reported by that exec, not here).
static void resolve_noalloc_scratch()
{
    const std::string keep = g_err;
    void *ws = nullptr;
    (void)noalloc_scratch(&ws);
    g_err = keep;
}

// split_hint = MFFT_SPLIT_TUNED: take split and chunk from the autotuner's cache.
static mfft_desc resolve_tuned(const mfft_desc *d, int nx, int ny, int64_t batch)
{
    mfft_desc r = *d;
    if (d->split_hint != MFFT_SPLIT_TUNED) return r;
    r.split_hint = 0;
    mfft_tune_entry e;
    std::string keep = g_err;
    if (mfft_tune_lookup(nullptr, nx, ny, batch, d, &e) == MFFT_OK) {
        r.split_hint = e.split_hint;
        r.workspace_limit = e.workspace_limit;
    }
    g_err = keep;
    return r;
}

static int create_1d(mfft_plan *plan, int n, int64_t batch, const mfft_desc *d_in, bool allow_onchip, bool allow_mixed = true)
{
    if (!plan || !d_in) return fail(MFFT_ERR_INVALID, "null argument");
    *plan = nullptr;
    if (n < 2 || batch < 1) return fail(MFFT_ERR_INVALID, "n=%d batch=%lld", n, (long long)batch);
    const mfft_desc dt = resolve_tuned(d_in, n, 0, batch);
    const mfft_desc *d = &dt;
    int rc = check_desc(d);
    if (rc) return rc;
    mfft_plan_s *p = new mfft_plan_s;
    p->kind = 1;
    p->n = n;
    p->batch = batch;
    p->d = *d;
    p->total = n;
    const bool rev = d->in_order == MFFT_ORDER_DIGIT_REVERSED;
    if (rev) {
        rev_radices(n, p->rev_list_axis[0]);
        gen_rev(n, p->rev_list_axis[0], p->rev_axis[0]);
    }
    if (allow_onchip && batch >= onchip_min_lines() && plan_onchip(p, d)) {
        rc = MFFT_OK;
    } else if (allow_onchip && n >= (1 << 19) && n <= (1 << 20) &&
               batch >= onchip_rows_min_lines(n / kOnchipColsN) && plan_onchip_rows(p, d)) {
        rc = MFFT_OK;
    } else if (rev && n > kMaxTile) {
        rc = plan_reversed_1d(p);
    } else {
        std::vector<Level> lines{Level{batch, n, n, true}};
        rc = plan_axis(p->passes, n, 1, 1, lines, BUF_IN, BUF_OUT, rev ? 0 : -1, d->split_hint, narrow_mid(d), false,
                       allow_mixed && find_mixed_kernel(d->precision, d->in_fmt, d->out_fmt) ? d->precision : -1);
    }
    if (!rc) rc = finalize_plan(p);
    if (!rc && allow_mixed && p->passes.size() == 1 && p->passes[0].mixed && fmt_bytes(d->in_fmt) != fmt_bytes(d->out_fmt)) {
        rc = create_1d(&p->aliased, n, batch, &dt, false, false);
        if (!rc && p->aliased->passes.size() == 1) {  // no better: a length without the two passes
            mfft_plan_destroy(p->aliased);
            p->aliased = nullptr;
        }
    }
    if (rc) {
        std::string msg = g_err;
        mfft_plan_destroy(p);
        g_err = msg;
        return rc;
    }
    resolve_noalloc_scratch();
    *plan = p;
    return MFFT_OK;
}

static bool has_onchip(const mfft_plan_s *p)
{
    for (auto &ps : p->passes)
        if (ps.onchip || ps.onchip_cols) return true;
    return false;
}

int mfft_plan_create_1d(mfft_plan *plan, int n, int64_t batch, const mfft_desc *d_in)
{
    int rc = create_1d(plan, n, batch, d_in, true);
    if (rc || !has_onchip(*plan)) return rc;
    mfft_plan p = *plan, q = nullptr;
    const long long below = n == kOnchipN ? onchip_min_lines() : onchip_rows_min_lines(n / kOnchipColsN);
    rc = create_1d(&q, n, below - 1, d_in, false);
    if (rc) {
        std::string msg = g_err;
        mfft_plan_destroy(p);
        *plan = nullptr;
        g_err = msg;
        return rc;
    }
    p->small = q;
    p->small_below = below;
    return MFFT_OK;
}

// conv: a transform of the conv operator, whose odd axes keep a streaming pass of their own (it
// takes the fused image load and filter product)
static int create_2d(mfft_plan *plan, int nx, int ny, int64_t batch, const mfft_desc *d_in, bool allow_onchip,
                     bool out_mid, bool conv)
{
    if (!plan || !d_in) return fail(MFFT_ERR_INVALID, "null argument");
    *plan = nullptr;
    if (nx < 2 || ny < 2 || batch < 1) return fail(MFFT_ERR_INVALID, "nx=%d ny=%d batch=%lld", nx, ny, (long long)batch);
    const mfft_desc dt = resolve_tuned(d_in, nx, ny, batch);
    const mfft_desc *d = &dt;
    int rc = check_desc(d);
    if (rc) return rc;
    mfft_plan_s *p = new mfft_plan_s;
    p->kind = 2;
    p->nx = nx;
    p->ny = ny;
    p->n = nx * ny;
    p->batch = batch;
    p->d = *d;
    p->total = (long long)nx * ny;
    bool rev = d->in_order == MFFT_ORDER_DIGIT_REVERSED;
    if (rev) {
        rev_radices(nx, p->rev_list_axis[0]);
        gen_rev(nx, p->rev_list_axis[0], p->rev_axis[0]);
        rev_radices(ny, p->rev_list_axis[1]);
        gen_rev(ny, p->rev_list_axis[1], p->rev_axis[1]);
    }
    // the column pass reads the x order itself when its kernel is the strided matrix-core
    // one (then up to 1024 points stay one pass); its input is the rows' intermediate
    DigitRev qx;
    const int col_in_fmt = d->mid_fmt >= 0                          ? d->mid_fmt
                           : d->precision == MFFT_PREC_FP16 ? MFFT_FMT_C16
                           : d->precision == MFFT_PREC_BF16 ? MFFT_FMT_CBF16
                                                            : MFFT_FMT_C32;
    const bool rev_cols = rev && fast_rev_ok(d->precision, col_in_fmt) && fast_rev_spec(nx, p->rev_list_axis[0], qx);
    long long NN = (long long)nx * ny;
    // rows (y axis, contiguous): lines = (x, b)
    std::vector<Level> rows{Level{nx, ny, ny, false}, Level{batch, NN, NN, true}};
    const int odd_hint = d->split_hint == 1 ? 1 : 0;  // 1 keeps odd * 2^a axes in one pass
    rc = plan_axis(p->passes, ny, 1, 1, rows, BUF_IN, BUF_WORK, rev ? 1 : -1, odd_hint, narrow_mid(d), false,
                   !conv && find_mixed_kernel(d->precision, d->in_fmt, col_in_fmt) ? d->precision : -1);
    const size_t nrow_passes = p->passes.size();
    // columns (x axis, stride ny): lines = (y, b)
    if (!rc) {
        // split_hint > 1: the first-pass length of the column axis when it is split
        const int col_hint = d->split_hint > 1 ? d->split_hint : odd_hint;
        std::vector<Level> cols{Level{ny, 1, 1, false}, Level{batch, NN, NN, true}};
        // 2048-point columns with 16-bit words on both sides, a multiple of 32 of them: one
        // pass of the on-chip column kernel (the split into a strided and a streaming pass
        // moves every point twice)
        const int fmt16 = d->precision == MFFT_PREC_BF16 ? MFFT_FMT_CBF16 : MFFT_FMT_C16;
        if (allow_onchip && nx == kOnchipColsN && ny % kOnchipColsLines == 0 && batch >= onchip_cols_min_images(ny) &&
            !rev && d->split_hint <= 1 && col_in_fmt == fmt16 && d->out_fmt == fmt16 &&
            find_onchip_cols_kernel(d->precision, fmt16)) {
            PassSpec ps;
            ps.R = nx;
            ps.ps_in = ps.ps_out = ny;
            ps.lines = cols;
            ps.src = BUF_WORK;
            ps.dst = BUF_OUT;
            ps.onchip_cols = true;
            p->passes.push_back(ps);
        } else {
            rc = plan_axis(p->passes, nx, ny, ny, cols, BUF_WORK, BUF_OUT, rev ? 0 : -1, col_hint, narrow_mid(d),
                           rev_cols,
                           !conv && find_mixed_kernel(d->precision, col_in_fmt, d->out_fmt) ? d->precision : -1);
        }
    }
    for (size_t i = nrow_passes; i < p->passes.size(); ++i) p->passes[i].col_axis = true;
    p->out_mid = out_mid;
    p->conv = conv;
    if (!rc) rc = finalize_plan(p);
    if (rc) {
        std::string msg = g_err;
        mfft_plan_destroy(p);
        g_err = msg;
        return rc;
    }
    resolve_noalloc_scratch();
    *plan = p;
    return MFFT_OK;
}

static int create_2d_all(mfft_plan *plan, int nx, int ny, int64_t batch, const mfft_desc *d_in, bool out_mid,
                         bool conv)
{
    int rc = create_2d(plan, nx, ny, batch, d_in, true, out_mid, conv);
    if (rc || !has_onchip(*plan)) return rc;
    mfft_plan p = *plan, q = nullptr;
    const long long below = onchip_cols_min_images(ny);
    rc = create_2d(&q, nx, ny, below - 1, d_in, false, out_mid, conv);
    if (rc) {
        std::string msg = g_err;
        mfft_plan_destroy(p);
        *plan = nullptr;
        g_err = msg;
        return rc;
    }
    p->small = q;
    p->small_below = below;
    return MFFT_OK;
}

int mfft_plan_create_2d(mfft_plan *plan, int nx, int ny, int64_t batch, const mfft_desc *d_in)
{
    return create_2d_all(plan, nx, ny, batch, d_in, false, false);
}

int mfft_plan_destroy(mfft_plan plan)
{
    if (!plan) return MFFT_OK;
    (void)hipDeviceSynchronize();
    if (plan->small) mfft_plan_destroy(plan->small);
    if (plan->aliased) mfft_plan_destroy(plan->aliased);
    for (void *ptr : plan->allocs) (void)hipFree(ptr);
    plan->ws_order.destroy();
    delete plan;
    return MFFT_OK;
}

}  // extern "C"

namespace mfft {
long long plan_scratch_bytes(mfft_plan p, bool in_place)
{
    return std::max({p->work_bytes, p->small ? p->small->work_bytes : 0LL, in_place && p->aliased ? p->aliased->work_bytes : 0LL});
}
}  // namespace mfft

extern "C" {

int mfft_plan_info(mfft_plan p, mfft_info *info)
{
    if (!p || !info) return fail(MFFT_ERR_INVALID, "null argument");
    memset(info, 0, sizeof *info);
    info->kind = p->kind;
    info->n = p->n;
    info->nx = p->nx;
    info->ny = p->ny;
    info->batch = p->batch;
    info->npasses = (int)std::min<size_t>(p->passes.size(), MFFT_MAX_PASSES);
    long long nchunks = (p->batch + p->chunk - 1) / p->chunk;
    for (int i = 0; i < info->npasses; ++i) {
        const PassSpec &ps = p->passes[i];
        mfft_pass_info &pi = info->pass[i];
        pi.R = ps.R;
        pi.lines_per_tile = ps.T;
        pi.lane_lines = ps.TL;
        pi.nstages = (int)ps.radix.size();
        for (int k = 0; k < pi.nstages && k < 8; ++k) pi.radix[k] = ps.radix[k];
        long long lines = 1;
        for (auto &l : ps.lines) lines *= l.batch ? p->chunk : l.count;
        long long c0 = ps.lines[ps.l0].batch ? p->chunk : ps.lines[ps.l0].count;
        int T = ps.T;
        if (ps.mixed && ps.mixed_cap) {
            T = mixed_col_tile(ps, c0, lines / c0);
        } else if (ps.mixed) {  // dense lines: tiled through all levels
            c0 = lines;
            T = mixed_tile_lines(ps.R, lines, ps.max_grid);
        }
        pi.lines_per_tile = T;
        pi.tiles = (lines / c0) * ((c0 + T - 1) / T);
        pi.generic = ps.generic;
        pi.in_elem_bytes = fmt_bytes(src_fmt(p, ps));
        pi.out_elem_bytes = fmt_bytes(dst_fmt(p, ps));
        pi.points = lines * ps.R;
        pi.kernel = ps.small ? MFFT_KERNEL_STREAM
                    : ps.mixed ? (ps.mixed_cap ? MFFT_KERNEL_MIXED_COLS : MFFT_KERNEL_MIXED_ROWS)
                    : ps.fast_kind == KIND_ROWS ? MFFT_KERNEL_ROWS
                    : ps.fast_kind == KIND_ROWS_TR ? MFFT_KERNEL_ROWS_TR
                    : ps.fast_kind == KIND_COLS ? MFFT_KERNEL_COLS
                    : ps.fast_kind == KIND_ONCHIP ? MFFT_KERNEL_ONCHIP
                    : ps.fast_kind == KIND_ONCHIP_COLS ? MFFT_KERNEL_ONCHIP_COLS
                    : ps.generic ? MFFT_KERNEL_GENERIC : MFFT_KERNEL_TILE;
    }
    info->out_scale = p->out_scale;
    // a caller-supplied workspace also serves the companion plans
    info->workspace_bytes = std::max(mfft::plan_scratch_bytes(p, false), mfft::plan_scratch_bytes(p, true));
    info->batch_chunk = p->chunk;
    info->launches_per_exec = nchunks * (long long)p->passes.size();
    return MFFT_OK;
}

static int exec_all(mfft_plan p, const void *in, void *out, void *stream, hipEvent_t *ev, long long batch = -1,
                    void *work = nullptr, const mfft::ExecFuse *fz = nullptr, int only = -1,
                    hipEvent_t kstart = nullptr, hipEvent_t kstop = nullptr)
{
    if (p->small && batch >= 0 && batch < p->small_below && only < 0 && !ev &&
        (!fz || !fz->input() || (p->small->passes.front().small && p->small->passes.front().src == BUF_IN)))
        return exec_all(p->small, in, out, stream, nullptr, batch, work, fz, -1, nullptr, nullptr);
    if (p->aliased && in == out) {
        // timed as the plan's one pass: all of the other plan's lies between the events
        const long long launches = ev ? ((batch < 0 ? p->batch : batch) + p->chunk - 1) / p->chunk : 0;
        if (ev) HIP_TRY(hipEventRecord(ev[0], (hipStream_t)stream));
        if (kstart) HIP_TRY(hipEventRecord(kstart, (hipStream_t)stream));
        const int rc = exec_all(p->aliased, in, out, stream, nullptr, batch, work);
        if (rc) return rc;
        if (kstop) HIP_TRY(hipEventRecord(kstop, (hipStream_t)stream));
        for (long long i = 1; i <= launches; ++i) HIP_TRY(hipEventRecord(ev[i], (hipStream_t)stream));
        return MFFT_OK;
    }
    if (p->out_mid && in == out)
        for (const PassSpec &ps : p->passes) {
            // a pass that reads the input (not a fused real source) and writes the output in
            // another format would overwrite lines it has not read yet
            const bool reads = !(fz && fz->real_src && &ps == &p->passes.front());
            if (reads && ps.src == BUF_IN && ps.dst == BUF_OUT && src_fmt(p, ps) != dst_fmt(p, ps))
                return fail(MFFT_ERR_INVALID, "plan keeps intermediates in the output buffer: in and out must differ");
        }
    std::unique_lock<std::mutex> lk(p->exec_mu, std::defer_lock);
    if (!work) lk.lock();  // the plan's own workspace is shared by its callers
    hipStream_t s = (hipStream_t)stream;
    long long ib = p->total * fmt_bytes(p->d.in_fmt), ob = p->total * fmt_bytes(p->d.out_fmt);
    if (batch < 0) batch = p->batch;
    if (!work && !p->work && p->work_bytes > 0) return fail(MFFT_ERR_INVALID, "plan needs a workspace (mfft_exec_ex)");
    // the plan's own workspace: an exec on another stream than the previous one runs
    // after it (two streams sharing p->work would otherwise overwrite each other's
    // intermediates between the passes)
    const bool own_ws = !work && p->work;
    if (own_ws) HIP_TRY(p->ws_order.acquire(s));
    int evi = 0, rc = MFFT_OK;
    for (long long b0 = 0; b0 < batch && !rc; b0 += p->chunk) {
        long long nb = std::min(p->chunk, batch - b0);
        rc = exec_chunk(p, (const char *)in + b0 * ib, (char *)out + b0 * ob, nb, s, ev, evi, work ? work : p->work, fz,
                        b0, only, kstart, kstop);
    }
    if (own_ws) {
        std::string keep = g_err;
        hipError_t e = p->ws_order.release(s);  // also after a partial enqueue
        if (!rc && e != hipSuccess) return fail(MFFT_ERR_HIP, "workspace order: %s", hipGetErrorString(e));
        if (rc) g_err = keep;
    }
    if (rc) return rc;
    if (ev) HIP_TRY(hipEventRecord(ev[evi++], s));
    return MFFT_OK;
}

int mfft_exec(mfft_plan p, const void *in, void *out, void *stream)
{
    if (!p || !in || !out) return fail(MFFT_ERR_INVALID, "null argument");
    return exec_all(p, in, out, stream, nullptr);
}

int mfft_exec_ex(mfft_plan p, const void *in, void *out, int64_t batch, void *workspace, void *stream)
{
    if (!p || !in || !out) return fail(MFFT_ERR_INVALID, "null argument");
    if (batch < 1 || batch > p->batch) return fail(MFFT_ERR_INVALID, "batch %lld outside 1..%lld", (long long)batch, p->batch);
    return exec_all(p, in, out, stream, nullptr, batch, workspace);
}

// ------------------------------------------------------------------ work-queue batcher
struct mfft_batcher_s {
    mfft_desc d{};
    int max_items = 0;
    DftOps *ops = nullptr;
    std::vector<float2 *> tables;  // stage twiddles of the lengths seen so far
    std::vector<float2 *> allocs;  // what holds them: one allocation per call that met new lengths
    std::vector<short> index = std::vector<short>(kMaxTile + 1, -1);  // length -> tables
    // the mixed-radix work-queue kernel, when it exists for the formats, and the schedules of
    // the lengths (entry i belongs to tables[i])
    const void *fn = nullptr;
    MixLen *lens = nullptr;
    struct Slot {
        TileArgs *h_jobs = nullptr, *d_jobs = nullptr;
        long long *h_first = nullptr, *d_first = nullptr;
        unsigned long long *counter = nullptr;
        MixItem *h_items = nullptr, *d_items = nullptr;  // max_items records, then their first tiles
        hipEvent_t done = nullptr;
        bool used = false;
    } slot[4];
    int next = 0;
    int grid = 0;
    std::mutex mu;
};

int mfft_batcher_destroy(mfft_batcher b)
{
    if (!b) return MFFT_OK;
    (void)hipDeviceSynchronize();
    (void)hipFree(b->ops);
    (void)hipFree(b->lens);
    for (float2 *t : b->allocs) (void)hipFree(t);
    for (auto &sl : b->slot) {
        (void)hipHostFree(sl.h_jobs);
        (void)hipHostFree(sl.h_first);
        (void)hipHostFree(sl.h_items);
        (void)hipFree(sl.d_jobs);
        (void)hipFree(sl.d_first);
        (void)hipFree(sl.d_items);
        (void)hipFree(sl.counter);
        if (sl.done) (void)hipEventDestroy(sl.done);
    }
    delete b;
    return MFFT_OK;
}

// Bytes of a slot's item records and first tiles; lengths 2^a 3^b 5^c 17^d up to kMaxTile: 195.
static size_t mix_items_bytes(int max_items) { return (sizeof(MixItem) + sizeof(int)) * (size_t)max_items; }
constexpr int kMixLengths = 256;

int mfft_batcher_create(mfft_batcher *out, const mfft_desc *d, int max_items)
{
    if (!out || !d || max_items < 1) return fail(MFFT_ERR_INVALID, "bad argument");
    int rc = check_desc(d);
    if (rc) return rc;
    if (ensure_w16()) return MFFT_ERR_HIP;
    mfft_batcher b = new mfft_batcher_s;
    b->d = *d;
    b->max_items = max_items;
    b->fn = find_mixed_queue_kernel(d->precision, d->in_fmt, d->out_fmt);
    hipError_t e = hipMalloc((void **)&b->ops, sizeof(DftOps));
    if (e == hipSuccess) e = gen_dft_ops(b->ops, d->direction, 0);
    if (b->fn) {
        if (e == hipSuccess) e = hipMalloc((void **)&b->lens, sizeof(MixLen) * kMixLengths);
        if (e == hipSuccess)
            e = hipFuncSetAttribute(b->fn, hipFuncAttributeMaxDynamicSharedMemorySize, mix_lds_max(0));
    }
    for (auto &sl : b->slot) {
        if (b->fn) {
            if (e == hipSuccess) e = hipHostMalloc((void **)&sl.h_items, mix_items_bytes(max_items), hipHostMallocDefault);
            if (e == hipSuccess) e = hipMalloc((void **)&sl.d_items, mix_items_bytes(max_items));
        } else {
            if (e == hipSuccess) e = hipHostMalloc((void **)&sl.h_jobs, sizeof(TileArgs) * max_items, hipHostMallocDefault);
            if (e == hipSuccess) e = hipHostMalloc((void **)&sl.h_first, sizeof(long long) * (max_items + 1), hipHostMallocDefault);
            if (e == hipSuccess) e = hipMalloc((void **)&sl.d_jobs, sizeof(TileArgs) * max_items);
            if (e == hipSuccess) e = hipMalloc((void **)&sl.d_first, sizeof(long long) * (max_items + 1));
        }
        if (e == hipSuccess) e = hipMalloc((void **)&sl.counter, sizeof(unsigned long long));
        if (e == hipSuccess) e = hipMemset(sl.counter, 0, sizeof(unsigned long long));
        if (e == hipSuccess) e = hipEventCreateWithFlags(&sl.done, hipEventDisableTiming);
    }
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) {
        mfft_batcher_destroy(b);
        return fail(MFFT_ERR_HIP, "batcher: %s", hipGetErrorString(e));
    }
    // the mixed-radix queue: up to four workgroups per compute unit take tiles from the counter
    b->grid = b->fn ? (int)(4 * device_cus()) : queue_grid(d->precision);
    *out = b;
    return MFFT_OK;
}

// Makes the tables (and entries of b->lens) of the items' lengths that are new to the batcher:
// generated together on the null stream and waited for once, so any stream may use them after.
static int batch_tables(mfft_batcher b, const mfft_batch_item *items, int nitems)
{
    std::vector<int> fresh;
    size_t words = 0;
    for (int i = 0; i < nitems; ++i)
        if (b->index[items[i].n] == -1) {
            b->index[items[i].n] = -2;  // seen in this call
            fresh.push_back(items[i].n);
            words += items[i].n;
        }
    if (fresh.empty()) return MFFT_OK;
    auto undo = [&](int code, const char *what, hipError_t e) {
        for (int n : fresh) b->index[n] = -1;
        return fail(code, "%s: %s", what, hipGetErrorString(e));
    };
    std::vector<MixLen> len(fresh.size());
    const size_t have = b->tables.size();
    float2 *tab = nullptr;
    hipError_t e = hipMalloc((void **)&tab, sizeof(float2) * words);
    if (e != hipSuccess) return undo(MFFT_ERR_NOMEM, "twiddle tables", e);
    float2 *t = tab;
    for (size_t i = 0; i < fresh.size() && e == hipSuccess; ++i) {
        len[i].tw = t;
        if (b->fn && (have + i >= kMixLengths ||
                      !mix_schedule(fresh[i], b->d.precision, b->d.scale == MFFT_SCALE_STAGE, MIX_16_LAST, len[i].sc)))
            e = hipErrorInvalidValue;
        else
            e = gen_twiddle(t, fresh[i], fresh[i], 1, b->d.direction, 0);
        t += fresh[i];
    }
    if (e == hipSuccess && b->fn)
        e = hipMemcpyAsync(b->lens + have, len.data(), sizeof(MixLen) * len.size(), hipMemcpyHostToDevice, 0);
    const hipError_t e2 = hipStreamSynchronize(0);
    if (e == hipSuccess) e = e2;
    if (e != hipSuccess) {
        (void)hipFree(tab);
        return undo(MFFT_ERR_HIP, "twiddle tables", e);
    }
    b->allocs.push_back(tab);
    for (size_t i = 0; i < fresh.size(); ++i) {
        b->index[fresh[i]] = (short)b->tables.size();
        b->tables.push_back(const_cast<float2 *>(len[i].tw));
    }
    return MFFT_OK;
}

// The next slot, once its previous launch has read its records.
static int batch_slot(mfft_batcher b, mfft_batcher_s::Slot **out)
{
    auto &sl = b->slot[b->next];
    if (sl.used) HIP_TRY(hipEventSynchronize(sl.done));
    b->next = (b->next + 1) % 4;
    *out = &sl;
    return MFFT_OK;
}

// The mixed-radix work queue. Up to kMixInline items travel in the kernel's arguments, and a
// launch whose tiles fit the grid hands out no further ones: such a call is one launch, with no
// copy, counter or slot.
static int batch_exec_mixed(mfft_batcher b, const mfft_batch_item *items, int nitems, hipStream_t s)
{
    long long points = 0;
    for (int i = 0; i < nitems; ++i) points += items[i].count * items[i].n;
    // points per tile: kMaxTile, less when that would leave compute units without a tile
    const long long cap = std::min<long long>(kMaxTile, std::max<long long>(kMixThreads, points / (b->grid / 2)));
    MixQueueArgs q;
    q.lens = b->lens;
    q.dft_ops = b->ops;
    q.items = nullptr;
    q.first = nullptr;
    q.counter = nullptr;
    q.nitems = nitems;
    q.sign = b->d.direction;
    memcpy(q.w16, g_w16, sizeof q.w16);
    mfft_batcher_s::Slot *sl = nullptr;
    MixItem *rec = q.item_in;
    int *first = q.first_in;
    if (nitems > kMixInline) {
        int rc = batch_slot(b, &sl);
        if (rc) return rc;
        rec = sl->h_items;
        first = (int *)(sl->h_items + b->max_items);
    }
    long long total = 0;
    int most = 0, longest = 0;
    for (int i = 0; i < nitems; ++i) {
        const mfft_batch_item &it = items[i];
        MixItem &m = rec[i];
        m.in = it.in;
        m.out = it.out;
        m.nlines = it.count;
        m.len = b->index[it.n];
        m.T = (int)std::max<long long>(1, std::min<long long>(it.count, cap / it.n));
        first[i] = (int)total;
        total += (it.count + m.T - 1) / m.T;
        if (total >= (1LL << 31)) return fail(MFFT_ERR_UNSUPPORTED, "%lld tiles in one launch", total);
        most = std::max(most, m.T * it.n);
        longest = std::max(longest, it.n);
    }
    q.total = (int)total;
    q.tw_at = (most + 1) & ~1;
    const int grid = (int)std::min<long long>(b->grid, total);
    if (total > grid && !sl) {
        int rc = batch_slot(b, &sl);
        if (rc) return rc;
    }
    if (sl) q.counter = (unsigned *)sl->counter;
    if (nitems > kMixInline) {
        HIP_TRY(hipMemcpyAsync(sl->d_items, sl->h_items, mix_items_bytes(b->max_items), hipMemcpyHostToDevice, s));
        q.items = sl->d_items;
        q.first = (const int *)(sl->d_items + b->max_items);
    }
    void *args[] = {&q};
    HIP_TRY(hipLaunchKernel(b->fn, dim3((unsigned)grid), dim3(kMixThreads), args, mix_lds_bytes(q.tw_at, longest), s));
    if (sl) {
        HIP_TRY(hipEventRecord(sl->done, s));
        sl->used = true;
    }
    return MFFT_OK;
}

int mfft_batcher_exec(mfft_batcher b, const mfft_batch_item *items, int nitems, void *stream)
{
    if (!b || (!items && nitems)) return fail(MFFT_ERR_INVALID, "null argument");
    if (nitems < 0 || nitems > b->max_items) return fail(MFFT_ERR_INVALID, "%d items (max %d)", nitems, b->max_items);
    if (nitems == 0) return MFFT_OK;
    std::lock_guard<std::mutex> lk(b->mu);
    hipStream_t s = (hipStream_t)stream;
    for (int i = 0; i < nitems; ++i) {
        const mfft_batch_item &it = items[i];
        std::vector<int> rad;
        if (it.n < 2 || it.n > kMaxTile || !line_radices(it.n, rad) || it.count < 1 || !it.in || !it.out)
            return fail(MFFT_ERR_INVALID, "item %d: n=%d count=%lld", i, it.n, (long long)it.count);
    }
    int rc = batch_tables(b, items, nitems);
    if (rc) return rc;
    if (trace_active()) {
        // one record for the call
        long long rd = 0, wr = 0;
        for (int i = 0; i < nitems; ++i) {
            rd += items[i].count * items[i].n * (long long)fmt_bytes(b->d.in_fmt);
            wr += items[i].count * items[i].n * (long long)fmt_bytes(b->d.out_fmt);
        }
        char name[64];
        snprintf(name, sizeof name, "queue %d items %s>%s", nitems, fmt_name(b->d.in_fmt), fmt_name(b->d.out_fmt));
        trace_launch(s, name, rd, wr);
    }
    if (b->fn) return batch_exec_mixed(b, items, nitems, s);
    mfft_batcher_s::Slot *slp = nullptr;
    rc = batch_slot(b, &slp);
    if (rc) return rc;
    auto &sl = *slp;
    long long total = 0;
    for (int i = 0; i < nitems; ++i) {
        const mfft_batch_item &it = items[i];
        std::vector<int> rad;
        line_radices(it.n, rad);
        TileArgs &a = sl.h_jobs[i];
        memset(&a, 0, sizeof a);
        a.in = it.in;
        a.out = it.out;
        a.in_fmt = b->d.in_fmt;
        a.out_fmt = b->d.out_fmt;
        a.R = it.n;
        a.nstages = (int)rad.size();
        for (int k = 0; k < a.nstages; ++k) {
            a.radix[k] = rad[k];
            a.stage_mul[k] = b->d.scale == MFFT_SCALE_STAGE ? 1.0f / rad[k] : 1.0f;
        }
        a.T = std::max(1, kMaxTile / it.n);
        a.TL = 1;
        a.c0 = (int)it.count;
        a.c1 = a.c2 = 1;
        a.in_s0 = a.out_s0 = it.n;
        a.in_ps = a.out_ps = 1;
        a.stage_tw = b->tables[b->index[it.n]];
        a.dft_ops = b->ops;
        a.out_mul = 1.0f;
        a.sign = b->d.direction;
        a.in_vec = ((uintptr_t)it.in & 15) == 0;
        a.out_vec = ((uintptr_t)it.out & 15) == 0;
        memcpy(a.w16, g_w16, sizeof a.w16);
        sl.h_first[i] = total;
        total += (it.count + a.T - 1) / a.T;
    }
    sl.h_first[nitems] = total;
    HIP_TRY(hipMemcpyAsync(sl.d_jobs, sl.h_jobs, sizeof(TileArgs) * nitems, hipMemcpyHostToDevice, s));
    HIP_TRY(hipMemcpyAsync(sl.d_first, sl.h_first, sizeof(long long) * (nitems + 1), hipMemcpyHostToDevice, s));
    int grid = (int)std::min<long long>(b->grid, total);
    HIP_TRY(launch_queue(b->d.precision, sl.d_jobs, sl.d_first, nitems, total, sl.counter, grid, s));
    HIP_TRY(hipEventRecord(sl.done, s));
    sl.used = true;
    return MFFT_OK;
}

int mfft_exec_pass(mfft_plan p, int pass, const void *in, void *out, void *stream, void *start_event, void *stop_event)
{
    if (!p || !in || !out) return fail(MFFT_ERR_INVALID, "null argument");
    if (pass < 0 || pass >= (int)p->passes.size())
        return fail(MFFT_ERR_INVALID, "pass %d of %d", pass, (int)p->passes.size());
    if ((start_event || stop_event) && p->chunk < p->batch)
        return fail(MFFT_ERR_UNSUPPORTED, "kernel events need a single-chunk plan (%lld per chunk, batch %lld)",
                    p->chunk, p->batch);
    return exec_all(p, in, out, stream, nullptr, -1, nullptr, nullptr, pass, (hipEvent_t)start_event,
                    (hipEvent_t)stop_event);
}

int mfft_exec_events(mfft_plan p, const void *in, void *out, void *stream, void **events, int nevents)
{
    if (!p || !in || !out || !events) return fail(MFFT_ERR_INVALID, "null argument");
    long long nchunks = (p->batch + p->chunk - 1) / p->chunk;
    long long need = nchunks * (long long)p->passes.size() + 1;
    if (nevents < need) return fail(MFFT_ERR_INVALID, "need %lld events, got %d", need, nevents);
    return exec_all(p, in, out, stream, (hipEvent_t *)events);
}

struct mfft_graph_s {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

int mfft_graph_create(mfft_graph *graph, mfft_plan p, const void *in, void *out, void *stream)
{
    if (!graph || !p || !in || !out) return fail(MFFT_ERR_INVALID, "null argument");
    *graph = nullptr;
    hipStream_t s = (hipStream_t)stream;
    hipStream_t cap = s;
    bool own = false;
    if (!cap) {  // the legacy default stream cannot be captured
        HIP_TRY(hipStreamCreateWithFlags(&cap, hipStreamNonBlocking));
        own = true;
    }
    mfft_graph g = new mfft_graph_s;
    hipError_t e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
    int rc = e == hipSuccess ? exec_all(p, in, out, cap, nullptr) : fail(MFFT_ERR_HIP, "begin capture: %s", hipGetErrorString(e));
    hipError_t e2 = hipStreamEndCapture(cap, &g->graph);
    if (!rc && e2 != hipSuccess) rc = fail(MFFT_ERR_HIP, "end capture: %s", hipGetErrorString(e2));
    if (!rc && hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0) != hipSuccess)
        rc = fail(MFFT_ERR_HIP, "graph instantiate");
    if (own) (void)hipStreamDestroy(cap);
    if (rc) {
        if (g->graph) (void)hipGraphDestroy(g->graph);
        delete g;
        return rc;
    }
    *graph = g;
    return MFFT_OK;
}

int mfft_graph_launch(mfft_graph g, void *stream)
{
    if (!g) return fail(MFFT_ERR_INVALID, "null graph");
    HIP_TRY(hipGraphLaunch(g->exec, (hipStream_t)stream));
    return MFFT_OK;
}

int mfft_graph_destroy(mfft_graph g)
{
    if (!g) return MFFT_OK;
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    delete g;
    return MFFT_OK;
}

int mfft_input_permutation(mfft_plan p, int axis, int *rev, int n)
{
    if (!p || !rev || axis < 0 || axis > 1) return fail(MFFT_ERR_INVALID, "bad argument");
    int len = p->kind == 1 ? p->n : (axis == 0 ? p->nx : p->ny);
    if (n != len) return fail(MFFT_ERR_INVALID, "length %d != %d", n, len);
    std::vector<int> rad, r;
    rev_radices(len, rad);
    gen_rev(len, rad, r);
    memcpy(rev, r.data(), sizeof(int) * len);
    return MFFT_OK;
}

int mfft_stage_convert(const void *src, int src_fmt, void *dst, int dst_fmt, int64_t n_inner, int64_t batch,
                       const int *perm_x, int nx, const int *perm_y, int ny, double scale, void *stream)
{
    if (!src || !dst || n_inner < 0 || batch < 0) return fail(MFFT_ERR_INVALID, "bad argument");
    if (src_fmt < 0 || src_fmt > 3 || dst_fmt < 0 || dst_fmt > 3) return fail(MFFT_ERR_INVALID, "format");
    if (perm_y && (ny <= 0 || n_inner % ny != 0)) return fail(MFFT_ERR_INVALID, "2D staging needs ny | n_inner");
    if (src == dst) return fail(MFFT_ERR_INVALID, "staging is out of place");
    if (trace_active()) {
        auto eb = [](int f) -> long long { return f == MFFT_FMT_C64 ? 16 : f == MFFT_FMT_C32 ? 8 : 4; };
        trace_launch((hipStream_t)stream, "stage_convert", batch * n_inner * eb(src_fmt), batch * n_inner * eb(dst_fmt));
    }
    HIP_TRY(stage_convert(src, src_fmt, dst, dst_fmt, n_inner, batch, perm_x, nx, perm_y, ny, scale,
                          (hipStream_t)stream));
    return MFFT_OK;
}

int mfft_trace_begin(void **events, mfft_launch_record *records, int capacity)
{
    if (!events || !records || capacity < 1) return fail(MFFT_ERR_INVALID, "trace: bad argument");
    if (mfft::trace_active()) return fail(MFFT_ERR_INVALID, "trace: already active on this thread");
    mfft_trace_reset((hipEvent_t *)events, records, capacity);
    return MFFT_OK;
}

int mfft_trace_end(void *stream, int *nlaunches)
{
    if (!nlaunches) return fail(MFFT_ERR_INVALID, "trace: null argument");
    int n = 0;
    bool overflow = false;
    hipEvent_t last = nullptr;
    hipError_t err = mfft_trace_stop(&n, &overflow, &last);
    *nlaunches = n;
    if (!last) return fail(MFFT_ERR_INVALID, "trace: not active on this thread");
    if (err != hipSuccess) return fail(MFFT_ERR_HIP, "trace: event record: %s", hipGetErrorString(err));
    HIP_TRY(hipEventRecord(last, (hipStream_t)stream));
    if (overflow) return fail(MFFT_ERR_INVALID, "trace: more launches than the %d records", n);
    return MFFT_OK;
}

const char *mfft_last_error(void) { return g_err.c_str(); }

const char *mfft_version(void) { return "mfft 0.1 (gfx950 matrix-core FFT)"; }

}  // extern "C"

namespace mfft {

void set_last_error(const char *msg) { g_err = msg ? msg : ""; }

void digit_reversal_radices(int n, std::vector<int> &out) { rev_radices(n, out); }

// ------------------------------------------------------------------ launch trace
namespace {
struct Trace {
    hipEvent_t *events = nullptr;
    mfft_launch_record *rec = nullptr;
    int cap = 0, n = 0;
    bool overflow = false;
    hipError_t err = hipSuccess;
};
thread_local Trace t_trace;
thread_local bool t_trace_on = false;
}  // namespace

bool trace_active() { return t_trace_on; }

void mfft_trace_reset(hipEvent_t *events, mfft_launch_record *rec, int cap)
{
    t_trace = Trace();
    t_trace.events = events;
    t_trace.rec = rec;
    t_trace.cap = cap;
    t_trace_on = true;
}

// ends the trace: n launches recorded; *last = the event to record after them (null when no
// trace was active)
hipError_t mfft_trace_stop(int *n, bool *overflow, hipEvent_t *last)
{
    *last = nullptr;
    if (!t_trace_on) return hipSuccess;
    t_trace_on = false;
    *n = t_trace.n;
    *overflow = t_trace.overflow;
    *last = t_trace.events[t_trace.n];
    return t_trace.err;
}

const char *fmt_name(int fmt) { return fmt == FMT_C16 ? "c16" : fmt == FMT_CBF16 ? "cbf16" : "c32"; }

void trace_launch(hipStream_t s, const char *kernel, long long bytes_read, long long bytes_written)
{
    if (!t_trace_on) return;
    Trace &t = t_trace;
    if (t.n >= t.cap) {
        t.overflow = true;
        return;
    }
    const hipError_t e = hipEventRecord(t.events[t.n], s);
    if (e != hipSuccess && t.err == hipSuccess) t.err = e;
    mfft_launch_record &r = t.rec[t.n];
    snprintf(r.kernel, sizeof r.kernel, "%s", kernel);
    r.bytes_read = bytes_read;
    r.bytes_written = bytes_written;
    ++t.n;
}

static bool capturing(hipStream_t s)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

hipError_t StreamOrder::acquire(hipStream_t s)
{
    if (!used || s == last || capturing(s)) return hipSuccess;
    if (ev) return hipStreamWaitEvent(s, ev, 0);
    hipError_t e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    return e;
}

hipError_t StreamOrder::release(hipStream_t s)
{
    if (capturing(s)) return hipSuccess;
    last = s;
    used = true;
    return ev ? hipEventRecord(ev, s) : hipSuccess;
}

void StreamOrder::destroy()
{
    if (ev) (void)hipEventDestroy(ev);
    ev = nullptr;
}

int plan_create_2d_conv(mfft_plan *plan, int nx, int ny, int64_t batch, const mfft_desc *d, bool out_mid)
{
    return create_2d_all(plan, nx, ny, batch, d, out_mid, true);
}

bool plan_first_pass_fusable(mfft_plan p)
{
    return p && !p->passes.empty() && p->passes.front().small && p->passes.front().src == BUF_IN;
}

// A pass on a matrix-core kernel that has a form with this end fused: transforms along l1, the same
// words on both sides.
static bool fast_ends_pass(mfft_plan p, const PassSpec &ps, int kind, int ends)
{
    return !p->small && p->d.precision == PREC_SPLIT && ps.fast_kind == kind && !ps.tw_N && !ps.rev_fast && ps.l1 >= 0 &&
           ps.lines[ps.l1].batch && src_fmt(p, ps) == dst_fmt(p, ps) && find_fast_ends(ps.R, ends, dst_fmt(p, ps)) != nullptr;
}

bool plan_takes_real(mfft_plan p, int f64, long long planes, int h, int w)
{
    if (plan_first_pass_fusable(p)) return true;
    return p && p->kind == 2 && !p->passes.empty() && !f64 && planes * h * w < (1LL << 29) &&
           p->passes.front().src == BUF_IN && p->passes.front().R == p->ny && p->passes.front().l2 < 0 &&
           fast_ends_pass(p, p->passes.front(), KIND_ROWS, ENDS_REAL);
}

// The last pass of the column axis, whole (R = nx) or the second of two (its l2 level is then the
// first pass's frequency).
bool plan_takes_crop(mfft_plan p, int f64, long long planes, int h, int w)
{
    if (!p || p->kind != 2 || p->passes.empty() || f64 || planes * h * w >= (1LL << 29)) return false;
    const PassSpec &ps = p->passes.back();
    if (!ps.col_axis || !fast_ends_pass(p, ps, KIND_COLS, ENDS_CROP)) return false;
    if (ps.R == p->nx) return ps.l2 < 0;
    return ps.l2 >= 0 && !ps.lines[ps.l2].batch && ps.lines[ps.l2].out_stride % p->ny == 0 && ps.ps_out % p->ny == 0;
}

int exec_fused(mfft_plan p, const void *in, void *out, int64_t batch, void *stream, const ExecFuse &f)
{
    const bool rows = !f.in_mul && !f.real_src2 && plan_takes_real(p, f.real_f64, (long long)f.real_b * f.real_c, f.real_h, f.real_w);
    if (f.input() && !rows && !plan_first_pass_fusable(p))
        return fail(MFFT_ERR_UNSUPPORTED, "first pass takes no fused input");
    if (f.crop_out && !plan_takes_crop(p, 0, f.crop_b ? (long long)f.crop_b * f.crop_c : p->batch, f.crop_h, f.crop_w))
        return fail(MFFT_ERR_UNSUPPORTED, "last pass takes no fused crop");
    if (batch < 1 || batch > p->batch) return fail(MFFT_ERR_INVALID, "batch %lld outside 1..%lld", (long long)batch, p->batch);
    return exec_all(p, in, out, stream, nullptr, batch, nullptr, &f);
}

}  // namespace mfft
