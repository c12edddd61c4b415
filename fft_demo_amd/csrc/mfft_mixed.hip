// Mixed-radix tile kernels: instantiations and the schedules of their lengths. Compiled once
// per part (MFFT_PART = 0: split fp16 with 16-bit ends and the host side; 1: split fp16 with
// 32-bit ends; 2: the single-word precisions), so the parts build in parallel.
#include "mfft_mixed_impl.h"

#include <algorithm>
#include <functional>

#ifndef MFFT_PART
#error "compile with -DMFFT_PART=0..2"
#endif

namespace mfft {

constexpr int kMixQueue = -1;

template <int PREC, int INF, int OUTF>
static const void *pick_mixed(int what)
{
    switch (what) {
    case 0: return (const void *)mixed::fft_mixed<PREC, INF, OUTF>;
    case kMixQueue: return (const void *)mixed::fft_mixed_queue<PREC, INF, OUTF>;
    case kMixColTiny: return (const void *)mixed::fft_mixed_cols<kMixColTiny, PREC, INF, OUTF>;
    case kMixColSmall: return (const void *)mixed::fft_mixed_cols<kMixColSmall, PREC, INF, OUTF>;
    case kMixColLarge: return (const void *)mixed::fft_mixed_cols<kMixColLarge, PREC, INF, OUTF>;
    default: return nullptr;
    }
}

#if MFFT_PART == 1
const void *find_mixed_split32(int inf, int outf, int what)
{
    if (inf == FMT_C16 && outf == FMT_C32) return pick_mixed<PREC_SPLIT, FMT_C16, FMT_C32>(what);
    if (inf == FMT_C32 && outf == FMT_C16) return pick_mixed<PREC_SPLIT, FMT_C32, FMT_C16>(what);
    if (inf == FMT_C32 && outf == FMT_C32) return pick_mixed<PREC_SPLIT, FMT_C32, FMT_C32>(what);
    return nullptr;
}
#elif MFFT_PART == 2
const void *find_mixed_plain(int prec, int inf, int outf, int what)
{
    if (prec == PREC_FP16 && inf == FMT_C16 && outf == FMT_C16) return pick_mixed<PREC_FP16, FMT_C16, FMT_C16>(what);
    if (prec == PREC_BF16 && inf == FMT_CBF16 && outf == FMT_CBF16)
        return pick_mixed<PREC_BF16, FMT_CBF16, FMT_CBF16>(what);
    if (prec == PREC_FP32 && inf == FMT_C32 && outf == FMT_C32) return pick_mixed<PREC_FP32, FMT_C32, FMT_C32>(what);
    return nullptr;
}
#else
const void *find_mixed_split32(int inf, int outf, int what);
const void *find_mixed_plain(int prec, int inf, int outf, int what);

static const void *find_mixed(int prec, int inf, int outf, int what)
{
    if (prec != PREC_SPLIT) return find_mixed_plain(prec, inf, outf, what);
    if (inf == FMT_C16 && outf == FMT_C16) return pick_mixed<PREC_SPLIT, FMT_C16, FMT_C16>(what);
    return find_mixed_split32(inf, outf, what);
}

const void *find_mixed_kernel(int prec, int inf, int outf, int cap) { return find_mixed(prec, inf, outf, cap); }
const void *find_mixed_queue_kernel(int prec, int inf, int outf) { return find_mixed(prec, inf, outf, kMixQueue); }

// Radices of n with the least sum of stage costs: a stage costs an LDS round trip of every
// point (about 20 issue slots a point) plus its butterfly. 16 is the matrix-core stage; 6, 10,
// 12 and 15 are coprime products, which save a round trip for a few additions.
bool mix_radices(int n, std::vector<int> &out, MixOrder order)
{
    if (order == MIX_16_EARLY) {
        std::vector<int> last;
        if (!mix_radices(n, last, MIX_16_LAST) || !mix_radices(n, out, MIX_16_AFTER_ODD)) return false;
        if (last.size() < out.size()) {
            const auto m16 = std::find(last.begin(), last.end(), 16);
            std::rotate(last.begin(), m16, m16 + 1);
            out = last;
        }
        return true;
    }
    static const struct { int r; float cost; } kRadix[] = {{17, 51}, {16, 28}, {15, 31}, {12, 28}, {10, 29}, {9, 35},
                                                           {8, 27},  {6, 26},  {5, 27},  {4, 24},  {3, 24},  {2, 23}};
    out.clear();
    if (n < 2 || n > kMaxTile) return false;
    std::vector<int> cur, best;
    float best_cost = 1e9f;
    std::function<void(int, size_t, float)> go = [&](int m, size_t from, float cost) {
        if (cost >= best_cost || cur.size() > (size_t)kMixStages) return;
        if (m == 1) {
            best = cur;
            best_cost = cost;
            return;
        }
        for (size_t i = from; i < sizeof kRadix / sizeof *kRadix; ++i) {
            const int r = kRadix[i].r;
            if (m % r || (order == MIX_NO16 && r == 16) || (order == MIX_16_AFTER_ODD && (r == 6 || r == 10 || r == 12))) continue;
            cur.push_back(r);
            go(m / r, i, cost + kRadix[i].cost);
            cur.pop_back();
        }
    };
    go(n, 0, 0.f);
    if (best.empty()) return false;
    // Order: radices with an odd factor first (the first stage writes LDS at a stride of its
    // radix, which an odd one spreads over the banks), then 8, 4 or 2, then the matrix-core
    // stages, whose last one stores 16 consecutive points per line segment. A power of two
    // starts with 16 (its four consecutive outputs per lane are 16-byte writes). A length of
    // one radix takes a copying first stage (radix 1).
    auto rank = [](int r) { return r == 16 ? 2 : (r & (r - 1)) == 0 ? 1 : 0; };
    std::stable_sort(best.begin(), best.end(), [&](int a, int b) { return rank(a) != rank(b) ? rank(a) < rank(b) : a > b; });
    if ((n & (n - 1)) == 0 && best.size() > 1 && order != MIX_NO16) {
        // [16, tail, 16, ...]; the lengths below 16 are one radix
        std::vector<int> o{16};
        for (int r : best)
            if (r != 16) o.push_back(r);
        while ((int)o.size() < (int)best.size()) o.push_back(16);
        best = o;
    }
    if (best.size() == 1) best.insert(best.begin(), 1);
    const auto m16 = std::find(best.begin(), best.end(), 16);
    if (order == MIX_16_AFTER_ODD && std::count(best.begin(), best.end(), 16) == 1)
        std::rotate(std::find_if(best.begin(), best.end(), [](int r) { return r % 2 == 0; }), m16, m16 + 1);
    out = best;
    return out.size() <= (size_t)kMixStages;
}

bool mix_schedule(int n, int prec, bool scale, MixOrder order, MixSched &sc)
{
    std::vector<int> r;
    if (!mix_radices(n, r, prec == PREC_FP32 ? MIX_16_LAST : order)) return false;
    sc = MixSched();
    sc.R = n;
    sc.nst = (int)r.size();
    // The vector-ALU stages' scales are one factor on the first stage's outputs: before the
    // matrix-core stages (fp16 operands), whose own scale stays with them, as every stage's
    // scale keeps values from growing past the input's magnitude. A last stage behind them has its own.
    float valu = 1.f;
    int s = 1;
    bool behind = false;
    for (int i = 0; i < sc.nst; ++i) {
        const bool mfma = r[i] == 16 && prec != PREC_FP32;
        sc.radix[i] = r[i];
        sc.cols[i] = n / r[i];
        sc.s[i] = s;
        sc.mul[i] = mfma ? (scale ? 1.f / 256 : 1.f / 16) : 1.f;  // the operands carry a factor 16
        if (scale && !mfma) (behind && i == sc.nst - 1 ? sc.mul[i] : valu) /= r[i];
        behind |= mfma;
        s *= r[i];
    }
    sc.mul[0] *= valu;
    return true;
}
#endif

}  // namespace mfft
