// Mixed-radix tile kernels for contiguous lines of 2^a 3^b 5^c 17^d points (mfft_mixed.hip).
#pragma once
#include "mfft_common.h"

#include <vector>

namespace mfft {

constexpr int kMixThreads = 512;
constexpr int kMixColTiny = 2048, kMixColSmall = 8192, kMixColLarge = 17408;  // points per tile of the strided kernels
constexpr int mix_col_threads(int cap) { return cap == kMixColTiny ? 256 : cap == kMixColSmall ? 512 : 1024; }
constexpr int kMixStages = 8;
constexpr int kMixInline = 64;  // work-queue items that travel in the kernel's arguments

// Stockham schedule of one line length, stage 0 first (the self-sorting order of the tile
// kernels). cols = R / radix; s = product of the earlier radices; mul multiplies the stage's
// outputs (scaling, and the 1/16 of the matrix-core operands).
struct MixSched {
    int R, nst;
    int radix[kMixStages], cols[kMixStages], s[kMixStages];
    float mul[kMixStages];
};

// One launch of lines of one length: nlines dense lines of R points, T per tile.
struct MixArgs {
    const void *in;
    void *out;
    long long nlines;
    const float2 *tw;      // W_R^e, e in [0, R), sign of the transform
    const void *dft_ops;   // DftOps
    int T, sign;
    float w16[3];
    MixSched sc;
};

// One launch of strided lines of one length (the columns of 2D transforms): transforms of c0
// adjacent lines each, T lines per tile (tiles0 tiles per transform).
struct MixColArgs {
    const void *in;
    void *out;
    const float2 *tw;
    const void *dft_ops;
    int T, sign, c0, tiles0;
    int ps_in, ps_out;           // elements between a line's points
    long long in_dist, out_dist; // elements between transforms
    float w16[3];
    MixSched sc;
};

// Work queue: an item is nlines dense lines of one registered length.
struct MixLen {
    const float2 *tw;
    MixSched sc;
};
struct MixItem {
    const void *in;
    void *out;
    long long nlines;
    int len, T;            // index into the length table; lines per tile
};
struct MixQueueArgs {
    const MixLen *lens;
    const void *dft_ops;
    const MixItem *items;      // more than kMixInline items: device arrays (else null)
    const int *first;          // first tile of each item
    unsigned *counter;         // {next tile, finished workgroups}, both 0 between launches
    int nitems, total, sign, tw_at;  // tw_at: LDS word where a tile's twiddle table starts
    float w16[3];
    int first_in[kMixInline];
    MixItem item_in[kMixInline];
};

// Where a single radix-16 stage, the one on the matrix cores, stands among the others (two or more
// always come last): its operands are 16-bit words, so what has been summed before it takes of fp16's
// range, and what a scaled stage has divided by is lost to fp16's smallest value.
enum MixOrder {
    MIX_16_LAST,       // the fastest
    MIX_16_AFTER_ODD,  // after the odd factors, before the even rest
    MIX_16_EARLY,      // that, or first of all where that takes fewer stages
    MIX_NO16,          // no such stage: all in fp32
};
// The radices of a length, stage order, as the kernels want them; false: not such a length.
bool mix_radices(int n, std::vector<int> &out, MixOrder order = MIX_16_LAST);
// Schedule of a length for a precision (scale: every stage multiplies by 1/radix).
bool mix_schedule(int n, int prec, bool scale, MixOrder order, MixSched &sc);
inline size_t mix_lds_bytes(int tile_points, int R) { return sizeof(float2) * ((size_t)tile_points + R); }
// The most that a launch of a kernel takes (cap as find_mixed_kernel's): its largest tile beside the
// longest line that comes in such tiles, 16 lines of 512 points or 8 of 2176, or a single one.
constexpr int mix_lds_max(int cap)
{
    return (int)sizeof(float2) * (!cap ? 2 * kMaxTile : cap + (cap == kMixColTiny ? kMixColTiny : cap == kMixColSmall ? kMixColSmall / 16 : kMixColLarge / 8));
}

// cap: 0 = contiguous lines, kMixColTiny, kMixColSmall or kMixColLarge = strided lines
const void *find_mixed_kernel(int prec, int in_fmt, int out_fmt, int cap = 0);
const void *find_mixed_queue_kernel(int prec, int in_fmt, int out_fmt);

}  // namespace mfft
