// How a batch of up to 64 requests is split when the kernels choose (kv_split
// = 0): the arithmetic that the kernels (auto_split) and the host's sizes of
// grid and workspace (split_plan) have to agree on.  Plain C++, so that a test
// can hold the sizes against the choice without a device.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define CAST_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define CAST_HOST_DEVICE inline
#endif

namespace cast {

constexpr int kSplitCandidates = 4;

// Items that splits below split_least tiles are made for: with fewer of them.
CAST_HOST_DEVICE int split_few(bool f32, int slots) { return f32 ? slots : 192; }
CAST_HOST_DEVICE int split_least(bool f32) { return f32 ? 4 : 8; }

// Tiles of 64 keys per split that the candidates start from.  share: the even
// share ceil(total / slots) of the batch's total tiles, per_few: total /
// split_few, smallest: tiles of the smallest chunk.
CAST_HOST_DEVICE int split_start(int share, int64_t total, int per_few, int smallest, bool f32, int slots) {
    const int least = split_least(f32);
    const int floor = total >= (int64_t)least * split_few(f32, slots) ? least : per_few > smallest ? per_few : smallest;
    return share > floor ? share : floor;
}
// Candidate w: {8, 9, 10, 12} / 8 of the start.
CAST_HOST_DEVICE int split_candidate(int start, int w) { return (start * (w < 3 ? 8 + w : 12) + 7) >> 3; }
// The candidate taken: the first whose items fit the slots, 10/8 where none does.
CAST_HOST_DEVICE int split_pick(bool fit0, bool fit1, bool fit2, bool fit3) {
    return fit0 ? 0 : fit1 ? 1 : fit2 ? 2 : fit3 ? 3 : 2;
}

// Whether a batch whose rows alone fill the device is so even that it is better
// left whole: its longest request (t_max tiles) no longer, against the average
// over row blocks, than what the partials of two splits cost beside the keys
// and values, less a tenth for what a split hides of latency
// (split_even_limit: rows x 2 x 8 bytes a head dim written and read against
// keys x 4; the host has the averages of both).
CAST_HOST_DEVICE bool split_even(int t_max, int rb_sum, int W, float limit) {
    return (float)t_max * (float)rb_sum <= limit * (float)W;
}
inline float split_even_limit(int64_t rows_avg, int64_t t_avg) { return 0.9f + 4.f * (float)rows_avg / (float)t_avg; }

// Bounds of that choice, with c >= L = total / slots tiles per split (total =
// Hkv * sum of row blocks x tiles) and RB >= sum rb: the items fit the slots,
// or c >= 10/8 L and they are Hkv * sum rb * ceil(tiles / c) <= 8/10 slots +
// Hkv * RB; an XCD takes at most ceil(groups / nx) groups of each request, so
// its slots are at most items / nx, plus RB where Hkv is no multiple of nx
// (workgroups past the last item cost their prologue at the end of the call:
// 2 us at the headline with a bound of 640 for 256); a request in ns > 1
// splits has ns - 1 < tiles / c and P <= rb * rows_wg / G, so the partial rows
// sum to less than rows_wg * slots / Hq plus the rows of the split requests,
// which are at most that many again.  (A batch left whole: Hkv * sum rb items.)
struct SplitBounds {
    int64_t part_rows;   // partial rows
    int64_t wgs;         // workgroups
};
inline SplitBounds split_bounds(int64_t batch, int64_t total_q, int64_t Hq, int64_t Hkv, int64_t rows_wg,
                                int64_t rbmax, int64_t slots, int64_t xcds) {
    const int64_t by_rows = total_q * (Hq / Hkv) / rows_wg + batch, by_pack = batch * rbmax;
    const int64_t rb_sum = by_rows < by_pack ? by_rows : by_pack;
    const int64_t once = (rows_wg * slots + Hq - 1) / Hq;
    const int64_t second = (slots * 8 + 9) / 10 + Hkv * rb_sum;
    const int64_t most = second > slots ? second : slots;
    return {once + (once < total_q ? once : total_q),
            xcds * ((most + xcds - 1) / xcds + (Hkv % xcds ? rb_sum : 0))};
}

}  // namespace cast
