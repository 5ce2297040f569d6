#pragma once
// How prefill kernels cut their work: functions of sizes alone (no GPU types), so that the
// rules can be checked on any host.
#include <algorithm>
#include <cstdint>

namespace q35k {

// ---------------------------------------------------------------- key ranges of the attention prefill
// waves per workgroup, 16 query rows each: with a bf16 cache two workgroups of 4 share a
// compute unit, and one's staging and barriers run under the other's products
constexpr int kBf16Waves = 4;
constexpr int flash_waves(bool kv_bf16) { return kv_bf16 ? kBf16Waves : 8; }
constexpr int kKT = 32;             // keys per tile
constexpr int kFlashPieces = 128;   // most pieces of a block
constexpr int kFlashSlots = 8192;   // most partial outputs ("slots": 16 rows of one piece; 135 MB)
constexpr int kFlashWhole = 64;     // blocks of up to so many tiles are never cut

// How the attention kernel splits a block of T tokens at pos0 over key ranges: tiles per piece,
// pieces of the longest row block (0: not split), the slots that takes, the expected time (in
// tiles; 0 where no split is considered), and the same were all pieces as long as the longest
// (whole rounds of workgroups).
struct FlashPlan {
    int piece, pieces, slots;
    double time, rounds;
};

// Cuts blocks into pieces where the longest block would outlast an even share of the work, into
// at most `room` slots on `n_cu` compute units.
// All times in tiles of 32 keys (5.9 us a tile of an fp32 cache, 3.1 us of a bf16 one). One
// workgroup runs per compute unit and they start longest first, so unsplit blocks take the
// longest of them or, with more blocks than compute units, the longest pair that shares one.
// Pieces of c tiles that all start at once take c and about one more for the query rows and
// the stores; more of them take an even share and about half a piece of unevenness. The merge
// and its launch are about four more, and a hundredth per piece for its 128 KB of partial
// output. Split when that is a tenth less. Blocks of up to 64 tiles (2048 keys) stay whole:
// their output keeps the same bits whatever workspace the caller gives.
inline FlashPlan flash_plan(int T, int NQ, int NKV, int pos0, bool kv_bf16, int n_cu, int64_t room = kFlashSlots) {
    const int waves = flash_waves(kv_bf16), kQT = 16 * waves;
    const int grp = NQ / NKV, rows = T * grp, nblk = (rows + kQT - 1) / kQT;
    const int64_t items = static_cast<int64_t>(nblk) * NKV;
    const int cu = n_cu * (8 / waves);  // workgroups that run at once
    room = std::min<int64_t>(room, kFlashSlots);
    // tiles of block b; rank r (longest first) is block nblk - 1 - r / NKV
    const auto tiles = [&](int64_t b) {
        return static_cast<int>((pos0 + std::min<int64_t>(rows - 1, b * kQT + kQT - 1) / grp) / kKT + 1);
    };
    FlashPlan p{0, 0, 0, 0.0, 0.0};
    const int most = tiles(nblk - 1);
    if (most <= kFlashWhole || items >= 2 * cu) return p;
    const auto ranked = [&](int64_t r) { return r < items ? tiles(nblk - 1 - r / NKV) : 0; };
    p.time = most;
    for (int i = 0; i < cu && cu + i < items; ++i) p.time = std::max<double>(p.time, ranked(cu - 1 - i) + ranked(cu + i));
    p.rounds = p.time;
    double best = 0.9 * p.time;
    for (int pieces = 2; pieces <= kFlashPieces && pieces * items * waves <= room; ++pieces) {
        const int c = (most + pieces - 1) / pieces;
        int64_t n = 0, all = 0;
        for (int b = 0; b < nblk; ++b) {
            n += static_cast<int64_t>((tiles(b) + c - 1) / c) * NKV;
            all += static_cast<int64_t>(tiles(b)) * NKV;
        }
        const double t = (n <= cu ? c + 1.0 : static_cast<double>(all + n) / cu + 0.6 * c) + 4.0 + 0.01 * n;
        if (t < best) {
            best = t;
            p = FlashPlan{c, (most + c - 1) / c, static_cast<int>((most + c - 1) / c * items * waves), t,
                          static_cast<double>((n + cu - 1) / cu * (c + 1))};
        }
    }
    return p;
}

// Workspace of the attention prefill in floats, all multiples of 16 bytes: the query rows; the
// keys and values of positions [0, pos0 + T) of an fp32 cache pre-split into the kernel's tile
// layout (K chunks [3 parts][2][32][16] of 16 bytes a tile, as many for V); the slots' partial
// outputs with their rows' maxima and sums.
constexpr int kImgK = 3 * 2 * 32 * 16;  // 16-byte chunks of a tile's K
constexpr int kImgTile = 2 * kImgK;
inline int64_t attn_prefill_workspace_floats(int NQ, int T) { return static_cast<int64_t>(NQ) * T * 256 + 64; }
inline int attn_prefill_image_tiles(int pos0, int T) {
    return static_cast<int>((static_cast<int64_t>(pos0) + T + kKT - 1) / kKT);
}
inline int64_t attn_prefill_image_floats(int NKV, int pos0, int T) {
    return static_cast<int64_t>(NKV) * attn_prefill_image_tiles(pos0, T) * kImgTile * 4;
}
inline int64_t attn_prefill_part_floats(int64_t slots) { return slots * 16 * (256 + 2); }

// What the attention prefill does with `floats` of workspace beyond its query rows: the tile
// image, then partial outputs in the rest, or without the image more of those. The image comes
// first unless that costs the cut more than it saves, and it saves what its readers, the row
// blocks of a head, would spend on splitting the tiles themselves: 5 to 20% of a cut of many
// blocks, 25 to 30% of uncut ones, nothing where fewer than 8 blocks read it. Which of two cuts is
// the faster one is told by their rounds. Over 1106 pairs (16 to 2000 tokens, 16 / 2 and 8 / 2
// heads, 2100 to 32000 positions, rooms between) the choice was within 2% of the one without the
// image or faster in all but two (7%), and on average 0.8% slower than the faster of the two: 700
// tokens of 16 heads at 16000 positions, image and 5632 slots 955 us against 1115 with 7744 slots
// alone; 1200 at 2100, image and 2400 slots 492, 3600 slots alone 427; 1500 at 8000, image and
// no cut 1263, 7520 slots alone 1399.
struct AttnRoom {
    bool image;
    FlashPlan plan;
};
inline AttnRoom attn_prefill_room(int T, int NQ, int NKV, int pos0, bool kv_bf16, int n_cu, int64_t floats) {
    const auto plan = [&](int64_t room) {
        return flash_plan(T, NQ, NKV, pos0, kv_bf16, n_cu, std::max<int64_t>(room, 0) / attn_prefill_part_floats(1));
    };
    const AttnRoom without{false, plan(floats)};
    const int64_t img = attn_prefill_image_floats(NKV, pos0, T);
    if (kv_bf16 || img > floats) return without;
    const AttnRoom with{true, plan(floats - img)};
    const int64_t blocks = (static_cast<int64_t>(T) * (NQ / NKV) + 16 * flash_waves(false) - 1) / (16 * flash_waves(false));
    const double gain = !with.plan.pieces ? 1.35 : blocks >= 8 ? 1.15 : 1.0;
    return with.plan.rounds <= gain * without.plan.rounds ? with : without;
}

// Slots a program that keeps one workspace for all blocks of up to T tokens within max_ctx
// positions sets aside: none where nothing is ever cut, no more than the most pieces of every
// row block, and at most half of kFlashSlots (68 MB; a cut into those is at most 1.3 times the
// time of the best one by the estimate above). Never less for more tokens or positions.
inline int attn_prefill_share_slots(int T, int NQ, int NKV, bool kv_bf16, int64_t max_ctx) {
    if (max_ctx <= kFlashWhole * kKT) return 0;
    const int waves = flash_waves(kv_bf16), kQT = 16 * waves;
    const int64_t items = (static_cast<int64_t>(T) * (NQ / NKV) + kQT - 1) / kQT * NKV;
    const int64_t pieces = std::min<int64_t>(kFlashPieces, (max_ctx + kKT - 1) / kKT);
    return static_cast<int>(std::min<int64_t>(items * waves * pieces, kFlashSlots / 2));
}

}  // namespace q35k
