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

// ---------------------------------------------------------------- few-token GEMM (k_gemm_small.hip)
enum SmallPath : int { kBf16 = 0, kF16 = 1, kF16Planes = 2 };  // X row-major / tiled (xt_off) / split (xp_off)
constexpr int kGemmSmallRows = 1024;
constexpr int kSmallBlk = 512;  // K of one partial sum
constexpr int kXcds = 8;        // XCDs: workgroups are dispatched to them in turn
constexpr int kSmallCus = 256;  // most compute units a plan counts on (its column tiles are bounded by that)

constexpr int max_waves(int mr, int nr) { return mr * nr <= 3 ? 12 : mr * nr <= 6 ? 8 : 4; }

// How the matrix is cut: row tiles of whole 16-row blocks (at most mr of them), column tiles
// of whole units of `unit` columns (at most 16 nr columns), both as even as they come.
struct SmallPlan {
    int mr, nr, rt, ct, unit;
};
constexpr int kSmallTiles[][2] = {{1, 1}, {1, 2}, {1, 3}, {1, 5}, {2, 2}, {2, 3}, {2, 4}, {2, 5}, {3, 3}, {3, 5}, {4, 3}, {4, 4}};

// The tile with the least expected time, or false where the 128 x 128 tiles are expected to
// be faster. The expected times are least-squares fits, in us, of this kernel's times over
// 96 products of 1 to 768 tokens (all twelve tiles, the six projection shapes of the 0.8B
// and 2B models, 10% rms): a launch, and for each 512-deep block of K the X and W lines of
// all tiles on the busiest compute unit, and the products and the split of X of its busiest
// SIMD. Coefficients of the fit, not costs one by one: X and its split both grow with the row
// blocks, which the fit cannot tell apart (it charges the split where X is already split, and not
// where the fp16 path splits it). The tile so chosen took on average 1.2% longer than the best of
// the twelve. The 128 x 128 kernel takes one time per tile alone on a compute unit and one per two
// that share it (128 tokens by 8224 x 2048: 65 tiles 53 us, 512 tokens: 260 tiles 82 us). It stays
// within 3% of its expected time, but with X as fp32 for the fp16 path and one or two blocks of K
// (below the fitted products) within 10%: 256 tokens by 7168 x 1024, 0.93 expected, took 6 us more
// than its 25, 384 by 5120 x 1024, 0.94, 3 us; at 0.9 and below at most 1.5 us, mostly less.
inline bool gemm_small_plan(int M, int N, int K, bool swiglu, int path, int n_cu, SmallPlan* best) {
    if (M > kGemmSmallRows) return false;  // from there on 128 x 128 tiles fill the chip for every N >= 2048
    // us per 512-deep block: X (16 rows), W (16 columns), products (16 x 16 block), split (16 rows)
    constexpr double kCost[3][4] = {{0.60, 0.43, 0.43, 0.43}, {0.42, 0.38, 0.41, 0.0}, {0.10, 0.41, 0.39, 0.21}};
    constexpr double kBig[3][2] = {{12.2, 20.5}, {10.2, 16.0}, {8.0, 12.7}};  // one tile, two tiles per CU
    constexpr double kLaunch = 4.5;
    const int cu = std::min(std::max(kXcds, n_cu), kSmallCus);
    const int nblk = (K + kSmallBlk - 1) / kSmallBlk, blocks = (M + 15) / 16;
    const int per_cu = (((N + 127) / 128) * ((M + 127) / 128) + cu - 1) / cu;
    double least = (path == kF16 && nblk <= 2 ? 0.90 : 0.97) * (kLaunch + nblk * (kBig[path][0] * (per_cu & 1) + kBig[path][1] * (per_cu >> 1)));
    bool found = false;
    for (const auto& t : kSmallTiles) {
        const int mr = t[0], nr = t[1];
        if (mr > blocks) continue;
        SmallPlan p{mr, nr, (blocks + mr - 1) / mr, (N + 16 * nr - 1) / (16 * nr), N % 4 == 0 ? 4 : swiglu ? 2 : 1};
        // workgroups of the busiest compute unit, and as many column tiles as that allows
        // (rt > 1: whole columns of row tiles per XCD)
        int k;
        if (p.rt == 1) {
            k = (p.ct + cu - 1) / cu;
            p.ct = cu * k;
        } else {
            const int cux = cu / kXcds, c8 = (p.ct + kXcds - 1) / kXcds;
            k = (c8 * p.rt + cux - 1) / cux;
            p.ct = std::max(c8, cux * k / p.rt) * kXcds;
        }
        p.ct = std::min(p.ct, (N + p.unit - 1) / p.unit);
        const int mw = max_waves(mr, nr), rounds = (nblk + mw - 1) / mw;
        const int simd = std::max((k * nblk + 3) / 4, rounds);  // K blocks of the busiest SIMD
        const double* c = kCost[path];
        const double us = kLaunch + k * nblk * (c[0] * ((blocks + p.rt - 1) / p.rt) + c[1] * N / (16.0 * p.ct)) +
                          simd * mr * (c[2] * nr + c[3]);
        if (us < least) {
            least = us;
            *best = p;
            found = true;
        }
    }
    return found;
}

// The most column tiles (so partial row maxima, SwiGLU) a plan for N columns has. A plan has the
// tiles that N needs, at most N / 16 + 1, rounded up to the compute units (one row tile: at most
// kSmallCus - 1 more) or, per XCD, to a share of its units over the row tiles.
inline int gemm_small_max_parts(int N) { return N / 16 + kSmallCus + 16; }

}  // namespace q35k
