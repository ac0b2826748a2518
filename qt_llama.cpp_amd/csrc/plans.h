// plans.h -- which kernel form a batched attention, a decode softmax or a
// batched product takes: the dispatch rules as host functions of sizes, types
// and positions (no HIP in here, so that a CPU test can evaluate them).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace mrml {

constexpr int kCUs = 256, kSIMDs = 4 * kCUs, kLdsBytes = 160 << 10;  // MI355X; LDS of a CU

// ---- decode softmax ------------------------------------------------------------
// The line lies on the widest window of the launch, not on the cache's
// capacity, and where the weights take as much LDS as LONG's chunk and flags:
// up to there the LDS form costs a batch no resident workgroup.  (A launch of
// one row has at most 256 workgroups, one a CU, and would have LDS for longer
// windows.)  Attention in caches
// of 8192 positions, LONG / LDS form: 5310 positions, 4 heads of 64 dims over
// Q4_0 rows 65.6 / 41.9 us; 2774, 8 heads of 128 over f16 36.8 / 25.4; a window
// of 1024, 16 heads of 128 over Q8_0/Q4_0 23.2 / 19.5.
constexpr int kSVShort = 10240;  // positions: 40 KiB of weights
#if defined(__HIPCC__)
__host__ __device__
#endif
constexpr bool sv_long(int span) { return span > kSVShort; }

constexpr int kSVD = 32;  // dims of a decode-form workgroup

// ---- attention of many query rows ------------------------------------------------
// `rows` rows at positions n_past0.., each seeing the last min(position + 1,
// wlimit) positions.
constexpr int kRowsP = 64;    // positions per score tile
constexpr int kRowsW = 4;     // waves per score workgroup
constexpr int kRowsQM = 4, kRowsQC = kRowsW * kRowsQM;  // quantised K: chain rows a wave, a pass

#if defined(__HIPCC__)
__host__ __device__
#endif
constexpr int rows_k_stride(int head_dim) { return head_dim * 2 + 16; }  // bytes of a staged f16 K row

constexpr int kRowsShortHD = 256, kRowsShortMax = 112;  // dims and positions of the short form

struct AttnRowsPlan {
    int span;             // the widest window
    int t_lo;             // the first row's window start
    bool one_row_scores;  // scores by the decode kernels, a workgroup a row, else by attn_rows.hip's:
    int score_m;          // chain rows (row x query head) a wave
    int score_reps;       // passes over a staged tile
    int tiles;            // score tiles dispatched a row block
    bool all_tiles;       // those are all from t_lo to the last row's position
    bool short_form;      // softmax and weighted sum in one launch (attn_rows_short_kernel), else
    bool rows_form;       // softmax and weighted sum as attn_rows.hip has them, else the decode form
    int softmax_threads;
    int pv_m, pv_d;       // weighted sum: chain rows a wave, dims a lane
    int score_blocks(int nchains) const
    {
        const int per = kRowsW * score_m * score_reps;
        return (nchains + per - 1) / per;
    }
};

// The weighted sum of the rows form reads the cache through one buffer descriptor (32-bit offsets).
inline bool attn_rows_v_ok(int n_kv_heads, int head_dim, int v_fmt, int capacity)
{
    const uint64_t block = v_fmt == 0 ? 64 : (v_fmt == 1 ? 34 : 18);
    return (uint64_t)capacity * n_kv_heads * (head_dim / 32) * block < (1ull << 32) - (1 << 20);
}

inline AttnRowsPlan attn_rows_plan(int n_past0, int rows, int n_heads, int n_kv_heads, int head_dim, int k_fmt,
                                   int v_fmt, int capacity, int wlimit)
{
    AttnRowsPlan p{};
    const int nchains = rows * (n_heads / n_kv_heads), count0 = n_past0 + 1;
    p.span = std::min(wlimit, n_past0 + rows);
    // positions tiled absolutely from row 0's window start to the last row's position
    p.t_lo = count0 > wlimit ? count0 - wlimit : 0;
    const int tiles = (n_past0 + rows - 1 - p.t_lo) / kRowsP + 1, group = n_heads / n_kv_heads;
    // the tiles that the chain rows' windows meet: (w + 62) / 64 of w positions on average
    const int64_t chain_tiles = (int64_t)n_kv_heads * nchains * std::min(tiles * kRowsP, wlimit + kRowsP - 2) / kRowsP;
    if (k_fmt != 0) {
        // passes over a staged tile: as many as leave four workgroups a CU
        p.score_m = kRowsQM;
        p.score_reps = (int)std::min<int64_t>(8, std::max<int64_t>(1, chain_tiles / (kRowsQC * 4 * kCUs)));
    } else {
        // Chain rows a wave: one while its workgroups are resident at once (four
        // a CU, fewer where a tile takes more of the 160 KB of LDS), two up to twice as
        // many, else four (77 rows of 8 heads at 377 positions: 9.6 us with
        // one, 11 with four; 80 rows of 8 x 512 dims over one kv head behind
        // 300 positions, 3840 chain tiles for 2 a CU: 45.5 / 41.6 / 43.4 at 1 / 2 /
        // 4).  Two sets of them a workgroup once the launch is many rounds of
        // the chip (512 rows behind 2048 positions: 10,240 workgroups, 7 us
        // less; 512 rows from the start: 2048, 2 us more).
        // (Past 256 dims a quarter later: 2176 chain tiles of 512 dims 42.1 / 44.3, 2880
        // 45.7 / 42.5.)
        const int64_t resident = (int64_t)kCUs * std::min(4, kLdsBytes / (kRowsP * rows_k_stride(head_dim)));
        const int64_t one = kRowsW * resident * (head_dim > 256 ? 5 : 4) / 4;
        p.score_m = chain_tiles >= 2 * one ? 4 : (chain_tiles >= one ? 2 : 1);
        p.score_reps = chain_tiles / (kRowsW * p.score_m) >= 8192 ? 2 : 1;
    }
    // A row block's tiles: its rows span wlimit positions and one more a row
    // after the first.  (All tiles of the launch a block left most workgroups
    // of a sliding window without work: 500 rows x 8 heads over a window of 20
    // took 48 us, 44 without them.)  With a whole number of rounds of the eight
    // XCDs over tiles and kv heads, where that adds at most a quarter, a tile
    // stays on its XCD from block to block (300 rows of 8 heads of 256
    // dims over a window of 512, Q8_0: 68 us, 70 at 11 tiles instead of 12).
    const int block_rows = (kRowsW * p.score_m * p.score_reps + group - 2) / group + 1;
    p.tiles = (wlimit + block_rows - 2) / kRowsP + 2;
    const int round = n_kv_heads % 8 == 0 ? 1 : n_kv_heads % 4 == 0 ? 2 : n_kv_heads % 2 == 0 ? 4 : 8;
    const int whole = (p.tiles + round - 1) / round * round;
    if (4 * whole <= 5 * p.tiles) p.tiles = whole;
    p.tiles = std::min(tiles, p.tiles);
    p.all_tiles = p.tiles == tiles;

    // Few rows: the decode kernels, which take a workgroup a row, kv head and
    // tile and have q in LDS, are done before attn_rows_scores_kernel at one
    // chain row a wave, whose scalar loads of q are waited for one after another
    // (whole attention, 8 / 4 heads of 256 dims: 16 rows at 100 positions 16.3 us
    // against 17.9, 1 row at 2500 26.5 against 27.8; 8 x 64 dims, 8 rows from 0
    // 11.1 / 11.6), up to four of these workgroups a CU (16 rows of 8 kv heads at 700,
    // 1536 of them: 39.3 / 37.9; 64 of 4 at 100, 768: 20.1 / 21.0; 128 of 4 from
    // 0, 1024: equal), eight for groups of four (16 / 4 heads, 1280: 86.8 / 87.9, 2560
    // level; 32 / 8 of 64 dims, 2560: 48.3 / 49.1).  Not for groups past four heads (two heads a wave there:
    // 16 / 2 heads of 128 14.1 / 12.8), 96 to 224 dims (8 of 128: 12.6 / 12.6)
    // or more (groups of 8 heads of 512: 25.4 / 16.9), quantised K (8 / 4 heads of
    // 256, Q8_0: 18.7 / 15.3), or windows whose last tile holds eight positions
    // or fewer, where a workgroup of the 256-dim kernel loads the last row for all
    // of the others (4 / 1 heads at a window of 200, 40 rows: 21.3 / 20.8; 8 / 8
    // heads 26.2 / 25.0; 8 / 8 heads of 64, 10 rows: 12.2 / 12.9).
    const int64_t one_row = (int64_t)((p.span + kRowsP - 1) / kRowsP) * n_kv_heads * rows;
    const int window0 = std::min(wlimit, count0);
    const bool thin = head_dim == 256 && (window0 - 1) % kRowsP < 8 && (group == 4 || (window0 == wlimit && rows > 8));
    p.one_row_scores = k_fmt == 0 && group <= 4 && (head_dim == 256 || head_dim <= 64) &&
                       one_row <= std::max(4, 2 * group) * kCUs && !thin;

    // The decode form's workgroups (32 dims of a row, 4.7 ns a position) go over
    // the CUs in rounds of 256, each round up to three on a CU adding to the
    // launch, the rows form's waves run over the whole window with less company.
    // So its line falls with the round and rises with the window.  Rows
    // form minus decode form, us (8 / 4 heads of 256 dims; other shapes
    // within 1 us), by workgroups and widest window:
    //   f16        60    120    200    500    700   1000   2000
    //    256     +2.2   +3.2   +5.1   +9.8  +13.4  +18.8
    //    512     -0.5   -1.1   +0.5   +4.3   +7.8  +10.9  +23.4
    //    768     -4.4   -4.5   -4.1   -1.8   +0.7   +2.8  +11.0
    //   1024     -8.1   -8.5   -8.4   -5.9   -5.6   -5.3   -1.5
    //   Q8_0
    //    256     +4.0   +5.5   +9.3  +18.9  +26.0  +36.2
    //    512     +1.6   +1.7   +4.5  +12.9  +19.6  +27.7
    //    768     -2.6   -1.7    0.0   +6.6  +13.0  +19.6
    //   1024     -6.5   -5.3   -4.7   +1.6   +5.6  +10.6
    //   1280    -11.2  -11.2  -10.3   -6.5   -3.3   +0.2  +18.4
    const int64_t wgs = (int64_t)rows * n_heads * (head_dim / kSVD);
    const int from = v_fmt == 0 ? (wgs <= 256 ? 0 : wgs <= 512 ? 150 : wgs <= 768 ? 650 : INT32_MAX)
                                : (wgs <= 256 ? 0 : wgs <= 512 ? 40 : wgs <= 768 ? 200 : wgs <= 1024 ? 430
                                                                    : wgs <= 1280 ? 1000 : INT32_MAX);
    p.rows_form = p.span <= from && attn_rows_v_ok(n_kv_heads, head_dim, v_fmt, capacity);

    // One launch for both, us against the choice above (8 / 8 heads, whole
    // attention): against the decode form in its first round of workgroups, 1 row at
    // 0 10.9 / 11.5, at 60 13.2 / 11.6; after it, 16 rows at 60 14.8 / 15.6, at 100
    // 16.0 / 15.8; 64 rows from 0 14.2 / 15.2, 50 at 60 18.2 / 17.4; a window of 60,
    // 64 rows 15.4 / 16.4, 130 22.1 / 22.6 (16 / 16 heads, 50: 19.4 / 18.9); of
    // 20, 200 rows 22.4 / 25.7.
    const int64_t heads = (int64_t)rows * n_heads;
    p.short_form = group == 1 && head_dim == kRowsShortHD && v_fmt == 0 &&
                   (wgs <= kCUs ? p.span <= 16
                                : p.span <= 32 || (p.span <= 64 && heads <= 3 * kCUs) ||
                                      (p.span <= kRowsShortMax && heads <= kCUs));

    // Windows up to 256 positions: one wave a row and head, no barrier to wait
    // at (200 rows x 8 heads, window 20: 29.7 us, 27.3 with it, whole attention).
    // Rows enough to fill the chip: small workgroups, more of them a CU, and
    // chunks past 1024 positions (512 rows x 8 heads of 2300 positions: 54 us,
    // 65 with 512 threads, 76 with 1024).  Few rows: the latency of one chunk
    // counts (4 rows of 3000 positions: 6 us with 1024 threads, 13 with 256).
    p.softmax_threads = p.span <= 256 ? 64
                        : p.span <= 1024 || (int64_t)rows * n_heads >= 1024 ? 256
                        : p.span <= 2048 ? 512 : 1024;

    // Weighted sum: the four-row forms issue the fewest conversions and loads a
    // product, the narrow ones keep more SIMDs busy, so a form is left once it
    // has more than about one wave a SIMD (1024).  us at (4,2) / (4,1) / (2,1) /
    // (1,1), whole attention:
    //   f16, 256 dims: 1280 waves of (1,1) behind 2500 positions 149 / 115 / 99 / 120,
    //     1024 behind 700 - / - / 35.5 / 34.4; (4,1) from 800 waves of it (960 behind
    //     700 - / 55.3 / 56.9, 640 38.2 / 33.3 / 32.8 / 37.5), later where a wave has
    //     a whole head (8 / 8 heads of 64, 1000: 274 / 236 / 223 / 296); (4,2) is
    //     level with (4,1) at 2000 waves of its own (behind 0 / 300 / 2500
    //     positions: 79 / 76, 105 / 104, 384 / 405);
    //   Q8_0, where a lane's one dim is a byte load: (4,1) is never the best,
    //     (4,2) is from 400 (behind 300, 320: 42.4 / 50.8 / 42.1 / 53.0, 600: 52 / 64 /
    //     60 / 84);
    //   Q4_0: (4,1) from 600 (640: 45.1 / 38.3 / 42.3 / 53.1, 512 with Q8_0 keys behind
    //     2500 - / 160 / 138); (4,2), a byte a lane, from 1000 where a head is two of its
    //     slices (1200 behind 2500: 340 / 376), later where it is one (16 / 4
    //     heads of 128, 2000: 178 / 167).
    // A lane of two dims needs 128 of them, but for Q8_0.  Windows up to 160
    // positions are mostly their ends, which few rows share: two rows a wave (200
    // rows, window 20, 24.4 at (4,1), 21.1; 150 from 0 over Q8_0 29.1 at (4,2),
    // 27.6), up to 1536 waves of (4,2) (window 100, Q8_0, 1200 41.2 / 42.8, 2000
    // 51.2 / 53.7).
    auto waves = [&](int m, int d) {
        return (int64_t)n_kv_heads * ((nchains + m - 1) / m) * ((head_dim + 64 * d - 1) / (64 * d));
    };
    const bool ends = p.span <= 160, lanes2 = head_dim > 64 || v_fmt == 1;
    const int min42 = ends ? 1536 : v_fmt == 0 ? 2 * kSIMDs : v_fmt == 1 ? 400 : head_dim >= 256 ? 1000 : 2400;
    const int min41 = v_fmt != 0 ? 600 : head_dim > 64 ? 800 : 1536;
    p.pv_m = 1, p.pv_d = 1;
    if (lanes2 && waves(4, 2) >= min42) p.pv_m = 4, p.pv_d = 2;
    else if (v_fmt != 1 && !ends && waves(4, 1) >= min41) p.pv_m = 4;
    else if (waves(1, 1) > kSIMDs) p.pv_m = 2;
    return p;
}

// ---- batched Q4_0 products ---------------------------------------------------------
constexpr int kGemmWaves = 4;  // 32-token groups per workgroup of the tile kernel, sharing one 32-row tile
constexpr int kFewRows = 16, kFewTokens = 16;  // of a few-token workgroup

inline int64_t few_workgroups(int32_t rows, int32_t batch)
{
    return (int64_t)((rows + kFewRows - 1) / kFewRows) * ((batch + kFewTokens - 1) / kFewTokens);
}

// Whether a product of nb-block rows runs as gemm_q4_0_few_kernel, whose fold
// is exact, or in tiles (relaxed: with their one-FMA fold; the entry that asks
// for that fold always gets it).  A few-token workgroup costs about 1 ns and
// 8.5e-5 us a block once the chip is full; the tile kernel takes 0.2 us a block
// for anything up to one wave a SIMD (a lone wave's step), so the line rises
// with K.  us, few / tiles / relaxed tiles, at 2048, 2304 and 2560 workgroups
// (4096, 4608, 5120 rows, 128 tokens):
//   K  512   13.3 / 13.6 / 13.0   14.1 / 13.5 / 13.0   14.7 / 13.6 / 13.2
//   K 2304   22.6 / 24.2 / 22.4   24.1 / 24.7 / 22.6   25.7 / 24.6 / 22.7
//   K 4096   29.2 / 35.3 / 31.6   31.2 / 36.0 / 32.1   33.5 / 35.8 / 32.3
//   K 9216   51.9 / 66.5 / 59.4   57.0 / 68.0 / 60.1   61.5 / 67.2 / 59.1
// Few tokens leave the tiles' workgroups of four token groups with less than
// four waves' work: 18432 rows x 32 tokens (2304) at K 2304 24.0 / 35.4 / 33.2.
inline bool gemm_few(int32_t rows, int nb, int32_t batch, bool relaxed)
{
    const int64_t w = few_workgroups(rows, batch), groups = (batch + 31) / 32;
    if (w <= 2048 || w > 2304) return w <= 2048;
    const int64_t waves = (int64_t)((rows + 31) / 32) * ((groups + kGemmWaves - 1) / kGemmWaves) * kGemmWaves;
    return waves > kSIMDs || nb >= (relaxed ? 112 : 64);
}

// And gate, up and activation together: the tiles pay twice and an
// elementwise pass (9216 x 2304 at 64 tokens, 2304 workgroups, 38.6 / 48.5 us; 4608 x
// 512 at 128 19.5 / 24.6).
inline bool gemm_few_glu(int32_t rows, int32_t batch) { return few_workgroups(rows, batch) <= 2304; }

// Producers of a few-token workgroup: 8 while the workgroups leave CUs their
// LDS (two of them a CU), else 4 (up to four a CU).  2304 x 9216 at 16 tokens
// (144 workgroups) 9.6 with 8, 12.6 us with 4; at 48 (432) 13.8 and 15.0; 4096
// x 2304 at 24 (512) 7.1 and 6.4.  GLU holds two products' terms, so it takes
// 4: 9216 x 2304 at 12 tokens 16.2 us, 21.0 with 8 (two tile products and the
// elementwise pass: 42.5).
inline int gemm_few_producers(bool glu, int32_t rows, int32_t batch)
{
    return !glu && few_workgroups(rows, batch) < 448 ? 8 : 4;
}

// Row tiles that the tile kernel runs as FULL waves, one per (row tile, token
// group).  When those number just over one per SIMD (2304 rows at 512 tokens:
// 1152 for 1024), the SIMDs holding two of them set the launch's time; then
// only as many row tiles as give every SIMD one FULL wave stay FULL and the
// rest run as HALF waves (two per token group), which add a little over half a
// wave's work to some SIMDs instead of a whole one.
inline int gemm_full_tiles(int32_t rows, int32_t batch)
{
    const int ng = (batch + 31) / 32, rt = (rows + 31) / 32, gq = (ng + kGemmWaves - 1) / kGemmWaves;
    const int64_t full_waves = (int64_t)rt * gq * kGemmWaves;
    return full_waves > kSIMDs && 2 * full_waves <= 3 * kSIMDs ? kSIMDs / (gq * kGemmWaves) : rt;
}

}  // namespace mrml
