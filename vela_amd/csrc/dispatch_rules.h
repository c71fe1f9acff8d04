// Rules of the automatic kernel choice that depend on sizes alone: plain host C++, no HIP, so that they can be
// compiled and checked without a GPU.
#pragma once
#include <algorithm>

namespace vk {

constexpr int NCU = 256;   // MI355X compute units

inline int cdiv(long long a, long long b) { return int((a + b - 1) / b); }

// int32 rows on 64 x 320 tiles in place of 64 x 128 ones (epilogue PLAIN, no K split): no more padding columns than
// 128-wide tiles have, and a last round of blocks (two per CU) at least three quarters full, since a round costs
// nearly the same with one block per CU. The wide tile fetches and quantises a row once for 320 columns, which pays
// with the depth of K, and has the longer epilogue, above all the one in 64-bit integers (large column constants), so
// below K = 1280 (640 for one column of tiles) the last round must be seven eighths full, and shallow K stays on the
// 64 x 128 tiles (64 x 128 first, us, residual and row maxima, the 64-bit epilogue in brackets):
//                          K = 160                   320                       640                       1280
//   512 tiles, N = 320    26.9 / 24.8 [40.5 / 40.6]   30.8 / 28.1 [44.1 / 43.3]   41.4 / 34.5 [53.5 / 49.5]   63.4 / 48.5 [73.8 / 62.3]
//   448 tiles, N = 320    25.7 / 24.5 [38.8 / 40.2]   29.7 / 26.8 [42.2 / 42.3]   39.3 / 32.7 [51.5 / 48.1]   58.0 / 46.1 [70.2 / 59.8]
//   384 tiles, N = 320    24.6 / 24.5 [35.0 / 39.8]   27.3 / 26.6 [38.2 / 42.2]   35.5 / 32.0 [46.0 / 47.6]   51.4 / 43.3 [63.2 / 58.5]
//   512 tiles, N = 1280   26.2 / 24.8 [38.2 / 40.7]   29.1 / 27.4 [41.1 / 42.9]   37.1 / 33.7 [49.5 / 48.9]   54.5 / 47.0 [66.1 / 61.7]
//   900 tiles, N = 1280   39.3 / 44.5 [60.5 / 76.1]   44.3 / 49.4 [65.4 / 80.5]   59.5 / 61.5 [78.9 / 91.2]   93.8 / 85.6 [109.8 / 114.8]
inline bool x32_wide_tiles(int M, int N, int Kp) {
    const int round = 2 * NCU, cols = cdiv(N, 320);
    if (cols * 320 > cdiv(N, 128) * 128) return false;
    const int last = int(((long long)cdiv(M, 64) * cols - 1) % round) + 1;
    if (last < round * 3 / 4) return false;
    if (Kp >= (cols == 1 ? 640 : 1280)) return true;
    return last >= round * 7 / 8 && (Kp >= 512 || (Kp >= 320 && N == 320));   // N < 320 pays for its padding at K = 320
}

// The row-stationary kernels' grid: blocks = row stripes x column ranges, as few column ranges as the table allows,
// raised until there are two blocks per CU. The column ranges, and the 64-column chunks of each.
constexpr int STRIPE_BM = 128, STRIPE_CH = 64;
constexpr int STRIPE_NCOLS = 1280;   // W rows per block, at most
struct StripeRanges { int cs, kper; };
inline StripeRanges stripe_ranges(int M, int N) {
    const int nch = cdiv(N, STRIPE_CH);
    const int cs = std::max(cdiv(nch, STRIPE_NCOLS / STRIPE_CH), std::min(nch, cdiv(2 * NCU, cdiv(M, STRIPE_BM)))), kper = cdiv(nch, cs);
    return {cdiv(nch, kper), kper};
}

// Rows with shifts (no residual) on the sixteen-row row-stationary kernel in place of the tile kernels: from 1024 rows
// and 960 64x128 tiles on (below, at 768 tiles, 16384 x 320 x 320 12.3 against 13.4 us on it), where a block has the
// chunks that pay for its set-up and the grid's rounds of two blocks a CU are filled. The kernel runs five K steps
// whatever Kp is, so Kp < 128 stays on the tiles but for wide GELU (61568 x 64 x 72 GEGLU 13.3 -> 19.6 us on it,
// 24576 x 64 x 512 PLAIN 17.2 -> 20.3, 9932 x 96 x 2560 GELU 48.7 -> 37.5). The lines are those of 4800 calls, K 64 to
// 320 and N 64 to 5120, in the integer form, the one in double (shifts up to 12) and the general one: those sent here
// take 0.78 of the tile kernels' time, 0.6 % of them over 1.02 and at most 1.09 (us below; in brackets in double).
// From 960 columns, where the tile kernels take 128x128 tiles:
//   GEGLU, one round      three chunks a block   8320 x 320 x 1280 23.5 -> 18.1 (19.7), two: 2944 x 320 x 2568 16.1 -> 16.2 (17.1)
//   GEGLU, more rounds    four                   6592 x 320 x 2560 35.0 -> 28.7 (32.5), three: 4713 x 320 x 2560 24.7 -> 25.2 (27.8)
//   PLAIN, GELU           two                    7040 x 320 x 1280 PLAIN 24.3 -> 20.4, 3136 x 320 x 2560 17.3 -> 15.6
// Below 960 columns:
//   one round             always                 61568 x 320 x 64 15.9 -> 13.7, 12352 x 320 x 640 18.1 -> 15.2
//   more rounds           by the share of the rounds' chunk slots that is used: half from five chunks a block on (GELU
//                         from three; 60 % at Kp = 128: 34188 x 128 x 640 GEGLU 1.13 times in double at 52 %), 55 % at
//                         four, 70 % at three: 38400 x 320 x 640 GEGLU 44 -> 33.5, 64000 x 320 x 320 39.4 -> 32.3;
//                         less, or two chunks: 14080 x 320 x 640 19.8 -> 20.4 (22.4), 16640 x 320 x 640 21.9 -> 23.2
//                         (26.1), 61568 x 320 x 72 16.5 -> 20.6
enum ShiftEpi { SHIFT_PLAIN, SHIFT_GEGLU, SHIFT_GELU };
inline bool stripe_shift_rows(ShiftEpi epi, int M, int N, int Kp) {
    if (M < 1024 || (long long)cdiv(M, 64) * cdiv(N, 128) < 15LL * NCU / 4) return false;
    const int kper = stripe_ranges(M, N).kper;
    const long long mt = cdiv(M, STRIPE_BM), rounds = cdiv(mt * stripe_ranges(M, N).cs, 2 * NCU);
    const bool gelu = epi == SHIFT_GELU;
    if (Kp < 128) return gelu && N >= 960 && kper >= 3;
    if (N >= 960) return kper >= (epi != SHIFT_GEGLU ? 2 : rounds == 1 ? 3 : 4);
    if (rounds == 1) return true;
    const double used = double(mt * cdiv(N, STRIPE_CH)) / double(rounds * 2 * NCU * kper);
    if (kper >= (gelu ? 3 : 5)) return used >= (gelu || Kp > 128 ? 0.5 : 0.6);
    return (kper == 4 && used >= 0.55) || (kper == 3 && used >= 0.7);
}

// Tiles of RT rows a block of the norms' row kernels takes (its four waves one each at a time), at most row_cap rows
// and 32: the number whose blocks end soonest when every CU takes a whole number of them, a block costing its rounds of
// four tiles and a set-up of `setup` rounds; a CU with one block (up to three) is `one` (`few`) times slower for the
// latency that nothing hides, and fewer tiles than fit have to save 5 %. 16320 rows of 1920: 510 blocks of 32 tiles, two
// a CU, GroupNorm + SiLU 77.7 us and LayerNorm to planes 70.8; 1360 of 12, five and a third a CU, 91.8 and 76.6. 2048
// rows of 640 as 64 blocks of 16 tiles: LayerNorm 18.2; as 256 blocks of four 8.0. The costs are fitted to every choice
// of 230 shapes, 700 to 40000 rows of 256 to 2560: the chosen tiles are within 1.5 % of the best on average.
struct NormCost { double setup, one, few; };
constexpr NormCost LNORM_COST = {0.05, 1.4, 1.1}, GN_APPLY_COST = {0.4, 1.6, 1.1};
inline int norm_tiles_per_block(long long M, int RT, long long row_cap, NormCost k) {
    const int most = int(std::max(1LL, std::min(32LL, row_cap) / RT));
    const long long tiles = (M + RT - 1) / RT;
    int best = most;
    double least = 0;
    for (int t = most; t >= 1; t = (t - 1) / 4 * 4) {
        const long long blocks = (tiles + t - 1) / t, per_cu = (blocks + NCU - 1) / NCU;
        const double cost = double(per_cu) * ((t + 3) / 4 + k.setup) * (per_cu == 1 ? k.one : per_cu <= 3 ? k.few : 1.0) * (t == most ? 0.95 : 1.0);
        if (t == most || cost < least) { best = t; least = cost; }
    }
    return best;
}

// The attention's form for Tkp padded keys: the waves that split a row's keys and the 64-key tiles of scores that each
// holds, or (multi) one wave that recomputes the scores in each pass. Up to 256 keys a wave holds all of its queries'
// scores, with a form of one tile for up to 64 keys (with two, 10 groups of 1024 x 20 in the general arithmetic 13.4 us
// in place of 11.3, 160 groups of 1024 x 64 in the integer one 39.6 in place of 28.7), up to 1024 two or four waves split
// the keys (80 groups of 1024 x 1024: 119 us, against 187 when every pass recomputes the scores); beyond, the recomputing
// form, as eight or sixteen waves to a row's scores leave 128 registers each, where they spill (4096 x 4096, 40 groups:
// 2350 us so, 1420 recomputed; 2795 in the form that recomputed them in double for every wave).
struct AttnForm { int tiles, waves; bool multi; };
inline AttnForm attn_form(int Tkp) {
    if (Tkp > 1024) return {1, 1, true};
    const int waves = Tkp <= 256 ? 1 : Tkp <= 512 ? 2 : 4;
    return {Tkp <= 64 ? 1 : Tkp <= 128 ? 2 : 4, waves, false};
}

}  // namespace vk
