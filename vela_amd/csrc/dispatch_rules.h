// Rules of the automatic kernel choice that depend on sizes alone: plain host C++, no HIP, so that they can be
// compiled and checked without a GPU.
#pragma once

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

}  // namespace vk
