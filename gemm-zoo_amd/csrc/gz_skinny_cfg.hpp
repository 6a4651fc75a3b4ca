// Host-side geometry of the weight-streaming (skinny M) rung, shared by the
// launcher and gz_plan.
#pragma once

#include "../../include/gemm_zoo.h"
#include "gz_mfma_cfg.hpp"

namespace gz {

constexpr int SKINNY_MAX_M = 128;      // most rows of activations the streaming kernels take
constexpr int SKINNY_REG_MAX_M = 16;   // activations in registers; above they are shared through LDS (stream_tile_kernel)
constexpr int SKINNY_K_STEP = 64;      // an explicitly named rung takes whole multiples of this K (of 16-bit elements)
// direct-to-LDS kernel: 256-byte K chunks of 4 NCP columns per stage.  A compute unit streams at its full rate with
// about 128 KiB in flight, and a narrow share of columns has few bytes per stage: more waves and more stages there.
constexpr int SKINNY_DTL_CHUNK_BYTES = 256;
struct SkinnyDtlShape { int waves, stages; };
constexpr SkinnyDtlShape skinny_dtl_shape(int ncp) {
  return ncp == 8 ? SkinnyDtlShape{4, 2} : ncp == 4 ? SkinnyDtlShape{8, 4} : SkinnyDtlShape{8, 6};
}
inline int skinny_dtl_copies(int cols) { return cols <= 4 ? 1 : cols <= 8 ? 2 : cols <= 16 ? 4 : 8; }
// (fragments are read for whole blocks of 16 columns: the ring of the last wave is followed by what a block is longer
// than its stage)
inline int skinny_dtl_lds_bytes(int ncp) {
  return skinny_dtl_shape(ncp).waves * skinny_dtl_shape(ncp).stages * ncp * 1024 + (ncp < 4 ? (4 - ncp) * 1024 : 0);
}
// producer / consumer tile kernel: 128 bytes of K per row and stage, at most 64 columns per work-group,
// four consumer and four producer waves, ring depth by number of 32-row blocks of A
constexpr int STREAM_TILE_ROW_BYTES = 128;
constexpr int STREAM_TILE_COLS = 64;
constexpr int STREAM_TILE_THREADS = 512;
constexpr int STREAM_TILE_STAGES_1 = 8, STREAM_TILE_STAGES_2 = 4, STREAM_TILE_STAGES_4 = 4;

// the same with wide column blocks and a split K (65 ... 128 rows, long K): 64 CB columns per work-group, CB = 2 ... 4,
// ring depth by CB; a work-group's partial sums are 4 waves x 2 row blocks x CB column blocks x 4 KiB
constexpr int STREAM_WIDE_K_STEP = 64;   // elements (16-bit) per stage
constexpr int STREAM_WIDE_MIN_K = 8192;
constexpr int STREAM_WIDE_MAX_CB = 4;
constexpr int STREAM_WIDE_STAGES_2 = 4, STREAM_WIDE_STAGES_3 = 3, STREAM_WIDE_STAGES_4 = 3;
inline int stream_wide_stages(int cb) { return cb == 2 ? STREAM_WIDE_STAGES_2 : cb == 3 ? STREAM_WIDE_STAGES_3 : STREAM_WIDE_STAGES_4; }
inline long long stream_wide_slot_bytes(int cb) { return 4LL * 2 * cb * 4 * 1024; }

enum { SKINNY_KIND_DTL = 1, SKINNY_KIND_TILE = 2, SKINNY_KIND_TILE_WIDE = 3 };

struct SkinnyCfg {
  int mb;             // rows of A the kernel instance covers: 16, 32, 64 or 128
  int cols_per_wave;  // columns that one wave works on
  int waves;          // wavefronts per work-group
  int cols_per_wg;
  int threads;
  int grid_n;         // work-groups along N
  int split_k;        // K slices (partial sums reduced by a second kernel when > 1)
  int k_per_split;
  int kind;           // SKINNY_KIND_*
  int lds_bytes;
  int cb;             // SKINNY_KIND_TILE_WIDE: 64-column blocks per work-group
  long long workspace_bytes;   // partial sums of a split K (0: none)
};

// Element types of the kernels, and those for which the rung can be named by the caller (the 8-bit ones come here through
// the launcher's own choice only).
constexpr bool skinny_rung_types(int types) { return types == GZ_BF16BF16F32 || types == GZ_BF16BF16BF16 || types == GZ_F16F16F16; }
constexpr bool skinny_stream_types(int types) {
  return skinny_rung_types(types) || types == GZ_S8S8S32 || types == GZ_E4M3E4M3F16 || types == GZ_E5M2E5M2F16;
}

// What the kernels can run: activations row-major (K contiguous), weights column-major (K contiguous), K in whole
// 16-byte pieces.
inline bool skinny_stream_supported(int types, int M, int N, int K, int layoutA, int layoutB) {
  if (!skinny_stream_types(types)) return false;
  if (layoutA != GZ_ROW_MAJOR || layoutB != GZ_COL_MAJOR) return false;
  const int es = skinny_rung_types(types) ? 2 : 1;
  if (M < 1 || M > SKINNY_MAX_M || N < 1 || K < 1) return false;
  if ((long long)K * es * SKINNY_MAX_M >= (1LL << 32)) return false;  // rows are addressed with 32-bit byte offsets
  return (long long)K * es % 16 == 0;
}
// What a caller that names the rung may ask for: 16-bit float inputs and whole 64-element super-steps of K.
inline bool skinny_supported(int types, int M, int N, int K, int layoutA, int layoutB) {
  return skinny_rung_types(types) && K >= SKINNY_K_STEP && K % SKINNY_K_STEP == 0 &&
         skinny_stream_supported(types, M, N, K, layoutA, layoutB);
}

// The streaming kernels copy 16-byte pieces of the rows of A and the columns of B and address them with 32-bit byte
// offsets from the first row (column of the work-group): leading dimensions of whole pieces, below 2^32 / (es * 128).
inline bool skinny_lines_ok(int es, long long lda, long long ldb) {
  return lda * es % 16 == 0 && ldb * es % 16 == 0 && lda * es * SKINNY_MAX_M < (1LL << 32) && ldb * es * SKINNY_MAX_M < (1LL << 32);
}

// What the launcher's own choice sends here: always the register-resident cases; the LDS-shared tile kernel only
// while the tiled MFMA rung could not give every compute unit a 128 x 128 tile of its own.
inline bool skinny_preferred(int types, int M, int N, int K, int layoutA, int layoutB, int num_cus) {
  if (!skinny_stream_supported(types, M, N, K, layoutA, layoutB)) return false;
  if (num_cus <= 0) num_cus = 256;
  return M <= 32 || (long long)((N + 127) / 128) <= num_cus;
}

// More columns than one work-group of the tile kernel per compute unit holds (64 each).  A second round of work-groups
// pays its fill and its stores again with nothing beside them, where the MFMA rung's tiles run several to a compute unit,
// and from 65 rows on each work-group takes in all of A as well.  Against that the streaming kernels read memory faster
// than the tiles do.  Whether the tiles win on the whole (geometric mean of both states of the cache); us, streaming / MFMA
// rung, operands just used; after 512 MiB of other data - they do: int8 16 x 28672 x 1024 8.7 / 7.0; 10.6 / 10.9,
// 32 x 16640 x 1024 8.6 / 6.7; 9.4 / 9.8, 128 x 20480 x 4096 31.7 / 20.8; 32.4 / 34.3; they do not: 16 x 32768 x 4096
// 21.4 / 21.3; 23.8 / 41.1, 32 x 20480 x 4096 17.6 / 16.6; 19.1 / 27.9, 64 x 28672 x 3072 21.8 / 16.6; 23.4 / 27.2,
// 65 x 24576 x 14336 83.1 / 83.5; 83.4 / 98.1.
inline bool skinny_wide_to_mfma(int types, int M, int N, int K, int num_cus) {
  if (num_cus <= 0) num_cus = 256;
  const double rounds = (double)N / (64.0 * num_cus);
  if (rounds <= 1.0) return false;
  const long long kb = (long long)K * (skinny_rung_types(types) ? 2 : 1);
  if (M <= 32) return kb <= 2048 && kb <= (M <= SKINNY_REG_MAX_M ? 640 : 1024) * rounds;
  // (a few columns past one round and a short K: 64 x 64 tiles, skinny_choose; e4m3 128 x 24576 x 512 streaming / MFMA rung /
  // 64 x 64 10.6 / 7.3 / 6.5; 11.8 / 10.0 / 9.6)
  return M > 64 && kb <= 8192 && (kb > 3072 || rounds > (kb <= 512 ? 1.5 : 1.125));
}

// equal column groups, one or more per compute unit, at most max_cols columns and a multiple of 4 each
inline int skinny_balanced_cols(int N, int num_cus, int max_cols) {
  if (num_cus <= 0) num_cus = 256;
  for (int w = 1; w <= 1024; w++) {
    const long long slots = (long long)num_cus * w;
    int per = (int)((N + slots - 1) / slots);
    per = (per + 3) / 4 * 4;
    if (per <= max_cols) return per;
  }
  return max_cols;
}

// Wide column blocks with a split K.  With 64 columns per work-group every compute unit pulls ALL of A from its L2
// beside its share of B, and at 65 ... 128 rows that, not HBM, sets the time (M = 128, N = 14336, K = 8192: 2 MiB of A
// and 0.9 MiB of B per compute unit, 60 us where the B stream alone is 42 at the 5.6 TB/s this part streams).  What a
// work-group takes in of A is rows x its K range, whatever its columns: splitting K in KS parts AND widening the column
// blocks KS-fold keeps one work-group per compute unit and divides the A traffic by KS.  The partial sums go to a workspace
// in the order the waves hold them (whole 1 KiB stores) and a second launch adds them in the order of the K parts - a fixed
// order, no waiting - and applies alpha, beta and the rounding.  Taken for 64 < M <= 128 from K = 8192 on where the column
// blocks come out at 65 ... 256 columns and the workspace fits.  The first launch then runs at the rate of the B stream (M
// = 128, N = 14336: 43 us at K = 8192, 75 at 14336); the second costs 8 us: 60.1 -> 53.9 us and 108.5 -> 83.1.
inline bool skinny_resolve_wide(int types, int M, int N, int K, int num_cus, unsigned long long ws_limit, int* split, int* cols) {
  if (num_cus <= 0) num_cus = 256;
  if (!skinny_rung_types(types) || M <= 64 || M > SKINNY_MAX_M || K < STREAM_WIDE_MIN_K || K % STREAM_WIDE_K_STEP) return false;
  // four parts where the column blocks allow it, else two (M = 128, N = 14336, us, two / four parts: K = 8192
  // 56.0 / 56.3, K = 14336 93.9 / 84.5, before the second launch wrote whole rows; at K = 4096 the split loses to the
  // one-launch kernel, 34.2 against 31.6)
  for (int ks = 4; ks >= 2; ks >>= 1) {
    if (num_cus % ks || (K / STREAM_WIDE_K_STEP) < 8 * ks) continue;
    const int groups = num_cus / ks;
    int per = (N + groups - 1) / groups;
    per = (per + 3) / 4 * 4;
    if (per <= STREAM_TILE_COLS || per > STREAM_TILE_COLS * STREAM_WIDE_MAX_CB) continue;
    const int cb = (per + STREAM_TILE_COLS - 1) / STREAM_TILE_COLS;
    const long long grid_n = (N + per - 1) / per;
    if ((unsigned long long)(grid_n * ks * stream_wide_slot_bytes(cb)) > ws_limit) continue;
    *split = ks;
    *cols = per;
    return true;
  }
  return false;
}

inline SkinnyCfg skinny_resolve(int types, int M, int N, int K, int num_cus, unsigned long long ws_limit = ~0ULL) {
  SkinnyCfg c;
  c.split_k = 1;
  c.k_per_split = K;
  c.cb = 1;
  c.workspace_bytes = 0;
  int wide_split = 1, wide_cols = 0;
  if (skinny_resolve_wide(types, M, N, K, num_cus, ws_limit, &wide_split, &wide_cols)) {
    c.kind = SKINNY_KIND_TILE_WIDE;
    c.mb = 128;
    c.cols_per_wg = wide_cols;
    c.cb = (wide_cols + STREAM_TILE_COLS - 1) / STREAM_TILE_COLS;
    c.cols_per_wave = 32 * c.cb;
    c.waves = STREAM_TILE_THREADS / 64;
    c.split_k = wide_split;
    c.k_per_split = K / wide_split;   // (whole 64-element stages are dealt as evenly as they divide)
    c.lds_bytes = stream_wide_stages(c.cb) * (128 + STREAM_TILE_COLS * c.cb) * STREAM_TILE_ROW_BYTES;
    c.threads = c.waves * 64;
    c.grid_n = (N + c.cols_per_wg - 1) / c.cols_per_wg;
    c.workspace_bytes = (long long)c.grid_n * c.split_k * stream_wide_slot_bytes(c.cb);
    return c;
  }
  if (M > SKINNY_REG_MAX_M) {
    c.kind = SKINNY_KIND_TILE;
    c.mb = M <= 32 ? 32 : M <= 64 ? 64 : 128;
    const int stages = c.mb == 32 ? STREAM_TILE_STAGES_1 : c.mb == 64 ? STREAM_TILE_STAGES_2 : STREAM_TILE_STAGES_4;
    c.cols_per_wg = skinny_balanced_cols(N, num_cus, STREAM_TILE_COLS);
    c.cols_per_wave = 32;
    c.waves = STREAM_TILE_THREADS / 64;
    c.lds_bytes = stages * (c.mb + STREAM_TILE_COLS) * STREAM_TILE_ROW_BYTES;
  } else {
    c.kind = SKINNY_KIND_DTL;
    c.mb = 16;
    c.cols_per_wg = skinny_balanced_cols(N, num_cus, 32);
    c.cols_per_wave = c.cols_per_wg;  // every wave of the work-group works on all of its columns (K is split)
    const int ncp = skinny_dtl_copies(c.cols_per_wg);
    c.waves = skinny_dtl_shape(ncp).waves;
    c.lds_bytes = skinny_dtl_lds_bytes(ncp);
  }
  c.threads = c.waves * 64;
  c.grid_n = (N + c.cols_per_wg - 1) / c.cols_per_wg;
  return c;
}

// The launcher's choice between the tile kernel above and the MFMA rung's 64 x 64 tiles for 17 ... 128 rows.  Every
// work-group of the tile kernel walks all of K and takes in all of A beside its share of the columns: with few columns
// per work-group and a long K it takes in mostly A, and the 64 x 64 tiles with a split K are faster; with many rows and a
// short K its fill and its one pass of stores are not paid back, and the same tiles unsplit are (below).  Measured, us, tile
// kernel / split K: bf16 20 x 2560 x 8192 18.2 / 14.6, 50 x 1024 x 8192 27.1 / 12.5, 100 x 2560 x 4096 20.3 / 14.0,
// 128 x 5120 x 4096 23.6 / 20.9, 20 x 5120 x 8192 19.6 / 22.3, 100 x 9600 x 4096 26.1 / 36; e4m3 50 x 2560 x 8192
// 16.3 / 12.3, 100 x 9600 x 8192 25.4 / 32.9.
inline double skinny_tile_estimate_us(int stages, int mb, int cols) {
  if (mb == 32) return 3.4 + stages * (cols < 26 ? 0.118 : 0.0046 * cols);   // (many columns: the rate of the B stream)
  if (mb == 64) return 3.2 + 0.015 * cols + stages * (0.185 + 0.0019 * cols);
  return 4.2 + 0.075 * cols + stages * (0.225 + 0.0026 * cols);
}
// 65 rows and more: up to how many 128-byte stages of K the unsplit 64 x 64 tiles are taken.  They win while the operands
// come from the cache and lose from memory, where the tile kernel's producers keep more in flight, so the line lies where
// the one outweighs the other (geometric mean), about alike for 8-bit and 16-bit elements.  us, tile kernel / 64 x 64
// tiles, operands just used; after 512 MiB of other data:
// up to 32 columns per work-group, 8 stages bf16 96 x 2560 6.1 / 4.9; 6.3 / 7.2, int8 128 x 2560 6.4 / 5.5; 7.0 / 7.5, 16 stages
// int8 128 x 2560 8.5 / 7.5; 9.1 / 11.4, bf16 128 x 5120 8.5 / 6.8; 9.5 / 11.9, 65 x 7168 8.5 / 6.9; 8.8 / 11.8;
// more, 4 stages bf16 128 x 9600 5.8 / 5.0; 6.5 / 6.6, e4m3 65 x 14336 5.6 / 5.6; 6.2 / 7.5, 8 stages int8 65 x 9600 6.9 / 7.3; 7.3 / 9.3,
// bf16 128 x 16384 7.5 / 6.5; 8.3 / 10.0, 16 stages int8 128 x 14336 11.2 / 10.8; 12.4 / 15.2, 24 stages bf16 128 x 16384
// 15.5 / 13.6; 17.2 / 21.0.
// Past one round of work-groups (skinny_wide_to_mfma) the tiles win up to a longer K, 64 x 64 ones while there are up to
// three to a compute unit: bf16 128 x 24576 x 1024 20.6 / 13.6; 21.6 / 20.9, 96 x 20480 x 1536 23.8 / 17.3; 25.0 / 26.4; beyond,
// those that the MFMA rung chooses: bf16 128 x 32768 x 1024, tile kernel / 64 x 64 / chosen 20.9 / 17.5 / 15.4; 21.9 / 28.6 / 22.2.
inline int skinny_tiles_max_stages(int cols, bool one_round) {
  if (!one_round) return 16 + cols / 4;
  return cols <= 32 ? 8 : 4;
}
enum { SKINNY_STREAM = 0, SKINNY_TILES_SPLITK = 1, SKINNY_TILES_64 = 2, SKINNY_TILES = 3, SKINNY_TILES_32 = 4 };   // (TILES: the MFMA rung's own choice)
inline int skinny_choose(int types, int M, int N, int K, int num_cus, unsigned long long ws_limit, SplitKPlan* split) {
  if (M <= SKINNY_REG_MAX_M) return SKINNY_STREAM;
  const SkinnyCfg c = skinny_resolve(types, M, N, K, num_cus, ws_limit);
  if (c.kind != SKINNY_KIND_TILE) return SKINNY_STREAM;
  const int es = skinny_rung_types(types) ? 2 : 1;
  const int stages = (int)(((long long)K * es + STREAM_TILE_ROW_BYTES - 1) / STREAM_TILE_ROW_BYTES);
  if (num_cus <= 0) num_cus = 256;
  // 32 x 32 tiles whose waves share out K, one launch.  Up to one tile per compute unit, and up to 1.75, or 32 rows, while K is
  // not so long that the tile kernel's spreading of the weights over all compute units, or a split K, outweighs its share of A
  // from memory (us, 32 x 32 / tile kernel / split K, operands just used; from memory: bf16 78 x 1024 x 2048 4.7 / 12.3 / 8.5;
  // 5.7 / 13.4 / 8.9, 100 x 2100 x 1136 6.3 / 9.0 / 9.7; 7.0 / 10.0 / 10.2, 36 x 7296 x 7168 24.8 / 29.3 / 21.5; 30.6 / 29.5 /
  // 26.2, int8 46 x 5632 x 10944 18.9 / 27.8 / 18.2; 29.1 / 28.6 / 24.3, e4m3 32 x 4096 x 11648 14.2 / 17.2 / -).
  const long long tiles32 = (long long)((M + 31) / 32) * ((N + 31) / 32);
  const double small_us = mfma_32_us(types, M, N, K, GZ_ROW_MAJOR, GZ_COL_MAJOR, num_cus);
  const double stream_us = skinny_tile_estimate_us(stages, c.mb, c.cols_per_wg);
  // (the rows of a short K below: 64 x 64 tiles that leave compute units idle are the slower ones - int8 65 x 1024 x 512
  // 3.4 / 2.8, bf16 70 x 2762 x 192 4.5 / 3.3)
  if (M > 64 && stages <= skinny_tiles_max_stages(c.cols_per_wg, c.grid_n <= num_cus)) {
    if (4 * tiles32 <= 3LL * num_cus && small_us < mfma_64_us(types, M, N, K, GZ_ROW_MAJOR, GZ_COL_MAJOR, num_cus)) return SKINNY_TILES_32;
    return 2LL * ((N + 63) / 64) <= 3LL * num_cus ? SKINNY_TILES_64 : SKINNY_TILES;
  }
  // (65 rows and more, rows of D that are not whole 16-byte pieces and a last stage that the end of K cuts: the tile kernel
  // up to 24 stages.  The figures are against it (bf16 70 x 1029 x 1136 8.3 / 4.5 on 32 x 32 tiles, 128 x 2100 x 1176 10.2
  // / 6.4): a test alone holds it, which takes this kernel's cut stages for such problems.)
  if (M > 64 && stages < 24 && N % 8 != 0 && (long long)K * es % STREAM_TILE_ROW_BYTES != 0) return SKINNY_STREAM;
  const bool split_ok = mfma_best_splitk(types, M, N, K, GZ_ROW_MAJOR, GZ_COL_MAJOR, num_cus, split) &&
                        (unsigned long long)split->workspace_bytes <= ws_limit;
  const bool small = ((M > 32 && tiles32 <= num_cus) || (4 * tiles32 <= 7LL * num_cus && stages <= 48)) && small_us < stream_us;
  if (small && (!split_ok || mfma_32_not_in_parts_us(types, M, N, K, GZ_ROW_MAJOR, GZ_COL_MAJOR, num_cus) < split->estimate_us))
    return SKINNY_TILES_32;
  // (0.9: bf16 30 x 1280 x 4224 tile kernel / split K 10.9 / 8.4, 36 x 7296 x 7168 above; e5m2 97 x 3456 x 3328 10.0 / 11.1)
  if (split_ok && split->estimate_us < 0.9 * stream_us) return SKINNY_TILES_SPLITK;
  return small ? SKINNY_TILES_32 : SKINNY_STREAM;
}

}  // namespace gz
