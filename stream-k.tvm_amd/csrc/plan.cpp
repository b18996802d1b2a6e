// Host-side Stream-K partitioner and kernel selection (pure integer code, no device access).
//
// The arithmetic restates streamk_fp32.py:30-54 of the reference for run-time shapes, with two
// changes: the persistent grid is a parameter instead of `total_sm = 108`, and the number of
// data-parallel waves is ceil(blocking_tiles / grid) with 0 allowed (the reference's
// max(blocking_tiles // total_sm, 1) walks out of range when there are no data-parallel tiles).
#include <math.h>
#include <string.h>

#include <mutex>

#include "kernel_table.h"
#include "streamk.h"

namespace sk {

constexpr int TABLE_MAX = 512;
static KernelInfo g_table[TABLE_MAX];
static int g_count = 0;
static std::once_flag g_table_once;

int tile_kernel_infos(KernelInfo *out, int max);
int tile_asm_kernel_infos(KernelInfo *out, int max);
int tile_asm8_kernel_infos(KernelInfo *out, int max);
int tile_q4_kernel_infos(KernelInfo *out, int max);
int tile_8bit_kernel_infos(KernelInfo *out, int max);
int skinny_kernel_infos(KernelInfo *out, int max);
int rows_q4_kernel_infos(KernelInfo *out, int max);
int stream_bytes_kernel_infos(KernelInfo *out, int max);
int tile_ring_kernel_infos(KernelInfo *out, int max);
int tile_wavek_kernel_infos(KernelInfo *out, int max);
int f32_kernel_infos(KernelInfo *out, int max);

const KernelInfo *kernel_table(int *count) {
  std::call_once(g_table_once, [] {
    int n = tile_kernel_infos(g_table, TABLE_MAX);
    n += tile_8bit_kernel_infos(g_table + n, TABLE_MAX - n);
    n += tile_asm_kernel_infos(g_table + n, TABLE_MAX - n);
    n += tile_asm8_kernel_infos(g_table + n, TABLE_MAX - n);
    n += tile_q4_kernel_infos(g_table + n, TABLE_MAX - n);
    n += skinny_kernel_infos(g_table + n, TABLE_MAX - n);
    n += rows_q4_kernel_infos(g_table + n, TABLE_MAX - n);
    n += stream_bytes_kernel_infos(g_table + n, TABLE_MAX - n);
    n += tile_ring_kernel_infos(g_table + n, TABLE_MAX - n);
    n += tile_wavek_kernel_infos(g_table + n, TABLE_MAX - n);
    n += f32_kernel_infos(g_table + n, TABLE_MAX - n);
    g_count = n;
  });
  if (count) *count = g_count;
  return g_table;
}

const KernelInfo *kernel_by_id(int id) {
  int n;
  const KernelInfo *t = kernel_table(&n);
  for (int i = 0; i < n; ++i)
    if (t[i].id == id) return &t[i];
  return nullptr;
}

// sk_config.reserved[0] of the operators' calls that name nothing: the fastest kernel there is, see sk_make_plan
constexpr int SK_VARIANT_OPERATOR = 12;

static int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// preference among kernel variants of one tile shape when the caller does not ask for one: the
// eight-wave direct-to-LDS tile kernels; the most specialised small-M kernel that accepts the shape
static int variant_rank(const KernelInfo &k) {
  // (small-M: general 0 < rows-of-A matrix-vector form 3 < single-row 1 < matrix-vector 2; the kernels that stream
  // the weights through LDS, variant 4, share tile shapes with general kernels and are taken when asked for by
  // variant, or by the default rule below)
  if (k.family == FAMILY_SKINNY)
    return k.variant == 4 ? -1 : (k.variant == 3 ? 1 : (k.variant == 0 ? 0 : k.variant + 1));
  return k.variant == 7 ? 4 : (k.variant == 4 ? 3 : (k.variant == 1 ? 2 : (k.variant == 2 ? 1 : 0)));
}
// kernels that a tile alone does not name: the Q4 ones whose waves stream K on their own, and the ones that stream one-byte
// weights through LDS, and the tile kernels for 65 to 128 rows
static bool by_variant_only(const KernelInfo &k) {
  return k.variant >= 9 || (k.family == FAMILY_SKINNY && (k.variant == 5 || k.variant == 8));
}
static bool accepts_shape(const KernelInfo &k, int64_t M, int64_t K) {
  // (the assembly-loop tile kernels have no K tail: other K go to the next-best variant of the tile)
  return (k.max_m == 0 || M <= k.max_m) && (k.max_ipt == 0 || (K + k.bk - 1) / k.bk <= k.max_ipt) &&
         (k.family != FAMILY_TILE || k.variant != 7 || K % k.k_align == 0);
}

// whether the kernel can run the grid or the fixed split that a configuration names
static bool takes_partition(const KernelInfo &k, int64_t M, int64_t N, int64_t K, const sk_config *cfg, int num_cus) {
  if (!cfg) return true;
  const int64_t most = (int64_t)num_cus * k.ctas_per_cu;
  if (cfg->grid > most) return false;
  if (cfg->schedule != SK_SCHED_SPLIT_K) return true;
  const int64_t split = cfg->reserved[1] > 0 ? cfg->reserved[1] : 1;
  return cdiv(K, k.bk) % split == 0 && cdiv(M, k.bm) * cdiv(N, k.bn) * split <= most;
}

// 65 to 96 rows of fp16 / bfloat16 (NT) whose 96 x 32 tiles fill the device in one round: see pick_kernel
static bool rows_65_to_96_stream(int64_t M, int64_t N, int dtype, int layout, int num_cus) {
  return (dtype == SK_F16 || dtype == SK_BF16) && layout == SK_LAYOUT_NT && M > 64 && M <= 96 && cdiv(N, 32) <= num_cus &&
         cdiv(N, 32) * 5 >= (int64_t)num_cus * 3;
}

static const KernelInfo *pick_kernel(int64_t M, int64_t N, int64_t K, int dtype, int layout,
                                     const sk_config *cfg, int num_cus) {
  int n;
  const KernelInfo *t = kernel_table(&n);
  const bool want_tile = cfg && cfg->bm > 0 && cfg->bn > 0;
  // cfg->reserved[0]: 0 = newest variant of the tile, v > 0 = variant v - 1
  const int want_variant = cfg ? cfg->reserved[0] - 1 : -1;
  if (want_tile) {
    const KernelInfo *found = nullptr;
    // (fp32 tiles that exist with two lengths of the K-iteration: the first that takes the caller's grid or split)
    for (int pass = dtype == SK_F32 ? 0 : 1; pass < 2 && !found; ++pass)
      for (int i = 0; i < n; ++i)
        if (t[i].dtype == dtype && t[i].layout == layout && t[i].bm == cfg->bm && t[i].bn == cfg->bn &&
            (cfg->bk <= 0 || t[i].bk == cfg->bk) &&
            (want_variant < 0 ? !by_variant_only(t[i]) : t[i].variant == want_variant) &&
            (pass > 0 || takes_partition(t[i], M, N, K, cfg, num_cus)) &&
            accepts_shape(t[i], M, K) && (found == nullptr || variant_rank(t[i]) > variant_rank(*found)))
          found = &t[i];
    return found;
  }
  // heuristic: small M -> weight-streaming kernels; otherwise the largest tile that still gives
  // every CU something to do
  const KernelInfo *best = nullptr;
  // (for 32 < M <= 64 the 64x64 LDS tile below is faster than streaming the weights past 64 rows)
  const bool q4 = dtype == SK_Q4 || dtype == SK_Q4_TILED || dtype == SK_Q4_ZP || dtype == SK_Q4_ZP_TILED;
  // (one-byte operands: up to 64 rows -- their tile kernels start at 128 rows)
  const bool one_byte = dtype == SK_F8E4M3 || dtype == SK_F8E5M2 || dtype == SK_I8;
  if (dtype == SK_Q4 && M > 64 && want_variant < 0) {
    // more rows than the weight-streaming kernels take: the tile kernels that dequantise B on its way into LDS.
    // 256 rows of A per tile as soon as M has them: a CTA decodes its BN weight rows whatever BM is, and the
    // four-wave 128 x 128 kernel waits for its loads (one wave per SIMD, a short iteration), so a 256 x 128 tile
    // takes no longer than a 128 x 128 one; where that leaves CUs without a tile the Stream-K schedule splits K
    // (N = K = 8192, M = 512: 73 us against 109 us on 128 x 128 tiles).  There is no 256 x 256 instance: eight waves
    // that decode and hold 128 x 64 accumulators each do not fit the register file (it spilled); large M is better
    // served by dequantising once and running the fp16 kernels, which is what streamk_q4 does from 1024 rows on.
    const int want_bm = M > 128 ? 256 : 128;
    const int want_bn = 128;
    for (int i = 0; i < n; ++i)
      if (t[i].family == FAMILY_TILE && t[i].dtype == SK_Q4 && t[i].bm == want_bm && t[i].bn == want_bn) return &t[i];
    return nullptr;
  }
  // (2 <= M <= 4 as well: the matrix-vector form with four rows of A (variant 3) is behind at every size measured,
  // weights from HBM -- 2 x 4096 x 4096 11.3 us against 8.7 us on 16 x 16 tiles, 4 x 11008 x 4096 23.0 / 17.5,
  // 4 x 4096 x 11008 26.9 / 17.4, 4 x 8192 x 8192 32.0 / 24.8 -- and stays as an explicit choice)
  // (one row: from 40 MB on -- 1 x 8192 x 8192 24.4 us against 28.9 us for the matrix-vector kernel, 1 x 14336 x 4096
  // 22.3 / 27.3, 1 x 4096 x 11008 17.3 / 19.9, 1 x 5120 x 5120 11.7 / 13.8, 1 x 11008 x 4096 17.5 / 17.2; 1 x 4096 x 4096
  // 8.6 / 8.1 stays with the matrix-vector kernel)
  const bool stream_rows = M >= 2 || N * K >= (int64_t)20 << 20;
  if ((dtype == SK_F16 || dtype == SK_BF16) && layout == SK_LAYOUT_NT && stream_rows && M <= 64 && want_variant < 0) {
    // 5 <= M <= 64 (fewer rows on large weights, above) with fp16 / bfloat16 weights: the kernels that stream the weights through LDS in contiguous loads
    // (tile_stream_pairs.h).  Tiles of 32 weight rows while one wave of them fits the device (N = 8192: one tile per
    // CU and no fix-up), 64 rows beyond; 64 rows of A exist with 32 weight rows only.
    // (more than 32 rows: 64 weight rows where they give three fifths of the CUs a tile -- A is then as many bytes
    // per CTA as the weights instead of twice as many; 64 x 16384 x 8192: 49 us against 56 us)
    const bool narrow = M > 32 ? cdiv(N, 64) * 5 < (int64_t)num_cus * 3 : cdiv(N, 32) <= num_cus;
    int bm = M <= 16 ? 16 : (M <= 32 ? 32 : 64), bn = narrow ? 32 : 64, bk = (bm == 16 && narrow) ? 512 : 256;
    // (up to 16 rows and no more than a tile of 16 weight rows per CU: K split over all four waves -- N = 4096 then
    // has a tile per CU; 16 x 4096 x 11008: 18.6 us against 21.4 us on 32-row tiles with a fix-up)
    if (bm == 16 && cdiv(N, 16) <= num_cus) bn = 16, bk = 1024;
    for (int i = 0; i < n; ++i)
      if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].variant == 4 && t[i].bm == bm && t[i].bn == bn &&
          t[i].bk == bk && accepts_shape(t[i], M, K))
        return &t[i];
  }
  // up to 64 rows of fp8 / int8: the same kernels on bytes, for a caller who names their variant alone (the operators
  // do, where no tuned configuration exists).  Up to 32 rows the narrowest tile of which every CU gets at
  // most one, beyond like the 16-bit ones (weights from HBM, e4m3, in us, tile_skinny.h's kernels / these:
  // 16 x 4096 x 4096 9.8 / 6.5, 16 x 8192 x 8192 22.5 / 14.3, 16 x 11008 x 4096 16.6 / 11.8 on 64-row tiles and 14.7 on
  // 32, 32 x 5120 x 5120 14.8 / 10.5 on 32 x 32 tiles and 12.8 on 32 x 64, 64 x 28672 x 8192 67.5 / 56.5,
  // 64 x 4096 x 4096 14.5 / 9.7 on 64 x 32 tiles and 13.0 on 64 x 64)
  if (one_byte && want_variant == 8) {
    if (M > 64) return nullptr;
    int bm = 64, bn = cdiv(N, 64) * 5 < (int64_t)num_cus * 3 ? 32 : 64, bk = 512;
    if (M <= 32) {
      bm = M <= 16 ? 16 : 32;
      bn = bm == 16 && cdiv(N, 16) <= num_cus ? 16 : (cdiv(N, 32) <= num_cus ? 32 : 64);
      bk = bn == 16 ? 2048 : (bn == 32 ? 1024 : 512);
    }
    for (int i = 0; i < n; ++i)
      if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].variant == 8 && t[i].bm == bm && t[i].bn == bn &&
          t[i].bk == bk)
        return &t[i];
    return nullptr;
  }
  // 65 to 96 rows of fp16 / bfloat16 where 96 x 32 tiles fill the device in one round (N = 8192 on 256 CUs): the
  // streaming kernel with three blocks of rows per wave -- A is three times the bytes of the weights per CTA, but the
  // weights still arrive in contiguous loads; 80 x 8192 x 8192 from HBM 38.5 us against 44.1 us on the tile kernels.
  // From three fifths of the CUs on (80 x 6144 x 4096: 19.6 / 27.1, 80 x 5120 x 5120: 24.0 / 33.5); other widths lose
  // to the tile kernels (96 x 11008 x 4096: 38.8 / 32.2, 80 x 4096 x 11008: 44.7 / 37.9, 80 x 16384 x 8192: 74.7 / 67.7).
  if (want_variant < 0 && rows_65_to_96_stream(M, N, dtype, layout, num_cus))
    for (int i = 0; i < n; ++i)
      if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].variant == 4 && t[i].bm == 96 && accepts_shape(t[i], M, K))
        return &t[i];
  if ((M <= (one_byte ? 64 : 32) && layout == SK_LAYOUT_NT) || q4) {
    // M == 1 with Q4 weights: the matrix-vector kernel with four waves splitting K (data-parallel
    // over 16-row tiles), the fastest instance at LLM-sized N and K.  Weights from HBM: from K = 14336 on eight waves
    // (1 x 16384 x 16384: 25.9 us against 28.7 us, 1 x 4096 x 14336: 7.9 / 9.0; 1 x 4096 x 11008: 8.2 / 7.4).  With more
    // 16-row tiles than CTAs of four waves stay resident (three per CU): K up to 6144 split over two waves, four
    // CTAs per CU (1 x 14336 x 4096: 7.7 us in one round against 10.8 us in two; 1 x 32000 x 4096: 14.6 / 16.2,
    // 1 x 65536 x 4096: 25.7 / 27.9), K from 8192 on over eight (1 x 28672 x 8192: 25.5 / 27.1).
    if (q4 && M == 1 && want_variant < 0) {
      int bk = 1024;
      if (K >= 14336) bk = 2048;
      else if (cdiv(N, 16) > (int64_t)num_cus * 3) bk = K <= 6144 ? 512 : (K >= 8192 ? 2048 : 1024);
      for (int pass = 0; pass < 2; ++pass, bk = 1024)
        for (int i = 0; i < n; ++i)
          if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].variant == 2 && t[i].bn == 16 &&
              t[i].bk == bk && accepts_shape(t[i], M, K))
            return &t[i];
    }
    // 2 <= M <= 16 with Q4 weights and per-group zero points: the kernels whose waves stream K on their own
    // (tile_rows_q4.h), as many rows of A staged as M needs, and the tile that gives the busiest CU the least to do -- a
    // round of tiles costs about 24 weight rows' time beside its own rows (ZP 16 x 28672 x 8192: two rounds of 64 rows
    // 40.7 us, three of 48 48.1, four of 32 49.3, seven of 16 61.0; 4 x 11008 x 4096: 48 rows 11.4, 64 rows 11.7, two
    // rounds of 32 12.5).  With one zero point for the matrix up to 8 rows, where 64-row tiles run in one round (beyond,
    // 4 x 28672 x 8192: 31.9 us on the general kernel against 38); 5 to 8 rows on 32-row tiles stay with the kernel
    // that streams through shared LDS where that one is taken, from 16 MB of weights on (8 x 5120 x 5120: 8.1 us against
    // 8.7, 8 x 8192 x 8192: 11.8 / 11.9; below, the general kernel / these: 8 x 5120 x 2048 5.4 / 4.9, 8 x 8192 x 1024 5.2 / 4.2).
    // (a caller's grid or fixed split that they cannot take -- more CTAs than stay resident, a factor that does not divide
    // their K-iterations -- goes to the kernels below)
    if ((dtype == SK_Q4_ZP || dtype == SK_Q4_ZP_TILED || (dtype == SK_Q4 && M <= 8 && cdiv(N, 64) <= num_cus)) && M > 1 && M <= 16 &&
        want_variant < 0) {
      int64_t least = 0;
      for (int i = 0; i < n; ++i) {
        if (t[i].family != FAMILY_SKINNY || t[i].dtype != dtype || t[i].variant != 5 || !accepts_shape(t[i], M, K)) continue;
        if (best && t[i].max_m > best->max_m) continue;
        const int64_t busiest = cdiv(cdiv(N, t[i].bn), num_cus) * (t[i].bn + 24);
        if (!best || t[i].max_m < best->max_m || busiest < least) {
          best = &t[i];
          least = busiest;
        }
      }
      const bool shared_lds = dtype == SK_Q4 && M > 4 && best && best->bn == 32 && K % 256 == 0 && N * K >= ((int64_t)16 << 20);
      if (best && takes_partition(*best, M, N, K, cfg, num_cus) && !shared_lds) return best;
      best = nullptr;
    }
    // 2 <= M <= 16 with row-major Q4 weights (scalar zero point), weights from HBM.  Where 64-row tiles give three
    // fifths of the CUs a tile the general kernel with 64 weight rows and K split over two waves, data-parallel
    // (16 x 28672 x 8192: 32.8 us; the 32-row kernel below: 48.5; 16 x 11008 x 4096: 10.7 / 14.8; 16 x 16384 x 16384:
    // 37.6 / 38.1).  Fewer rows and 16 MB of weights or more: the kernel that streams the packed weights through
    // LDS in contiguous loads, 32 weight rows per tile (tile_stream_q4.h; 16 x 8192 x 8192: 12.2 us against 14.2,
    // 16 x 4096 x 11008: 13.3 / 15.3; 16 x 4096 x 4096: 6.9 / 7.3).
    if (dtype == SK_Q4 && M > 1 && M <= 16 && want_variant < 0) {
      if (cdiv(N, 64) * 5 >= (int64_t)num_cus * 3) {
        for (int i = 0; i < n; ++i)
          if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].variant == 0 && t[i].bm == 16 &&
              t[i].bn == 64 && t[i].bk == 512 && accepts_shape(t[i], M, K))
            return &t[i];
      } else if (N * K >= ((int64_t)16 << 20) && K % 256 == 0) {
        for (int i = 0; i < n; ++i)
          if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].variant == 4 && t[i].bn == 32 &&
              accepts_shape(t[i], M, K))
            return &t[i];
      }
    }
    // 2 <= M <= 16 with Q4 weights: eight waves per CTA (two per SIMD cover each other's waits),
    // 32 weight rows, K split over four waves
    if (((dtype == SK_Q4 && M > 1) || dtype == SK_Q4_ZP || dtype == SK_Q4_ZP_TILED) && M <= 16 && want_variant < 0)
      for (int i = 0; i < n; ++i)
        if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].variant == 0 && t[i].bm == 16 &&
            t[i].bn == 32 && t[i].bk == 1024 && accepts_shape(t[i], M, K))
          return &t[i];
    // 2 <= M <= 4 with fp16 / bfloat16 weights: the matrix-vector form with four rows of A
    if ((dtype == SK_F16 || dtype == SK_BF16) && M >= 2 && M <= 4 && want_variant < 0)
      for (int i = 0; i < n; ++i)
        if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].layout == layout && t[i].variant == 3 &&
            t[i].bn == 16 && t[i].bk == 512 && accepts_shape(t[i], M, K))
          return &t[i];
    // M == 1 with fp16 / bfloat16 weights: the same structure, K split over four waves
    if ((dtype == SK_F16 || dtype == SK_BF16) && M == 1 && want_variant < 0)
      for (int i = 0; i < n; ++i)
        if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].layout == layout && t[i].variant == 2 &&
            t[i].bn == 16 && t[i].bk == 512 && accepts_shape(t[i], M, K))
          return &t[i];
    int mb = M <= 16 ? 16 : (M <= 32 ? 32 : 64);
    for (int i = 0; i < n; ++i)
      if (t[i].family == FAMILY_SKINNY && t[i].dtype == dtype && t[i].bm == mb && t[i].bn == 64 &&
          accepts_shape(t[i], M, K) && (want_variant < 0 || t[i].variant == want_variant) &&
          t[i].variant <= 2 && (best == nullptr || t[i].variant > best->variant))
        best = &t[i];
    if (best) return best;
    if (q4) return nullptr;
  }
  if (dtype == SK_F32) {
    // (a schedule or a grid without a tile; with nothing given model_pick_f32 chooses)
    // 32 x 256 tiles for M <= 32 (a quarter of the wasted rows of a 128-row tile), else 128 x 128
    const int want_bm = M <= 32 ? 32 : 128;
    const KernelInfo *any = nullptr;
    for (int i = 0; i < n; ++i)
      if (t[i].dtype == SK_F32 && t[i].layout == layout && t[i].bm == want_bm && t[i].bn == (want_bm == 32 ? 256 : 128)) {
        if (takes_partition(t[i], M, N, K, cfg, num_cus)) return &t[i];
        if (!any) any = &t[i];
      }
    return any;
  }
  // 256x256 tiles when they fill the device; else 128x128, else 64x64.  The smaller tiles run one
  // or two waves per SIMD, where the four-stage (BK = 32) pipeline hides the load latency better;
  // it exists for the NT layout only.
  const int64_t tiles256 = cdiv(M, 256) * cdiv(N, 256), tiles128 = cdiv(M, 128) * cdiv(N, 128);
  // (256x256: the four-wave kernel with the K loop in assembly where it applies -- K a multiple of 64 --
  // else the eight-wave 16x16x32-MFMA form)
  int pref[3][4] = {{256, 256, 64, 4}, {128, 128, 32, 3}, {64, 64, 32, 3}};  // bm, bn, bk, variant
  if (K % 64 == 0 && (dtype == SK_F16 || dtype == SK_BF16)) pref[0][3] = 7;
  const int first = tiles256 * 4 >= (int64_t)num_cus * 3 ? 0 : (tiles128 * 2 >= num_cus ? 1 : 2);
  const int order[3][3] = {{0, 1, 2}, {1, 2, 0}, {2, 1, 0}};  // smaller tiles first, then larger ones
  for (int oi = 0; oi < 3 && !best; ++oi) {
    const int pi = order[first][oi];
    for (int pass = 0; pass < 2 && !best; ++pass) {  // pass 1: any variant / BK of the tile shape
      for (int i = 0; i < n; ++i) {
        if (t[i].family != FAMILY_TILE || t[i].dtype != dtype || t[i].layout != layout) continue;
        if (t[i].bm != pref[pi][0] || t[i].bn != pref[pi][1]) continue;
        if (want_variant >= 0 ? t[i].variant != want_variant : by_variant_only(t[i])) continue;
        if (pass == 0 && want_variant < 0 && (t[i].bk != pref[pi][2] || t[i].variant != pref[pi][3])) continue;
        if (!accepts_shape(t[i], M, K)) continue;
        if (best == nullptr || variant_rank(t[i]) > variant_rank(*best)) best = &t[i];
      }
    }
  }
  return best;
}

// ---- which tile kernel and which split of K, when the caller leaves both open (M > 64) ----
// A cost model with four constants per kernel family, fitted to 80 shapes x 5 families x splits 1, 2, 4 timed on
// an MI355X (mean |log error| 5-10 %):
//     time = rounds * (n * tau * clock + o) + phi * log2(split)
//   n       K-iterations per CTA (iterations per tile / split)
//   clock   1 + 0.4 * (busy CUs / CUs)^2: the part is power-limited, busy CUs slow each other down
//   rounds  CTAs the busiest CU runs one after another; a family whose CTAs share a CU (occ > 1) is charged
//           1 + (rounds - 1) * gamma for them
//   o       prologue and epilogue of a CTA, phi one exchange of half tiles between the CTAs of a split tile (a
//           tile cut in two takes one, a tile cut in four two in a row: see run_persistent)
// Choosing by it is within 5 % of the fastest of the candidates on average (worst case 23 %) on those shapes, where
// the earlier rule (largest tile that fills the device, Stream-K for what is left) was 49 % behind on average.
static int gcd_int(int a, int b) {
  while (b) {
    const int r = a % b;
    a = b;
    b = r;
  }
  return a;
}

// The automatic schedule of a tile kernel with more tiles than CTAs; *sk_tiles: how many tiles it splits.
// Data-parallel when the last wave of tiles is at least 90 % full.  Else Stream-K over the remainder plus one
// wave of tiles (`sk2`, streamk_fp32.py:37-43; with fewer than two waves that is every tile, `basic` -- the
// reference's formula would split the remainder alone there, 2 tiles over 256 CTAs for 258 tiles, and the ordered
// fix-up has one CTA add up 63 partial tiles per tile: 1243 us against 130 us) -- but only where the CTAs of an
// XCD stay close to lock-step on K, which the L2 reuse of the tile kernels depends on: either every CTA range
// starts at the beginning or in the middle of a tile (grid / gcd(Stream-K tiles, grid) <= 2), or consecutive
// ranges start within ipt / 2 iterations of each other across the grid / 8 CTAs of an XCD.  Measured against
// data-parallel: 3-22 % faster where admitted; 4 or 8 distinct offsets between 8 % faster and 40 % slower;
// ranges that start anywhere up to 1.5x slower.  `interleave` (may be null: not offered) opens a third way for a
// one-CTA-per-CU kernel: with g = gcd(Stream-K tiles, grid) >= 8 the interleaved tile order puts the g CTAs that
// start at the same offset side by side on one XCD, which restores their lock-step (fp16 256 x 256 tiles, every
// tile split: 4096 x 5120 x 5120 172 us against 203 us in raster order, 3000 x 6144 x 4096 132 against 172,
// 2048 x 11008 x 4096 171 against 172; the best data-parallel plan of any tile: 215 / 160 / 178 us).
static int auto_tile_schedule(int64_t total, int grid, int ipt, int *sk_tiles, int *interleave = nullptr) {
  *sk_tiles = 0;
  if (interleave) *interleave = 0;
  const int64_t waves = (total + grid - 1) / grid;
  if (total < grid || total * 10 >= waves * grid * 9 || ipt < 64) return SK_SCHED_DP;  // (short K: the fix-up outweighs the tail)
  const int sched = total >= 2 * (int64_t)grid ? SK_SCHED_SK_TWO_TILE : SK_SCHED_SK_BASIC;
  const int skt = (int)(total % grid) + grid;
  const int64_t iters = (int64_t)skt * ipt;          // spread over `grid` CTAs
  const double per_cta = (double)iters / grid;       // in [ipt, 2 ipt)
  const double r = per_cta - ipt;                    // how far consecutive ranges drift apart, in iterations
  const double d = r < ipt - r ? r : ipt - r;
  const bool aligned = grid / gcd_int(skt, grid) <= 2;
  const bool close = d * (grid / 8 > 0 ? grid / 8 : 1) <= ipt / 2.0;
  if (!aligned && !close) {
    const int g = gcd_int(skt, grid);
    if (!interleave || g < 8 || skt / g < 2) return SK_SCHED_DP;
    *interleave = 1;
  }
  *sk_tiles = skt;
  return sched;
}

// A time of the model is of warm weights.  `measured`: what the times of 1 600 sizes of 65 to 1100 rows, their rows multiples of 128
// bytes, are of it, with the weights from the Infinity Cache (three sets of operands in turn) and from HBM (600 MB of them)
// (standard deviations 5 to 10 % and 5 to 20 %).
enum { FROM_CACHE, FROM_HBM };
struct Times {
  double us[2];
};
struct TileFamily {
  int bm, bn, bk, variant, occ, max_split;  // variant -1: the preferred variant of the tile
  float tau, gamma, o, phi, measured[2];
};
static const TileFamily kFamilies16[] = {
    {256, 256, 64, 7, 1, 4, 0.919f, 0.20f, 6.4f, 6.9f, {1.08f, 1.12f}},   // four waves, K loop in assembly (K % 64 == 0)
    {256, 256, 64, 4, 1, 2, 1.080f, 0.20f, 9.3f, 10.0f, {1.08f, 1.12f}},  // eight waves, for the other K
    {128, 128, 64, 4, 2, 4, 0.497f, 0.47f, 4.9f, 5.1f, {0.93f, 1.06f}},
    {128, 128, 32, 5, 2, 4, 0.218f, 0.89f, 3.8f, 4.5f, {1.00f, 1.21f}},   // four stages of 32 (NT only)
    {64, 128, 32, 5, 3, 4, 0.154f, 0.89f, 3.5f, 3.2f, {1.01f, 1.17f}},
    {128, 256, 64, 4, 1, 4, 0.689f, 1.00f, 6.0f, 5.9f, {1.06f, 1.25f}},
    {256, 128, 64, 4, 1, 4, 0.685f, 0.20f, 5.3f, 5.8f, {1.02f, 1.13f}},
};
// one-byte operands (BK = 128), fitted the same way to 36 shapes each (64 x 128: to 42 shapes with M <= 1024)
static const TileFamily kFamiliesF8[] = {
    {256, 256, 128, -1, 1, 4, 0.934f, 1.00f, 8.8f, 6.1f, {1.05f, 1.14f}},
    {128, 128, 128, -1, 2, 2, 0.435f, 0.52f, 6.3f, 6.6f, {1.00f, 1.20f}},
    {128, 256, 128, -1, 1, 2, 0.580f, 0.20f, 9.3f, 6.7f, {1.10f, 1.34f}},
    {256, 128, 128, -1, 1, 2, 0.608f, 1.00f, 7.2f, 7.8f, {0.95f, 1.17f}},
    {64, 128, 128, -1, 2, 2, 0.335f, 0.46f, 4.3f, 6.5f, {0.89f, 1.08f}},
    {128, 128, 64, 5, 2, 4, 0.218f, 0.88f, 2.3f, 11.0f, {1.06f, 1.33f}},  // four stages of 64 (fitted to 48 shapes with M <= 1024)
    {64, 128, 64, 5, 3, 4, 0.135f, 1.00f, 2.9f, 8.6f, {1.10f, 1.37f}},
};
static const TileFamily kFamiliesI8[] = {
    {256, 256, 128, -1, 1, 4, 0.876f, 0.20f, 13.3f, 4.2f, {1.06f, 1.09f}},
    {128, 128, 128, -1, 2, 2, 0.531f, 0.52f, 2.3f, 6.4f, {1.33f, 1.53f}},
    {128, 256, 128, -1, 1, 2, 0.674f, 0.20f, 6.5f, 6.5f, {1.16f, 1.40f}},
    {256, 128, 128, -1, 1, 2, 0.700f, 1.00f, 4.9f, 6.5f, {1.13f, 1.35f}},
    {64, 128, 128, -1, 2, 2, 0.392f, 0.39f, 3.3f, 4.0f, {0.95f, 1.15f}},
    {128, 128, 64, 5, 2, 4, 0.222f, 0.77f, 4.7f, 3.9f, {0.98f, 1.25f}},   // four stages of 64 (fitted to 48 shapes with M <= 1024)
    {64, 128, 64, 5, 3, 4, 0.143f, 0.88f, 4.0f, 4.1f, {1.01f, 1.19f}},
};

static const KernelInfo *model_pick(int64_t M, int64_t N, int64_t K, int dtype, int layout, int num_cus, int *split,
                                    int *sched, Times *times = nullptr) {
  const TileFamily *fams = kFamilies16;
  int nfams = (int)(sizeof(kFamilies16) / sizeof(kFamilies16[0]));
  if (dtype == SK_F8E4M3 || dtype == SK_F8E5M2) {
    fams = kFamiliesF8;
    nfams = (int)(sizeof(kFamiliesF8) / sizeof(kFamiliesF8[0]));
  } else if (dtype == SK_I8) {
    fams = kFamiliesI8;
    nfams = (int)(sizeof(kFamiliesI8) / sizeof(kFamiliesI8[0]));
  }
  const KernelInfo *best = nullptr;
  const TileFamily *best_family = nullptr;
  double best_time = 0;
  bool have_asm = false;
  for (int fi = 0; fi < nfams; ++fi) {
    const TileFamily &f = fams[fi];
    sk_config want;
    memset(&want, 0, sizeof(want));
    want.bm = f.bm; want.bn = f.bn; want.bk = f.bk;
    want.reserved[0] = f.variant + 1;
    const KernelInfo *k = pick_kernel(M, N, K, dtype, layout, &want, num_cus);
    if (!k || k->family != FAMILY_TILE || K % k->k_align != 0) continue;
    if (f.variant == 7) have_asm = true;
    if (f.variant == 4 && f.bm == 256 && f.bn == 256 && have_asm) continue;  // the assembly kernel applies
    const int64_t tiles = cdiv(M, f.bm) * cdiv(N, f.bn);
    const int64_t ipt = cdiv(K, f.bk);
    for (int s = 1; s <= f.max_split; s *= 2) {
      if (ipt % s != 0 || (s > 1 && ipt / s < 8)) continue;
      const int64_t ctas = tiles * s;
      if (s > 1 && ctas > (int64_t)num_cus * k->ctas_per_cu) continue;  // the CTAs of a split tile wait for each other
      const double busy = ctas < num_cus ? (double)ctas / num_cus : 1.0;
      const double clock = 1.0 + 0.4 * busy * busy;
      const int64_t rounds = ctas > num_cus ? cdiv(ctas, num_cus) : 1;
      const double eff = f.occ == 1 ? (double)rounds : 1.0 + (rounds - 1) * f.gamma;
      const double time = eff * ((double)(ipt / s) * f.tau * clock + f.o) + (s == 1 ? 0.0 : (s == 2 ? f.phi : 2.0 * f.phi));
      if (!best || time < best_time) {
        best = k;
        best_family = &f;
        best_time = time;
        *split = s;
        *sched = s > 1 ? SK_SCHED_SPLIT_K : SK_SCHED_DP;
      }
    }
    // more tiles than CUs on a one-CTA-per-CU kernel, and a Stream-K schedule that the automatic rule admits: the
    // iterations spread evenly over the CUs, plus one exchange of partial tiles (the rule is applied again below,
    // to the same effect, when the plan is made)
    int skt = 0;
    int ilv = 0;
    int *offer = f.bm == 256 && f.bn == 256 ? &ilv : nullptr;  // (the interleaved order: measured on these tiles)
    if (f.occ == 1 && tiles > num_cus && auto_tile_schedule(tiles, num_cus, (int)ipt, &skt, offer) != SK_SCHED_DP) {
      const double time = (double)tiles * ipt / num_cus * f.tau * 1.4 + f.o * (double)cdiv(tiles, num_cus) + 2.0 * f.phi;
      if (!best || time < best_time) {
        best = k;
        best_family = &f;
        best_time = time;
        *split = 1;
        *sched = SK_SCHED_AUTO;
      }
    }
  }
  for (int from = FROM_CACHE; times && best && from <= FROM_HBM; ++from) times->us[from] = best_time * best_family->measured[from];
  return best;
}

// ---- 65 to 128 rows of fp16 / bfloat16, NT: the ring kernels' tile and split of K ----
// time = o + rounds * iterations * (t + u * busy CUs / CUs) + fix-up(split), fitted to 60 timings, weights from HBM
// (within 6 % of each); a split that does not divide the iterations costs 3 to 5 us more, as its CTAs cross from one tile into
// the next (100 x 11008 x 4160, 65 iterations: 128-wide tiles in two 38.7, whole 64-wide ones 35.7).  100 rows, the tile kernels of the table above / these, in us: 4096 x 11008 42.0 / 33.5,
// 2048 x 8192 29.1 / 21.4, 5120 x 5120 35.2 / 27.2, 8192 x 8192 48.9 / 40.2, 28672 x 8192 130 / 98, 11008 x 4096 36.7 / 33.0.
struct RingFamily {
  int bn;
  double o, t, u, fix, per_log2, uneven;
};
static const RingFamily kFamiliesRing[] = {{64, 3.9, 0.395, 0.09, 2.6, 2.6, 3.0}, {128, 2.4, 0.55, 0.22, 3.5, 4.3, 5.0}};
// Short K and few columns give a CTA too few iterations for its deep ring to fill: there the tile kernels stay (100 rows, tile
// kernels / these, in us: K = 1024: 1024 wide 8.8 / 10.3, 28672 20.4 / 21.6; K = 1536: 1024 wide 10.8 / 13.1, 4096 14.6 / 15.0,
// 11008 20.0 / 17.5, 28672 29.2 / 29.0; K = 2048: 256 to 1024 wide 11.8 / 12.0, 1536 15.1 / 13.0, 4096 16.7 / 15.4; K = 2176:
// 256 to 1024 wide 12.2 / 14.4; K = 2816: 777 wide 14.2 / 14.5, 1024 15.1 / 13.8; K = 3000: 777 wide 23.6 / 18.8; K = 3072:
// 256 wide 14.2 / 13.3, 1024 16.4 / 14.5; 66 and 128 rows alike).
static bool ring_pays(int64_t N, int64_t K) { return K >= 2880 || (K >= 2048 && N >= 1536) || (K >= 1536 && N >= 8192); }
static const KernelInfo *model_pick_ring(int64_t N, int64_t K, int dtype, int num_cus, sk_config *out, Times *times = nullptr) {
  const KernelInfo *best = nullptr;
  double best_time = 0;
  int count;
  const KernelInfo *t = kernel_table(&count);
  for (const RingFamily &f : kFamiliesRing) {
    const KernelInfo *k = nullptr;
    for (int i = 0; i < count && !k; ++i)
      if (t[i].family == FAMILY_TILE && t[i].variant == 9 && t[i].dtype == dtype && t[i].bn == f.bn) k = &t[i];
    if (!k) continue;
    const int64_t tiles = cdiv(N, f.bn), ipt = cdiv(K, k->bk);
    for (int s = 1; s <= 8; s *= 2) {
      if (s > 1 && (tiles * s > num_cus || ipt / s < 8)) continue;
      const double busy = tiles * s < num_cus ? (double)(tiles * s) / num_cus : 1.0;
      const bool even = ipt % s == 0;
      const double time = f.o + (double)cdiv(tiles * s, num_cus) * ((double)ipt / s) * (f.t + f.u * busy) +
                          (s == 1 ? 0.0 : f.fix + f.per_log2 * (s == 2 ? 1 : (s == 4 ? 2 : 3)) + (even ? 0 : f.uneven));
      if (best && time >= best_time) continue;
      best = k;
      best_time = time;
      out->schedule = s == 1 ? SK_SCHED_DP : (even ? SK_SCHED_SPLIT_K : SK_SCHED_SK_BASIC);
      out->grid = s > 1 && !even ? (int)(tiles * s) : 0;
      out->reserved[1] = s > 1 && even ? s : 0;
    }
  }
  if (best) {
    out->bm = best->bm;
    out->bn = best->bn;
    out->bk = best->bk;
    out->reserved[0] = best->variant + 1;
    // (measured as in TileFamily; whatever the rows' alignment)
    if (times) *times = Times{{0.90 * best_time, 0.97 * best_time}};
  }
  return best;
}

// ---- a middling number of rows: the tiles whose waves stream K on their own (tile_wavek.h, tile_wavek_q4.h) ----
// Model, fitted to 33 000 timings each with the weights from the Infinity Cache (three sets of operands in turn; weights below 85 MB)
// and from HBM (600 MB of them): 16-bit, one-byte, Q4 and [K, N] weights, 1 to 1100 rows, 200 to 28672 columns, K from 512 to 16384;
// mean |log error| 4 to 5 and 5 to 9 %:
//     time = start + round (rounds - 1) + (core^1.6 + memory^1.6)^(1/1.6) + split + log2 (log2 of the split)
//   core    rounds x iterations x (iter + busy x busy CUs / CUs): one CTA per CU, every tile of a round side by side; longer where
//           rows of operands are no multiple of 128 bytes, because a wave's pieces then share lines with its neighbours', who drift
//           away from it in the course of K: `off` of it for rows of 16 KB and proportionally less for shorter ones (half of it for
//           odd multiples of 64 bytes), and `line` wherever that is so (fp16 63 x 1408 x 15096 on 32 x 32 tiles 49.6 us from HBM
//           and 34.0 from the cache, 35.9 and 22.4 with K = 15104); shorter by `empty` of the share of its operands that are rows of A past M, which are not fetched
//   memory  the operands and C once at `rate` TB/s, from HBM the higher the more weight rows a CTA has
struct WaveKFamily {
  int bm, bn;
  float start, round, split, log2;
  struct {
    float iter, busy, rate;
  } k[2];
};
struct WaveKRows {
  float off, line, empty;
};
static const WaveKFamily kFamiliesWaveK16[] = {
    {32, 32, 2.48f, 1.50f, 2.32f, 0.47f, {{0.317f, 0.043f, 9.3f}, {0.419f, 0.018f, 5.8f}}},
    {32, 64, 2.87f, 1.69f, 2.34f, 0.61f, {{0.431f, 0.111f, 9.0f}, {0.573f, 0.105f, 5.8f}}},
    {64, 32, 2.98f, 1.74f, 2.27f, 0.68f, {{0.427f, 0.095f, 10.4f}, {0.539f, 0.046f, 5.1f}}},
    {64, 48, 3.33f, 1.78f, 2.37f, 0.82f, {{0.511f, 0.099f, 9.8f}, {0.676f, 0.019f, 5.7f}}},
    {64, 64, 3.78f, 1.92f, 2.34f, 0.90f, {{0.553f, 0.133f, 10.0f}, {0.700f, 0.126f, 6.2f}}},
    {64, 80, 4.34f, 2.47f, 2.25f, 1.05f, {{0.664f, 0.127f, 9.2f}, {0.844f, 0.106f, 6.1f}}},
    {64, 96, 4.68f, 2.68f, 2.34f, 1.10f, {{0.724f, 0.129f, 9.5f}, {1.056f, 0.000f, 6.5f}}},
    {64, 112, 5.54f, 3.23f, 2.51f, 1.14f, {{0.782f, 0.295f, 9.2f}, {1.270f, 0.000f, 7.1f}}},
    {64, 128, 5.98f, 3.49f, 2.43f, 1.19f, {{0.840f, 0.298f, 10.7f}, {1.350f, 0.000f, 7.1f}}},
    {96, 32, 3.43f, 1.76f, 2.36f, 0.82f, {{0.536f, 0.141f, 11.4f}, {0.687f, 0.030f, 4.8f}}},
    {96, 64, 4.88f, 2.79f, 2.35f, 1.10f, {{0.704f, 0.126f, 10.0f}, {0.956f, 0.000f, 6.0f}}},
    {128, 32, 3.92f, 2.04f, 2.24f, 1.02f, {{0.698f, 0.117f, 10.2f}, {0.856f, 0.032f, 4.9f}}},
    {128, 48, 5.48f, 2.97f, 2.33f, 1.01f, {{0.877f, 0.095f, 9.9f}, {1.016f, 0.106f, 6.0f}}},
    {128, 64, 6.19f, 3.37f, 2.52f, 1.21f, {{0.824f, 0.276f, 8.9f}, {1.241f, 0.000f, 6.0f}}},
};
// [K, N] weights
static const WaveKFamily kFamiliesWaveKNN[] = {
    {32, 32, 2.08f, 0.94f, 2.32f, 0.62f, {{0.475f, 0.058f, 6.8f}, {0.629f, 0.014f, 4.5f}}},
    {32, 64, 2.53f, 1.25f, 2.18f, 0.76f, {{0.559f, 0.076f, 7.3f}, {0.752f, 0.026f, 5.2f}}},
    {32, 128, 3.49f, 1.76f, 2.46f, 0.78f, {{0.817f, 0.100f, 8.7f}, {0.931f, 0.212f, 5.9f}}},
    {64, 32, 2.51f, 1.35f, 2.15f, 0.90f, {{0.587f, 0.087f, 6.9f}, {0.736f, 0.059f, 4.7f}}},
    {64, 64, 3.47f, 1.45f, 2.24f, 1.06f, {{0.668f, 0.106f, 8.5f}, {0.848f, 0.117f, 5.7f}}},
    {96, 64, 4.74f, 1.96f, 2.28f, 1.16f, {{0.816f, 0.125f, 9.6f}, {0.938f, 0.210f, 6.0f}}},
    {128, 32, 3.32f, 1.49f, 2.41f, 1.15f, {{0.877f, 0.079f, 6.5f}, {0.950f, 0.111f, 3.6f}}},
};
static const WaveKFamily kFamiliesWaveK8[] = {
    {32, 32, 2.43f, 1.00f, 2.29f, 0.47f, {{0.342f, 0.061f, 8.6f}, {0.409f, 0.047f, 5.2f}}},
    {32, 64, 2.96f, 1.47f, 2.28f, 0.64f, {{0.430f, 0.141f, 9.0f}, {0.532f, 0.135f, 5.5f}}},
    {64, 32, 3.05f, 1.41f, 2.37f, 0.62f, {{0.427f, 0.108f, 10.5f}, {0.495f, 0.086f, 5.0f}}},
    {64, 48, 3.53f, 1.71f, 2.28f, 0.75f, {{0.496f, 0.121f, 10.0f}, {0.591f, 0.103f, 5.4f}}},
    {64, 64, 4.05f, 2.07f, 2.18f, 0.88f, {{0.531f, 0.138f, 10.1f}, {0.595f, 0.204f, 6.0f}}},
    {64, 80, 4.59f, 2.54f, 1.95f, 1.02f, {{0.657f, 0.137f, 9.7f}, {0.741f, 0.193f, 6.0f}}},
    {64, 96, 4.98f, 2.91f, 2.15f, 1.01f, {{0.700f, 0.150f, 9.8f}, {0.946f, 0.097f, 6.6f}}},
    {64, 112, 5.86f, 3.64f, 2.16f, 1.14f, {{0.849f, 0.176f, 9.9f}, {1.233f, 0.004f, 7.0f}}},
    {64, 128, 6.34f, 3.58f, 2.20f, 1.15f, {{0.792f, 0.325f, 11.9f}, {1.238f, 0.101f, 7.2f}}},
    {96, 32, 3.62f, 1.60f, 2.24f, 0.77f, {{0.501f, 0.164f, 13.4f}, {0.571f, 0.159f, 5.2f}}},
    {96, 64, 5.09f, 2.92f, 2.16f, 1.05f, {{0.666f, 0.161f, 11.0f}, {0.878f, 0.079f, 6.3f}}},
    {128, 32, 4.18f, 1.98f, 2.28f, 0.88f, {{0.647f, 0.161f, 12.6f}, {0.725f, 0.153f, 5.3f}}},
    {128, 48, 5.56f, 2.97f, 2.33f, 0.93f, {{0.942f, 0.039f, 10.0f}, {0.981f, 0.152f, 6.7f}}},
    {128, 64, 6.45f, 3.44f, 2.36f, 1.17f, {{0.869f, 0.220f, 11.7f}, {1.099f, 0.144f, 6.9f}}},
};
static const WaveKFamily kFamiliesWaveKQ4[] = {
    {32, 32, 3.02f, 1.42f, 2.28f, 0.63f, {{0.662f, 0.061f, 11.7f}, {0.684f, 0.065f, 5.0f}}},
    {32, 64, 3.64f, 1.86f, 2.20f, 0.79f, {{0.947f, 0.109f, 9.6f}, {0.990f, 0.124f, 4.6f}}},
    {64, 32, 3.66f, 1.76f, 2.41f, 0.71f, {{0.825f, 0.093f, 9.5f}, {0.846f, 0.127f, 4.3f}}},
    {64, 64, 4.50f, 2.26f, 2.40f, 0.93f, {{1.269f, 0.084f, 6.7f}, {1.322f, 0.076f, 3.9f}}},
    {64, 96, 5.17f, 3.09f, 2.67f, 1.06f, {{1.680f, 0.186f, 6.7f}, {1.767f, 0.205f, 4.2f}}},
    {128, 32, 4.59f, 1.71f, 2.50f, 0.83f, {{1.291f, 0.223f, 9.5f}, {1.323f, 0.226f, 3.0f}}},
};
static const WaveKRows kRowsWaveK16[2] = {{0.41f, 0.097f, 0.49f}, {0.35f, 0.136f, 0.48f}};
static const WaveKRows kRowsWaveKNN[2] = {{0.00f, 0.200f, 0.39f}, {0.06f, 0.094f, 0.19f}};
static const WaveKRows kRowsWaveK8[2] = {{0.36f, 0.093f, 0.36f}, {0.40f, 0.139f, 0.37f}};
static const WaveKRows kRowsWaveKQ4[2] = {{0.00f, 0.000f, 0.18f}, {0.00f, 0.000f, 0.19f}};   // (rows of whole scale groups: aligned)
// whether some sets of the weights stay in the Infinity Cache between calls (else the times from HBM alone count)
static bool from_cache(int64_t N, int64_t K, int dtype) {
  const bool q4 = dtype == SK_Q4 || dtype == SK_Q4_ZP, b16 = dtype == SK_F16 || dtype == SK_BF16;
  return (q4 ? 0.52 : (b16 ? 2.0 : 1.0)) * N * K < 85e6;
}
static double unaligned_rows(const WaveKRows &m, int64_t pitch) {
  if (pitch % 128 == 0) return 1;
  return 1 + m.line + m.off * (pitch % 64 == 0 ? 0.5 : 1.0) * (pitch < 16384 ? pitch / 16384.0 : 1.0);
}
static const KernelInfo *model_pick_wavek(int64_t M, int64_t N, int64_t K, int dtype, int layout, int num_cus, sk_config *out,
                                          Times *times) {
  const bool q4 = dtype == SK_Q4 || dtype == SK_Q4_ZP, one_byte = dtype == SK_F8E4M3 || dtype == SK_F8E5M2 || dtype == SK_I8;
  const WaveKFamily *fams = kFamiliesWaveK16;
  int nfams = (int)(sizeof(kFamiliesWaveK16) / sizeof(kFamiliesWaveK16[0]));
  const WaveKRows *mem = kRowsWaveK16;
  if (layout == SK_LAYOUT_NN) {
    fams = kFamiliesWaveKNN;
    nfams = (int)(sizeof(kFamiliesWaveKNN) / sizeof(kFamiliesWaveKNN[0]));
    mem = kRowsWaveKNN;
  } else if (q4) {
    fams = kFamiliesWaveKQ4;
    nfams = (int)(sizeof(kFamiliesWaveKQ4) / sizeof(kFamiliesWaveKQ4[0]));
    mem = kRowsWaveKQ4;
  } else if (one_byte) {
    fams = kFamiliesWaveK8;
    nfams = (int)(sizeof(kFamiliesWaveK8) / sizeof(kFamiliesWaveK8[0]));
    mem = kRowsWaveK8;
  }
  const double weight_bytes = q4 ? 0.52 : (one_byte ? 1 : 2), a_bytes = one_byte ? 1 : 2, c_bytes = dtype == SK_I8 ? 4 : 2;
  const double bytes = weight_bytes * N * K + a_bytes * M * K + c_bytes * M * N;
  const int64_t pitch = layout == SK_LAYOUT_NN ? 2 * N : (one_byte ? K : 2 * K);
  const bool cached = from_cache(N, K, dtype);
  const KernelInfo *best = nullptr;
  double best_time = 0;
  int count;
  const KernelInfo *t = kernel_table(&count);
  for (int fi = 0; fi < nfams; ++fi) {
    const WaveKFamily &f = fams[fi];
    const KernelInfo *k = nullptr;
    for (int i = 0; i < count && !k; ++i)
      if (t[i].family == FAMILY_TILE && t[i].variant == 10 && t[i].dtype == dtype && t[i].layout == layout && t[i].bm == f.bm && t[i].bn == f.bn) k = &t[i];
    if (!k || K % k->k_align != 0) continue;
    const int64_t tiles = cdiv(M, f.bm) * cdiv(N, f.bn), ipt = cdiv(K, k->bk);
    for (int s = 1; s <= 8; s *= 2) {
      if (s > 1 && (ipt % s != 0 || tiles * s > num_cus)) continue;
      const double busy = tiles * s < num_cus ? (double)(tiles * s) / num_cus : 1.0;
      const double rounds = (double)cdiv(tiles * s, num_cus);
      const double past_m = (1 - (double)M / (cdiv(M, f.bm) * f.bm)) * f.bm / (f.bm + (q4 ? 0.5 : 1.0) * f.bn);
      Times time;
      for (int from = FROM_CACHE; from <= FROM_HBM; ++from) {
        const double core = rounds * ((double)ipt / s) * (f.k[from].iter + f.k[from].busy * busy) * unaligned_rows(mem[from], pitch) *
                            (1 - mem[from].empty * past_m);
        const double memory = bytes / (f.k[from].rate * 1e6);
        time.us[from] = f.start + f.round * (rounds - 1) + pow(pow(core, 1.6) + pow(memory, 1.6), 1 / 1.6) +
                        (s == 1 ? 0.0 : f.split + f.log2 * (s == 2 ? 1 : (s == 4 ? 2 : 3)));
      }
      // (both count alike; within 2 % the larger tile: fewer bytes of the operands through the caches)
      const double both = cached ? sqrt(time.us[FROM_CACHE] * time.us[FROM_HBM]) : time.us[FROM_HBM];
      if (best && both >= best_time * (f.bm * f.bn > best->bm * best->bn ? 1.02 : (f.bm * f.bn < best->bm * best->bn ? 0.98 : 1.0))) continue;
      best = k;
      best_time = both;
      *times = time;
      out->schedule = s == 1 ? SK_SCHED_DP : SK_SCHED_SPLIT_K;
      out->reserved[1] = s > 1 ? s : 0;
    }
  }
  if (best) {
    out->bm = best->bm;
    out->bn = best->bn;
    out->bk = best->bk;
    out->reserved[0] = best->variant + 1;
  }
  return best;
}

// The kernels that such calls of up to 64 rows (96 on 96 x 32 tiles) take otherwise, fitted to 2 300 of the same timings (mean |log
// error| 2 to 8 %):
//     time = start + sqrt(core^2 + memory^2) + (where tiles are split) fixup + share x CTAs per tile
//   core    iterations of the busiest CTA x (iter + busy x CTAs / CUs)
//   memory  the operands once at `rate` TB/s, at 15 times the share of the CUs that has a CTA where that is less
enum RowsOperands { ROWS_16, ROWS_8, ROWS_Q4, ROWS_Q4_ZP, ROWS_NN };
struct RowsFamily {
  int operands, bm, bn;
  struct {
    float start, iter, busy, rate, fixup, share;
  } t[2];
};
static const RowsFamily kFamiliesRows[] = {
    {ROWS_8, 32, 32, {{3.09f, 0.471f, 0.329f, 8.00f, 3.89f, 0.32f}, {2.87f, 0.556f, 0.948f, 8.00f, 4.10f, 0.34f}}},
    {ROWS_8, 32, 64, {{2.79f, 0.044f, 0.948f, 8.00f, 4.00f, 0.00f}, {3.31f, 0.403f, 0.706f, 8.00f, 4.26f, 0.55f}}},
    {ROWS_8, 64, 32, {{2.84f, 0.587f, 0.106f, 7.56f, 4.81f, 0.17f}, {2.89f, 0.591f, 0.148f, 5.56f, 5.23f, 0.16f}}},
    {ROWS_8, 64, 64, {{3.55f, 0.000f, 1.217f, 8.00f, 4.00f, 0.00f}, {4.64f, 0.441f, 0.812f, 8.00f, 4.17f, 0.28f}}},
    {ROWS_16, 32, 32, {{2.61f, 0.248f, 0.113f, 8.00f, 2.87f, 0.35f}, {2.30f, 0.381f, 0.320f, 8.00f, 3.30f, 0.34f}}},
    {ROWS_16, 32, 64, {{2.79f, 0.000f, 0.889f, 8.00f, 4.00f, 0.00f}, {3.66f, 0.556f, 0.440f, 8.00f, 4.00f, 0.00f}}},
    {ROWS_16, 64, 32, {{3.22f, 0.411f, 0.024f, 6.27f, 3.92f, 0.33f}, {3.35f, 0.397f, 0.000f, 4.63f, 4.28f, 0.31f}}},
    {ROWS_16, 64, 64, {{3.47f, 0.000f, 1.020f, 8.00f, 4.00f, 0.00f}, {5.24f, 0.372f, 0.779f, 8.00f, 4.00f, 0.00f}}},
    {ROWS_16, 96, 32, {{3.85f, 0.819f, 0.000f, 6.33f, 4.00f, 0.00f}, {4.09f, 0.926f, 0.000f, 5.68f, 4.00f, 0.00f}}},
    {ROWS_NN, 128, 128, {{2.38f, 0.458f, 0.430f, 6.66f, 0.69f, 1.45f}, {2.36f, 0.635f, 0.430f, 8.00f, 0.93f, 1.52f}}},
    {ROWS_Q4, 32, 64, {{4.52f, 0.368f, 0.217f, 4.53f, 3.53f, 0.47f}, {4.41f, 0.469f, 0.341f, 5.83f, 3.54f, 0.48f}}},
    {ROWS_Q4, 64, 64, {{4.99f, 0.849f, 0.256f, 5.09f, 4.49f, 1.11f}, {5.37f, 0.816f, 0.353f, 5.05f, 4.62f, 1.12f}}},
    {ROWS_Q4_ZP, 32, 64, {{5.15f, 0.448f, 0.000f, 3.24f, 3.23f, 0.54f}, {5.28f, 0.504f, 0.352f, 5.44f, 3.37f, 0.52f}}},
    {ROWS_Q4_ZP, 64, 64, {{5.42f, 0.756f, 0.420f, 4.84f, 5.17f, 1.17f}, {5.90f, 0.747f, 0.512f, 4.96f, 5.38f, 1.16f}}},
};
static bool rows_times(const KernelInfo &k, const sk_plan &p, int num_cus, Times *times) {
  const bool zp = p.dtype == SK_Q4_ZP, q4 = zp || p.dtype == SK_Q4, b16 = p.dtype == SK_F16 || p.dtype == SK_BF16;
  const bool nn = p.layout == SK_LAYOUT_NN;
  const int operands = q4 ? (zp ? ROWS_Q4_ZP : ROWS_Q4) : (b16 ? (nn ? ROWS_NN : ROWS_16) : ROWS_8);
  if (!nn && k.variant != (q4 ? 0 : (b16 ? 4 : 8))) return false;
  const double per_cta = p.streamk_tiles > 0 ? (double)p.total_tiles * p.iters_per_tile / p.grid : (double)cdiv(p.total_tiles, p.grid) * p.iters_per_tile;
  const double bytes = (q4 ? (zp ? 0.54 : 0.52) : (b16 ? 2 : 1)) * p.N * p.K + (q4 || b16 ? 2.0 : 1.0) * p.M * p.K;
  const double cus = p.grid < num_cus ? (double)p.grid / num_cus : 1.0;
  for (const RowsFamily &f : kFamiliesRows) {
    if (f.operands != operands || f.bm != k.bm || f.bn != k.bn) continue;
    for (int from = FROM_CACHE; from <= FROM_HBM; ++from) {
      const auto &t = f.t[from];
      const double core = per_cta * (t.iter + t.busy * p.grid / num_cus), memory = bytes / ((t.rate < 15 * cus ? t.rate : 15 * cus) * 1e6);
      times->us[from] = t.start + sqrt(core * core + memory * memory) + (p.streamk_tiles > 0 ? t.fixup + t.share * p.grid / p.total_tiles : 0);
    }
    return true;
  }
  return false;
}
// the Q4 tile kernels that decode into LDS: fitted like the others, 128 x 128 tiles up to 128 rows, 256 x 128 beyond (mean
// |log error| 6 and 4 %)
static double q4_tile_us(int64_t M, int64_t N, int64_t K, int num_cus) {
  const int bm = M > 128 ? 256 : 128, occ = bm == 256 ? 1 : 2;
  const int64_t tiles = cdiv(M, bm) * cdiv(N, 128), ipt = K / 64;
  int split = 1;
  for (int s = 2; tiles < num_cus && s <= 4; s *= 2)
    if (tiles * s <= (int64_t)num_cus * occ && ipt % s == 0 && ipt / s >= 8) split = s;
  int skt;
  const bool even = tiles > num_cus && auto_tile_schedule(tiles, num_cus * occ, (int)ipt, &skt) != SK_SCHED_DP;
  const double rounds = even ? (double)tiles / num_cus : (double)cdiv(tiles * split, num_cus);
  const double busy = tiles * split < num_cus ? (double)(tiles * split) / num_cus : 1.0;
  const double per = bm == 256 ? 0.667 + 0.316 * busy : 0.664 + 0.105 * busy;
  return (bm == 256 ? 5.24 : 2.45) + rounds * ((double)ipt / split) * per +
         (split == 1 ? 0.0 : (bm == 256 ? 4.8 : 5.0) * (split == 2 ? 1 : 2));
}
// Whether a problem whose tile, variant, schedule and grid are open goes to them: wavek's times against those of the kernel that it
// takes otherwise (`other`, its plan), with the weights from the cache and from HBM; a call must win by both, because its caller's
// other weights decide which it is.  The margins cover the models' errors: of
// 6 600 random sizes that go to them 25 are behind the other kernel by more than 3 % in either, by 11 % at most, and by type they take
// .47 to .64 of its time on average.
static bool wavek_pays(const sk_plan &other, int num_cus, const Times &wavek) {
  const KernelInfo *k = kernel_by_id(other.kernel_id);
  if (!k) return false;
  const int64_t M = other.M, N = other.N, K = other.K;
  const int dtype = other.dtype, layout = other.layout;
  const bool q4 = dtype == SK_Q4 || dtype == SK_Q4_ZP, b16 = dtype == SK_F16 || dtype == SK_BF16, nn = layout == SK_LAYOUT_NN;
  Times times;
  double margin;
  if (k->family == FAMILY_SKINNY || (nn && M <= 64)) {
    if (!rows_times(*k, other, num_cus, &times)) return false;
    // (per-group zero points and a long K: two arrays beside the nibbles, 8 % more from HBM than the model of both says.  Of 51 sizes
    // with K from 7500 on those below 0.85 of the other's predicted time took .59 to .90 of it, the others 1.06: 23 x 10144 x 14720
    // 40.6 us there and 50.3 here)
    margin = dtype == SK_Q4_ZP && K >= 7500 ? 0.85 : (q4 ? 1.0 : (nn ? 0.97 : 0.95));
  } else if (dtype == SK_Q4) {
    times.us[FROM_CACHE] = times.us[FROM_HBM] = q4_tile_us(M, N, K, num_cus);
    margin = 0.97;
  } else {
    // (the tile kernels' rows suffer from their alignment as the wave-K tiles' do, the ring kernels' hardly)
    sk_config c;
    int split, sched;
    const bool ring = k->variant == 9;
    if (!(ring ? model_pick_ring(N, K, dtype, num_cus, &c, &times) : model_pick(M, N, K, dtype, layout, num_cus, &split, &sched, &times))) return true;
    const WaveKRows *rows = nn ? kRowsWaveKNN : (b16 ? kRowsWaveK16 : kRowsWaveK8);
    for (int from = FROM_CACHE; from <= FROM_HBM && !ring; ++from)
      times.us[from] *= unaligned_rows(rows[from], nn ? 2 * N : (b16 ? 2 * K : K));
    // ([K, N] weights and up to 128 rows, which fill the others' tiles: 128 x 5120 x 5120 from HBM 30.1 us on those, 35.3 here against a
    // predicted 29, from the cache 25.2 / 23.1)
    margin = ring ? 0.97 : (nn ? (M <= 128 ? 0.85 : 0.93) : 0.95);
    // (products that take the others several full rounds: predicted closer than that they took 1.0 of the time from the cache and .97
    // from HBM, 1.4 at worst, int8 534 x 24608 x 9056 183 us there and 255 here)
    if ((double)M * N * K > 1.5e10 && margin > 0.88) margin = 0.88;
  }
  return (!from_cache(N, K, dtype) || wavek.us[FROM_CACHE] < margin * times.us[FROM_CACHE]) && wavek.us[FROM_HBM] < margin * times.us[FROM_HBM];
}

// ---- fp32: tile, schedule and grid, when the caller leaves all three open ----
// The matrix pipe is slow enough (64 FLOP per cycle and SIMD) that tiles of 64 x 64 keep it busy; what decides is how
// many CTAs there are and whether two of them share a CU (one computes while the other waits at its barrier).  Model,
// fitted to 590 timings of every tile and schedule on 18 shapes in both layouts, weights from HBM, on one device with the
// 32 x 256 tiles' ring eight slots deep (mean |log error| 4 %).  On the kernels as they are its choice is 2.1 % behind the
// fastest candidate on average over 20 shapes in both layouts, 12 % at worst (profiles/planner_f32_choice.md); the rule
// before -- 128 x 128 tiles, 32 x 256 up to 32 rows, split in two or four -- was 1.1 to 5.8 times behind:
//     time = o + (compute^4 + memory^4)^(1/4) + fix-up
//   compute  tiles of the busiest CU x the tile's FLOP at 0.614 TFLOP/s per CU, over `one` (a CTA alone on its CU) or
//            `two`; up to 16 rows a 32-row tile computes 16 rows only
//   memory   the operands once at 5.1 TB/s, slower by 1.53 x busy CUs / CUs below two thirds of the CUs
//   fix-up   1.7 us + 0.34 us per 32 KB of partial tile and contributor
struct F32Family {
  int bm, bn;
  double one, two;
};
static const F32Family kFamiliesF32[] = {
    {32, 64, 0.52, 0.65}, {32, 256, 0.59, 0.59}, {64, 64, 0.68, 0.87}, {64, 128, 0.77, 0.90}, {128, 128, 0.80, 0.91},
};
static const KernelInfo *model_pick_f32(int64_t M, int64_t N, int64_t K, int layout, int num_cus, sk_config *out) {
  const KernelInfo *best = nullptr;
  double best_time = 0;
  int count;
  const KernelInfo *t = kernel_table(&count);
  for (const F32Family &f : kFamiliesF32) {
    if ((f.bm == 32 && M > 64) || (f.bm == 128 && M <= 32)) continue;
    const KernelInfo *k = nullptr;
    for (int i = 0; i < count; ++i)   // (the instance with the longest K-iteration: see kernels_f32.hip)
      if (t[i].dtype == SK_F32 && t[i].layout == layout && t[i].bm == f.bm && t[i].bn == f.bn && (!k || t[i].bk > k->bk)) k = &t[i];
    if (!k) continue;
    // (a tile that gains nothing from a second CTA on its CU is offered one: 16 x 16384 x 8192 on 256 CTAs of 32 x 256
    // 99.7 us, on 512 110)
    const int ctas = f.two > f.one ? k->ctas_per_cu : 1;
    const int64_t tiles = cdiv(M, f.bm) * cdiv(N, f.bn), ipt = cdiv(K, k->bk), cap = (int64_t)num_cus * ctas;
    const double tile_us = (double)(f.bm == 32 && M <= 16 ? 16 : f.bm) * f.bn * K * 2 / 0.614e6;
    const double bytes_us = 4.0 * ((double)N * K + (double)M * K + (double)M * N) / 5.1e6 / (f.bn == 256 ? 1.05 : 1.0);
    auto consider = [&](int sched, int64_t grid, int split) {
      double comp, fix = 0;
      const double contributors = (double)grid / tiles;
      if (sched == SK_SCHED_DP) {
        comp = (double)cdiv(tiles, num_cus) * tile_us / (tiles > num_cus && ctas > 1 ? f.two : f.one);
      } else {
        comp = (double)cdiv(grid, num_cus) / contributors * tile_us / (grid > num_cus ? f.two : f.one);
        fix = 1.7 + 0.34 * f.bm * f.bn / 8192 * (contributors > 1 ? contributors : 1);
      }
      const double busy = 1.53 * grid / num_cus;
      const double mem = bytes_us / (busy < 1 ? busy : 1);
      const double c2 = comp * comp, m2 = mem * mem, time = 5.2 + sqrt(sqrt(c2 * c2 + m2 * m2)) + fix;
      if (best && time >= best_time) return;
      best = k;
      best_time = time;
      out->schedule = sched;
      out->grid = sched == SK_SCHED_SK_BASIC ? (int)grid : 0;
      out->reserved[1] = split > 1 ? split : 0;
    };
    consider(SK_SCHED_DP, tiles < cap ? tiles : cap, 1);
    for (int s = 2; s <= 16; s *= 2)
      if (ipt % s == 0 && ipt / s >= 4 && tiles * s <= cap) consider(SK_SCHED_SPLIT_K, tiles * s, s);
    // every tile split evenly over one or two CTAs per CU, at least four iterations each, at most 16 per tile
    for (int64_t g = num_cus; g <= cap; g += num_cus)
      if (tiles * ipt >= 4 * g && tiles * 16 >= g && tiles < 2 * g && tiles != g) consider(SK_SCHED_SK_BASIC, g, 1);
    if (tiles * 8 < num_cus && ipt >= 32) consider(SK_SCHED_SK_BASIC, tiles * 8, 1);
  }
  if (best) {
    out->bm = best->bm;
    out->bn = best->bn;
    out->bk = best->bk;
  }
  return best;
}

}  // namespace sk

using namespace sk;

extern "C" int sk_selfcheck(void) {
  int n;
  const KernelInfo *t = kernel_table(&n);
  if (n <= 0 || n >= TABLE_MAX) return SK_ERR_CONFIG;
  for (int i = 0; i < n; ++i) {
    if (t[i].id < 0 || t[i].id >= 1024 || !t[i].name || !t[i].name[0]) return SK_ERR_CONFIG;
    for (int j = 0; j < i; ++j)
      if (t[j].id == t[i].id) return SK_ERR_CONFIG;
  }
  return SK_OK;
}

extern "C" int sk_make_plan(int64_t M, int64_t N, int64_t K, int dtype, int layout, const sk_config *cfg,
                            int num_cus, sk_plan *out) {
  if (!out) return SK_ERR_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return SK_ERR_SHAPE;
  if (dtype != SK_F16 && dtype != SK_F32 && dtype != SK_Q4 && dtype != SK_BF16 && dtype != SK_Q4_TILED &&
      dtype != SK_F8E4M3 && dtype != SK_I8 && dtype != SK_Q4_ZP && dtype != SK_F8E5M2 && dtype != SK_Q4_ZP_TILED)
    return SK_ERR_CONFIG;
  if ((dtype == SK_F8E4M3 || dtype == SK_F8E5M2 || dtype == SK_I8) && layout != SK_LAYOUT_NT) return SK_ERR_CONFIG;
  if (layout != SK_LAYOUT_NT && layout != SK_LAYOUT_NN) return SK_ERR_CONFIG;
  if (num_cus <= 0) return SK_ERR_DEVICE;
  // tile, variant, schedule and grid all left open for a 16-bit or one-byte problem with more rows than the
  // weight-streaming kernels take: the cost models choose kernel and split.  The kernels whose waves stream K on their own and
  // the ring kernels add up fp32 partial tiles: a fix-up that adds packed 16-bit partials into C, or exchanges them in 16 bits,
  // is a matter of the other tile kernels.  The former are for a caller who asks for SK_VARIANT_OPERATOR: a plan without it
  // takes the kernels that plans have taken so far.
  sk_config modelled, wavek;
  // (the tiled layout of Q4 weights takes what the row-major one does, so that both give the same bits)
  const int as_rows = dtype == SK_Q4_TILED ? (int)SK_Q4 : (dtype == SK_Q4_ZP_TILED ? (int)SK_Q4_ZP : dtype);
  const bool q4_rows = as_rows == SK_Q4 || as_rows == SK_Q4_ZP, b16 = dtype == SK_F16 || dtype == SK_BF16;
  const bool one_byte = dtype == SK_F8E4M3 || dtype == SK_F8E5M2 || dtype == SK_I8;
  const bool by_operator = cfg && cfg->reserved[0] == SK_VARIANT_OPERATOR && cfg->bm == 0 && cfg->bn == 0;
  const bool open = !cfg || (cfg->bm == 0 && cfg->bn == 0 && cfg->bk == 0 && (cfg->reserved[0] == 0 || by_operator) &&
                             cfg->schedule == SK_SCHED_AUTO && cfg->grid == 0);
  const bool few = M <= 64;
  if (by_operator) {
    modelled = *cfg;
    modelled.reserved[0] = one_byte && few ? 9 : 0;
    cfg = &modelled;
  }
  const int want_fixup = cfg ? cfg->fixup : SK_FIXUP_AUTO;
  const bool fp32_partials = want_fixup == SK_FIXUP_AUTO || want_fixup == SK_FIXUP_REDUCE || want_fixup == SK_FIXUP_ATOMIC;
  if (open && fp32_partials && by_operator && (layout == SK_LAYOUT_NT ? M > 16 : b16) && (b16 || q4_rows || one_byte)) {
    Times times;
    wavek = *cfg;
    sk_plan other;   // what a call takes otherwise, if any kernel runs it in one launch
    if (model_pick_wavek(M, N, K, as_rows, layout, num_cus, &wavek, &times) &&
        (sk_make_plan(M, N, K, as_rows, layout, cfg, num_cus, &other) != SK_OK || wavek_pays(other, num_cus, times)))
      cfg = &wavek;
  }
  if (open && cfg != &wavek && (b16 || one_byte) && !few && !rows_65_to_96_stream(M, N, dtype, layout, num_cus)) {
    if (cfg) modelled = *cfg; else memset(&modelled, 0, sizeof(modelled));
    if (b16 && layout == SK_LAYOUT_NT && M <= 128 && ring_pays(N, K) && fp32_partials &&
        model_pick_ring(N, K, dtype, num_cus, &modelled)) {
      cfg = &modelled;
    } else {
      int split = 1, model_sched = SK_SCHED_AUTO;
      if (const KernelInfo *mk = model_pick(M, N, K, dtype, layout, num_cus, &split, &model_sched)) {
        modelled.bm = mk->bm; modelled.bn = mk->bn; modelled.bk = mk->bk;
        modelled.reserved[0] = mk->variant + 1;
        modelled.schedule = model_sched;
        if (split > 1) modelled.reserved[1] = split;
        cfg = &modelled;
      }
    }
  }
  if (dtype == SK_F32 && (!cfg || (cfg->bm == 0 && cfg->bn == 0 && cfg->bk == 0 && cfg->reserved[0] == 0 &&
                                   cfg->schedule == SK_SCHED_AUTO && cfg->grid == 0))) {
    if (cfg) modelled = *cfg; else memset(&modelled, 0, sizeof(modelled));
    if (model_pick_f32(M, N, K, layout, num_cus, &modelled)) cfg = &modelled;
  }
  const KernelInfo *k = pick_kernel(M, N, K, dtype, layout, cfg, num_cus);
  if (!k) return SK_ERR_CONFIG;
  if (K % k->k_align != 0) return SK_ERR_ALIGN;

  memset(out, 0, sizeof(*out));
  out->M = M; out->N = N; out->K = K;
  out->dtype = dtype; out->layout = layout;
  out->bm = k->bm; out->bn = k->bn; out->bk = k->bk;
  out->kernel_id = k->id; out->threads = k->threads; out->lds_bytes = k->lds_bytes;
  out->num_block_m = (int32_t)cdiv(M, k->bm);
  out->num_block_n = (int32_t)cdiv(N, k->bn);
  out->iters_per_tile = (int32_t)cdiv(K, k->bk);
  if (k->max_ipt > 0 && out->iters_per_tile > k->max_ipt) return SK_ERR_CONFIG;
  const int64_t total64 = (int64_t)out->num_block_m * out->num_block_n;
  if (total64 * out->iters_per_tile > 0x7fffffff) return SK_ERR_SHAPE;
  const int total = (int)total64;
  out->total_tiles = total;

  // every CTA of the Stream-K wave may wait for another one, so the grid is capped at what the
  // device keeps resident
  const int occ = k->ctas_per_cu;
  const int max_grid = num_cus * occ;
  int grid = cfg && cfg->grid > 0 ? cfg->grid : max_grid;
  if (grid > max_grid) return SK_ERR_CONFIG;
  int sched = cfg ? cfg->schedule : SK_SCHED_AUTO;
  if (!(cfg && cfg->grid > 0)) {
    const int64_t iters = total64 * out->iters_per_tile;
    // (the kernels that stream the weights through LDS are bound by memory: with tiles for three fifths of the CUs --
    // fp16 / bfloat16: two fifths -- they run data-parallel rather than pay a fix-up; Q4 16 x 11008 x 4096: 11.5 us
    // against 14.3 us, fp16 16 x 2048 x 8192 on 128 tiles: 11.5 against 14.1, 32 x 11008 x 4096 on 172 tiles of 32 x 64:
    // 19.2 against 22.7; not the 64 x 32 tiles, where the split wins)
    // (one-byte weights through LDS: always up to 16 rows -- 16 x 1024 x 16384 on 64 tiles 11.2 us against 11.5, at worst
    // 16 x 520 x 16384 10.8 / 10.0 -- and on 32 and 64 rows unless a CTA would run many iterations while others idle, data-parallel /
    // split: 32 x 520 x 8192 9.2 us / 9.2, 32 x 2048 x 8192 11.9 / 11.8, 32 x 520 x 16384 18.5 / 13.6, 32 x 2048 x 16384 19.5 / 15.0,
    // 64 x 4096 x 4096 9.7 / 11.9, 64 x 5120 x 5120 11.9 / 15.4, 64 x 4096 x 11008 20.2 / 18.9, 64 x 2048 x 8192 15.0 / 12.7)
    const bool stream_bytes = k->family == FAMILY_SKINNY && k->variant == 8;
    // (the Q4 kernels whose waves stream K on their own, variant 5: from two fifths on; ZP 8 x 2048 x 8192 on 128 tiles
    // 8.8 us against 10.2, 16 x 1024 x 16384 on 64 tiles 15.0 / 11.3)
    const bool stream_dp =
        k->family == FAMILY_SKINNY &&
        (stream_bytes ? k->bm == 16 || total64 >= num_cus || out->iters_per_tile * (num_cus - total64) <= 8 * num_cus
         : k->variant == 5 ? total64 * 5 >= (int64_t)num_cus * 2
                         : (k->variant == 4 || k->dtype == SK_Q4) && k->max_m >= 16 &&
                               (k->bm == 16 || (k->variant == 4 && k->dtype != SK_Q4 && !(k->bm == 64 && k->bn == 32))) &&
                               total64 * 5 >= (int64_t)num_cus * (k->variant == 4 && k->dtype != SK_Q4 ? 2 : 3));
    const bool q4_gemv = k->family == FAMILY_SKINNY && k->variant == 2 && k->max_m == 1 &&
                         (k->dtype == SK_Q4 || k->dtype == SK_Q4_ZP || k->dtype == SK_Q4_TILED || k->dtype == SK_Q4_ZP_TILED);
    if ((total64 >= num_cus || stream_dp) && total64 <= max_grid) {
      grid = (int)total64;  // one tile per CTA, all resident: a single data-parallel wave
    } else if (q4_gemv && total64 > max_grid) {
      // more tiles than resident CTAs: as few CTAs as finish in the same number of rounds, so that every CTA walks
      // (nearly) the same number of tiles -- a CTA's later tiles find their first loads in flight (mac_tiles)
      grid = (int)cdiv(total64, cdiv(total64, max_grid));
    } else if (total64 < num_cus) {
      // fewer tiles than CUs: one CTA per CU, but a split tile keeps at least 4 K-iterations per CTA
      // and there are never fewer CTAs than tiles
      int64_t want = iters / 4 < num_cus ? iters / 4 : num_cus;
      if (want < total64) want = total64;
      grid = (int)(want > 8 && want != total64 ? want / 8 * 8 : want);
      // (nor by the rounding, where nothing is split: 8 CTAs for 9 tiles took fp8 18 x 264 x 3072 7.6 us, 9 4.1)
      if (sched == SK_SCHED_DP && grid < total64) grid = (int)total64;
      if (grid > max_grid) grid = max_grid;
    }
  }
  if (sched == SK_SCHED_SPLIT_K) {
    // fixed split: the grid follows from the split factor, a caller's grid is not consulted
    const int ipt = out->iters_per_tile;
    int split = cfg ? cfg->reserved[1] : 0;
    if (split < 0) return SK_ERR_CONFIG;
    if (split == 0) {
      split = 1;
      for (int s = 2; s <= ipt / 4 && total64 * s <= max_grid; ++s)
        if (ipt % s == 0) split = s;
    }
    if (ipt % split != 0 || total64 * split > max_grid) return SK_ERR_CONFIG;
    grid = (int)(total64 * split);
  }
  int auto_interleave = 0;  // the automatic schedule asks for the interleaved order of its Stream-K tiles
  if (sched == SK_SCHED_AUTO) {
    // data-parallel when the last wave of tiles is (nearly) full: Stream-K's fix-up and the L2
    // reuse it gives up cost more than a tail of under 10 %.  Otherwise Stream-K, splitting only
    // the remainder tiles when there are at least two full waves beside them.
    const int64_t waves = (total64 + grid - 1) / grid;
    if (total64 * 10 >= waves * grid * 9) sched = SK_SCHED_DP;
    else sched = total64 >= 2 * (int64_t)grid ? SK_SCHED_SK_ONE_TILE : SK_SCHED_SK_TWO_TILE;
    // (the kernels that stream the weights through LDS are bound by memory, not by the busiest CU: an uneven last
    // wave costs them less than the fix-up; 16 x 28672 x 8192: 77.8 us data-parallel against 83.6 us.  With 64 rows of
    // A on 64 x 32 tiles it is the other way round, 110 us against 103 us; on 64 x 64 tiles 91.5 against 92.6)
    if (k->family == FAMILY_SKINNY && k->variant >= 4 && (k->bm == 16 || k->bn == 64) && total64 >= grid) sched = SK_SCHED_DP;
    // (the same for the Q4 matrix-vector kernels: 1 x 28672 x 8192 on 1792 tiles 28.0 us data-parallel against 31.2 us,
    // 1 x 14336 x 4096 with K split over four waves 10.8 against 16.1)
    if (k->family == FAMILY_SKINNY && k->variant == 2 && k->max_m == 1 && total64 >= grid &&
        (k->dtype == SK_Q4 || k->dtype == SK_Q4_ZP || k->dtype == SK_Q4_TILED || k->dtype == SK_Q4_ZP_TILED))
      sched = SK_SCHED_DP;
    if (k->family == FAMILY_TILE && sched != SK_SCHED_DP) {
      // Fewer tiles than CUs: the idle CUs are put to work by an aligned split in two or four, never by CTA ranges
      // that start anywhere.  More tiles than CTAs: see
      // auto_tile_schedule.
      if (total64 < num_cus && !(cfg && cfg->grid > 0)) {
        const int ipt = out->iters_per_tile, max_split = 4;
        int split = 1;
        for (int s = 2; s <= max_split && total64 * s <= max_grid; s *= 2)
          if (ipt % s == 0 && ipt / s >= 8) split = s;
        sched = split > 1 ? SK_SCHED_SPLIT_K : SK_SCHED_DP;
        grid = split > 1 ? (int)(total64 * split) : grid;
      } else {
        int skt;
        sched = auto_tile_schedule(total64, grid, out->iters_per_tile, &skt, occ == 1 && k->bm == 256 && k->bn == 256 ? &auto_interleave : nullptr);  // (measured on these)
      }
    }
  }
  // a data-parallel-only launch never has more CTAs than tiles (idle CTAs would also skew the
  // CTA -> XCD mapping: the low logical ids sit on the first XCDs)
  if (sched == SK_SCHED_DP && grid > total) grid = total;
  int sk_tiles;
  switch (sched) {
    case SK_SCHED_DP: sk_tiles = 0; break;
    case SK_SCHED_SK_TWO_TILE:  // streamk_fp32.py:37-43
      sk_tiles = total % grid;
      if (total - sk_tiles > grid) sk_tiles += grid;
      break;
    case SK_SCHED_SK_ONE_TILE: sk_tiles = total % grid; break;
    case SK_SCHED_SK_BASIC: sk_tiles = total; break;
    case SK_SCHED_SPLIT_K: sk_tiles = grid == total ? 0 : total; break;  // split 1 is data-parallel
    default: return SK_ERR_CONFIG;
  }
  out->schedule = sched;
  out->grid = grid;
  out->streamk_tiles = sk_tiles;
  out->blocking_tiles = total - sk_tiles;
  out->streamk_iters = sk_tiles * out->iters_per_tile;
  out->streamk_full_tiles = out->streamk_iters / grid;
  out->streamk_partial_tiles = out->streamk_iters % grid;
  out->dp_waves = (int32_t)cdiv(out->blocking_tiles, grid);
  int fixup = cfg ? cfg->fixup : SK_FIXUP_AUTO;
  if (fixup == SK_FIXUP_AUTO) fixup = SK_FIXUP_REDUCE;
  if (fixup != SK_FIXUP_ATOMIC && fixup != SK_FIXUP_REDUCE && fixup != SK_FIXUP_ATOMIC_C && fixup != SK_FIXUP_REDUCE16)
    return SK_ERR_CONFIG;
  // partial sums exchanged in 16 bits: the assembly-loop kernels for fp16 / bfloat16, every Stream-K tile cut into two
  // or four equal segments (what the device side's exchange of half tiles handles)
  if (fixup == SK_FIXUP_REDUCE16 &&
      !(k->family == FAMILY_TILE && k->variant == 7 && (dtype == SK_F16 || dtype == SK_BF16) && sk_tiles > 0 &&
        out->streamk_partial_tiles == 0 &&
        (2 * out->streamk_full_tiles == out->iters_per_tile || 4 * out->streamk_full_tiles == out->iters_per_tile)))
    return SK_ERR_CONFIG;
  // packed 16-bit atomics into C: the 16-bit tile kernels with 16x16 accumulator blocks
  if (fixup == SK_FIXUP_ATOMIC_C &&
      !(k->family == FAMILY_TILE && (k->variant == 4 || k->variant == 5 || k->variant == 7) &&
        (dtype == SK_F16 || dtype == SK_BF16) && N % 2 == 0))
    return SK_ERR_CONFIG;
  out->fixup = fixup;
  out->spin_limit = cfg && cfg->spin_limit > 0 ? cfg->spin_limit : (1 << 22);
  out->interleave = 0;
  if (cfg && cfg->reserved[2] != 0 && cfg->reserved[2] != 1) return SK_ERR_CONFIG;
  if ((cfg && cfg->reserved[2] == 1) || auto_interleave) {
    int g = sk_tiles, b = grid;  // gcd
    while (b) { const int t = g % b; g = b; b = t; }
    if (sk_tiles > 0 && g > 1 && sk_tiles / g > 1) out->interleave = sk_tiles / g;
  }
  out->raster = cfg ? cfg->raster : 0;
  if (out->raster < 0) return SK_ERR_CONFIG;
  // default tile order of the LDS-tiled 16-bit and fp8 kernels: groups of 8 tile rows.  Concurrent CTAs
  // then share B tiles as well as A tiles in the L2s: 0-20 % faster than row-major order on every shape
  // measured (no effect on the fp32 kernels, which keep the reference's order).
  if (out->raster == 0 && k->family == FAMILY_TILE && dtype != SK_F32 && out->num_block_m > 1) {
    out->raster = 8;
    // (wave-K tiles, more than eight rows of them: groups alike.  The tiles of a short last group share little with each other and
    // read the weights once more than they need: bf16 277 x 1792 x 15616 on nine rows of 32 x 64 tiles, 8 + 1 rows 52.2 us from the
    // cache and 52.8 from HBM, 5 + 4 37.5 and 48.1; 530 x 1792 x 4096, nine of 64 x 64, 18.4 / 18.2 and 15.5 / 17.6; 600 x 1536 x 8192,
    // ten of them, 26.2 / 29.0 and 25.2 / 28.5)
    if (k->variant == 10 && out->num_block_m > 8) out->raster = (int)cdiv(out->num_block_m, cdiv(out->num_block_m, 8));
  }

  // workspace: status block, fixed-size flag area, fp32 partial tiles
  int64_t ws = 0;
  // (CTA ranges that are whole tiles -- e.g. `basic` on a tile count that is a multiple of the grid, which only
  // changes which tiles a CTA takes -- never reach the fix-up: no workspace)
  const bool whole_tiles = out->streamk_partial_tiles == 0 && out->streamk_full_tiles % out->iters_per_tile == 0;
  if (sk_tiles > 0 && fixup != SK_FIXUP_ATOMIC_C && !whole_tiles) {
    const int64_t nflags = (fixup == SK_FIXUP_REDUCE || fixup == SK_FIXUP_REDUCE16) ? grid : sk_tiles;
    if (nflags > WS_MAX_FLAGS) return SK_ERR_CONFIG;
    ws = WS_PART_OFF + nflags * (int64_t)k->partial_elems * 4;
  }
  out->workspace_bytes = ws;
  return SK_OK;
}

extern "C" int sk_plan_cta_range(const sk_plan *p, int pid, int32_t *start, int32_t *last) {
  if (!p || !start || !last) return SK_ERR_NULL;
  if (pid < 0 || pid >= p->grid) return SK_ERR_CONFIG;
  const int full = p->streamk_full_tiles, part = p->streamk_partial_tiles;
  *start = pid * full + (pid < part ? pid : part);              // streamk_fp32.py:93
  *last = (pid + 1) * full + (pid + 1 < part ? pid + 1 : part);  // streamk_fp32.py:94-96
  return SK_OK;
}

extern "C" int sk_plan_tile_coords(const sk_plan *p, int tile, int32_t *pid_m, int32_t *pid_n) {
  if (!p || !pid_m || !pid_n) return SK_ERR_NULL;
  if (tile < 0 || tile >= p->total_tiles) return SK_ERR_CONFIG;
  if (p->interleave > 1 && tile < p->streamk_tiles)
    tile = (tile % p->interleave) * (p->streamk_tiles / p->interleave) + tile / p->interleave;
  if (p->raster <= 0) {  // streamk_fp32.py:106-107
    *pid_m = tile / p->num_block_n;
    *pid_n = tile % p->num_block_n;
  } else {  // triton_impl.py:14-28
    const int width = p->raster * p->num_block_n;
    const int group = tile / width;
    const int first_m = group * p->raster;
    const int gsize = p->num_block_m - first_m < p->raster ? p->num_block_m - first_m : p->raster;
    const int r = tile - group * width;
    *pid_m = first_m + r % gsize;
    *pid_n = r / gsize;
  }
  return SK_OK;
}

extern "C" size_t sk_workspace_bytes(const sk_plan *p) { return p ? (size_t)p->workspace_bytes : 0; }
