// Up to 16 rows of A against Q4 weights [N, K/2], one zero point for the matrix or one per scale group: every wave
// streams its own share of K through LDS of its own, and the main loop has no barrier.
//
//  * CTA = WAVES waves that split K between them, one 128-wide scale group per wave and iteration, and one more wave that
//    stages the tile's scales in LDS (another one: the zero points), transposed to [group][row], while the others' first
//    loads are on their way.  Every wave multiplies all NB blocks of 16 weight rows of the tile with its K-values; the sums are added
//    through LDS when the segment ends (the reference's "block reduction", streamk_fp16_block_reduce.py:45,235-306).
//  * A ring of S slots per wave, private to it: NB KB of weights (16 rows x 64 bytes per block, one direct-to-LDS load
//    each) and MR rows of A x 256 bytes (four rows per load).  What orders a slot's loads, reads and refill is the wave's
//    own vmcnt / lgkmcnt, so a wave never waits for another one's loads; WAVES * S * (NB + MR / 4) KB are in flight per
//    CTA, which for the sizes of a model's layers is most of what a CU reads at all.
//  * A load of weights reads 64 contiguous bytes of 16 rows, four lanes of a row side by side (one row per lane, the MFMA's
//    own order, streams 1.8 times slower, see tile_gemv_q4.h); piece p of row r is kept at position p ^ (r / 4) of the row,
//    piece p of a row of A at p ^ row: the 16 lanes served together then read 16 different bank groups.  Rows of A beyond
//    the MR staged ones repeat them: they only reach rows of the result that are not stored.  TILED_: the weights come in
//    tiles of 16 rows x 64 bytes (see tile_skinny.h), a load then reads one of them; everything else is the same.
//  * The nibbles become the exact integers q - zero (1024 + q and 64 + q minus 1024 + zero and 64 + zero in fp16).  With
//    one zero point for the matrix they go into the MFMA as they are and the group's scale multiplies the fp32 group sum,
//    so no weight is rounded.  With per-group zero points (ZP_) the contract for more than one row is the rounded weights
//    bit for bit -- what the dequantiser and the kernels for more rows give, blocks of one call among them: they are
//    multiplied by the scale in fp16 first and the sums run on in the accumulators.
//
// What bounds it: launch, arguments and the first trip to memory are about 4 us, then the weights stream; with zero points
// 4 x 11008 x 4096 takes 11.5 us (11.1 with unrounded weights; of these 9.0 without the decode and the MFMAs, 11.0 without
// the loads of A; one row: 7.2).  Weights from HBM, in us, the kernels that ran these shapes before (tile_skinny.h, with a
// zero point for the matrix tile_stream_q4.h) -> these: per-group zero points 4 x 11008 x 4096 16.9 -> 11.5,
// 4 x 4096 x 11008 18.4 -> 10.6, 16 x 4096 x 4096 9.3 -> 7.3, 16 x 14336 x 4096 20.9 -> 12.9, 16 x 16384 x 16384 52 -> 47;
// one zero point 4 x 4096 x 11008 15.3 -> 10.2, 4 x 4096 x 4096 6.9 -> 6.2, 8 x 2048 x 8192 11.1 -> 7.9,
// 8 x 16384 x 16384 40.0 -> 36.7.  Counters: profiles/rows_q4zp_M4_N11008_K4096.md.
// (Sixteen waves do not fit a workgroup beside the staging ones; twelve with 64 weight rows 11.8 against 12.0, eight
// slots instead of four for 16 weight rows 12.8 against 11.9 at 4 x 4096 x 11008.)
//
// Epilogue, partial tiles and fix-ups are those of tile_stream_pairs.h (wave j holds the sums of block j).
// Replaces the reference's decode-then-MMA step (streamk_fp16_ladder_block_reduce_q4.py:283-294).
#pragma once
#include "q4_dequant.h"
#include "tile_stream_pairs.h"

namespace sk {

template <int MR_, int NB_, int S_, bool ZP_, int GROUPS_MAX_, bool TILED_ = false>
struct TileRowsQ4 : TileStreamPairs<1, 1, NB_, 1, 3, false> {
  typedef TileStreamPairs<1, 1, NB_, 1, 3, false> Base;
  typedef typename Base::Args Args;
  typedef typename Base::Acc Acc;
  typedef typename Base::AccV AccV;
  static constexpr bool ZP_ARGS = ZP_;
  static constexpr int MR = MR_, NB = NB_, S = S_, WAVES = 8, STAGERS = ZP_ ? 2 : 1, NT = 64 * (WAVES + STAGERS);
  static constexpr int BM = 16, BN = 16 * NB, MAX_M = MR;
  static constexpr int BKC = 128 * WAVES, MAX_ITERS = GROUPS_MAX_ / WAVES, GROUPS_MAX = MAX_ITERS * WAVES;
  static constexpr int W_BYTES = NB * 1024, A_BYTES = MR * 256, SLOT = W_BYTES + A_BYTES, RING = S * SLOT;
  static constexpr int LDS_RINGS = WAVES * RING, LDS_SC = GROUPS_MAX * BN * 2;
  static constexpr int LDS_BYTES = LDS_RINGS + (ZP_ ? 2 : 1) * LDS_SC, LDS_TOTAL = LDS_BYTES;
  static_assert(MR == 4 || MR == 8 || MR == 16, "rows of A staged: whole loads of four rows");
  static_assert(LDS_BYTES <= 160 * 1024, "the rings must fit the LDS of a CU");
  static_assert(WAVES * NB * 1024 <= LDS_RINGS && NB <= WAVES, "the waves' sums pass through the rings");
  static constexpr int CTAS_PER_CU_LDS = (160 * 1024) / (LDS_BYTES + 64), CTAS_PER_CU = CTAS_PER_CU_LDS < 1 ? 1 : (CTAS_PER_CU_LDS > 2 ? 2 : CTAS_PER_CU_LDS);
  static constexpr int WAVES_PER_EU = (CTAS_PER_CU * (WAVES + STAGERS) + 3) / 4;
  static constexpr int TILE_ELEMS = BM * BN, LOADS = NB + MR / 4;

  // an extra wave: scales (or zero points) of groups [g0, g0 + count) of the tile's rows to lds[group - g0][row]
  static __device__ __forceinline__ void stage_groups(half_t *lds, const half_t *tile, int rows, int groups, int g0, int count) {
    const BufferRsrc rsrc = make_rsrc(tile, (uint32_t)(rows * groups * 2));
    const int lane = threadIdx.x & 63, pieces = BN * ((count + 7) >> 3);
    for (int idx0 = 0; idx0 < pieces; idx0 += 64 * 4) {
      uint4v v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {   // eight groups of one row, where they are whole
        const int idx = idx0 + u * 64 + lane, r = idx % BN, c = idx / BN * 8;
        v[u] = buffer_load_16(rsrc, c + 8 <= count ? (uint32_t)(r * groups + g0 + c) * 2 : OOB_OFFSET, 0);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int idx = idx0 + u * 64 + lane, r = idx % BN, c = idx / BN * 8;
        if (c >= count) continue;
        half_t *dst = lds + c * BN + r;
        if (c + 8 <= count) {
          const half8v h = __builtin_bit_cast(half8v, v[u]);
#pragma unroll
          for (int e = 0; e < 8; ++e) dst[e * BN] = h[e];
        } else {
          // (fewer than eight left: one by one -- a 16-byte load could cross the end of the array)
          for (int e = 0; c + e < count; ++e)
            dst[e * BN] = __builtin_bit_cast(half_t, __builtin_amdgcn_raw_buffer_load_b16(rsrc, (uint32_t)(r * groups + g0 + c + e) * 2, 0, 0));
        }
      }
    }
  }

  static __device__ __forceinline__ void mac(const Args &a, Acc &acc, int /*pm: one row of tiles*/, int pn, int k0, int n, char *smem) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    half_t *lds_s = reinterpret_cast<half_t *>(smem + LDS_RINGS), *lds_z = lds_s + GROUPS_MAX * BN;
    const int g0 = k0 * WAVES, rows_w = min(BN, a.N - pn * BN);
    const int fi = lane & 15, fg = lane >> 4;
    AccV part[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) part[j] = AccV{0, 0, 0, 0};

    if (wave >= WAVES) {
      const int count = min(a.groups - g0, n * WAVES);
      const half_t *from = ZP_ && wave > WAVES ? a.zeros : a.scales;
      stage_groups(ZP_ && wave > WAVES ? lds_z : lds_s, from + (int64_t)pn * BN * a.groups, rows_w, a.groups, g0, count);
      __syncthreads();
    } else {
      const uint32_t ldw_bytes = (uint32_t)a.ldw, lda_bytes = (uint32_t)a.lda * 2;
      // (bytes from one block of 16 rows to the next, and from one group to the next)
      const uint32_t block_bytes = TILED_ ? (uint32_t)a.groups * 1024 : 16 * ldw_bytes, group_bytes = TILED_ ? 1024 : 64;
      const uint4v rsrc_w = uniform_rsrc(
          make_rsrc_words(reinterpret_cast<const char *>(a.W) + (int64_t)pn * NB * block_bytes,
                          TILED_ ? (uint32_t)((rows_w + 15) / 16) * block_bytes : (uint32_t)rows_w * ldw_bytes));
      const uint4v rsrc_a = uniform_rsrc(make_rsrc_words(a.A, (uint32_t)min(a.M, MR) * lda_bytes));
      const uint32_t ring = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_address(smem) + (uint32_t)wave * RING));
      const uint32_t voff_w = (uint32_t)(lane >> 2) * (TILED_ ? 64 : ldw_bytes) + 16 * ((lane & 3) ^ (lane >> 4));
      uint32_t voff_a[MR / 4];
#pragma unroll
      for (int j = 0; j < MR / 4; ++j) voff_a[j] = (uint32_t)(4 * j + fg) * lda_bytes + 16 * (fi ^ (4 * j + fg));
      const int rot = rotation_of(pn, n);
      // iteration t of the segment, this wave's group of it (loads past the segment or past K fetch nothing: zeros arrive
      // and the wait counts stay exact)
      auto group_of = [&](int t) { return (k0 + rotated_iteration(t, rot, n)) * WAVES + wave; };
      auto issue = [&](int t, int slot) {
        const int g = group_of(t);
        const bool live = t < n && g < a.groups;
        const uint32_t gl = live ? (uint32_t)g : 0, dst = ring + (uint32_t)slot * SLOT;
#pragma unroll
        for (int j = 0; j < NB; ++j) dma_load_16(rsrc_w, dst + j * 1024, live ? voff_w : OOB_OFFSET, gl * group_bytes + (uint32_t)j * block_bytes);
#pragma unroll
        for (int j = 0; j < MR / 4; ++j) dma_load_16(rsrc_a, dst + W_BYTES + j * 1024, live ? voff_a[j] : OOB_OFFSET, gl * 256);
      };
#pragma unroll
      for (int t = 0; t < S; ++t) issue(t, t);

      // fragments: lane (i, g) takes piece g of weight row i, 32 K-values, and the same K-values of A's row i: pieces
      // 4 g .. 4 g + 3
      const char *w_rd = smem + wave * RING + fi * 64 + 16 * (fg ^ (fi >> 2));
      const char *a_rd[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) a_rd[q] = smem + wave * RING + W_BYTES + (fi % MR) * 256 + 16 * ((4 * fg + q) ^ (fi % MR));
      // scales: of the four weight rows whose sums the lane holds, or of the weight row it decodes (ZP_)
      const half_t *s_rd = lds_s + (ZP_ ? fi : 4 * fg), *z_rd = lds_z + fi;
      Q4Consts qc;
      q4_pin_patterns(qc);
      uint32_t magic_hi = 0x54005400u;   // fp16 64.0: 64 + q for the nibbles at bits 4..7 of a half
      asm volatile("" : "+v"(magic_hi));
      __syncthreads();   // the scales are there

      int slot = 0;
      for (int t = 0; t < n; ++t) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * LOADS) : "memory");
        const int sofs = slot * SLOT;
        uint4v wf[NB];
        half8v fa[4];
#pragma unroll
        for (int j = 0; j < NB; ++j) wf[j] = *reinterpret_cast<const uint4v *>(w_rd + sofs + j * 1024);
#pragma unroll
        for (int q = 0; q < 4; ++q) fa[q] = *reinterpret_cast<const half8v *>(a_rd[q] + sofs);
        const int g = group_of(t), gs = min(g, a.groups - 1) - g0;   // (a wave without a group reads zeros and any scale)
        half4v sc[NB];
        half_t z[NB], s[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          if constexpr (ZP_) {
            s[j] = s_rd[gs * BN + 16 * j];
            z[j] = z_rd[gs * BN + 16 * j];
          } else {
            sc[j] = *reinterpret_cast<const half4v *>(s_rd + gs * BN + 16 * j);
          }
        }
        // the slot is read: refill it
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(t + S, slot);
        if (g < a.groups) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {   // element order 0,4,1,5,2,6,3,7
            const uint4v v = __builtin_bit_cast(uint4v, fa[q]);
            uint4v p;
            p[0] = __builtin_amdgcn_perm(v[2], v[0], 0x05040100u);
            p[1] = __builtin_amdgcn_perm(v[2], v[0], 0x07060302u);
            p[2] = __builtin_amdgcn_perm(v[3], v[1], 0x05040100u);
            p[3] = __builtin_amdgcn_perm(v[3], v[1], 0x07060302u);
            fa[q] = __builtin_bit_cast(half8v, p);
          }
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            const half_t zero = ZP_ ? z[j] : (half_t)(float)a.zero;
            const half_t lo = (half_t)1024.f + zero, hi = (half_t)64.f + zero;   // exact
            const half2v lo2 = half2v{lo, lo}, hi2 = half2v{hi, hi};
            AccV sum = ZP_ ? part[j] : AccV{0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              union {
                uint32_t u[4];
                half2v h[4];
                half8v v;
              } r;
              const uint32_t w = wf[j][q], t8 = w >> 8;
              r.u[0] = and_or(w, qc.mask_lo, qc.magic);
              r.u[1] = and_or(w, qc.mask_hi, magic_hi);
              r.u[2] = and_or(t8, qc.mask_lo, qc.magic);
              r.u[3] = and_or(t8, qc.mask_hi, magic_hi);
              r.h[0] = r.h[0] - lo2;
              r.h[1] = r.h[1] - hi2;
              r.h[2] = r.h[2] - lo2;
              r.h[3] = r.h[3] - hi2;
              if constexpr (ZP_) {
                const half2v s2 = half2v{s[j], s[j]};
#pragma unroll
                for (int e = 0; e < 4; ++e) r.h[e] = r.h[e] * s2;
              }
              sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(r.v, fa[q], sum, 0, 0, 0);
            }
            if constexpr (ZP_) {
              part[j] = sum;
            } else {
#pragma unroll
              for (int r = 0; r < 4; ++r) part[j][r] = __builtin_fmaf(sum[r], (float)sc[j][r], part[j][r]);
            }
          }
        }
        slot = slot + 1 == S ? 0 : slot + 1;
      }
      // the loads still in flight (they fetch nothing) write LDS: let them land before the rings are reused
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();

    // ---- add up the waves' sums: wave j finishes block j ----
    float *red = reinterpret_cast<float *>(smem);
    if (wave < WAVES) {
#pragma unroll
      for (int j = 0; j < NB; ++j) *reinterpret_cast<AccV *>(red + ((wave * NB + j) * 64 + lane) * 4) = part[j];
    }
    __syncthreads();
    if (wave < NB) {
      AccV sum = AccV{0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < WAVES; ++r) sum += *reinterpret_cast<const AccV *>(red + ((r * NB + wave) * 64 + lane) * 4);
      acc.c[0][0] = sum;
    }
    __syncthreads();
  }
};

}  // namespace sk
