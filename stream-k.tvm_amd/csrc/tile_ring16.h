// 65 to 128 rows of fp16 / bfloat16 against weights [N, K] (NT): tiles of BM rows, operands through direct-to-LDS rings of
// different depths.
//
// With this many rows the weights still come from HBM once and A, small enough for the L2s, again and again: a CU has to
// have about 60 KB of weights on their way to keep HBM busy, but only one or two iterations of A.  One ring of whole
// stages spends two thirds of its LDS on A; here the weights have WD slots and A has AD.
//
//  * An iteration is 64 K-values: LDS rows of 128 bytes, piece p (16 bytes) of row r at position p ^ ((r >> 1) & 7).
//    Loads are issued in the order A(t + AD - 1), B(t + WD - 1) in iteration t and complete in that order; one wait
//    (vmcnt) and one barrier per iteration, as in tile_stream_pairs.h.
//  * WM x WN waves of 16x16x32 MFMAs, times KH = 2: two waves share the two K-steps of an iteration (their sums are added
//    through LDS at the end of the segment), which keeps two waves on a SIMD without more fragment reads.
//  * Partial tiles travel with device-scope accesses, the owner of a tile adds them up.
//
// What bounds it: a CU gets 30 to 65 GB/s of A and weights together, where its direct loads reach 107 GB/s on rows of 128
// bytes in the L2 and 25 on every CU at once from HBM (profiles/lds_direct_load_rate.md), so neither limit is met: the waves
// wait (two fifths of their cycles for a counter or the barrier, profiles/ring_bf16_M100_N11008_K4096.md) on iterations that
// start with the slowest wave's loads, and widths that are no multiple of the CUs leave some idle.  The depths of the rings do
// not matter much (128 x 64 tiles: 12 + 3, 9 + 5 and 7 + 6 slots within 2 % of each other; 128 K-values per iteration with
// four waves per K sub-block 6 % slower; all tiles starting at the same K no faster).  Weights from HBM, bfloat16, 100 rows,
// the four-stage tile kernels -> these: 4096 x 11008 41.9 -> 33.5 us, 28672 x 8192 135 -> 99 (4.7 TB/s), 2048 x 8192
// 29.2 -> 21.8, 5120 x 5120 35.0 -> 28.1, 11008 x 4096 36.7 -> 33.0; with bias and GELU 44.0 -> 36.6, 140 -> 108,
// 31.3 -> 25.3, 36.9 -> 31.0, 39.9 -> 39.1.  128 x 32 tiles are not built (11008 x 4096 57 us).
#pragma once
#include <type_traits>

#include "sk_device.h"
#include "tile_f16.h"

namespace sk {

template <int BM_, int BN_, int BK_, int WM_, int WN_, int KH_, int WD_, int AD_, bool BF16_>
struct TileRing16 {
  typedef GemmArgs Args;
  static constexpr bool LEAN_ENTRY = true;            // see run_persistent
  static constexpr bool COHERENT_PARTIALS = true;
  static constexpr bool FIXUP_WORD_IN_LDS = true;     // the rings are dead between two calls of mac
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, KH = KH_, WD = WD_, AD = AD_, BK = BK_;
  static constexpr int WAVES = WM * WN * KH, NT = 64 * WAVES, FM = BM / (WM * 16), FN = BN / (WN * 16), STEPS = BK / 32 / KH;
  static_assert(BM % (WM * 16) == 0 && BN % (WN * 16) == 0 && STEPS * KH * 32 == BK && (BK == 64 || BK == 128), "tile shape");
  static constexpr int ROW = BK * 2, PR = BK / 8, ROWS_PER_LOAD = 1024 / ROW;   // bytes and 16-byte pieces of an LDS row
  static constexpr int A_SLOT = BM * ROW, B_SLOT = BN * ROW, LDS_B = WD * B_SLOT, LDS_BYTES = LDS_B + AD * A_SLOT, LDS_TOTAL = LDS_BYTES;
  static constexpr int LA = A_SLOT / 1024 / WAVES, LB = B_SLOT / 1024 / WAVES;   // wave-wide loads per wave and iteration
  static_assert(LA * WAVES * 1024 == A_SLOT && LB * WAVES * 1024 == B_SLOT, "the loads are shared out evenly");
  static_assert(WD > AD && AD >= 2 && LDS_BYTES <= 160 * 1024, "rings");
  static_assert((KH - 1) * WM * WN * FM * FN * 1024 <= LDS_BYTES, "the sums pass through the rings");
  static constexpr int CTAS_PER_CU = 1, WAVES_PER_EU = WAVES / 4;
  static constexpr int NTP = WM * WN * 64, NV4 = FM * FN, TILE_ELEMS = BM * BN;
  static constexpr int OUTSTANDING = LB + (AD - 2) * (LA + LB);

  // c[i][j][e] = C[pm*BM + (wm*FM + i)*16 + lane%16][pn*BN + (wn*FN + j)*16 + 4*(lane/16) + e], in the kh == 0 waves
  struct Acc {
    floatx4 c[FM][FN];
  };

  static __device__ __forceinline__ int swizzle(int row) { return PR == 8 ? (row >> 1) & 7 : row & 15; }

  static __device__ __forceinline__ void mac(const Args &a, Acc &acc, int pm, int pn, int k0, int n, char *smem) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wm = wave % WM, wn = (wave / WM) % WN, kh = wave / (WM * WN);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc.c[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    // ---- descriptors: rows past M / N read as zero ----
    const uint32_t lda_bytes = (uint32_t)a.lda * 2, ldb_bytes = (uint32_t)a.ldb * 2;
    const uint4v rsrc_a = uniform_rsrc(make_rsrc_words(a.A + (int64_t)pm * BM * a.lda, (uint32_t)min(BM, a.M - pm * BM) * lda_bytes));
    const uint4v rsrc_b = uniform_rsrc(make_rsrc_words(a.B + (int64_t)pn * BN * a.ldb, (uint32_t)min(BN, a.N - pn * BN) * ldb_bytes));
    // load G of a slot: ROWS_PER_LOAD rows from ROWS_PER_LOAD G on, lane l writes position l % PR of row l / PR of them
    uint32_t off_a[LA], off_b[LB];
    int ka[LA], kb[LB];
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      const int row = (wave * LA + j) * ROWS_PER_LOAD + lane / PR, piece = (lane % PR) ^ swizzle(row);
      off_a[j] = (uint32_t)row * lda_bytes + (uint32_t)piece * 16;
      ka[j] = piece * 8;
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const int row = (wave * LB + j) * ROWS_PER_LOAD + lane / PR, piece = (lane % PR) ^ swizzle(row);
      off_b[j] = (uint32_t)row * ldb_bytes + (uint32_t)piece * 16;
      kb[j] = piece * 8;
    }
    const int rot = a.M <= BM ? rotation_of(pn, n) : 0;   // one row of tiles: see rotation_of
    const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_address(smem));
    // iterations past the segment and pieces past K fetch nothing (zeros arrive, the wait counts stay exact)
    auto issue_a = [&](int t, int slot) {
      const int kk = t < n ? (k0 + rotated_iteration(t, rot, n)) * BK : 0, left = t < n ? a.K - kk : 0;
      const uint32_t kbytes = (uint32_t)__builtin_amdgcn_readfirstlane(kk * 2), dst = base + (uint32_t)(LDS_B + slot * A_SLOT);
#pragma unroll
      for (int j = 0; j < LA; ++j) dma_load_16(rsrc_a, dst + (uint32_t)(wave * LA + j) * 1024, ka[j] < left ? off_a[j] : OOB_OFFSET, kbytes);
    };
    auto issue_b = [&](int t, int slot) {
      const int kk = t < n ? (k0 + rotated_iteration(t, rot, n)) * BK : 0, left = t < n ? a.K - kk : 0;
      const uint32_t kbytes = (uint32_t)__builtin_amdgcn_readfirstlane(kk * 2), dst = base + (uint32_t)(slot * B_SLOT);
#pragma unroll
      for (int j = 0; j < LB; ++j) dma_load_16(rsrc_b, dst + (uint32_t)(wave * LB + j) * 1024, kb[j] < left ? off_b[j] : OOB_OFFSET, kbytes);
    };
    // fragments: lane (i, g) takes piece 4 s + g of its row for K-step s
    const int fi = lane & 15, fg = lane >> 4;
    int rd[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) rd[s] = fi * ROW + ((4 * (kh * STEPS + s) + fg) ^ swizzle(fi)) * 16;
    const char *b_rd = smem + wn * FN * 16 * ROW, *a_rd = smem + LDS_B + wm * FM * 16 * ROW;
    // what the iterations -(WD - 1) .. -1 would have issued
#pragma unroll
    for (int j = 1 - WD; j < 0; ++j) {
      if (j + AD - 1 >= 0) issue_a(j + AD - 1, j + AD - 1);
      issue_b(j + WD - 1, j + WD - 1);
    }
    int bs = 0, as = 0;   // slots of iteration t: t % WD, t % AD
    for (int t = 0; t < n; ++t) {   // (n is the same for every wave of the CTA: the barriers stay matched)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(OUTSTANDING) : "memory");
      __syncthreads();   // everybody's loads of the iteration have landed; everybody has read the slots refilled next
      issue_a(t + AD - 1, as == 0 ? AD - 1 : as - 1);
      issue_b(t + WD - 1, bs == 0 ? WD - 1 : bs - 1);
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        half8v fa[FM], fb[FN];
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[j] = *reinterpret_cast<const half8v *>(b_rd + bs * B_SLOT + rd[s] + j * 16 * ROW);
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[i] = *reinterpret_cast<const half8v *>(a_rd + as * A_SLOT + rd[s] + i * 16 * ROW);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            if constexpr (BF16_) {
              typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
              acc.c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fb[j]), __builtin_bit_cast(bf16x8, fa[i]),
                                                                    acc.c[i][j], 0, 0, 0);
            } else {
              acc.c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[j], fa[i], acc.c[i][j], 0, 0, 0);
            }
          }
      }
      // the fragments are in registers before the next barrier hands the slots back to the loads
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      bs = bs + 1 == WD ? 0 : bs + 1;
      as = as + 1 == AD ? 0 : as + 1;
    }
    // the loads still in flight (they fetch nothing) write LDS: let them land before the rings are reused
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if constexpr (KH > 1) {   // the kh == 0 waves take the sums of their partners
      floatx4 *red = reinterpret_cast<floatx4 *>(smem) + lane;
      if (kh > 0) {
#pragma unroll
        for (int v = 0; v < NV4; ++v) red[((wave - WM * WN) * NV4 + v) * 64] = acc.c[v / FN][v % FN];
      }
      __syncthreads();
      if (kh == 0) {
#pragma unroll
        for (int h = 0; h < KH - 1; ++h)
#pragma unroll
          for (int v = 0; v < NV4; ++v) acc.c[v / FN][v % FN] += red[((h * WM * WN + wave) * NV4 + v) * 64];
      }
      __syncthreads();
    }
  }

  // (two copies behind one uniform branch: the epilogue without a bias carries none of its code)
  static __device__ __forceinline__ void store_c(const Args &a, const Acc &acc, int pm, int pn, char *, const void *bias) {
    if (bias == nullptr)
      store_c_impl<false>(a, acc, pm, pn, nullptr);
    else
      store_c_impl<true>(a, acc, pm, pn, bias);
  }
  template <bool BIAS>
  static __device__ __forceinline__ void store_c_impl(const Args &a, const Acc &acc, int pm, int pn, const void *epi) {
    const half_t *bias = BIAS ? epi_bias(epi) : nullptr;
    const int act = BIAS ? epi_act(epi) : 0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (wave >= WM * WN) return;
    const int wm = wave % WM, wn = wave / WM;
    const bool vec_ok = (a.ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(a.C) & 7) == 0);
    // (the bias once per column block, all loads at once: fetched per element it cost 7 us at 100 x 11008 x 4096, so 2 to 3)
    float bcol[FN][4];
    if constexpr (BIAS) {
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int col = pn * BN + (wn * FN + j) * 16 + 4 * (lane >> 4) + e;
          bcol[j][e] = bias_at<BF16_>(bias, min(col, a.N - 1), a.N);
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = pm * BM + (wm * FM + i) * 16 + (lane & 15);
      if (row >= a.M) continue;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = pn * BN + (wn * FN + j) * 16 + 4 * (lane >> 4);
        if (col >= a.N) continue;
        half4v h;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float x = acc.c[i][j][e];
          if constexpr (BIAS) x = activate(x + bcol[j][e], act);
          if constexpr (BF16_) {
            const __bf16 b = (__bf16)x;
            h[e] = __builtin_bit_cast(half_t, b);  // C carries 16-bit patterns
          } else {
            h[e] = (half_t)x;
          }
        }
        half_t *dst = a.C + (int64_t)row * a.ldc + col;
        if (vec_ok && col + 4 <= a.N) {
          *reinterpret_cast<half4v *>(dst) = h;
        } else {
          for (int e = 0; e < 4 && col + e < a.N; ++e) dst[e] = h[e];
        }
      }
    }
  }

  // Partial tiles: block v = i FN + j of thread t (one of the NTP threads of the kh == 0 waves) at (v NTP + t) 4; the
  // accumulating form keeps element e of it at (v 4 + e) NTP + t.
  static __device__ __forceinline__ void store_partial(const Acc &acc, float *dst) {
    if (threadIdx.x >= NTP) return;
    const BufferRsrc r = make_rsrc(dst, TILE_ELEMS * 4);
#pragma unroll
    for (int v = 0; v < NV4; ++v) st_coherent16(r, threadIdx.x * 16, v * NTP * 16, __builtin_bit_cast(uint4v, acc.c[v / FN][v % FN]));
  }
  static __device__ __forceinline__ void add_partial(Acc &acc, const float *src) {
    if (threadIdx.x >= NTP) return;
    const BufferRsrc r = make_rsrc(src, TILE_ELEMS * 4);
    floatx4 x[NV4];
#pragma unroll
    for (int v = 0; v < NV4; ++v) x[v] = __builtin_bit_cast(floatx4, ld_coherent16(r, threadIdx.x * 16, v * NTP * 16));
#pragma unroll
    for (int v = 0; v < NV4; ++v) acc.c[v / FN][v % FN] += x[v];
  }
  static __device__ __forceinline__ void atomic_partial(const Acc &acc, float *dst) {
    if (threadIdx.x >= NTP) return;
#pragma unroll
    for (int v = 0; v < NV4; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) atomic_add_f32(dst + (size_t)(v * 4 + e) * NTP + threadIdx.x, acc.c[v / FN][v % FN][e]);
  }
  static __device__ __forceinline__ void take_partial(Acc &acc, float *src) {
    if (threadIdx.x >= NTP) return;
#pragma unroll
    for (int v = 0; v < NV4; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float *p = src + (size_t)(v * 4 + e) * NTP + threadIdx.x;
        acc.c[v / FN][v % FN][e] = ld_coherent_scalar(p);
        st_coherent(p, 0.f);
      }
  }
};

}  // namespace sk
