// fp32 tile arithmetic on v_mfma_f32_16x16x4_f32: B as [K,N] (the reference's layout, streamk_fp32.py:74) or [N,K].
// Replaces the T.gemm of the reference's fp32 kernel (streamk_fp32.py:109-125).
//
// An fp32 MFMA takes 32 cycles for 2048 FLOP, so the LDS reads of even a 32 x 32 wave tile are a third of the LDS
// bandwidth: what bounds these kernels is the matrix pipe (157 TFLOP/s) for many rows of A and the stream of B from HBM
// for few.  Both want the same thing, loads far ahead of their use without registers to hold them: a ring of STAGES
// slots of BK K-values of A and B, filled by direct global -> LDS loads (16 bytes per lane), one wait (vmcnt, in order)
// and one barrier per iteration, STAGES - 1 iterations in flight.  Tile shapes differ in how many CTAs a problem gives:
// 128 x 128 where that fills the device, 64 x 64 / 64 x 128 where it does not or M <= 64, 32 x 64 / 32 x 256 for
// M <= 32 (see the planner's kFamiliesF32).  Measured (B [K,N], weights from HBM) against the register-staged two-slot
// kernels this replaced, in us: 16 x 16384 x 8192 120 -> 92 (5.8 TB/s), 16 x 4096 x 4096 59.8 -> 20.7, 64 x 4096 x 4096
// 97 -> 28, 256 x 1024 x 512 23.1 -> 10.0, 512 x 4096 x 4096 163 -> 133, 4096^3 1019 -> 961 (143 TFLOP/s); as [N,K]
// 149 -> 97, 64.8 -> 20.2, 98 -> 28, 23.4 -> 10.8, 167 -> 131, 1061 -> 933 (147 TFLOP/s).  (One device; between devices and
// runs the first varies from 92 to 95, those the matrix pipe bounds by up to 12 %; profiles/f32_M16_N16384_K8192.md.)
//
// LDS layout of a slot: BM rows of A of BK * 4 bytes, then B: [N,K] BN rows like A's, [K,N] BK rows of BN * 4 bytes.
// 16-byte piece p of a row of 4 / 8 / 16 pieces is kept at position p ^ swizzle(row) ((row >> 2) & 3, (row >> 1) & 7,
// row & 15: the 16 lanes served together read 16 rows on distinct banks); piece p of K-row k of a [K,N] stage at
// p ^ 4 ((k >> 2) & 3): the four lane groups of a fragment read, four K-rows apart, fall on the four 64-byte quarters of
// the 64 banks.
//
// Fragments: lane (i = lane % 16, g = lane / 16) takes piece 4 s + g of its row for K-step s of 16, four consecutive
// K-values, and feeds them to four MFMAs: MFMA e contracts K = 16 s + {e, 4 + e, 8 + e, 12 + e}; from a [K,N] stage it reads the
// same four K-values of its column one by one.
#pragma once
#include "sk_device.h"

namespace sk {

struct GemmArgsF32 {
  const float *A;
  const float *B;
  float *C;
  int M, N, K;
  int64_t lda, ldb, ldc;
};

template <bool B_KN_, int BM_, int BN_, int BK_, int WM_, int WN_, int STAGES_, int CTAS_>
struct TileF32 {
  typedef GemmArgsF32 Args;
  static constexpr bool LEAN_ENTRY = true;            // see run_persistent
  static constexpr bool COHERENT_PARTIALS = true;     // partials travel with device-scope accesses
  static constexpr bool FIXUP_WORD_IN_LDS = true;     // the ring is dead between two calls of mac
  static constexpr bool B_KN = B_KN_;
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, S = STAGES_;
  static constexpr int NT = 256, FM = BM / (WM * 16), FN = BN / (WN * 16), STEPS = BK / 16;
  static_assert(WM * WN == 4 && BM % (WM * 16) == 0 && BN % (WN * 16) == 0 && BN % 64 == 0, "tile shape");
  static_assert(BK == 16 || BK == 32 || BK == 64, "rows of 4, 8 or 16 pieces");
  static constexpr int ROW = BK * 4, PR = BK / 4;             // bytes / 16-byte pieces of an LDS row along K
  static constexpr int A_BYTES = BM * ROW, B_BYTES = BN * ROW, SLOT = A_BYTES + B_BYTES;
  static constexpr int NA = A_BYTES / 1024, NB = B_BYTES / 1024;  // wave-wide loads of a slot
  // (a slot of A may hold fewer loads than there are waves: the other waves repeat them, which keeps the counts equal)
  static constexpr int LA = NA >= 4 ? NA / 4 : 1, LB = NB / 4, LOADS = LA + LB;
  static_assert((NA % 4 == 0 || 4 % NA == 0) && NB % 4 == 0, "the loads are shared out evenly");
  static constexpr int LDS_BYTES = S * SLOT, LDS_TOTAL = LDS_BYTES;
  static_assert(LDS_BYTES * CTAS_ <= 160 * 1024, "the rings must fit the LDS of a CU");
  static constexpr int CTAS_PER_CU = CTAS_, WAVES_PER_EU = CTAS_;
  static constexpr int TILE_ELEMS = BM * BN, NV4 = FM * FN;
  static constexpr int OUTSTANDING = (S - 2) * LOADS;

  // c[i][j][e] = C[pm*BM + (wm*FM + i)*16 + lane%16][pn*BN + (wn*FN + j)*16 + 4*(lane/16) + e]
  struct Acc {
    floatx4 c[FM][FN];
  };

  static __device__ __forceinline__ int swizzle(int row) {
    return PR == 4 ? (row >> 2) & 3 : (PR == 8 ? (row >> 1) & 7 : row & 15);
  }

  static __device__ __forceinline__ void mac(const Args &a, Acc &acc, int pm, int pn, int k0, int n, char *smem) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc.c[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // ---- descriptors: rows past M / N and K-rows past K read as zero ----
    const int rows_a = min(BM, a.M - pm * BM), cols_b = min(BN, a.N - pn * BN);
    const uint32_t lda_bytes = (uint32_t)a.lda * 4, ldb_bytes = (uint32_t)a.ldb * 4;
    const uint4v rsrc_a = uniform_rsrc(make_rsrc_words(a.A + (int64_t)pm * BM * a.lda, (uint32_t)rows_a * lda_bytes));
    const uint4v rsrc_b = uniform_rsrc(
        B_KN ? make_rsrc_words(a.B + (int64_t)pn * BN, (uint32_t)(((int64_t)(a.K - 1) * a.ldb + cols_b) * 4))
             : make_rsrc_words(a.B + (int64_t)pn * BN * a.ldb, (uint32_t)cols_b * ldb_bytes));

    // ---- this lane's source of each of its wave's loads: byte offset at K = 0 and its K-values (for the K tail) ----
    uint32_t off_a[LA], off_b[LB];
    int ka[LA], kb[LB];
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      const int x = ((wave * LA + j) % NA) * 64 + lane, row = x / PR, piece = (x % PR) ^ swizzle(row);
      off_a[j] = (uint32_t)row * lda_bytes + (uint32_t)piece * 16;
      ka[j] = piece * 4;
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const int x = (wave * LB + j) * 64 + lane;
      if constexpr (B_KN) {
        const int k = x / (BN / 4), piece = (x % (BN / 4)) ^ (4 * ((k >> 2) & 3));
        off_b[j] = piece * 4 < cols_b ? (uint32_t)k * ldb_bytes + (uint32_t)piece * 16 : OOB_OFFSET;
        kb[j] = 0;   // (K-rows past K lie past the descriptor's end)
      } else {
        const int row = x / PR, piece = (x % PR) ^ swizzle(row);
        off_b[j] = (uint32_t)row * ldb_bytes + (uint32_t)piece * 16;
        kb[j] = piece * 4;
      }
    }
    // one row of tiles over [N,K] weights: every tile starts K at a different offset (see rotation_of)
    const int rot = (!B_KN && a.M <= BM) ? rotation_of(pn, n) : 0;
    const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_address(smem));
    auto issue = [&](int t, int slot) {
      // (past the segment K = 0: the offset of a load that fetches nothing stays at OOB_OFFSET, far past any descriptor)
      const int kk = t < n ? (k0 + rotated_iteration(t, rot, n)) * BK : 0;
      const uint32_t kbytes = (uint32_t)__builtin_amdgcn_readfirstlane(kk * 4);
      const uint32_t kb_bytes = B_KN ? (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)kk * ldb_bytes)) : kbytes;
      const uint32_t dst = base + (uint32_t)(slot * SLOT);
      if (t < n && kk + BK <= a.K) {
#pragma unroll
        for (int j = 0; j < LB; ++j) dma_load_16(rsrc_b, dst + A_BYTES + (uint32_t)(wave * LB + j) * 1024, off_b[j], kb_bytes);
#pragma unroll
        for (int j = 0; j < LA; ++j) dma_load_16(rsrc_a, dst + (uint32_t)((wave * LA + j) % NA) * 1024, off_a[j], kbytes);
      } else {
        // the K tail, and iterations past the segment: nothing is fetched for K-values past the end (zeros arrive)
        const int left = t < n ? a.K - kk : 0;
#pragma unroll
        for (int j = 0; j < LB; ++j)
          dma_load_16(rsrc_b, dst + A_BYTES + (uint32_t)(wave * LB + j) * 1024, kb[j] < left ? off_b[j] : OOB_OFFSET, kb_bytes);
#pragma unroll
        for (int j = 0; j < LA; ++j)
          dma_load_16(rsrc_a, dst + (uint32_t)((wave * LA + j) % NA) * 1024, ka[j] < left ? off_a[j] : OOB_OFFSET, kbytes);
      }
    };

    // ---- fragment addresses ----
    const int fi = lane & 15, fg = lane >> 4;
    int rd_a[STEPS], rd_b[STEPS], rd_bt[FN];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int pos = ((4 * s + fg) ^ swizzle(fi)) * 16;
      rd_a[s] = (wm * FM * 16 + fi) * ROW + pos;
      rd_b[s] = A_BYTES + (wn * FN * 16 + fi) * ROW + pos;
    }
    if constexpr (B_KN) {
#pragma unroll
      for (int j = 0; j < FN; ++j) rd_bt[j] = A_BYTES + (4 * fg * BN + ((16 * (wn * FN + j) + fi) ^ (16 * fg))) * 4;
    }
    auto compute = [&](const char *st, auto rows_active) {
      constexpr int FMA = decltype(rows_active)::value;
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        floatx4 fa[FMA], fb[FN];
#pragma unroll
        for (int i = 0; i < FMA; ++i) fa[i] = *reinterpret_cast<const floatx4 *>(st + rd_a[s] + i * 16 * ROW);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          if constexpr (B_KN) {
#pragma unroll
            for (int e = 0; e < 4; ++e) fb[j][e] = *reinterpret_cast<const float *>(st + rd_bt[j] + (16 * s + e) * BN * 4);
          } else {
            fb[j] = *reinterpret_cast<const floatx4 *>(st + rd_b[s] + j * 16 * ROW);
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < FMA; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              acc.c[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][e], fa[i][e], acc.c[i][j], 0, 0, 0);
      }
    };

#pragma unroll
    for (int j = 0; j < S - 1; ++j) issue(j, j);
    int slot = 0;
    // (M <= 16 on a tile of 32 rows: the second block of rows is left out)
    const bool half = FM == 2 && WM == 1 && a.M <= 16;
    for (int t = 0; t < n; ++t) {   // (n is the same for every wave of the CTA: the barriers stay matched)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(OUTSTANDING) : "memory");
      __syncthreads();   // everybody's loads of the iteration have landed; everybody has read the slot refilled next
      issue(t + S - 1, slot == 0 ? S - 1 : slot - 1);
      const char *st = smem + slot * SLOT;
      if (FM == 2 && WM == 1 && half)
        compute(st, std::integral_constant<int, 1>{});
      else
        compute(st, std::integral_constant<int, FM>{});
      // the fragments are in registers before the next barrier hands the slot back to the loads
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      slot = slot + 1 == S ? 0 : slot + 1;
    }
    // the loads still in flight (they fetch nothing) write LDS: let them land before the ring is reused
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }

  static __device__ __forceinline__ void store_c(const Args &a, const Acc &acc, int pm, int pn, char *,
                                                 const void * /*bias: not offered for fp32*/) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const bool vec_ok = (a.ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(a.C) & 15) == 0);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = pm * BM + (wm * FM + i) * 16 + (lane & 15);
      if (row >= a.M) continue;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = pn * BN + (wn * FN + j) * 16 + 4 * (lane >> 4);
        float *dst = a.C + (int64_t)row * a.ldc + col;
        if (vec_ok && col + 4 <= a.N) {
          *reinterpret_cast<floatx4 *>(dst) = acc.c[i][j];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (col + e < a.N) dst[e] = acc.c[i][j][e];
        }
      }
    }
  }

  // Partial tiles: block v = i FN + j of thread t at (v NT + t) 4; the accumulating form keeps element e of it at
  // (v 4 + e) NT + t.  Every access is of device scope (write-through stores, loads that bypass the XCD's L2): no CTA
  // writes back or invalidates an L2 (128 x 128 tiles split in four used to spend 40 us on that).
  static __device__ __forceinline__ void store_partial(const Acc &acc, float *dst) {
    const BufferRsrc r = make_rsrc(dst, TILE_ELEMS * 4);
#pragma unroll
    for (int v = 0; v < NV4; ++v)
      st_coherent16(r, threadIdx.x * 16, v * NT * 16, __builtin_bit_cast(uint4v, acc.c[v / FN][v % FN]));
  }
  static __device__ __forceinline__ void add_partial(Acc &acc, const float *src) {
    const BufferRsrc r = make_rsrc(src, TILE_ELEMS * 4);
    constexpr int GROUP = NV4 < 16 ? NV4 : 16;   // loads in flight before their sums
#pragma unroll
    for (int v0 = 0; v0 < NV4; v0 += GROUP) {
      floatx4 x[GROUP];
#pragma unroll
      for (int v = 0; v < GROUP; ++v)
        x[v] = __builtin_bit_cast(floatx4, ld_coherent16(r, threadIdx.x * 16, (v0 + v) * NT * 16));
#pragma unroll
      for (int v = 0; v < GROUP; ++v) acc.c[(v0 + v) / FN][(v0 + v) % FN] += x[v];
    }
  }
  static __device__ __forceinline__ void atomic_partial(const Acc &acc, float *dst) {
    dst = pin_here(dst);
#pragma unroll
    for (int v = 0; v < NV4; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) atomic_add_f32(dst + (size_t)(v * 4 + e) * NT + threadIdx.x, acc.c[v / FN][v % FN][e]);
  }
  static __device__ __forceinline__ void take_partial(Acc &acc, float *src) {
    src = pin_here(src);
#pragma unroll
    for (int v = 0; v < NV4; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float *p = src + (size_t)(v * 4 + e) * NT + threadIdx.x;
        acc.c[v / FN][v % FN][e] = ld_coherent_scalar(p);
        st_coherent(p, 0.f);
      }
  }
};

}  // namespace sk
