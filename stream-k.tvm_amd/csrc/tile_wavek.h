// Tiles for a middling number of rows of A (NT): every wave of a CTA multiplies the whole tile with its own share of K.
//
//  * CTA = four waves, one per SIMD.  An iteration is four chunks of 128 bytes of K per row (64 16-bit or 128 one-byte
//    K-values), one per wave.  A wave fetches the BM + BN rows of its chunk straight into a ring of LDS of its own (loads of
//    8 rows x 128 bytes), reads the fragments back, refills what it has read and multiplies.  What orders a ring's loads, reads
//    and refills is the wave's own vmcnt / lgkmcnt: the main loop has no barrier, no wave waits for another one's loads, and
//    the CTA has most of its 160 KB of LDS in flight all the time.  Every fragment is read from LDS once per CTA.
//  * The fragments of a chunk are read beside the MFMAs of the first half of the chunk before, its place is refilled beside those
//    of the second half: a wave that has its SIMD for itself issues one instruction in four cycles, a quarter of an MFMA.
//  * The ring is a ring of loads, R KB long, a chunk being L of them: for tiles whose chunks are larger than 20 KB, R is no
//    multiple of L, and part of the chunk after next is in flight.
//  * When the segment ends every wave puts its sums into its own ring and every thread adds the four waves' values of its share
//    of the tile: pieces of 16 bytes along the rows of C, whose stores fill whole lines.
//
// What bounds it: a CU takes in 60 to 100 GB/s of operands (bf16 100 x 11008 x 4096 60, fp16 256 x 4096 x 4096 88, 1024 x 1024 x 8192
// 100; its direct loads alone 107, profiles/lds_direct_load_rate.md), through LDS or through registers alike, and 3 to 4 us pass
// before and behind the loop.  So it serves what fits one or two rounds of tiles.  Every XCD walks K from a start of its own
// (start_of), because all CTAs of one share A as well as the weights (a start per column of tiles: 2048 x 1024 x 4096 45 us, so 28).
// Graphs of launches, the kernels that such calls took before / these, in us, with three sets of operands in turn and with 600 MB of
// weights in rotation, which come from HBM: fp16 64 x 4096 x 4096 13.5 / 8.5 and 14.9 / 11.7, 128 x 2048 x 2048 13.0 / 5.6 and
// 13.8 / 6.9, 128 x 4096 x 4096 19.0 / 11.8 and 19.4 / 15.2, 256 x 4096 x 4096 21.4 / 15.9 and 28.4 / 19.3, 1024 x 1024 x 8192
// 32.9 / 26.8 and 38.8 / 30.5, 80 x 8192 x 8192 41.2 / 32.8 and 39.4 / 32.7; bf16 100 x 11008 x 4096 with bias and GELU 35.1 / 26.5
// and 36.1 / 27.8; int8 100 x 4096 x 4096 12.6 / 7.3 and 16.9 / 8.7, 128 x 8192 x 8192 21.5 / 16.0 and 30.0 / 21.3; fp8
// 100 x 512 x 8192 17.4 / 7.9 and 25.0 / 8.8, 256 x 1024 x 8192 24.7 / 8.6 and 40.2 / 10.7.
#pragma once
#include <type_traits>

#include "sk_device.h"
#include "tile_f16.h"

namespace sk {

enum WaveKType { WK_F16 = 0, WK_BF16 = 1, WK_F8E4M3 = 2, WK_F8E5M2 = 3, WK_I8 = 4, WK_Q4 = 5, WK_Q4ZP = 6 };

struct WaveKArgs : GemmArgs {
  uint32_t start_scale;   // 2^32 x tiles of a column in a raster group / tiles of a round of the launch, rounded up (start_of)
};
// Q4 weights: with the array of zero points where every group has its own
struct WaveKQ4Args : WaveKArgs {
  const half_t *zeros;
};

// what the kernels of this file share: who holds which block of the tile, the sums over the waves, epilogue, partial tiles
template <int TYPE_, int FM_, int FN_>
struct WaveKTile {
  typedef typename std::conditional<(TYPE_ >= WK_Q4), WaveKQ4Args, WaveKArgs>::type Args;
  static constexpr bool LEAN_ENTRY = true;            // see run_persistent
  static constexpr bool COHERENT_PARTIALS = true;
  static constexpr bool FIXUP_WORD_IN_LDS = true;     // the rings are dead between two calls of mac
  static constexpr int TYPE = TYPE_, FM = FM_, FN = FN_, BM = 16 * FM_, BN = 16 * FN_, WAVES = 4, NT = 256;
  static constexpr int TILE_ELEMS = BM * BN, NB = FM * FN, NQ = NB / WAVES;   // blocks of the tile, of a wave's quarter
  static_assert(NB % WAVES == 0, "the waves share out the blocks evenly");
  static constexpr bool I8 = TYPE_ == WK_I8, BF16 = TYPE_ == WK_BF16, F8 = TYPE_ == WK_F8E4M3 || TYPE_ == WK_F8E5M2;
  typedef int intx4 __attribute__((ext_vector_type(4)));
  typedef typename std::conditional<I8, intx4, floatx4>::type AccV;
  typedef typename std::conditional<I8, int, float>::type AccT;

  // What a thread ends up with: pieces of PW columns of one row, 16 bytes of C where the tile's size allows.  Piece u of thread t is
  // number u NT + t of the tile's, along its rows.
  static constexpr int PV = !I8 && NQ % 2 == 0 ? 2 : 1, PW = 4 * PV, PIECES = NQ / PV, PPR = BN / PW;   // PPR pieces make a row
  struct Acc {
    AccV c[NQ];
    half_t bias __attribute__((ext_vector_type(PW)));   // (prefetch_bias)
  };
  static __device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }
  static __device__ __forceinline__ int piece_row(int u, int tid) { return (int)((unsigned)(u * NT + tid) / (unsigned)PPR); }
  static __device__ __forceinline__ int piece_col(int u, int tid) { return (int)((unsigned)(u * NT + tid) % (unsigned)PPR); }
  static constexpr bool ONE_COL = NT % PPR == 0;        // the thread's pieces stand below each other

  // The iteration of a segment of n that a tile of column pn starts with: the XCDs' starts are spread over the segment, and a tile takes
  // that of the XCD which holds the first tile of its column -- its own XCD's but where a column straddles two, or goes on in another
  // group of rows.  So all tiles of a column add up K in one order: equal rows of A give equal bits, wherever they stand in it.
  // (pn * start_scale: how far the first tile is into its round of the launch, as a fraction of 2^32)
  static __device__ __forceinline__ int start_of(const Args &a, int pn, int n) {
    return (int)((((uint32_t)pn * a.start_scale) >> 29) * (uint32_t)n >> 3);
  }

  // c: the wave's sums of all blocks, lane l of block v holding C[16 (v / FN) + l % 16][16 (v % FN) + 4 (l / 16) + e].  Every wave
  // puts them into its own ring -- row r of a block's 16 at place r ^ key, so that the eight pieces along a row that are read
  // together stand in eight different 16-byte places -- and after one barrier every thread adds the four waves' values of its
  // pieces, (w0 + w1) + (w2 + w3).
  template <int RING>
  static __device__ __forceinline__ void add_waves(const AccV (&c)[NB], Acc &acc, char *smem) {
    static_assert(NB * 1024 <= RING, "a wave's sums fit its ring");
    constexpr int KM = PPR >= 8 ? 1 : (PPR >= 4 ? 2 : 4);
    const int tid = pin_here((int)threadIdx.x), lane = tid & 63;   // (pinned: no address is held through the loop)
    char *mine = smem + wave_id() * RING + (lane >> 4) * 256;
    static_for<0, NB>([&](auto v) {
      constexpr int j = v % FN;
      const int key = ((PV == 2 ? 2 * j + (lane >> 5) : 4 * j + (lane >> 4)) * KM) & 7;
      *reinterpret_cast<AccV *>(mine + v * 1024 + ((lane & 15) ^ key) * 16) = c[v];
    });
    __syncthreads();
    static_for<0, PIECES>([&](auto u) {
      const int row = piece_row(u, tid), p = piece_col(u, tid);
      static_for<0, PV>([&](auto h) {
        const int col4 = p * PV + h;
        const char *from = smem + (((row >> 4) * FN + (col4 >> 2)) * 64 + (col4 & 3) * 16 + ((row & 15) ^ ((p * KM) & 7))) * 16;
        const AccV w0 = *reinterpret_cast<const AccV *>(from), w1 = *reinterpret_cast<const AccV *>(from + RING);
        const AccV w2 = *reinterpret_cast<const AccV *>(from + 2 * RING), w3 = *reinterpret_cast<const AccV *>(from + 3 * RING);
        acc.c[u * PV + h] = (w0 + w1) + (w2 + w3);
      });
    });
    __syncthreads();   // the rings may be filled again
  }

  // The bias of the thread's pieces, requested before the tile's loop: behind it the trip to memory would be waited for.  Whole
  // aligned pieces of one column only; the others are read in the epilogue.
  static __device__ __forceinline__ bool whole_bias(const Args &a, const half_t *bias) {
    return ONE_COL && !I8 && bias != nullptr && a.N % PW == 0 && (reinterpret_cast<uintptr_t>(bias) & (2 * PW - 1)) == 0;
  }
  static __device__ __forceinline__ void prefetch_bias(const Args &a, Acc &acc, int pn, const void *epi) {
    const half_t *bias = epi_bias(epi);
    if (whole_bias(a, bias)) acc.bias = *reinterpret_cast<const decltype(acc.bias) *>(bias + min(pn * BN + piece_col(0, threadIdx.x) * PW, a.N - PW));
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
    const int act = BIAS ? epi_act(epi) : 0, tid = pin_here((int)threadIdx.x);
    typedef half_t HalfP __attribute__((ext_vector_type(PW)));
    const uintptr_t at = reinterpret_cast<uintptr_t>(a.C);
    const bool wide = a.ldc % PW == 0 && (at & (I8 ? 15 : 2 * PW - 1)) == 0, vec_ok = a.ldc % 4 == 0 && (at & (I8 ? 15 : 7)) == 0;
    floatx4 b4[NQ];
    if constexpr (BIAS && !I8) {
      if (whole_bias(a, bias)) {
#pragma unroll
        for (int x = 0; x < PW; ++x) {
          const half_t h = acc.bias[x];
          const float f = BF16 ? __builtin_bit_cast(float, (uint32_t)__builtin_bit_cast(uint16_t, h) << 16) : (float)h;
#pragma unroll
          for (int u = 0; u < PIECES; ++u) b4[u * PV + x / 4][x % 4] = f;
        }
      } else {   // all loads at once
#pragma unroll
        for (int u = 0; u < NQ; ++u) b4[u] = bias4_at<BF16>(bias, pn * BN + piece_col(u / PV, tid) * PW + 4 * (u % PV), a.N);
      }
    }
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
      const int row = pm * BM + piece_row(u, tid), col = pn * BN + piece_col(u, tid) * PW;
      if (row >= a.M || col >= a.N) continue;
      if constexpr (I8) {   // int32 C straight from the accumulators (ldc counts int32 elements)
        int *dst = reinterpret_cast<int *>(a.C) + (int64_t)row * a.ldc + col;
        if (vec_ok && col + 4 <= a.N) {
          *reinterpret_cast<intx4 *>(dst) = acc.c[u];
        } else {
          for (int e = 0; e < 4 && col + e < a.N; ++e) dst[e] = acc.c[u][e];
        }
      } else {
        HalfP h;
#pragma unroll
        for (int e = 0; e < PW; ++e) {
          float x = acc.c[u * PV + e / 4][e % 4];
          if constexpr (F8) x *= a.alpha;
          if constexpr (BIAS) x = activate(x + b4[u * PV + e / 4][e % 4], act);
          if constexpr (BF16) {
            const __bf16 b = (__bf16)x;
            h[e] = __builtin_bit_cast(half_t, b);  // C carries 16-bit patterns
          } else {
            h[e] = (half_t)x;
          }
        }
        half_t *dst = a.C + (int64_t)row * a.ldc + col;
        if (wide && col + PW <= a.N) {
          *reinterpret_cast<HalfP *>(dst) = h;
        } else {
#pragma unroll
          for (int q = 0; q < PW; q += 4) {
            if (vec_ok && col + q + 4 <= a.N) {
              *reinterpret_cast<half4v *>(dst + q) = half4v{h[q], h[q + 1], h[q + 2], h[q + 3]};
            } else {
#pragma unroll
              for (int e = q; e < q + 4; ++e)
                if (col + e < a.N) dst[e] = h[e];
            }
          }
        }
      }
    }
  }

  // Partial tiles: four columns u of thread t at (u NT + t) 4; the accumulating form keeps element e of it at (u 4 + e) NT + t.
  static __device__ __forceinline__ void store_partial(const Acc &acc, float *dst) {
    const BufferRsrc r = make_rsrc(dst, TILE_ELEMS * 4);
#pragma unroll
    for (int u = 0; u < NQ; ++u) st_coherent16(r, threadIdx.x * 16, u * NT * 16, __builtin_bit_cast(uint4v, acc.c[u]));
  }
  static __device__ __forceinline__ void add_partial(Acc &acc, const float *src) {
    const BufferRsrc r = make_rsrc(src, TILE_ELEMS * 4);
    AccV x[NQ];
#pragma unroll
    for (int u = 0; u < NQ; ++u) x[u] = __builtin_bit_cast(AccV, ld_coherent16(r, threadIdx.x * 16, u * NT * 16));
#pragma unroll
    for (int u = 0; u < NQ; ++u) acc.c[u] += x[u];
  }
  static __device__ __forceinline__ void atomic_partial(const Acc &acc, float *dst_) {
    AccT *dst = reinterpret_cast<AccT *>(dst_);
#pragma unroll
    for (int u = 0; u < NQ; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (I8)
          atomic_add_i32(dst + (size_t)(u * 4 + e) * NT + threadIdx.x, acc.c[u][e]);
        else
          atomic_add_f32(dst + (size_t)(u * 4 + e) * NT + threadIdx.x, acc.c[u][e]);
      }
  }
  static __device__ __forceinline__ void take_partial(Acc &acc, float *src_) {
    AccT *src = reinterpret_cast<AccT *>(src_);
#pragma unroll
    for (int u = 0; u < NQ; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        AccT *p = src + (size_t)(u * 4 + e) * NT + threadIdx.x;
        acc.c[u][e] = ld_coherent_scalar(p);
        st_coherent(p, (AccT)0);
      }
  }
};

// dma_load_16 (sk_device.h) to lds_base + IMM: one scalar instruction for the address.  A wave has its SIMD for itself in these
// kernels and issues one instruction in four cycles, so what a load costs in them is what it takes from the MFMAs.
template <int IMM>
static __device__ __forceinline__ void wavek_dma_16(uint4v rsrc, uint32_t lds_base, uint32_t lane_off, uint32_t uniform_off) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds_base), "v"(lane_off), "s"(rsrc), "s"(uniform_off), "n"(IMM)
               : "memory", "m0", "scc");
}
// two bytes per lane, zero-extended to four: lane l's value lands at lds_base + IMM + 4 l
template <int IMM>
static __device__ __forceinline__ void wavek_dma_2(uint4v rsrc, uint32_t lds_base, uint32_t lane_off, uint32_t uniform_off) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_ushort %1, %2, %3 offen lds"
               :
               : "s"(lds_base), "v"(lane_off), "s"(rsrc), "s"(uniform_off), "n"(IMM)
               : "memory", "m0", "scc");
}

template <int N>
static __device__ __forceinline__ void wavek_wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory");
}

// NN_: the weights are [K, N] (16-bit operands).  A chunk's weights are 64 rows of K of BN columns, and their fragments are read
// with ds_read_b64_tr_b16: a 16-lane group that points at a 4 (K) x 16 (N) patch receives, per lane, 4 consecutive K of one column.
// 16-byte piece c of K-row k stands at position c ^ 2 f(k) of the row, so that the 32 lanes served together -- 2 groups x 4
// rows x 32 bytes, the groups 8 rows apart -- read 8 different 32-byte slots of the 256 bytes of banks; f by the length of a row.
template <int TYPE_, int FM_, int FN_, bool NN_ = false>
struct TileWaveK : WaveKTile<TYPE_, FM_, FN_> {
  typedef WaveKTile<TYPE_, FM_, FN_> Base;
  typedef typename Base::Args Args;
  typedef typename Base::Acc Acc;
  typedef typename Base::AccV AccV;
  static constexpr int FM = FM_, FN = FN_, BM = Base::BM, BN = Base::BN, WAVES = Base::WAVES, NT = Base::NT, NB = Base::NB;
  static constexpr int KV = 64, BK = KV * WAVES;      // 16-bit units of K: of a chunk, of an iteration
  static constexpr int L = 2 * (FM + FN);             // loads of a chunk
  static constexpr bool NN = NN_;
  static_assert(!NN || ((TYPE_ == WK_F16 || TYPE_ == WK_BF16) && (BN == 32 || BN == 64 || BN == 128)), "[K, N] weights: 16-bit, loads of whole rows");
  static constexpr int R = L > 20 && !NN ? 40 : (L * 4 < 40 ? L * 4 : 40 / L * L);   // loads of a wave's ring (at most 160 KB / 4 waves, four chunks)
  static constexpr int S = R / L, PART = R % L;       // whole chunks in the ring, loads of one more
  static_assert(S >= 1 && (L % 2) == 0 && (R % 2) == 0, "a 16-row block of a chunk stays together in the ring");
  static constexpr int RING = R * 1024, LDS_BYTES = WAVES * RING, LDS_TOTAL = LDS_BYTES;
  static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
  static constexpr int CTAS_PER_CU = 1, WAVES_PER_EU = 1;
  static constexpr int NMFMA = Base::F8 ? NB : 2 * NB;   // MFMAs of a chunk
  static constexpr int H = NMFMA / 2, HR = H - (H + 3) / 4;   // of a phase, of those that have fragments read beside them

  // the loads of a chunk behind which `left` more chunks of the segment follow (the last PART loads of a segment fetch nothing)
  static __device__ __forceinline__ void wait_chunk(int left) {
    if (left >= S - 1) wavek_wait_loads<R - L>();
    else if (left == 0) wavek_wait_loads<PART>();
    else if (left == 1) wavek_wait_loads<L + PART>();
    else wavek_wait_loads<2 * L + PART>();
  }
  struct Frags {
    half8v a[FM][2], b[FN][2];   // [K-step]
  };
  static __device__ __forceinline__ int nn_swizzle(int k) {   // 2 f(k)
    return BN == 32 ? (k >> 2) & 2 : (BN == 64 ? (k & 2) | ((k >> 1) & 4) : 2 * (k & 3) | (k & 8));
  }
  // MFMA m of a chunk
  template <int m>
  static __device__ __forceinline__ void mfma(AccV (&c)[NB], const Frags &f) {
    constexpr int v = m % NB, s = m / NB, i = v / FN, j = v % FN;
    if constexpr (Base::F8) {
      typedef int intx8 __attribute__((ext_vector_type(8)));
      struct Pair { half8v v[2]; };
      const intx8 b = __builtin_bit_cast(intx8, Pair{{f.b[j][0], f.b[j][1]}}), x = __builtin_bit_cast(intx8, Pair{{f.a[i][0], f.a[i][1]}});
      constexpr int FMT = TYPE_ == WK_F8E4M3 ? 0 : 1;
      c[v] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b, x, c[v], FMT, FMT, 0, 0, 0, 0);
    } else if constexpr (Base::I8) {
      typedef typename Base::intx4 intx4;
      c[v] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(intx4, f.b[j][s]), __builtin_bit_cast(intx4, f.a[i][s]), c[v], 0, 0, 0);
    } else if constexpr (Base::BF16) {
      typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
      c[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f.b[j][s]), __builtin_bit_cast(bf16x8, f.a[i][s]), c[v], 0, 0, 0);
    } else {
      c[v] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.b[j][s], f.a[i][s], c[v], 0, 0, 0);
    }
  }

  static __device__ __forceinline__ void mac(const Args &a, Acc &acc, int pm, int pn, int k0, int n, char *smem) {
    const int lane = threadIdx.x & 63, wave = Base::wave_id();
    AccV c[NB];
    static_for<0, NB>([&](auto v) { c[v] = AccV{0, 0, 0, 0}; });
    // ---- descriptors: rows past M / N read as zero ----
    const uint32_t lda_bytes = (uint32_t)a.lda * 2, ldb_bytes = (uint32_t)a.ldb * 2;
    const uint4v rsrc_a = uniform_rsrc(make_rsrc_words(a.A + (int64_t)pm * BM * a.lda, (uint32_t)min(BM, a.M - pm * BM) * lda_bytes));
    const int rows_b = min(BN, a.N - pn * BN);
    // (NN: to the tile's last element of row K - 1, so that rows past K read as zero)
    const uint4v rsrc_b = NN ? uniform_rsrc(make_rsrc_words(a.B + (int64_t)pn * BN, (uint32_t)(((int64_t)(a.K - 1) * a.ldb + rows_b) * 2)))
                             : uniform_rsrc(make_rsrc_words(a.B + (int64_t)pn * BN * a.ldb, (uint32_t)rows_b * ldb_bytes));
    // load l of a chunk: rows 8 l .. 8 l + 7 (A's first), lane's row lane / 8, piece p (16 bytes) of row r of a block at position
    // p ^ ((r >> 1) & 7)
    const int row8 = lane >> 3;
    uint32_t off[L];
    int kp[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) kp[e] = ((lane & 7) ^ (4 * e + (row8 >> 1))) * 8;
    static_for<0, L>([&](auto l) {
      off[l] = l < 2 * FM ? (uint32_t)(8 * l + row8) * lda_bytes + (uint32_t)kp[l & 1] * 2
                          : (uint32_t)(8 * (l - 2 * FM) + row8) * ldb_bytes + (uint32_t)kp[l & 1] * 2;
      if constexpr (NN && l >= 2 * FM) {   // 512 / BN rows of K, BN / 8 lanes to a row
        const int k = (l - 2 * FM) * (512 / BN) + lane / (BN / 8), c = lane % (BN / 8) ^ nn_swizzle(k);
        // (a row past K of a problem shorter than a chunk: k * ldb_bytes may wrap around into the descriptor)
        off[l] = 8 * c < rows_b && k < a.K ? (uint32_t)k * ldb_bytes + (uint32_t)c * 16 : OOB_OFFSET;
      }
    });
    const uint32_t ring = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_address(smem) + wave * RING);
    // one row of tiles: see rotation_of.  Several: the CTAs of an XCD share A as well as the weights and stay on the same K
    // ([K, N] weights: the CTAs of a row of tiles read neighbouring pieces of the same rows and stay together too)
    const int rot = a.M <= BM && !NN ? rotation_of(pn, n) : Base::start_of(a, pn, n);
    // load l of a chunk that starts kbytes into the rows and `left` 16-bit units before K's end, pos: where the chunk starts in
    // the ring.  (Pieces past K fetch nothing: zeros arrive and the wait counts stay exact.)
    struct Chunk {
      uint32_t kbytes, kbytes_b;
      int left, pos;
      uint32_t base;   // LDS address of load 0, were the ring long enough
    };
    auto chunk = [&](int t, int pos) {
      const int kk = ((k0 + rotated_iteration(t, rot, n)) * WAVES + wave) * KV, left = t < n ? a.K - kk : 0;
      // (a chunk past K or past the segment must not carry its offset either)
      const uint32_t kbytes = (uint32_t)__builtin_amdgcn_readfirstlane(left > 0 ? kk * 2 : 0);
      return Chunk{kbytes, NN ? kbytes * (uint32_t)a.ldb : kbytes, left, pos, ring + (uint32_t)pos * 1024};
    };
    auto issue = [&](auto li, const Chunk &q) {
      constexpr int l = decltype(li)::value;
      uint32_t base = q.base;
      if (R % L != 0) base = q.pos >= R - l ? base - R * 1024 : base;
      if constexpr (NN && l >= 2 * FM)   // (the descriptor ends with K)
        wavek_dma_16<l * 1024>(rsrc_b, base, q.left > 0 ? off[l] : OOB_OFFSET, q.kbytes_b);
      else
        wavek_dma_16<l * 1024>(l < 2 * FM ? rsrc_a : rsrc_b, base, q.left >= KV || kp[l & 1] < q.left ? off[l] : OOB_OFFSET, q.kbytes);
    };
#pragma unroll
    for (int t = 0; t < S; ++t)
      if (t < n) {
        const Chunk q = chunk(t, t * L);
        static_for<0, L>([&](auto l) { issue(l, q); });
      }
    {
      const Chunk q = chunk(S, S * L);
      static_for<0, PART>([&](auto l) { issue(l, q); });
    }

    // fragments: lane (i, g) takes piece 4 s + g of its row for K-step s
    const int fi = lane & 15, fg = lane >> 4;
    const char *rd0 = smem + wave * RING + fi * 128 + ((fg ^ ((fi >> 1) & 7)) * 16), *rd1 = smem + wave * RING + fi * 128 + (((4 + fg) ^ ((fi >> 1) & 7)) * 16);
    // (NN: lane L of group g points at row 8 g + L / 4 of K, columns 4 (L % 4) .. of the block; four rows further on the other half)
    const char *rd_nn[FN];
    if constexpr (NN) {
      const int k = 8 * fg + (fi >> 2);
      static_for<0, FN>([&](auto j) {
        rd_nn[j] = smem + wave * RING + 2 * FM * 1024 + k * (BN * 2) + ((2 * j + ((fi & 3) >> 1)) ^ nn_swizzle(k)) * 16 + (fi & 1) * 8;
      });
    }
    auto read = [&](auto ri, Frags &f, int pos) {
      constexpr int r = decltype(ri)::value, s = r / (FM + FN), b = r % (FM + FN);   // block b of the chunk: A's, then the weights'
      if constexpr (NN && b >= FM) {
        typedef short short4v __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) short4v *lds_s4;
        const char *from = rd_nn[b - FM] + pos * 1024 + 32 * s * (BN * 2);
        union { short4v s[2]; half8v h; } u;
        u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)from);
        u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(from + 4 * (BN * 2)));
        f.b[b - FM][s] = u.h;
        return;
      }
      const char *from = (s ? rd1 : rd0) + pos * 1024;
      if (R % L != 0) from = pos >= R - 2 * b ? from - R * 1024 : from;
      const half8v x = *reinterpret_cast<const half8v *>(from + 2 * b * 1024);
      if constexpr (b < FM) f.a[b][s] = x;
      else f.b[b - FM][s] = x;
    };
    int pos = 0;   // of the chunk that is read next
    auto advance = [&] {
      pos += L;
      if (pos >= R) pos -= R;
    };
    // the place of the chunk just read (t) takes the rest of chunk t + S and the first PART loads of chunk t + S + 1
    Chunk q0, q1;
    auto refill_begin = [&](int t) {
      int p = pos + S * L;
      if (p >= R) p -= R;
      q0 = chunk(t + S, p);
      p += L;
      if (p >= R) p -= R;
      if (PART > 0) q1 = chunk(t + S + 1, p);
    };
    auto refill = [&](auto xi) {
      constexpr int x = decltype(xi)::value;
      if constexpr (x < L - PART) issue(std::integral_constant<int, x + PART>{}, q0);
      else issue(std::integral_constant<int, x - (L - PART)>{}, q1);
    };
    // X: fragments of chunk t, Y: of chunk t + 1, read while the first half of chunk t is multiplied; their place is refilled
    // during the second half
    auto body = [&](int t, const Frags &x, Frags &y) {
      if (t + 1 < n) {
        wait_chunk(n - 2 - t);
        static_for<0, H>([&](auto m) {
          mfma<m>(c, x);
          // (none beside the last MFMAs: they are waited for behind those)
          static_for<(m * L / HR < L ? m * L / HR : L), ((m + 1) * L / HR < L ? (m + 1) * L / HR : L)>([&](auto r) { read(r, y, pos); });
          __builtin_amdgcn_sched_barrier(0);
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      } else {
        static_for<0, H>([&](auto m) { mfma<m>(c, x); });
      }
      if (t + 1 + S < n) {
        refill_begin(t + 1);
        static_for<0, NMFMA - H>([&](auto m) {
          mfma<H + m>(c, x);
          static_for<m * L / (NMFMA - H), (m + 1) * L / (NMFMA - H)>([&](auto l) { refill(l); });
          __builtin_amdgcn_sched_barrier(0);
        });
      } else {
        static_for<H, NMFMA>([&](auto m) { mfma<m>(c, x); });
      }
      advance();
    };
    Frags x, y;
    wait_chunk(n - 1);
    static_for<0, L>([&](auto r) { read(r, x, pos); });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (S < n) {
      refill_begin(0);
      static_for<0, L>([&](auto l) { refill(l); });
    }
    advance();
    for (int t = 0;;) {
      body(t, x, y);
      if (++t == n) break;
      body(t, y, x);
      if (++t == n) break;
    }
    wavek_wait_loads<0>();   // the loads past the segment write LDS too
    Base::template add_waves<RING>(c, acc, smem);
  }
};

}  // namespace sk
