// Q4 weights against a middling number of rows of A: tiles whose waves stream K on their own, as in tile_wavek.h.
//
//  * An iteration is four scale groups of 128 K-values, one per wave.  A wave fetches its group in two halves of 64 K-values of
//    A (loads of 8 rows x 128 bytes, a ring of DA halves) and the group's nibbles (loads of 16 rows x 64 bytes) and scales and
//    zero points (one 2-byte value per lane into four bytes of LDS) in a ring of DW groups.
//  * Every weight is decoded once per CTA, by the wave that multiplies it, right before the MFMA: the rounded weights bit for bit
//    (q4_dequant.h), whatever the number of rows.
//  * The fragments of a half are read beside the MFMAs of the first step of the half before, their place is refilled beside those of
//    the second; beside a block's MFMAs stands the decode of the next block.
//
// What bounds it: with few rows what a CU takes in of A and nibbles (tile_wavek.h), with 64 rows and more the decode -- 17 vector
// instructions per fragment of 16 x 32 weights, whose FM MFMAs are four issue slots each.  128 x 64 and 64 x 128 tiles
// are not built: two fragment buffers beside 128 accumulators make the compiler move registers in the loop (512 x 4096 x 4096 42 and
// 57 us, 30 on 64 x 64 tiles).  The kernels before (up to 64 rows tile_skinny.h, beyond the decode into LDS of tile_f16_dma.h) /
// these, in us, three sets of operands in turn and from HBM: 64 x 4096 x 4096 15.7 / 8.5 and 15.9 / 9.6, 64 x 8192 x 8192 26.2 / 18.7
// and 26.6 / 22.8, 128 x 4096 x 4096 25.5 / 11.3 and 25.9 / 12.6, 128 x 8192 x 8192 42.1 / 27.1 and 41.8 / 29.5, 256 x 4096 x 4096
// 27.3 / 15.6 and 28.5 / 16.4.
#pragma once
#include "q4_dequant.h"
#include "tile_wavek.h"

namespace sk {

// TILED_: the nibbles in tiles of 16 rows x one scale group, the tiles of 16 rows behind each other.  A load reads one of them, and
// every lane gets the bytes that it gets from the row-major array: equal plans give equal bits.
template <int TYPE_, int FM_, int FN_, bool TILED_ = false>
struct TileWaveKQ4 : WaveKTile<TYPE_, FM_, FN_> {
  typedef WaveKTile<TYPE_, FM_, FN_> Base;
  typedef typename Base::Args Args;
  typedef typename Base::Acc Acc;
  typedef typename Base::AccV AccV;
  static constexpr bool ZP = TYPE_ == WK_Q4ZP;
  static constexpr int FM = FM_, FN = FN_, BM = Base::BM, BN = Base::BN, WAVES = Base::WAVES, NT = Base::NT, NB = Base::NB;
  static constexpr int BK = 128 * WAVES;              // K-values of an iteration
  static constexpr int LA = 2 * FM, LW = FN, LS = (BN + 63) / 64, LWS = LW + LS * (ZP ? 2 : 1);   // loads: half of A, nibbles, scales, all of a group
  static constexpr int W_SLOT = LW * 1024 + (LWS - LW) * 256, A_SLOT = LA * 1024;
  static constexpr int MOST = 40 * 1024;              // a wave's share of the LDS
  static constexpr int rings() {                      // 10 DA + DW, the largest that fits with DW = DA / 2, rounded up
    int best = 0;
    for (int da = 2; da <= 6; ++da)
      if (da * A_SLOT + (da + 1) / 2 * W_SLOT <= MOST) best = 10 * da + (da + 1) / 2;
    return best;
  }
  static constexpr int DA = rings() / 10, DW = rings() % 10;
  static_assert(DA >= 2 && DW == (DA + 1) / 2, "two halves of A and a group of weights at least");
  static constexpr int RING_W = DA * A_SLOT, RING = RING_W + DW * W_SLOT;
  static constexpr int LDS_BYTES = WAVES * RING, LDS_TOTAL = LDS_BYTES;
  static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
  static constexpr int CTAS_PER_CU = 1, WAVES_PER_EU = 1;
  static constexpr bool PERM_W = FM >= FN;   // the four permutations of a fragment on the side that has fewer of them

  static constexpr int least(int x, int y) { return x < y ? x : y; }
  // Half x of the segment is read when everything up to the refill behind the reading of half x - 1 has been issued: A's half
  // h behind the reading of half h - DA, group u's weights before A's half behind that of half 2 (u - DW) + 1.  The loads that may
  // then still be under way, by how many iterations follow (none: only what is left of this one; a few: not all of the next loads
  // exist, and fewer than that are waited for).
  static __device__ __forceinline__ void wait_even(int left) {   // half 2 t: A and the group's weights
    constexpr int steady = least((DA - 1) * LA + DA / 2 * LWS, (2 * DW - 1) * LA + (DW - 1) * LWS);
    constexpr int some = least(least(DA - 1, 3), 2 * DW - 1) * LA;
    if (left >= DW) wavek_wait_loads<steady>();
    else if (left > 0) wavek_wait_loads<some>();
    else wavek_wait_loads<LA>();
  }
  static __device__ __forceinline__ void wait_odd(int left) {
    constexpr int steady = (DA - 1) * LA + (DA - 1) / 2 * LWS, some = least(DA - 1, 2) * LA;
    if (left > DW) wavek_wait_loads<steady>();
    else if (left > 0) wavek_wait_loads<some>();
    else wavek_wait_loads<0>();
  }

  struct Frags {   // of a half: A's for two MFMA steps, eight nibbles per step of each weight row
    half8v a[FM][2];
    uint2 w[FN];
  };
  struct Group {
    half_t s[FN], z[ZP ? FN : 1];
  };

  static __device__ __forceinline__ void mac(const Args &a, Acc &acc, int pm, int pn, int k0, int n, char *smem) {
    const int lane = threadIdx.x & 63, wave = Base::wave_id();
    AccV c[NB];
    static_for<0, NB>([&](auto v) { c[v] = AccV{0, 0, 0, 0}; });
    // ---- descriptors: rows past M / N read as zero ----
    const uint32_t lda_bytes = (uint32_t)a.lda * 2, ldb_bytes = (uint32_t)a.ldb, groups_bytes = (uint32_t)a.groups * 2;
    const int rows_w = min(BN, a.N - pn * BN);
    const uint4v rsrc_a = uniform_rsrc(make_rsrc_words(a.A + (int64_t)pm * BM * a.lda, (uint32_t)min(BM, a.M - pm * BM) * lda_bytes));
    // (tiled weights have whole blocks of 16 rows)
    const uint4v rsrc_w = uniform_rsrc(make_rsrc_words(reinterpret_cast<const char *>(a.B) + (int64_t)pn * BN * a.ldb,
                                                       (uint32_t)(TILED_ ? (rows_w + 15) & ~15 : rows_w) * ldb_bytes));
    const uint4v rsrc_s = uniform_rsrc(make_rsrc_words(a.scales + (int64_t)pn * BN * a.groups, (uint32_t)rows_w * groups_bytes));
    uint4v rsrc_z = rsrc_s;
    if constexpr (ZP) rsrc_z = uniform_rsrc(make_rsrc_words(a.zeros + (int64_t)pn * BN * a.groups, (uint32_t)rows_w * groups_bytes));
    // lane's part of a load.  A: row lane / 8, piece p (16 bytes) of row r of a block at position p ^ ((r >> 1) & 7); nibbles: row
    // lane / 4, piece p of row r of a block at p ^ (r >> 2); scales: row lane
    const int row8 = lane >> 3;
    uint32_t off_a[LA], off_w[LW], off_s[LS];
    static_for<0, LA>([&](auto l) { off_a[l] = (uint32_t)(8 * l + row8) * lda_bytes + (uint32_t)((lane & 7) ^ (4 * (l & 1) + (row8 >> 1))) * 16; });
    static_for<0, LW>([&](auto l) {
      off_w[l] = (uint32_t)(16 * l) * ldb_bytes + (uint32_t)(lane >> 2) * (TILED_ ? 64u : ldb_bytes) + (uint32_t)((lane & 3) ^ (lane >> 4)) * 16;
    });
    static_for<0, LS>([&](auto l) { off_s[l] = 64 * l + lane < BN ? (uint32_t)(64 * l + lane) * groups_bytes : OOB_OFFSET; });
    const uint32_t ring = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_address(smem) + wave * RING);
    const int rot = a.M <= BM ? rotation_of(pn, n) : Base::start_of(a, pn, n);
    auto group_of = [&](int t) { return (k0 + rotated_iteration(t, rot, n)) * WAVES + wave; };
    // (a group past K fetches nothing: zeros arrive and the wait counts stay exact; it must not carry its offset either)
    struct Where {
      uint32_t bytes, slot;
      bool live;
    };
    auto where_a = [&](int h, int slot) {
      const int g = group_of(h >> 1);
      const bool live = g < a.groups;
      return Where{(uint32_t)__builtin_amdgcn_readfirstlane(live ? g * 256 + (h & 1) * 128 : 0), ring + (uint32_t)slot * A_SLOT, live};
    };
    auto where_w = [&](int t, int slot) {
      const int g = group_of(t);
      const bool live = g < a.groups;
      return Where{(uint32_t)__builtin_amdgcn_readfirstlane(live ? g : 0), ring + RING_W + (uint32_t)slot * W_SLOT, live};
    };
    auto issue_a = [&](auto li, const Where &q) {
      constexpr int l = decltype(li)::value;
      wavek_dma_16<l * 1024>(rsrc_a, q.slot, q.live ? off_a[l] : OOB_OFFSET, q.bytes);
    };
    auto issue_w = [&](auto li, const Where &q) {
      constexpr int l = decltype(li)::value;
      if constexpr (l < LW) wavek_dma_16<l * 1024>(rsrc_w, q.slot, q.live ? off_w[l] : OOB_OFFSET, q.bytes * (TILED_ ? 1024 : 64));
      else if constexpr (l < LW + LS) wavek_dma_2<LW * 1024 + (l - LW) * 256>(rsrc_s, q.slot, q.live ? off_s[l - LW] : OOB_OFFSET, q.bytes * 2);
      else wavek_dma_2<LW * 1024 + (l - LW) * 256>(rsrc_z, q.slot, q.live ? off_s[l - LW - LS] : OOB_OFFSET, q.bytes * 2);
    };
    // what the readings of the halves -2 DW .. -1 would have issued
    static_for<0, 2 * DW>([&](auto x) {
      constexpr int e = x - 2 * DW;
      if constexpr (x % 2 == 1) {
        constexpr int u = x / 2;
        if (u < n) {
          const Where q = where_w(u, u);
          static_for<0, LWS>([&](auto l) { issue_w(l, q); });
        }
      }
      if constexpr (e + DA >= 0) {
        if (e + DA < 2 * n) {
          const Where q = where_a(e + DA, e + DA);
          static_for<0, LA>([&](auto l) { issue_a(l, q); });
        }
      }
    });

    const int fi = lane & 15, fg = lane >> 4;
    const char *mine = smem + wave * RING;
    // A: lane (i, g) takes piece 2 g + q of its row for step q; nibbles: bytes 32 (h & 1) + 8 g of its row
    const char *rd_a[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) rd_a[q] = mine + fi * 128 + ((2 * fg + q) ^ ((fi >> 1) & 7)) * 16;
    const char *rd_w[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) rd_w[h] = mine + RING_W + fi * 64 + ((2 * h + (fg >> 1)) ^ (fi >> 2)) * 16 + (fg & 1) * 8;
    const char *rd_s = mine + RING_W + LW * 1024 + fi * 4;
    constexpr int READS = 2 * FM + FN;
    // read r of a half: A's fragments, then the nibbles (HALF: which half of the group)
    auto read = [&](auto ri, auto half, Frags &f, int sa, int sw) {
      constexpr int r = decltype(ri)::value;
      if constexpr (r < 2 * FM) f.a[r / 2][r % 2] = *reinterpret_cast<const half8v *>(rd_a[r % 2] + sa * A_SLOT + r / 2 * 2048);
      else f.w[r - 2 * FM] = *reinterpret_cast<const uint2 *>(rd_w[decltype(half)::value] + sw * W_SLOT + (r - 2 * FM) * 1024);
    };
    auto read_group = [&](auto j, Group &g, int sw) {
      g.s[j] = *reinterpret_cast<const half_t *>(rd_s + sw * W_SLOT + j * 64);
      if constexpr (ZP) g.z[j] = *reinterpret_cast<const half_t *>(rd_s + sw * W_SLOT + LS * 256 + j * 64);
    };
    Q4Consts qc = q4_consts(ZP ? 0 : a.zero);
    auto decode = [&](const Frags &f, const Group &g, auto ji, int q) {
      constexpr int j = decltype(ji)::value;
      const half2v s2 = half2v{g.s[j], g.s[j]};
      const uint32_t w = q ? f.w[j].y : f.w[j].x;
      half8v x;
      if constexpr (ZP) {
        const half_t lo = (half_t)1024.f + g.z[j], hi = (half_t)-64.f - g.z[j];   // exact
        x = dequant_word_q4(w, qc, s2, half2v{lo, lo}, half2v{hi, hi});
      } else {
        x = dequant_word_q4(w, qc, s2);
      }
      if constexpr (PERM_W) {   // the decode's element order to A's
        const uint4v v = __builtin_bit_cast(uint4v, x);
        uint4v p;
        p[0] = __builtin_amdgcn_perm(v[1], v[0], 0x05040100u);
        p[1] = __builtin_amdgcn_perm(v[3], v[2], 0x05040100u);
        p[2] = __builtin_amdgcn_perm(v[1], v[0], 0x07060302u);
        p[3] = __builtin_amdgcn_perm(v[3], v[2], 0x07060302u);
        x = __builtin_bit_cast(half8v, p);
      }
      return x;
    };
    auto permute = [&](const half8v &x) {   // A's element order to the decode's, 0,4,1,5,2,6,3,7
      if constexpr (PERM_W) return x;
      const uint4v v = __builtin_bit_cast(uint4v, x);
      uint4v p;
      p[0] = __builtin_amdgcn_perm(v[2], v[0], 0x05040100u);
      p[1] = __builtin_amdgcn_perm(v[2], v[0], 0x07060302u);
      p[2] = __builtin_amdgcn_perm(v[3], v[1], 0x05040100u);
      p[3] = __builtin_amdgcn_perm(v[3], v[1], 0x07060302u);
      return __builtin_bit_cast(half8v, p);
    };
    // slots of the next half of A and of the group whose nibbles are read next
    int sa = 0, sw = 0;
    Group g, gn;
    // Half x of the segment (HALF: x & 1), whose fragments are f: step 0 while the fragments of half x + 1 are read into y, step 1
    // while what that frees is refilled.  A wave has its SIMD for itself, so beside the MFMAs of a block of weight rows stand the
    // decode of the next block and a share of the permutations of A's fragments for the next step.
    half8v pa[FM], pb[FM], w;   // A for step 0 and 1 in the decode's element order; the block of weights to multiply next
    auto body = [&](int t, auto half, auto refill, auto steady, const Frags &f, Frags &y) {
      constexpr int HALF = decltype(half)::value;
      constexpr bool REFILL = decltype(refill)::value;
      constexpr std::integral_constant<int, 1 - HALF> next;
      const int left = decltype(steady)::value ? DW + 1 : n - 1 - t;   // (any number from there on is the same)
      // (behind the last half nothing comes: what is read and decoded then is never used)
      if constexpr (HALF == 0) wait_odd(left);
      else if (left > 0) wait_even(left - 1);
      static_for<0, FN>([&](auto j) {
        half8v wn;
        if constexpr (j + 1 < FN) wn = decode(f, g, std::integral_constant<int, j + 1>{}, 0);
        else wn = decode(f, g, std::integral_constant<int, 0>{}, 1);
        static_for<j * FM / FN, (j + 1) * FM / FN>([&](auto i) { pb[i] = permute(f.a[i][1]); });
        static_for<0, FM>([&](auto i) { c[i * FN + j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, pa[i], c[i * FN + j], 0, 0, 0); });
        // (none beside the last block: they are waited for behind it)
        static_for<least(READS, j * READS / (FN - 1)), least(READS, (j + 1) * READS / (FN - 1))>([&](auto r) { read(r, next, y, sa, sw); });
        if constexpr (HALF == 1 && j == 0) static_for<0, FN>([&](auto jj) { read_group(jj, gn, sw); });
        w = wn;
        __builtin_amdgcn_sched_barrier(0);
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      // half x + 1 is read: its place takes half x + 1 + DA, and with a second half the group's place group t + DW
      const int nsa = sa + 1 == DA ? 0 : sa + 1, nsw = sw + 1 == DW ? 0 : sw + 1;
      Where qw, qa;
      if constexpr (REFILL) qa = where_a(2 * t + HALF + 1 + DA, sa);
      if constexpr (REFILL && HALF == 0) qw = where_w(t + DW, sw);
      static_for<0, FN>([&](auto j) {
        half8v wn;
        if constexpr (j + 1 < FN) wn = decode(f, g, std::integral_constant<int, j + 1>{}, 1);
        else wn = decode(y, HALF == 0 ? g : gn, std::integral_constant<int, 0>{}, 0);
        static_for<j * FM / FN, (j + 1) * FM / FN>([&](auto i) { pa[i] = permute(y.a[i][0]); });
        static_for<0, FM>([&](auto i) { c[i * FN + j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, pb[i], c[i * FN + j], 0, 0, 0); });
        // (a group's weights before the half of A)
        if constexpr (REFILL) {
          constexpr int FIRST = HALF == 0 ? LWS : 0, TOTAL = FIRST + LA, l0 = j * TOTAL / FN, l1 = (j + 1) * TOTAL / FN;
          static_for<(l0 < FIRST ? l0 : FIRST), (l1 < FIRST ? l1 : FIRST)>([&](auto l) { issue_w(l, qw); });
          static_for<(l0 > FIRST ? l0 - FIRST : 0), (l1 > FIRST ? l1 - FIRST : 0)>([&](auto l) { issue_a(l, qa); });
        }
        w = wn;
        __builtin_amdgcn_sched_barrier(0);
      });
      sa = nsa;
      if constexpr (HALF == 0) sw = nsw;
    };
    Frags x, y;
    wait_even(n - 1);
    static_for<0, READS>([&](auto r) { read(r, std::integral_constant<int, 0>{}, x, 0, 0); });
    static_for<0, FN>([&](auto j) { read_group(j, g, 0); });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (DA < 2 * n) {
      const Where q = where_a(DA, 0);
      static_for<0, LA>([&](auto l) { issue_a(l, q); });
    }
    sa = 1;
    static_for<0, FM>([&](auto i) { pa[i] = permute(x.a[i][0]); });
    w = decode(x, g, std::integral_constant<int, 0>{}, 0);
    // group t + DW and half 2 t + 1 + DA, half 2 t + 2 + DA: both, the first alone, neither of them is still to be fetched.  (Loops of
    // their own: with the choice inside, the compiler moves the accumulators between its two register files every iteration.)
    auto iteration = [&](int t, auto refill0, auto refill1, auto steady) {
      body(t, std::integral_constant<int, 0>{}, refill0, steady, x, y);
      body(t, std::integral_constant<int, 1>{}, refill1, steady, y, x);
      g = gn;
    };
    int t = 0;
    for (; 2 * t + 2 + DA < 2 * n; ++t) iteration(t, std::true_type{}, std::true_type{}, std::bool_constant<(2 * DW - DA < 1)>{});
    if constexpr (DA == 2 * DW)
      if (t + DW < n) iteration(t++, std::true_type{}, std::false_type{}, std::false_type{});
    for (; t < n; ++t) iteration(t, std::false_type{}, std::false_type{}, std::false_type{});
    Base::template add_waves<RING>(c, acc, smem);
  }
};

}  // namespace sk
