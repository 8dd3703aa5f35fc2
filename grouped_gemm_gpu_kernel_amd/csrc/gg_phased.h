// gg_phased.h -- the k-loop of the full 256 x 256 work tile (32-bit addressing).
//
// The tile's 64-deep stages are staged and multiplied in quarters: the loads
// are issued evenly through the loop, more than a stage of them stays in
// flight in 128 KB of LDS, and fragments are read a quarter ahead of the MFMAs
// that use them.  With whole stages (all loads of the next stage issued at the
// top of a step, one stage in flight) the waves spent a third of a step blocked
// on issuing loads and as much waiting for them: a stage took 4,030 cycles
// where its MFMAs need 2,048; here it takes 2,900 to 3,100 traced.  Same card: 64 x
// 2048^3 1221 -> 1005 us, one 8192^3 problem 991 -> 814 us (1350 TFLOP/s).  On random
// data the clock falls to 1.7 GHz under the chip's power limit (zeros: 595 us at 2.4
// GHz, with the same 73% of the SIMDs' cycles in MFMAs), so what bounds the loop is
// energy per product: without its loads it takes 16% less time, without its
// fragment reads 17%.
#pragma once

#include <type_traits>

#include "gg_common.h"

namespace gg {

// Waits until at most N (0..15) LDS operations of this wave are in flight.
template <int N>
__device__ __forceinline__ void wait_lgkmcnt() {
  __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4) | (N << 8));
}

// Workgroup barrier that waits for nothing of this wave's own (see the waits
// before each use); the empty asm keeps LDS accesses on their side of it.
__device__ __forceinline__ void phase_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// One stage (k0 .. k0 + 63) is four 16 KB units, in the order the loop reads
// them:
//   A0, A1  rows 64 i .. 64 i + 63 of each 128-row half of the tile, 64 deep
//           (a wave's 128 rows are 64 of unit A0 and 64 of A1; local row
//           64 h + r of unit i is tile row 128 h + 64 i + r)
//   B0, B1  k-rows 32 j .. 32 j + 31 of the stage, all 256 columns
// A 128-byte row segment of A and whole 512-byte rows of B: every line of L2
// is asked for once.  LDS holds two stages, [parity][A0, B0, B1, A1].
//
// A phase multiplies one pair (A half i, B half j): 64 rows x 64 columns x 32
// deep per wave, 16 MFMAs.  The pairs follow (0,0), (0,1), (1,0), (1,1), so
// every accumulator meets k in ascending order and a fragment read from LDS
// serves two phases.  Phase f reads the fragments of unit f + 2 into
// registers nothing uses any more (phases 0..3 of stage t: B1 of t, A1 of t,
// A0 of t + 1, B0 of t + 1) and issues the loads of unit f + 8, into the slot
// whose fragments were read in phase f - 2.  Its end waits until this wave's
// loads of unit f + 3 have landed (five units stay in flight) and until its
// LDS reads of the phases before have returned (a phase makes eight); one
// barrier then tells every wave both.
template <class G>
struct PhasedLoader {
  static constexpr int UNIT = 128 * 64;  // values of a unit
  static constexpr int A0 = 0, B0 = UNIT, B1 = 2 * UNIT, A1 = 3 * UNIT, PARITY = 4 * UNIT;
  static_assert(G::BM == 256 && G::BN == 256 && G::BK == 64 && G::THREADS == 512, "the full work tile");
  static_assert(2 * PARITY <= G::LDS_HALVES, "two stages");
  static constexpr int WAVES = 8;
  static constexpr int LOADS = 2;  // load instructions per unit and wave
  static constexpr uint32_t kOutOfRange = DmaLoader<G>::kOutOfRange;

  int m, n, k, ldb;
  const uint16_t* a_tile;  // A at (m0, 0)
  uint32_t a_n;            // bytes from a_tile to the end of A
  const uint16_t* b_tile;  // B at (0, n0)
  int64_t b_bytes;         // bytes from b_tile to the end of B
  uint32_t a_row64;        // bytes of 64 rows of A
  uint32_t b_row16;        // bytes of 16 rows of B
  uint32_t a_off, b_off;   // this thread's byte offset within a unit's first rows
  int a_col8;              // its piece's first k within a stage, over 8
  int wave;
  int m0, n0;
  int last_stage;
  bool fix_a, fix_b;  // the units of the last stage need repair (see repair_a, repair_b)

  __device__ __forceinline__ PhasedLoader(const gg_device_problem_desc& p, int m0_, int n0_, int wave_)
      : m(p.m), n(p.n), k(p.k), ldb(p.ldb), wave(wave_), m0(m0_), n0(n0_) {
    const int tid = opaque_tid(wave);
    a_tile = static_cast<const uint16_t*>(p.a) + (int64_t)m0 * p.lda;
    a_n = DmaLoader<G>::records(2 * ((int64_t)(p.m - 1 - m0) * p.lda + p.k));
    b_tile = static_cast<const uint16_t*>(p.b) + n0;
    b_bytes = 2 * ((int64_t)(p.k - 1) * p.ldb + p.n - n0);
    // Piece tid of a unit's first half: A row tid / 8, B row tid / 32; the
    // second half lies 64 (A) or 16 (B) local rows on, where the swizzles
    // repeat.
    const int a_row = tid / 8;
    a_col8 = (tid & 7) ^ G::a_swizzle(a_row);
    const int b_row = tid / 32;
    const int b_col8 = (tid & 31) ^ (G::b_swizzle(b_row) >> 1);
    a_off = 2u * ((uint32_t)a_row * (uint32_t)p.lda + 8u * (uint32_t)a_col8);
    b_off = n0 + 8 * b_col8 < p.n ? 2u * ((uint32_t)b_row * (uint32_t)p.ldb + 8u * (uint32_t)b_col8) : kOutOfRange;
    a_row64 = 128u * (uint32_t)p.lda;
    b_row16 = 32u * (uint32_t)p.ldb;
    last_stage = (p.k - 1) / G::BK;
    // A pieces that straddle K hold the next row's head past it; B rows at
    // k >= K lie past the matrix (and read as zero) unless rows overlap; the
    // last value of B reads as zero when its dword straddles the matrix end
    // (odd N; that of A does for odd K, which k & 7 covers).
    fix_a = (p.k & 7) != 0;
    fix_b = ((p.n & 1) != 0 && n0 + G::BN >= p.n) || (p.ldb < p.n && p.k % G::BK != 0);
  }

  // Load `i` (0, 1) of unit A`half` of stage kt into the unit at `unit`.
  __device__ __forceinline__ void issue_a(int kt, int half, uint16_t* unit, int i) const {
    const uint32_t voff = kt * G::BK + 8 * a_col8 < k ? a_off : kOutOfRange;
    load_to_lds16(a_tile, a_n, lds_address(unit) + 1024u * (uint32_t)(i * WAVES + wave), voff,
                  2u * G::BK * (uint32_t)kt + (uint32_t)(2 * i + half) * a_row64);
  }
  // Load `i` of unit B`half` of stage kt.
  __device__ __forceinline__ void issue_b(int kt, int half, uint16_t* unit, int i) const {
    const int64_t skip = 2 * (int64_t)G::BK * kt * ldb;
    load_to_lds16(b_tile + skip / 2, DmaLoader<G>::records(b_bytes - skip),
                  lds_address(unit) + 1024u * (uint32_t)(i * WAVES + wave), b_off, (uint32_t)(2 * half + i) * b_row16);
  }

  // Repairs this thread's pieces of a unit of the last stage after they have
  // landed: values at k >= K become zero, and a matrix's last value is put
  // back where its straddling dword read as zero.
  __device__ __forceinline__ void repair_a(const gg_device_problem_desc& p, int half, uint16_t* unit) const {
    const int tid = opaque_tid(wave);
    const int a_row = tid / 8;
    const int col = last_stage * G::BK + 8 * ((tid & 7) ^ G::a_swizzle(a_row));
    const uint32_t last =
        (k & 1) != 0 ? load_value_uniform(static_cast<const uint16_t*>(p.a) + (int64_t)(m - 1) * p.lda + (k - 1)) : 0u;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      u32x4_t* slot = reinterpret_cast<u32x4_t*>(unit + i * (UNIT / 2) + 8 * tid);
      const int row = m0 + 128 * i + 64 * half + a_row;
      u32x4_t val = keep_values(*slot, k - col);
      val = put_value(val, (k & 1) != 0 && row == m - 1 ? k - 1 - col : -1, last);
      *slot = val;
    }
    wait_lgkmcnt<0>();  // written before the barrier that follows
  }
  __device__ __forceinline__ void repair_b(const gg_device_problem_desc& p, int half, uint16_t* unit) const {
    const int tid = opaque_tid(wave);
    const int b_row = tid / 32;
    const int col = n0 + 8 * ((tid & 31) ^ (G::b_swizzle(b_row) >> 1));
    const bool odd = (n & 1) != 0 && n0 + G::BN >= n;
    const uint32_t last =
        odd ? load_value_uniform(static_cast<const uint16_t*>(p.b) + (int64_t)(k - 1) * ldb + (n - 1)) : 0u;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      u32x4_t* slot = reinterpret_cast<u32x4_t*>(unit + i * (UNIT / 2) + 8 * tid);
      const int krow = last_stage * G::BK + 32 * half + 16 * i + b_row;
      const u32x4_t zero = {0u, 0u, 0u, 0u};
      u32x4_t val = krow < k ? *slot : zero;
      val = put_value(val, odd && krow == k - 1 ? n - 1 - col : -1, last);
      *slot = val;
    }
    wait_lgkmcnt<0>();  // written before the barrier that follows
  }
};

// Runs the k-loop of the full work tile at (m0, n0) for wave `wave`, at block row
// wm (128 rows) and block column wn (64 columns); on_start as in the other
// k-loops.
template <class G, class OnStart, class Stamps>
__device__ __forceinline__ void run_k_loop_phased(const gg_device_problem_desc& p, int m0, int n0, uint16_t* lds,
                                                  int wave, int wm, int wn, floatx4_t (&acc)[8][4], OnStart&& on_start,
                                                  const Stamps& stamps) {
  using L = PhasedLoader<G>;
  const int nk = (p.k + G::BK - 1) / G::BK;
  if (nk <= 0) {
    on_start();
    return;
  }
  const L loader(p, m0, n0, wave);

  half8_t a[2][4][2];  // [A half][16-row block][32-deep k-step]
  half8_t b[2][4];     // [B half, one k-step][16-column block]
  const int lane = opaque_lane();
  const int g = lane >> 4, j = lane & 15;
  // LDS byte address of the lane's fragment in the first units: block 0, k-step 0
  // (operand layouts as in MfmaTile).
  const uint32_t a_lane = lds_address(lds) + 2u * (uint32_t)G::a_piece(wm * 64 + j, g);
  const uint32_t b_lane =
      lds_address(lds) + 2u * (uint32_t)G::b_chunk(8 * g + (j >> 2), wn * 64 + 4 * (j & 3));

  // Fragment read r (0..7) of the unit at offset `unit` (values) of a stage at
  // byte offset `stage` of the ring.
  static_assert((2 * L::UNIT) % kStageAlign == 0, "a unit keeps the address bits that select a fragment");
  auto read_a = [&](int half, int unit, uint32_t stage, int r) {
    const int fm = r & 3, s = r >> 2;
    a[half][fm][s] = *(const GG_LDS half8_t*)(uintptr_t)G::a_fragment(a_lane + stage, s, unit + fm * 16 * G::SA);
  };
  short4_t b_lo;
  auto read_b = [&](int half, int unit, uint32_t stage, int r) {
    const int fn = r >> 1;
    const uint32_t at = G::b_fragment(b_lane + stage, fn, unit);
    if ((r & 1) == 0) {
      b_lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((GG_LDS short4_t*)(uintptr_t)at);
    } else {
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((GG_LDS short4_t*)(uintptr_t)(at + 8u * G::SB));
      b[half][fn] = __builtin_bit_cast(half8_t, __builtin_shufflevector(b_lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };
  // The 16 MFMAs of (A half, B half).  Each of the first 8 is followed by
  // read(r) of a later unit, so that the fragments the next phase starts with
  // have landed by then; issue(0) and issue(1) ask for the two loads of a unit
  // later still, where no LDS read waits behind them (8192^3: 814 us; issued
  // after MFMAs 3 and 9, 834; with the reads at every other MFMA, 834).
  // Consecutive MFMAs share an operand: columns go back and forth.
  auto phase = [&](int ah, int bh, auto&& issue, auto&& read) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int fm = r >> 2, fn = (fm & 1) != 0 ? 3 - (r & 3) : r & 3;
      acc[4 * ah + fm][fn] =
          __builtin_amdgcn_mfma_f32_16x16x32_f16(b[bh][fn], a[ah][fm][bh], acc[4 * ah + fm][fn], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (r < 8) read(r);
      if (r == 8) issue(0);
      if (r == 12) issue(1);
      __builtin_amdgcn_sched_barrier(0);
    }
    wait_lgkmcnt<8>();
  };

  // The claim request comes after the first units: the waits below let it
  // stay in flight until the loads behind it are needed.
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    uint16_t* const st = lds + t * L::PARITY;
#pragma unroll
    for (int i = 0; i < 2; ++i) loader.issue_a(t, 0, st + L::A0, i);
#pragma unroll
    for (int i = 0; i < 2; ++i) loader.issue_b(t, 0, st + L::B0, i);
#pragma unroll
    for (int i = 0; i < 2; ++i) loader.issue_b(t, 1, st + L::B1, i);
#pragma unroll
    for (int i = 0; i < 2; ++i) loader.issue_a(t, 1, st + L::A1, i);
  }
  const bool extra = __builtin_amdgcn_readfirstlane(on_start() ? 1 : 0) != 0;
  if (extra) {
    wait_vmcnt<6 * L::LOADS + 1>();
  } else {
    wait_vmcnt<6 * L::LOADS>();
  }
  stamps.mark(GGK_PHASE_FIRST_STAGE);
  const bool single = nk == 1;
  if (single && loader.fix_a) loader.repair_a(p, 0, lds + L::A0);
  if (single && loader.fix_b) loader.repair_b(p, 0, lds + L::B0);
  phase_barrier();
  stamps.mark(GGK_PHASE_K_LOOP);
#pragma unroll
  for (int r = 0; r < 8; ++r) read_a(0, L::A0, 0, r);
#pragma unroll
  for (int r = 0; r < 8; ++r) read_b(0, L::B0, 0, r);
  wait_vmcnt<5 * L::LOADS>();
  if (single && loader.fix_b) loader.repair_b(p, 1, lds + L::B1);
  wait_lgkmcnt<0>();
  phase_barrier();

  // One stage.  ISSUE: the loads of stage kt + 2 are issued; otherwise kt is
  // one of the last two stages, everything has been issued and the waits count
  // down, the last stage's units being repaired as they land.  LAST: nothing
  // more is read.  The step stamps of a traced launch follow the four phases.
  auto stage = [&](int kt, auto issue_tag, auto last_tag) {
    constexpr bool ISSUE = decltype(issue_tag)::value, LAST = decltype(last_tag)::value;
    constexpr int N = L::LOADS;
    const int here = (kt & 1) * L::PARITY;
    const uint32_t rd = 2u * (uint32_t)here, rn = 2u * (uint32_t)(L::PARITY - here);
    uint16_t* const st = lds + here;
    uint16_t* const nx = lds + (L::PARITY - here);
    const bool stamped = kt == nk / 2;  // the step whose timing a traced launch records
    if (stamped) stamps.step_mark(0);
    phase(0, 0, [&](int i) { if constexpr (ISSUE) loader.issue_a(kt + 2, 0, st + L::A0, i); },
          [&](int r) { read_b(1, L::B1, rd, r); });
    wait_vmcnt<ISSUE ? 5 * N : LAST ? 0 : 4 * N>();
    if (LAST && loader.fix_a) loader.repair_a(p, 1, st + L::A1);
    phase_barrier();
    if (stamped) stamps.step_mark(1);
    phase(0, 1, [&](int i) { if constexpr (ISSUE) loader.issue_b(kt + 2, 0, st + L::B0, i); },
          [&](int r) { read_a(1, L::A1, rd, r); });
    if constexpr (!LAST) {
      wait_vmcnt<ISSUE ? 5 * N : 3 * N>();
      if (!ISSUE && loader.fix_a) loader.repair_a(p, 0, nx + L::A0);
      phase_barrier();
    }
    if (stamped) stamps.step_mark(2);
    phase(1, 0, [&](int i) { if constexpr (ISSUE) loader.issue_b(kt + 2, 1, st + L::B1, i); },
          [&](int r) { if constexpr (!LAST) read_a(0, L::A0, rn, r); });
    if constexpr (!LAST) {
      wait_vmcnt<ISSUE ? 5 * N : 2 * N>();
      if (!ISSUE && loader.fix_b) loader.repair_b(p, 0, nx + L::B0);
      phase_barrier();
    }
    if (stamped) stamps.step_mark(3);
    phase(1, 1, [&](int i) { if constexpr (ISSUE) loader.issue_a(kt + 2, 1, st + L::A1, i); },
          [&](int r) { if constexpr (!LAST) read_b(0, L::B0, rn, r); });
    if constexpr (!LAST) {
      wait_vmcnt<ISSUE ? 5 * N : N>();
      if (!ISSUE && loader.fix_b) loader.repair_b(p, 1, nx + L::B1);
      phase_barrier();
    }
    if (stamped) stamps.step_mark(4);
    // A traced launch's k-loop ends when every wave's does.
    if constexpr (LAST && !std::is_same_v<Stamps, NoStamps>) phase_barrier();
  };
  int kt = 0;
#pragma unroll 1
  for (; kt < nk - 2; ++kt) stage(kt, std::true_type{}, std::false_type{});
  if (nk >= 2) stage(kt++, std::false_type{}, std::false_type{});
  stage(kt, std::false_type{}, std::true_type{});  // a single stage also waits for the (empty) loads past K
}

}  // namespace gg
