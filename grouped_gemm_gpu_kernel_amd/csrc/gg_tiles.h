// gg_tiles.h -- macro-tile compute for the gfx950 grouped GEMM.
//
// The MFMA path loads its stages straight into LDS and multiplies them a phase
// behind the fragment reads (run_k_loop_halves here, run_k_loop_phased in
// gg_phased.h for the full 256 x 256 work tile), as the FMA path does
// (run_k_loop_fma).  The 64-bit addressing forms stage through registers: each
// K stage is read from global memory into registers while the previous stage,
// held in LDS, is being multiplied; the registers are then written to the
// other LDS buffer and one barrier ends the stage.  The reference's
// equivalents are compute_gemm_tile_tensor_core and compute_gemm_tile_simt
// (src/grouped_gemm.cu:373-626); the k-loop structure, register blocking and LDS
// layout here are gfx950's own.
#pragma once

#include "gg_common.h"
#include "gg_phased.h"

namespace gg {

// Runs the staged k-loop of one tile in the 64-bit addressing form:
// compute(stage_pointer) is called once per stage with that stage's LDS buffer,
// and on_start() once, by every thread, after the first loads are on their way
// (the persistent scheduler requests its next tile there, so that the request's
// latency overlaps this tile's).  on_start returns whether the calling wave
// issued one global memory request of its own.
//
// Stage s is fetched into register set s % DEPTH.  While stage k is
// multiplied out of LDS buffer k % 2, the loads of stage k + DEPTH - 1 are
// issued and stage k + 1 (issued DEPTH - 1 stages earlier) is written to the
// other LDS buffer; one barrier closes the step.  Loads and LDS writes are
// issued for every step, also for stages past K (which read as zero without
// touching memory and land in a buffer nobody reads): a load under a branch
// would make the compiler wait for every load in flight before the next LDS
// write, and only DEPTH - 1 = 1 stage could ever be in flight.  The main loop
// runs whole groups of DEPTH steps with no branch; the last steps of a tile
// are guarded.  The body is unrolled DEPTH times so that every register set
// is addressed statically.
template <class G, class Compute, class OnStart, class Stamps>
__device__ __forceinline__ void run_k_loop(const gg_device_problem_desc& p, int m0, int n0, uint16_t* lds,
                                           int wave, Compute&& compute, OnStart&& on_start, const Stamps& stamps) {
  constexpr int D = G::DEPTH;
  const int nk = (p.k + G::BK - 1) / G::BK;
  if (nk <= 0) {
    on_start();
    return;
  }
  const StageLoader<G> loader(p, m0, n0, wave);
  RawStage<G> ring[D];
#pragma unroll
  for (int s = 0; s < D - 1; ++s) loader.issue(s, ring[s]);
  on_start();  // the compiler's waits count the request like any other load
  loader.store(ring[0], 0, lds, 0);
  stamps.mark(GGK_PHASE_FIRST_STAGE);
  __syncthreads();
  stamps.mark(GGK_PHASE_K_LOOP);
  auto step = [&](int k, int u) {
    loader.issue(k + D - 1, ring[(u + D - 1) % D]);
    compute(lds + (k & 1) * G::STAGE);
    loader.store(ring[(u + 1) % D], k + 1, lds, (k + 1) & 1);
    __syncthreads();
  };
  int k0 = 0;
  for (; k0 + D <= nk; k0 += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) step(k0 + u, u);
  }
#pragma unroll
  for (int u = 0; u < D - 1; ++u) {
    if (k0 + u < nk) step(k0 + u, u);
  }
}

// The k-loop with stage loads straight into LDS (32-bit offsets) of wave
// blocks of up to 64 x 64, BUFFERS LDS buffers of one stage each.
//
// A stage is multiplied in two phases, its k-halves (32 deep, FM x 4 MFMAs per
// wave); each phase reads the fragments of the next half into the registers
// the phase before used, so no MFMA waits for a read that was issued just
// before it.  The second half's fragments are read in phase 0, so a stage's
// buffer is free from phase 1 on: the loads of stage t + BUFFERS go there in
// phase 1 of stage t and (where more than one stage stays in flight) phase 0
// of stage t + 1.  One wait and one barrier per stage, at the end of phase 0:
// the wave's loads of stage t + 1 have landed (the stage holding K - 1 is
// repaired then), and its reads of stage t are done.
//
// Stages past K are never asked for: a problem of fewer stages than BUFFERS
// issues what it has and waits for all of it.
//
// These tiles are bound by latency and by what they stream rather than by the
// matrix cores.  Against whole stages read and multiplied in one go, same
// card: a 24-problem ragged set (half of it edge classes) 168.5 -> 146.9 us, 16
// problems of at most 256 in each dimension 14.0 -> 12.7, mixed-512 222.9 ->
// 220.5.
//
// on_start runs after the first barrier: the request it makes is then the
// youngest operation in flight, and the first stage's wait lets it stay there.
template <class G, int WM, class OnStart, class Stamps>
__device__ __forceinline__ void run_k_loop_halves(const gg_device_problem_desc& p, int m0, int n0, uint16_t* lds,
                                                  int wave, int wm, int wn, floatx4_t (&acc)[WM / 16][4], OnStart&& on_start,
                                                  const Stamps& stamps) {
  using L = DmaLoader<G>;
  constexpr int NBUF = G::BUFFERS;
  constexpr int FM = WM / 16;
  constexpr int LOADS = L::LOADS;
  // Loads of a stage issued in phase 1; the rest follow in the next phase 0.
  constexpr int FIRST = NBUF > 2 ? LOADS / 2 : LOADS;
  const int nk = (p.k + G::BK - 1) / G::BK;
  if (nk <= 0) {
    on_start();
    return;
  }
  const L loader(p, m0, n0, wave);
  const bool deep = nk >= NBUF;  // every buffer gets a stage
#pragma unroll
  for (int s = 0; s < NBUF - 1; ++s) {
    if (s < nk) loader.issue(s, lds + s * G::STAGE);
  }
  if (deep) {
#pragma unroll
    for (int l = 0; l < FIRST; ++l) loader.issue_load(NBUF - 1, lds + (NBUF - 1) * G::STAGE, l);
    wait_vmcnt<(NBUF - 2) * LOADS + FIRST>();
  } else {
    wait_vmcnt<0>();
  }
  stamps.mark(GGK_PHASE_FIRST_STAGE);
  if (loader.last_stage == 0) loader.fix_last_stage(0, lds);
  stage_barrier();
  stamps.mark(GGK_PHASE_K_LOOP);
  const bool extra = __builtin_amdgcn_readfirstlane(on_start() ? 1 : 0) != 0;

  half8_t a[2][FM];  // [k-half][16-row block]
  half8_t b[2][4];   // [k-half][16-column block]
  const int lane = opaque_lane();
  const int g = lane >> 4, j = lane & 15;
  // LDS byte address of the lane's fragments of block 0, k-half 0 (operand layouts as in MfmaTile).
  const uint32_t a_lane = lds_address(lds) + 2u * (uint32_t)G::a_piece(wm * WM + j, g);
  const uint32_t b_lane = lds_address(lds) + 2u * (uint32_t)(G::A_STAGE + G::b_chunk(8 * g + (j >> 2),
                                                                                      wn * 64 + 4 * (j & 3)));
  // Fragment read r (0..FM + 7) of k-half h of the stage at byte offset `at`
  // of the ring.
  short4_t b_lo;
  auto read = [&](int h, uint32_t at, int r) {
    if (r < 8) {
      const int fn = r >> 1;
      const uint32_t addr = G::b_fragment(b_lane + at, fn, 32 * h * G::SB);
      if ((r & 1) == 0) {
        b_lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((GG_LDS short4_t*)(uintptr_t)addr);
      } else {
        const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((GG_LDS short4_t*)(uintptr_t)(addr + 8u * G::SB));
        b[h][fn] = __builtin_bit_cast(half8_t, __builtin_shufflevector(b_lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    } else {
      const int fm = r - 8;
      a[h][fm] = *(const GG_LDS half8_t*)(uintptr_t)G::a_fragment(a_lane + at, h, 16 * fm * G::SA);
    }
  };
  // The MFMAs of k-half h, among them the reads of the next half and
  // issue(0 .. LOADS_N - 1).
  auto phase = [&](int h, auto&& read_next, auto loads_tag, auto&& issue) {
    constexpr int N = FM * 4;                         // MFMAs
    constexpr int READS = FM + 8;
    constexpr int LOADS_N = decltype(loads_tag)::value;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int fm = i >> 2, fn = (fm & 1) != 0 ? 3 - (i & 3) : i & 3;
      acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[h][fn], a[h][fm], acc[fm][fn], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < READS; ++r) {
        if (r * (N * 3 / 4) / READS == i) read_next(r);  // within the first three quarters
      }
#pragma unroll
      for (int l = 0; l < LOADS_N; ++l) {
        if (N - LOADS_N + l == i) issue(l);  // the last ones
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const auto nothing = [](int) {};
#pragma unroll
  for (int r = 0; r < FM + 8; ++r) read(0, 0, r);

  int t = 0, u = 0;  // stage and its buffer
  // Stages with all the loads that follow still to be issued.
#pragma unroll 1
  for (; t < nk - NBUF; ++t) {
    const int un = u == NBUF - 1 ? 0 : u + 1, ul = u == 0 ? NBUF - 1 : u - 1;
    const uint32_t here = 2u * (uint32_t)(u * G::STAGE), next = 2u * (uint32_t)(un * G::STAGE);
    const bool stamped = t == nk / 2;  // the step whose timing a traced launch records
    if (stamped) stamps.step_mark(0);
    const auto second = [&](int l) { loader.issue_load(t + NBUF - 1, lds + ul * G::STAGE, FIRST + l); };
    phase(0, [&](int r) { read(1, here, r); }, std::integral_constant<int, LOADS - FIRST>{}, second);
    if (stamped) stamps.step_mark(1);
    if (t == 0 && extra) {
      wait_vmcnt<(NBUF - 2) * LOADS + 1>();
    } else {
      wait_vmcnt<(NBUF - 2) * LOADS>();
    }
    if (stamped) stamps.step_mark(2);
    stage_barrier();
    if (stamped) stamps.step_mark(3);
    const auto first = [&](int l) { loader.issue_load(t + NBUF, lds + u * G::STAGE, l); };
    phase(1, [&](int r) { read(0, next, r); }, std::integral_constant<int, FIRST>{}, first);
    if (stamped) stamps.step_mark(4);
    u = un;
  }
  // The last stages: the rest of the last one's loads, then only waits.
  const int tail = t;
#pragma unroll 1
  for (; t < nk; ++t) {
    const int un = u == NBUF - 1 ? 0 : u + 1, ul = u == 0 ? NBUF - 1 : u - 1;
    const uint32_t here = 2u * (uint32_t)(u * G::STAGE), next = 2u * (uint32_t)(un * G::STAGE);
    const bool stamped = t == nk / 2;
    if (stamped) stamps.step_mark(0);
    if (FIRST < LOADS && t == tail && deep) {
#pragma unroll
      for (int l = FIRST; l < LOADS; ++l) loader.issue_load(t + NBUF - 1, lds + ul * G::STAGE, l);
    }
    phase(0, [&](int r) { read(1, here, r); }, std::integral_constant<int, 0>{}, nothing);
    if (stamped) {
      stamps.step_mark(1);
      stamps.step_mark(2);
    }
    if (t + 1 < nk) {
      // Loads of the stages after t + 1 may stay in flight, and the request made at the start.
      const bool young = t == 0 && extra;
      if (NBUF >= 4 && deep && t == tail) {
        if (young) wait_vmcnt<2 * LOADS + 1>(); else wait_vmcnt<2 * LOADS>();
      } else if (NBUF >= 3 && deep && t == tail + NBUF - 3) {
        if (young) wait_vmcnt<LOADS + 1>(); else wait_vmcnt<LOADS>();
      } else {
        if (young) wait_vmcnt<1>(); else wait_vmcnt<0>();
      }
      if (t + 1 == loader.last_stage) loader.fix_last_stage(t + 1, lds + un * G::STAGE);
      stage_barrier();
    }
    if (stamped) stamps.step_mark(3);
    phase(1, [&](int r) { read(0, next, r); }, std::integral_constant<int, 0>{}, nothing);  // past K: unused
    if (stamped) stamps.step_mark(4);
    u = un;
  }
  // A traced launch's k-loop ends when every wave's does.
  if constexpr (!std::is_same_v<Stamps, NoStamps>) phase_barrier();
}

// The FMA path's k-loop with stage loads straight into LDS:
// compute(stage, first k, issue) once per stage, which calls issue(l) for l = 0
// .. LOADS - 1 somewhere in it.  Stages t and t + 1 share two buffers: while
// stage t is multiplied, issue asks for the loads of stage t + 1, into the
// buffer that every wave has left since the barrier before (the first two
// stages are asked for ahead of the loop).  One wait and one barrier a stage.
// No load waits in registers, and one copy of the multiplying code serves every
// stage: staged through a ring of three register sets it came in five copies
// (40 KB).  256 problems of 16 to 256 in each dimension (893 tiles): 31.2 ->
// 29.3 us, with FmaTile's vector epilogue 26.0, with every tile fixed 21.2, with
// the unrolled slices 20.8.  A launch like that is bound by each tile's own
// chain: a 64 x 64 tile 256 deep takes 6.8 us of FMAs, all tiles together 5.9 us
// of the chip.
template <class G, class Compute, class OnStart, class Stamps>
__device__ __forceinline__ void run_k_loop_fma(const gg_device_problem_desc& p, int m0, int n0, uint16_t* lds,
                                               int wave, Compute&& compute, OnStart&& on_start, const Stamps& stamps) {
  using L = DmaLoader<G>;
  constexpr int NBUF = G::BUFFERS;
  constexpr int LOADS = L::LOADS;
  static_assert(NBUF == 2, "the waits below are those of two buffers");
  const int nk = (p.k + G::BK - 1) / G::BK;
  if (nk <= 0) {
    on_start();
    return;
  }
  const L loader(p, m0, n0, wave);
  loader.issue(0, lds);
  if (nk > 1) loader.issue(1, lds + G::STAGE);
  const bool extra = __builtin_amdgcn_readfirstlane(on_start() ? 1 : 0) != 0;
  // In flight behind the loads of stage 0: those of stage 1 and the request.
  if (nk == 1) {
    if (extra) wait_vmcnt<1>(); else wait_vmcnt<0>();
  } else {
    if (extra) wait_vmcnt<LOADS + 1>(); else wait_vmcnt<LOADS>();
  }
  stamps.mark(GGK_PHASE_FIRST_STAGE);
  if (loader.last_stage == 0) loader.fix_last_stage(0, lds);
  stage_barrier();
  stamps.mark(GGK_PHASE_K_LOOP);
#pragma unroll 1
  for (int t = 0; t < nk; ++t) {
    uint16_t* const stage = lds + (t & 1) * G::STAGE;
    uint16_t* const next = lds + ((t + 1) & 1) * G::STAGE;
    const bool ask = t > 0 && t + 1 < nk;
    compute(stage, t * G::BK, [&](int l) {
      if (ask) loader.issue_load(t + 1, next, l);
    });
    if (t + 1 < nk) {
      // The loads of stage t + 1; the request made at the start may stay in flight once.
      if (t == 0 && extra) wait_vmcnt<1>(); else wait_vmcnt<0>();
      if (t + 1 == loader.last_stage) loader.fix_last_stage(t + 1, next);
      stage_barrier();
    }
  }
}

// ---------------------------------------------------------------------------
// MFMA tile: v_mfma_f32_16x16x32_f16, (BM/WM) x (BN/64) waves, each owning a
// WM x 64 block of D held as (WM/16) x 4 16x16 accumulators.  Per product the
// 16x16x32 form reads and writes half the accumulators of the 32x32x16 one: on
// random data, where the chip's power sets the clock, one 8192^3 problem took
// 836 us with it against 873 us (though 630 against 590 us on zeros, where the
// clock is at its limit).  Both give the same bits.
//
// D is computed transposed, with B as the instruction's first operand and A as
// its second: a lane then holds 4 consecutive columns of one row of D, as the
// epilogue reads C and writes D.
//
// Operand layouts of v_mfma_f32_16x16x32_f16 (lane l of 64):
//   A: row l%16, k = 8*(l/16) + e, e = 0..7 (one 16-byte read of an A row)
//   B: col l%16, k = 8*(l/16) + e
//   D: acc[r] = D[l%16][4*(l/16) + r], r = 0..3
// B sits in LDS row-major ([k][n]); ds_read_b64_tr_b16 turns four k-rows of
// 16 columns into the k-contiguous operand.  Within each group of 16 lanes it
// returns, to lane i, element i%4 of the 8-byte chunk addressed by lane
// 4*e + i/4 of the group, for e = 0..3.  Lane j of the group therefore
// addresses row kb + j/4, columns nb + 4*(j%4), and lane i receives
// B[kb + e][nb + i].
// ---------------------------------------------------------------------------
// Epilogue chunks of C requested ahead of the one being written (for blocks
// written in three or more chunks): C comes from HBM, and with two chunks in
// flight its latency is paid about half as often.
#ifndef GG_EPI_AHEAD
#define GG_EPI_AHEAD 2
#endif
template <class G, int WM_>
struct MfmaTile {
  static constexpr int WM = WM_;
  static constexpr int WN = 64;
  static constexpr int WAVES_M = G::BM / WM;
  static constexpr int WAVES_N = G::BN / WN;
  static constexpr int FM = WM / 16;
  static constexpr int FN = WN / 16;
  static_assert(WAVES_M * WAVES_N * kWave == G::THREADS, "one wave per block of D");
  static_assert(WM % 32 == 0, "whole 16-row blocks, in pairs");
  // The full 256 x 256 work tile in 128 x 64 wave blocks.
  static constexpr bool PHASED = G::BM == 256 && G::BN == 256 && G::BK == 64 && G::THREADS == 512 && WM == 128;
  // 16-row blocks of D per epilogue chunk: the whole block up to 64 rows (16 C
  // vectors, 64 registers), 32 rows per chunk for larger blocks, which hold
  // more registers.
  static constexpr int EPI_BLOCKS = FM <= 4 ? FM : 2;
  static_assert(FM % EPI_BLOCKS == 0, "whole chunks");
  // Blocks written in one chunk (64 registers of C) ask for their C before the
  // k-loop's first loads, so that it arrives with them instead of after the
  // last stage: mixed-512 217.2 -> 214.0 us, a ragged 24-problem set 142.2 ->
  // 140.5.  The 128 x 64 blocks have no registers left for it.
  static constexpr bool EARLY_C = FM <= 4;

  // Multiplies one LDS stage into acc (64-bit addressing form).  All MFMAs of a
  // stage are issued unconditionally; skipping is decided once per tile for the
  // whole wave.
  __device__ __forceinline__ static void compute_stage(const uint16_t* stage, int lane, int wm, int wn,
                                                       floatx4_t (&acc)[FM][FN]) {
    const uint16_t* as = stage;
    const uint16_t* bs = stage + G::A_STAGE;
    lane = opaque_lane();
    const int g = lane >> 4;
    const int j = lane & 15;
    // Operand fragments of k-step s (32 deep) of the stage.
    auto load_frags = [&](int s, half8_t (&af)[FM], half8_t (&bf)[FN]) {
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) {
        const uint16_t* src = as + G::a_piece(wm * WM + fm * 16 + j, 4 * s + g);
        af[fm] = *reinterpret_cast<const half8_t*>(src);
      }
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
        const int kb = s * 32 + 8 * g;
        // Rows kb + j/4 and kb + 4 + j/4 share one swizzle.
        const uint16_t* src = bs + G::b_chunk(kb + (j >> 2), wn * WN + fn * 16 + 4 * (j & 3));
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((GG_LDS short4_t*)(src));
        const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((GG_LDS short4_t*)(src + 4 * G::SB));
        bf[fn] = __builtin_bit_cast(half8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    constexpr int STEPS = G::BK / 32;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      half8_t af[FM];
      half8_t bf[FN];
      load_frags(s, af, bf);
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) {
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
          acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[fn], af[fm], acc[fm][fn], 0, 0, 0);
        }
      }
    }
  }

  // Computes the work tile at (m0, n0) as wave `wave`; on_start as in the k-loops, and
  // after_k_loop() once by every thread when the k-loop is over (no LDS read
  // of this tile follows it: the epilogue works from registers).
  template <bool WIDE, class OnStart, class AfterKLoop, class Stamps>
  __device__ __forceinline__ static void run(const gg_device_problem_desc& p, int m0, int n0, uint16_t* lds,
                                             int wave, OnStart&& on_start, AfterKLoop&& after_k_loop,
                                             const Stamps& stamps) {
    const int lane = opaque_lane();
    const int wm = wave / WAVES_N;
    const int wn = wave % WAVES_N;
    // A wave whose block starts past the problem's edge has nothing to store; it
    // still stages its share of A and B for the others.  The pipelined k-loops
    // multiply for it all the same.  A branch past the MFMAs of such waves took
    // 64 experts' 1.24 MFMAs per useful one down (2427 -> 2400 us), but breaks up
    // the interleaving of MFMAs, reads and loads: 24 ragged problems 140.5 -> 143, a
    // 16-expert layer 29.9 -> 31.2, column-edge tiles 3 to 5% slower.
    const bool live = m0 + wm * WM < p.m && n0 + wn * WN < p.n;

    floatx4_t acc[FM][FN];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const bool use_c = p.c != nullptr && p.beta != 0.0f;
    const int r0 = m0 + wm * WM, c0 = n0 + wn * WN;
    CVectors early;
    if constexpr (!WIDE && EARLY_C) {
      if (live && use_c) load_c(p, r0, c0, lane, 0, early);
    }

    auto compute = [&](const uint16_t* stage) {
      if (live) compute_stage(stage, lane, wm, wn, acc);
    };
    if constexpr (WIDE) {
      run_k_loop<G>(p, m0, n0, lds, wave, compute, on_start, stamps);
    } else if constexpr (PHASED) {
      run_k_loop_phased<G>(p, m0, n0, lds, wave, wm, wn, acc, on_start, stamps);
    } else {
      run_k_loop_halves<G, WM>(p, m0, n0, lds, wave, wm, wn, acc, on_start, stamps);
    }
    after_k_loop();

    if (live) store_tile<WIDE>(p, r0, c0, lane, acc, use_c, early);
    stamps.wave_done();
  }

  // 4 x 4 transpose across the 4 lanes of a quad: lane q holds x[k] = M[q][k]
  // and receives M[k][q], in two exchange steps (partner q^1, then q^2).
  __device__ __forceinline__ static void quad_transpose(float (&x)[4], int q) {
    const auto xor1 = [](float v) {
      return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));
    };
    const auto xor2 = [](float v) {
      return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xf, 0xf, true));
    };
    // Exchanged by every lane (a lane that is switched off would send zeros), then selected.
    const float s0 = xor1(x[1]), s1 = xor1(x[0]), s2 = xor1(x[3]), s3 = xor1(x[2]);
    const bool odd = (q & 1) != 0, high = (q & 2) != 0;
    const float y0 = odd ? s0 : x[0];
    const float y1 = odd ? x[1] : s1;
    const float y2 = odd ? s2 : x[2];
    const float y3 = odd ? x[3] : s3;
    const float t0 = xor2(y2), t1 = xor2(y3), t2 = xor2(y0), t3 = xor2(y1);
    x[0] = high ? t0 : y0;
    x[1] = high ? t1 : y1;
    x[2] = high ? y2 : t2;
    x[3] = high ? y3 : t3;
  }

  // D = alpha * acc + beta * C for the wave's block at (r0, c0).
  //
  // Lane (g, j) = (lane / 16, lane % 16) holds, of 16x16 block (fm, fn), row
  // 16 fm + j, columns 16 fn + 4 g .. + 3.  A 4 x 4 transpose in each quad of
  // lanes (over fn, for each of the 4 columns) gives lane (g, 4 jj + q) the
  // rows 16 fm + 4 jj + r, r = 0..3, columns 16 q + 4 g .. + 3: C is read and
  // D written as 16-byte vectors (a dword access costs the address unit as
  // much as a 16-byte one), and one access instruction covers 4 rows x 64
  // columns, 256 contiguous bytes of each row.  Rows of tightly packed matrices
  // (ldc = ldd = N) seldom start on a 128-byte line, and 256 contiguous bytes of
  // such a row span 3 lines where four separate 64-byte pieces span 6.
  //
  // With 32-bit addressing C is read through a buffer resource from (r0, c0)
  // to the end of C: rows past M read as zero, so the loads need no branch.
  // The block is written in chunks of EPI_BLOCKS 16-row blocks, and all C
  // vectors of the next chunk (two, for blocks of three or more chunks) are
  // requested before the current one is written, so their latencies overlap.
  // Stores go through the same kind of resource; columns that cross N go
  // element by element.
  // C vectors of a chunk: [16-row block][row of the lane].
  struct CVectors {
    floatx4_t v[EPI_BLOCKS][4];
  };

  // Requests the C vectors of a chunk of the block at (r0, c0).
  __device__ __forceinline__ static void load_c(const gg_device_problem_desc& p, int r0, int c0, int lane, int chunk,
                                                CVectors& dst) {
    const int row_lane = 4 * ((lane >> 2) & 3);           // first of the lane's 4 rows in a 16-row block
    const int col = 16 * (lane & 3) + 4 * (lane >> 4);  // first of its 4 columns in the wave block
    const __amdgpu_buffer_rsrc_t crs =
        buffer_rsrc(p.c + ((int64_t)r0 * p.ldc + c0), 4 * ((int64_t)(p.m - 1 - r0) * p.ldc + (p.n - c0)));
#pragma unroll
    for (int i = 0; i < EPI_BLOCKS; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = (chunk * EPI_BLOCKS + i) * 16 + row_lane + r;
        // Vectors wholly past N would read the next row's head: an offset past the resource.
        const uint32_t off =
            c0 + col < p.n ? 4u * ((uint32_t)row * (uint32_t)p.ldc + col) : DmaLoader<G>::kOutOfRange;
        dst.v[i][r] = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(crs, (int)off, 0, 0));
      }
  }

  template <bool WIDE>
  __device__ __forceinline__ static void store_tile(const gg_device_problem_desc& p, int r0, int c0, int lane,
                                                    const floatx4_t (&acc)[FM][FN], bool use_c,
                                                    const CVectors& early) {
    if constexpr (!WIDE) {
      const int q = lane & 3;
      const int row_lane = 4 * ((lane >> 2) & 3);   // first of the lane's 4 rows in a 16-row block
      const int col = 16 * q + 4 * (lane >> 4);     // first of its 4 columns in the wave block
      const int ncol = p.n - (c0 + col);            // how many of them lie inside the matrix
      const __amdgpu_buffer_rsrc_t drs =
          buffer_rsrc(p.d + ((int64_t)r0 * p.ldd + c0), 4 * ((int64_t)(p.m - 1 - r0) * p.ldd + (p.n - c0)));
      constexpr int CHUNKS = FM / EPI_BLOCKS;
      constexpr int AHEAD = CHUNKS >= 3 ? GG_EPI_AHEAD : 1;
      CVectors cv[AHEAD + 1];
      auto request_c = [&](int chunk, CVectors& dst) {
        if (use_c) {
          load_c(p, r0, c0, lane, chunk, dst);
        } else {
#pragma unroll
          for (int i = 0; i < EPI_BLOCKS; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) dst.v[i][r] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
      };
      if constexpr (EARLY_C) {
        if (use_c) {
          cv[0] = early;
        } else {
          request_c(0, cv[0]);
        }
      } else {
#pragma unroll
        for (int c = 0; c < AHEAD; ++c) {
          if (c < CHUNKS) request_c(c, cv[c]);
        }
      }
#pragma unroll
      for (int chunk = 0; chunk < CHUNKS; ++chunk) {
        if (chunk + AHEAD < CHUNKS) request_c(chunk + AHEAD, cv[(chunk + AHEAD) % (AHEAD + 1)]);
#pragma unroll
        for (int i = 0; i < EPI_BLOCKS; ++i) {
          const int fm = chunk * EPI_BLOCKS + i;
          float v[4][4];  // [column of the lane][row of the lane]
#pragma unroll
          for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int fn = 0; fn < 4; ++fn) v[e][fn] = acc[fm][fn][e];
            quad_transpose(v[e], q);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = fm * 16 + row_lane + r;
            floatx4_t out;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              out[e] = epilogue_value(v[e][r], cv[chunk % (AHEAD + 1)].v[i][r][e], p.alpha, use_c ? p.beta : 0.0f);
            }
            if (r0 + row >= p.m || ncol <= 0) continue;
            const uint32_t off = 4u * ((uint32_t)row * (uint32_t)p.ldd + col);
            if (ncol >= 4) {
              __builtin_amdgcn_raw_buffer_store_b128(
                  __builtin_bit_cast(__attribute__((ext_vector_type(4))) int, out), drs, (int)off, 0, 0);
            } else {
#pragma unroll
              for (int e = 0; e < 3; ++e) {
                if (e < ncol) __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(out[e]), drs, (int)(off + 4 * e), 0, 0);
              }
            }
          }
        }
        // Keep each chunk's loads and stores in place: hoisting every C load
        // to the top would hold the whole block's C in registers.
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) {
        const int row = r0 + fm * 16 + (lane & 15);
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
          const int col = c0 + fn * 16 + 4 * (lane >> 4);
          const int ncol = p.n - col;
          if (row >= p.m || ncol <= 0) continue;
          g_cf32_t* crow = (g_cf32_t*)p.c + ((int64_t)row * p.ldc + col);
          g_f32_t* drow = (g_f32_t*)p.d + ((int64_t)row * p.ldd + col);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (e < ncol) {
              drow[e] = epilogue_value(acc[fm][fn][e], use_c ? crow[e] : 0.0f, p.alpha, use_c ? p.beta : 0.0f);
            }
          }
        }
      }
    }
  }
};

// ---------------------------------------------------------------------------
// FMA tile: 256 threads as a 16 x 16 grid, thread (tm, tn) owns rows
// tm*RM .. tm*RM+RM-1 and columns tn*RN .. tn*RN+RN-1 of the macro-tile, with
// RM = BM/16, RN = BN/16 float32 accumulators.  Per 8-deep k slice a thread
// reads one 16-byte piece of each of its A rows and one RN-wide piece of each
// B row from LDS, then issues RM*RN*8 fused multiply-adds in ascending k.
// Used when MFMA is not requested (use_tensor_cores = false).
//
// The slices of a stage are unrolled and left to the compiler to schedule.
// Reading each slice ahead of the one being multiplied needs another RM*4 +
// RN*4 registers: the larger tiles then hold two workgroups a CU instead of
// three, and every tile pays in issue slots.  37 problems of 300 to 1400 rows and
// columns, K 256 to 512: 64x64x16 348 -> 333 us, 128x64x32 374 -> 350, 64x128x32
// 358 -> 340; 300 problems of 16 to 400: 41.3 -> 40.4, 65 -> 62, 64.8 -> 54.8.
// ---------------------------------------------------------------------------
template <class G>
struct FmaTile {
  static constexpr int RM = G::BM / 16;
  static constexpr int RN = G::BN / 16;
  static_assert(RN == 4 || RN == 8, "column block must be one or two LDS chunks");
  static_assert(G::THREADS == 256, "16 x 16 thread grid");

  // One accumulator tile of 4 x 4 leaves registers for C beside the k-loop's.
  static constexpr bool SMALL = RM * RN <= 16;
  static constexpr int SLICES = G::BK / 8;
  static constexpr int LOADS = DmaLoader<G>::LOADS;
  static_assert(LOADS <= SLICES, "a stage's loads go out one a slice");

  // Multiplies a stage whose first krem values of k lie inside the problem.
  // issue(l) asks for load l of the next stage: one a slice behind its operand
  // reads in the 4 x 4 form, where a lone workgroup has nothing else to hide
  // them behind (64 problems 1024 to 4096 deep: 193 -> 181 us), else all ahead of
  // the slices (the larger tiles lose up to 4% with the loads spread out).
  template <class Issue>
  __device__ __forceinline__ static void compute_stage(const uint16_t* stage, int krem, int tm, int tn,
                                                       float (&acc)[RM][RN], Issue&& issue) {
    using brow_t = std::conditional_t<RN == 4, half4_t, half8_t>;
    if constexpr (!SMALL) issue_all(issue);
#pragma unroll
    for (int k8 = 0; k8 < SLICES; ++k8) {
      if (k8 * 8 >= krem) break;  // loads follow full stages only
      half8_t av[RM];
      brow_t bv[8];
#pragma unroll
      for (int i = 0; i < RM; ++i) av[i] = *reinterpret_cast<const half8_t*>(stage + G::a_piece(tm * RM + i, k8));
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        bv[kk] = *reinterpret_cast<const brow_t*>(stage + G::A_STAGE + G::b_chunk(k8 * 8 + kk, tn * RN));
      }
      if constexpr (SMALL) {
        if (k8 < LOADS) issue(k8);
      }
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
#pragma unroll
        for (int i = 0; i < RM; ++i) {
          const float a = (float)av[i][kk];
#pragma unroll
          for (int j = 0; j < RN; ++j) acc[i][j] = __builtin_fmaf(a, (float)bv[kk][j], acc[i][j]);
        }
      }
    }
  }
  template <class Issue>
  __device__ __forceinline__ static void issue_all(Issue&& issue) {
#pragma unroll
    for (int l = 0; l < LOADS; ++l) issue(l);
  }

  // Computes the work tile at (m0, n0); on_start and after_k_loop as in
  // MfmaTile::run.
  template <bool WIDE, class OnStart, class AfterKLoop, class Stamps>
  __device__ __forceinline__ static void run(const gg_device_problem_desc& p, int m0, int n0, uint16_t* lds,
                                             int wave, OnStart&& on_start, AfterKLoop&& after_k_loop,
                                             const Stamps& stamps) {
    const int tid = threadIdx.x;
    const int tm = tid >> 4;
    const int tn = tid & 15;
    // Wave w holds tm = 4w .. 4w+3, i.e. rows [4w*RM, 4w*RM + 4*RM) of the tile.
    const bool active = m0 + (tid / kWave) * 4 * RM < p.m;

    float acc[RM][RN];
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int j = 0; j < RN; ++j) acc[i][j] = 0.0f;

    // The thread's part of C, as 16-byte vectors through a buffer resource from
    // the wave's first row (vectors past N read as zero).  The 4 x 4 form asks
    // for it before the k-loop's loads (read and written as dwords after the
    // k-loop: 29.3 us where this takes 26.0, 256 problems of 16 to 256 in each
    // dimension), the others, which have no registers left for it beside three
    // waves per SIMD, when the k-loop ends, ahead of the hand-over.
    const bool use_c = p.c != nullptr && p.beta != 0.0f;
    const int r0 = __builtin_amdgcn_readfirstlane(m0 + (tid / kWave) * 4 * RM);
    floatx4_t cv[RM][RN / 4];
    auto request_c = [&](int t) {
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int v = 0; v < RN / 4; ++v) cv[i][v] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
      if (WIDE || !use_c || !active) return;
      const __amdgpu_buffer_rsrc_t crs =
          buffer_rsrc(p.c + ((int64_t)r0 * p.ldc + n0), 4 * ((int64_t)(p.m - 1 - r0) * p.ldc + (p.n - n0)));
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int v = 0; v < RN / 4; ++v) {
          const int row = ((t & (kWave - 1)) >> 4) * RM + i, col = (t & 15) * RN + 4 * v;
          const uint32_t off = n0 + col < p.n ? 4u * ((uint32_t)row * (uint32_t)p.ldc + (uint32_t)col)
                                              : DmaLoader<G>::kOutOfRange;
          cv[i][v] = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(crs, (int)off, 0, 0));
        }
    };
    if constexpr (SMALL) request_c(tid);

    if constexpr (WIDE) {
      int kt = 0;
      run_k_loop<G>(p, m0, n0, lds, wave, [&](const uint16_t* stage) {
        if (active) compute_stage(stage, p.k - kt * G::BK, tm, tn, acc, [](int) {});
        ++kt;
      }, on_start, stamps);
    } else {
      run_k_loop_fma<G>(p, m0, n0, lds, wave, [&](const uint16_t* stage, int k0, auto&& issue) {
        if (active) {
          compute_stage(stage, p.k - k0, tm, tn, acc, issue);
        } else {
          issue_all(issue);
        }
      }, on_start, stamps);
    }
    if constexpr (!SMALL) request_c(opaque_tid(wave));
    after_k_loop();

    if (!active) {
      stamps.wave_done();
      return;
    }
    if constexpr (WIDE) {
      g_cf32_t* cptr = (g_cf32_t*)p.c;
      g_f32_t* dptr = (g_f32_t*)p.d;
#pragma unroll
      for (int i = 0; i < RM; ++i) {
        const int row = m0 + tm * RM + i;
        if (row >= p.m) continue;
        float ce[RN];
#pragma unroll
        for (int j = 0; j < RN; ++j) {
          const int col = n0 + tn * RN + j;
          ce[j] = (use_c && col < p.n) ? cptr[(int64_t)row * p.ldc + col] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < RN; ++j) {
          const int col = n0 + tn * RN + j;
          if (col >= p.n) continue;
          dptr[(int64_t)row * p.ldd + col] = epilogue_value(acc[i][j], ce[j], p.alpha, use_c ? p.beta : 0.0f);
        }
      }
    } else {
      const int t = opaque_tid(wave);  // its parts are not held through the k-loop
      const __amdgpu_buffer_rsrc_t drs =
          buffer_rsrc(p.d + ((int64_t)r0 * p.ldd + n0), 4 * ((int64_t)(p.m - 1 - r0) * p.ldd + (p.n - n0)));
#pragma unroll
      for (int i = 0; i < RM; ++i) {
        const int row = ((t & (kWave - 1)) >> 4) * RM + i;
        if (r0 + row >= p.m) continue;
#pragma unroll
        for (int v = 0; v < RN / 4; ++v) {
          const int col = (t & 15) * RN + 4 * v;
          const int ncol = p.n - (n0 + col);
          const uint32_t off = 4u * ((uint32_t)row * (uint32_t)p.ldd + (uint32_t)col);
          floatx4_t out;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            out[e] = epilogue_value(acc[i][4 * v + e], cv[i][v][e], p.alpha, use_c ? p.beta : 0.0f);
          }
          if (ncol >= 4) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) int, out), drs,
                                                   (int)off, 0, 0);
          } else {
#pragma unroll
            for (int e = 0; e < 3; ++e) {
              if (e < ncol) __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(out[e]), drs, (int)(off + 4 * e), 0, 0);
            }
          }
        }
      }
    }
    stamps.wave_done();
  }
};

// The tile code of kernel shape S (gg_common.h).
template <class S, int PATH> struct TileFor;
template <class S> struct TileFor<S, GGK_PATH_MFMA> { using type = MfmaTile<typename S::G, S::WAVE_M>; };
template <class S> struct TileFor<S, GGK_PATH_FMA> { using type = FmaTile<typename S::G>; };

// LDS (binary16 values) a kernel of shape S needs: the largest stage ring of
// the forms its work tiles take.
template <class S, bool CLASSES = S::CLASSES>
struct KernelLds {
  static constexpr int HALVES = S::G::LDS_HALVES;
};
template <class S>
struct KernelLds<S, true> {
  static constexpr int a = S::G::LDS_HALVES, r = S::GR::LDS_HALVES, c = S::GC::LDS_HALVES, rc = S::GRC::LDS_HALVES;
  static constexpr int ab = a > r ? a : r;
  static constexpr int cd = c > rc ? c : rc;
  static constexpr int HALVES = ab > cd ? ab : cd;
  static_assert(2 * HALVES <= 150 * 1024, "the stage rings and the scheduler's words fit the 160 KB of LDS");
};

// Computes the work tile at (m0, n0): in the edge class its extent inside the
// problem selects (KernelShape::CLASSES), else in the kernel's own form.  The
// class is uniform across the workgroup (scalar descriptor and origin).
template <class S, int PATH, bool WIDE, class OnStart, class AfterKLoop, class Stamps = NoStamps>
__device__ __forceinline__ void run_work_tile(const gg_device_problem_desc& p, int m0, int n0,
                                              StageRing<KernelLds<S>::HALVES>& ring, int wave, OnStart&& on_start,
                                              AfterKLoop&& after_k_loop, const Stamps& stamps = Stamps{}) {
  uint16_t* const lds = ring.values;
  if constexpr (PATH == GGK_PATH_MFMA && !WIDE && S::CLASSES) {
    const bool rows = p.m - m0 <= S::G::BM / 2;
    const bool cols = p.n - n0 <= S::G::BN / 2;
    // The full form first: its code then follows the dispatch as it would
    // without the edge classes.
    if (__builtin_expect(!rows && !cols, 1)) {
      TileFor<S, PATH>::type::template run<false>(p, m0, n0, lds, wave, on_start, after_k_loop, stamps);
    } else if (!cols) {
      MfmaTile<typename S::GR, S::WAVE_M_R>::template run<false>(p, m0, n0, lds, wave, on_start, after_k_loop, stamps);
    } else if (!rows) {
      MfmaTile<typename S::GC, S::WAVE_M_C>::template run<false>(p, m0, n0, lds, wave, on_start, after_k_loop, stamps);
    } else {
      MfmaTile<typename S::GRC, S::WAVE_M_RC>::template run<false>(p, m0, n0, lds, wave, on_start, after_k_loop, stamps);
    }
  } else {
    TileFor<S, PATH>::type::template run<WIDE>(p, m0, n0, lds, wave, on_start, after_k_loop, stamps);
  }
}

}  // namespace gg
