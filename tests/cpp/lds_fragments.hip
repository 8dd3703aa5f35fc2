// Host check of the fragment addresses the k-loops read operands at: each one
// is the place the LDS layout gives that fragment, for every wave, lane, stage
// and fragment of every work-tile form, wherever the stage buffers start.  Runs
// on the CPU (the address functions are host functions as well).
#include <stdio.h>

#include "gg_tiles.h"

using namespace gg;

static long long checked = 0, wrong = 0;

static void expect(uint32_t got, uint32_t want) {
  ++checked;
  if (got != want && wrong++ < 10) printf("fragment at %u, the layout has it at %u\n", got, want);
}

// run_k_loop_halves: WM x 64 wave blocks, stages of A then B.
template <class G, int WM>
static void check_halves(uint32_t base) {
  for (int wm = 0; wm < G::BM / WM; ++wm)
    for (int wn = 0; wn < G::BN / 64; ++wn)
      for (int lane = 0; lane < kWave; ++lane)
        for (int u = 0; u < G::BUFFERS; ++u)
          for (int h = 0; h < 2; ++h) {
            const int g = lane >> 4, j = lane & 15;
            const uint32_t stage = base + 2u * (uint32_t)(u * G::STAGE);
            for (int fm = 0; fm < WM / 16; ++fm) {
              expect(G::a_fragment(stage + 2u * (uint32_t)G::a_piece(wm * WM + j, g), h, 16 * fm * G::SA),
                     stage + 2u * (uint32_t)G::a_piece(wm * WM + 16 * fm + j, 4 * h + g));
            }
            for (int fn = 0; fn < 4; ++fn)
              for (int four = 0; four < 2; ++four) {
                const int k = 8 * g + (j >> 2), n = wn * 64 + 4 * (j & 3);
                expect(G::b_fragment(stage + 2u * (uint32_t)(G::A_STAGE + G::b_chunk(k, n)), fn, 32 * h * G::SB) +
                           8u * (uint32_t)(four * G::SB),
                       stage + 2u * (uint32_t)(G::A_STAGE + G::b_chunk(32 * h + k + 4 * four, n + 16 * fn)));
              }
          }
}

// run_k_loop_phased: units of 128 A rows or 32 B rows.
template <class G>
static void check_phased(uint32_t base) {
  using L = PhasedLoader<G>;
  for (int wave = 0; wave < 8; ++wave)
    for (int lane = 0; lane < kWave; ++lane)
      for (int parity = 0; parity < 2; ++parity) {
        const int wm = wave / 4, wn = wave % 4, g = lane >> 4, j = lane & 15;
        const uint32_t stage = base + 2u * (uint32_t)(parity * L::PARITY);
        for (int unit : {L::A0, L::A1})
          for (int fm = 0; fm < 4; ++fm)
            for (int s = 0; s < 2; ++s) {
              expect(G::a_fragment(stage + 2u * (uint32_t)G::a_piece(wm * 64 + j, g), s, unit + fm * 16 * G::SA),
                     stage + 2u * (uint32_t)(unit + G::a_piece(wm * 64 + 16 * fm + j, 4 * s + g)));
            }
        for (int unit : {L::B0, L::B1})
          for (int fn = 0; fn < 4; ++fn)
            for (int four = 0; four < 2; ++four) {
              const int k = 8 * g + (j >> 2), n = wn * 64 + 4 * (j & 3);
              expect(G::b_fragment(stage + 2u * (uint32_t)G::b_chunk(k, n), fn, unit) + 8u * (uint32_t)(four * G::SB),
                     stage + 2u * (uint32_t)(unit + G::b_chunk(k + 4 * four, n + 16 * fn)));
            }
      }
}

// Bases the type allows: wherever StageRing may be placed.
template <int V>
static void check_variant() {
  using S = KernelShape<V, GGK_PATH_MFMA>;
  constexpr size_t align = alignof(StageRing<KernelLds<S>::HALVES>);
  for (uint32_t base : {0u, (uint32_t)align, 3u * (uint32_t)align, 37u * (uint32_t)align}) {
    if constexpr (S::CLASSES) {
      check_phased<typename S::G>(base);
      check_halves<typename S::GR, S::WAVE_M_R>(base);
      check_halves<typename S::GC, S::WAVE_M_C>(base);
      check_halves<typename S::GRC, S::WAVE_M_RC>(base);
    } else {
      check_halves<typename S::G, S::WAVE_M>(base);
    }
  }
}

int main() {
  check_variant<GGK_VARIANT_64x64x16>();
  check_variant<GGK_VARIANT_128x64x32>();
  check_variant<GGK_VARIANT_64x128x32>();
  check_variant<GGK_VARIANT_64x64x16_SMALL>();
  check_variant<GGK_VARIANT_128x64x32_SMALL>();
  check_variant<GGK_VARIANT_64x128x32_SMALL>();
  printf("%lld fragment addresses checked, %lld wrong\n", checked, wrong);
  return wrong == 0 ? 0 : 1;
}
