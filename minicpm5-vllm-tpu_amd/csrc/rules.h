// Launch rules that are plain arithmetic on sizes (no HIP types: the CPU tests compile this header too).
#pragma once

#include <stddef.h>

namespace mk {

enum class GemmIn { I8, BF16, F8 };   // operands of a GEMM; F8: OCP e4m3 operands, f32 accumulation

// Whether GEMM tile `id` (GemmArgs::cfg) is built.  The SiLU epilogues need waves that hold whole 64-column
// [gate | up] blocks, which 5, 8, 9 and 10 have not; 6, 11 and 13 are never the faster choice for them, 12 only
// for them.  fp8 stages are one wide k-step held in four operand sets: with the 256x320 tile's 160 accumulators
// they exceed a wave's 256 registers.
constexpr bool gemm_tile_built(int id, bool silu, GemmIn in) {
  return silu ? id == 2 || id == 3 || id == 4 || id == 7 || id == 12
              : id >= 2 && id <= 13 && id != 12 && !(id == 8 && in == GemmIn::F8);
}

// Tile configuration for a problem: M x N outputs, kb bytes of K.  The busiest CU runs ceil(tiles / 256) tiles (the
// order spreads them evenly), so the estimate is ceil(tiles / 256) * tile area / relative throughput, the throughputs
// measured on MI355X at the model's shapes (random data): the 8-wave ping-pong 256x256 tile is fastest per tile,
// except for the SiLU epilogue, whose VALU work is hidden better by two co-resident 256x128 workgroups.  The 256x320
// tile's 1.14: the QKV shape M = 8192, N = 2560, K = 1536 (dequantising epilogue, no routing) takes 40.9 us on it,
// 48.6 us on 256x192 tiles (1.75 rounds) and 52.3 us on 256x256 ones (1.25 rounds); with 128-byte stages 37.5 against
// 39.5 us, and 41.9 on 256x192.  The SiLU 256x256 tile's 1.10 (1.15 fits its own times, 125 us for the 1B gate/up at
// M = 8192 against 130 on 256x128 pairs): inside the model the pairs take 127 us there against 130, and the attention
// next to them 231 against 240.
inline int gemm_tile(bool silu, GemmIn in, int M, int N, int kb) {
  const bool line = kb % 128 == 0;   // whole 128-byte stages
  const int lines = kb / 128;
  auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  auto fits = [&](int bm, int bn) { return tiles(bm, bn) <= 256; };
  // Few tiles (short prompts): the smallest tile whose tiling fits one round of 256 CUs, on whole-line stages.
  // Measured on MI355X over M = 40 .. 3072 at the model's shapes, us warm / with cold weights, against the next
  // larger choice:
  //   32x64   1B down M = 256  17.8 / 19.3 (64x64 17.8 / 23.2), 2B down M = 128  21.9 / 25.0 (22.1 / 31.3)
  //   64x64   1B down M = 512  19.1 / 23.4 (64x128 25.4 / 33.5), 1B QKV M = 384  6.5 / 7.1 (8.1 / 9.7)
  //   64x128  1B down M = 1024  27.3 / 32.9 (64x128 with 64-byte stages 30.5 / 43.6); K loops of 32 or more
  //           lines only: at 12 (int8, K = 1536) the 64-byte stages start sooner, 7.5 against 8.3 at M = 512
  //   128x128 1B down M = 2048  40.4 / 43.6 (64-byte stages 44.3 / 55.0), likewise for 32 or more lines
  // The SiLU epilogues need 64-column waves: 64x128 with 64-byte stages (1B gate/up M = 128  6.9 / 11.8 against
  // 7.9 / 9.9 on whole lines), then 128x128 with three workgroups per CU (M = 256  9.6 / 14.2 against
  // 13.7 / 17.8 on 256x128 tiles, M = 384  11.0 / 14.6 against 14.8 / 17.9).
  if (!silu && line) {
    if (fits(32, 64)) return 10;
    if (fits(64, 64)) return 9;
    if (lines >= 32 && fits(64, 128)) return 11;
  }
  if (kb >= 1024 && fits(64, 128)) return 7;
  if (!silu && line && lines >= 32 && fits(128, 128)) return 6;
  // up to two 128x128 workgroups per CU: 1B down at M = 4096 72.3 -> 60.4 us (before: one 256x128 tile per CU),
  // O at M = 3072 34.5 -> 29.5, QKV at M = 2500 19.4 -> 18.0, 2B down at M = 4096 103 -> 96.9 (256x256 109)
  if (!silu && line && !fits(128, 128) && tiles(128, 128) <= 512) return 13;
  if (silu && fits(128, 128)) return 3;
  struct Opt { int id, bm, bn; double eff; };
  const Opt opts[6] = {{4, 256, 256, silu ? 1.10 : 1.33}, {2, 256, 128, 1.0}, {3, 128, 128, 0.85},
                       {5, 256, 192, 1.25},               {8, 256, 320, 1.14}, {12, 192, 128, 1.0}};
  int best = 2;
  double bt = 1e300;
  for (const Opt& o : opts) {
    if (!gemm_tile_built(o.id, silu, in)) continue;
    if (silu && o.id == 3) continue;   // the problems it is the faster SiLU tile for are above
    // 192x128 pairs fill rounds the larger tiles leave half empty: 2B gate/up at M = 1536 52.0 -> 43.9 us, at
    // M = 3072 88.4 -> 82.6, 1B gate/up at M = 6000 103 -> 96.7
    if (o.id == 12 && !line) continue;
    // but alone on its CU, three rows of int8 tiles lose to two of 256x128: 1B gate/up at M = 400 15.3 us, now 14.8
    // (M = 576, three rows either way, 15.1 against 16.6; bf16 24.0 against 27.2)
    if (o.id == 12 && in == GemmIn::I8 && fits(192, 128) && M > 384 && M <= 512) continue;
    const long rounds = (tiles(o.bm, o.bn) + 255) / 256;
    const double t = (double)rounds * o.bm * o.bn / o.eff;
    if (t < bt * 0.999) {
      bt = t;
      best = o.id;
    }
  }
  return best;
}

// Byte ranges that otherwise idle workgroups of a launch read and drop (attn.hip): a hint that leaves the
// data in the memory-side cache for the launches that follow.  No result depends on it.
struct PrefetchRanges {
  const void* p[4];
  size_t bytes[4];   // 0: unused
};

// The ranges that `spare` workgroups can read while an attention launch over sequences of S tokens runs anyway;
// the launch lasts until the last of them is done.  One workgroup reads 72 - 75 KB/us (8 of them took 111 us for
// the 2B layer's 64 MB); 64 KB/us are counted, over 8 us and, at hd 128, 1.25 us per 64-key tile of the longest
// q tile.  Ranges are taken whole or left out: a GEMM waits for the cold rest of its weights as for all of them
// (2B (12, 128), us per forward: nothing read 7029, 55 of 64 MB 7255, all 6948).  Forwards, us, without a
// prefetch / all ranges / this rule: 2B (31, 128) 12844 / 17265 / 12841, (6, 640) 13047 / 14489 / 12957,
// (1, 1920) 8959 / 9957 / 9133, (20, 128) 10469 / 9920 / 9938, (8, 128) 5555 / 5213 / 5212; 1B (31, 128)
// 5164 / 6748 / 5192, (12, 128) 3189 / 3075 / 3077, (1, 512) 2119 / 1893 / 1894.
inline PrefetchRanges prefetch_fit(PrefetchRanges pf, int spare, int hd, int S) {
  const double us = 8.0 + 1.25 * hd / 128 * (S / 64);
  double left = spare * 64.0 * 1024 * us;
  for (int r = 0; r < 4; ++r) {
    if ((double)pf.bytes[r] > left) {
      pf.p[r] = nullptr;
      pf.bytes[r] = 0;
    }
    left -= (double)pf.bytes[r];
  }
  return pf;
}

inline bool prefetch_any(const PrefetchRanges& pf) {
  return pf.bytes[0] || pf.bytes[1] || pf.bytes[2] || pf.bytes[3];
}

// Waves per attention workgroup: 8, or 4, which doubles the items (items8 of 8 waves) and leaves one wave per SIMD.
// A lone wave's step is 5 - 25 % shorter, so the longest q tile finishes sooner while every item has a CU to itself
// (us, 8 then 4 waves: 64 items hd 128 31.3, 25.8, hd 96 23.2, 21.5; 128 items hd 128 51.9, 45.1, hd 96 39.5, 37.7).
// Beyond that some CUs take a second item, which mostly costs more than it gains ((4, 768), 192 items: hd 128 27.3,
// 33.6, hd 96 20.8, 27.9; (2, 1536): hd 96 32.6, 36.8).  At hd 128 a batch of one or two long sequences has few long
// tiles and the second items are its short ones: there 4 waves still win, with the K / V preparation, up to 15/16 of
// the CUs for one sequence ((1, 3200) 80.1, 74.3; (1, 3584) 87.8, 84.5; (1, 3840) 94.0, 93.5; (1, 3968) 97.5, 98.5)
// and below 3/4 for two ((2, 1216) 41.2, 39.4; (2, 1344) 44.5, 42.8; (2, 1536) 48.6, 49.9).  Inside a model the CUs
// that 8 waves leave free read the next weights, which is worth more from 3/4 of the CUs on for one sequence and at
// any size for two (forwards, ms, 8 then 4 waves: 2B (1, 3456) 13.7, 14.2, (1, 3840) 15.2, 15.9, (2, 1280) 10.6, 11.4; 1B
// (1, 3456) 6.50, 6.48, (1, 3840) 6.53, 6.89, (2, 1280) 4.06, 4.29).
inline int attn_waves(int items8, int ncu, int hd, int B, bool prefetch) {
  if (2 * items8 <= ncu) return 4;
  if (hd == 128 && B == 1 && 16 * items8 <= (prefetch ? 12 : 15) * ncu) return 4;
  if (hd == 128 && B == 2 && 4 * items8 < 3 * ncu && !prefetch) return 4;
  return 8;
}

// Whether a pass of the LM head over `rows` rows (V columns, K elements) takes the skinny kernel: no barriers to pay
// for and 64 columns per workgroup, where the batch kernel's workgroups hold 128.  So it wins while few rows share
// the weights and its workgroups all run in one round of 256 CUs (us, skinny then batch kernel: V = 8192, H = 1536,
// 1 row 10.3, 13.5, 8 rows 11.9, 13.5, 16 rows 13.7, 13.6; H = 4096, 2 rows 27.8, 33.6, 16 rows 31.5, 33.7;
// V = 16384, H = 2048, 2 rows 8 % apart), but not beyond (V = 20480: the batch kernel takes 0.77 times as long).
// There it wins for one row over more than six chunks of K (V = 130560, H = 2048: 93.4, 96.5), and for two where the
// batch kernel's workgroups fill whole rounds of three per CU or more (95.7, 98.6; V = 65536: 9 % slower).
inline bool lm_head_skinny(int rows, int V, int K) {
  if (V <= 64 * 256 && rows <= (8 + K / 384 < 16 ? 8 + K / 384 : 16)) return true;
  return K > 1536 && (rows == 1 || (rows == 2 && V >= 3 * 128 * 256));
}

}  // namespace mk
