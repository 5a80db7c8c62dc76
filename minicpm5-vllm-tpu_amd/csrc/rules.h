// Launch rules that are plain arithmetic on sizes (no HIP types: the CPU tests compile this header too).
#pragma once

#include <stddef.h>

namespace mk {

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
// and below 3/4 for two ((2, 1216) 41.2, 39.4; (2, 1344) 44.5, 42.8; (2, 1536) 48.6, 49.9).  Inside a model the CUs that 8
// waves leave free read the next weights, which is worth more from 3/4 of the CUs on for one sequence (2B forward:
// (1, 3456) 13.96 ms, 14.40; (1, 3840) 15.3, 15.9) and for two (1B (2, 1280) 3.98, 4.67).
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
