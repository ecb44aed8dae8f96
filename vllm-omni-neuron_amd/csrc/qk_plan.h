// Launch rules of the Q/K pass (norm, RoPE, key-norm maximum) and of the maximum alone. Plain C++ without HIP, so that it is checked on
// the CPU.
#pragma once

#include <stdint.h>

namespace wanmi {

struct QKPlan {
  int chunks;           // kernel instantiation: registers for this many chunks of four heads
  int waves;            // waves per workgroup
  int tokens_per_wave;
};

// `heads` a multiple of 4, at most 128; `rows`: tokens times parts; `maxnorm`: with the key-norm maximum.
//
// Tokens each wave walks. A token is one latency chain (its row, the reduction, the fp64 root, the
// write), so a wave's tokens are served one after another while other waves hide the latency: as many
// waves as one round holds (four workgroups of four waves per CU) come first, and only a sequence longer
// than that gives a wave more than one token. At most 8: an S = 32760 launch is then one resident
// round, and the gamma copy is shared by four waves' tokens. With 8 tokens per wave throughout, 512 / 1560 /
// 3600 tokens ran 34 / 43 / 47 us: 16 / 49 / 113 workgroups on 256 CUs, each eight such chains long. One
// token per wave took 24 us off the first, 22 off the second, 21 off the third (the block's
// cross-attention K/V 94 -> 69 us, row_mx_qkv_proj of 3600 tokens 387 -> 344).
//
// Waves per workgroup. With the key-norm maximum every workgroup ends in atomics on the same 160 bytes, which
// the XCDs' separate L2s leave to the memory side: about 45 ns a workgroup, one after another, so half as
// many workgroups of eight waves take half of it off (16 waves: as good, and 392 against 356 us at 75600
// tokens). With 4 / 8 waves, 40 heads: 19.0 / 16.2 us at 2500 tokens, 28.7 / 22.5 at 4096, 37.5 / 31.1 at
// 7800. Not once every wave has its 8 tokens (more than 28672): the pass is then bound by memory, and larger
// workgroups lengthen its end: 16 heads 49.7 / 51.0 us at 32760 tokens and 122.8 / 129.6 at 75600, 12 heads 96.5 /
// 99.5, 32 heads 270 / 278, 40 heads 338 / 338 (halves 352 / 356). Up to 8 heads the atomics still bound it: 71.3 /
// 62.5, 4 heads 46.2 / 41.1.
// The instantiation is the smallest that holds the heads, for every pass: with the key-norm maximum 16 heads of
// 32760 tokens, halves, took 59.8 us with the registers and the gamma copy of 40 heads, 52.4 with their own.
inline QKPlan qk_plan(int heads, int64_t rows, bool maxnorm, int64_t cus) {
  constexpr int64_t kTokensPerWaveMax = 8;
  const int64_t resident = cus * 4 * 4;
  const int64_t n = (rows + resident - 1) / resident;
  QKPlan p{};
  p.tokens_per_wave = (int)(n < 1 ? 1 : n > kTokensPerWaveMax ? kTokensPerWaveMax : n);
  p.chunks = heads <= 16 ? 4 : heads <= 40 ? 10 : heads <= 64 ? 16 : 32;
  p.waves = maxnorm && heads <= 40 && (p.tokens_per_wave < kTokensPerWaveMax || heads <= 8) ? 8 : 4;
  return p;
}

// Waves per workgroup of the key-norm maximum alone over `rows` tokens: eight, which halve its atomics as above
// (4 / 8 waves, 40 heads: 9.2 / 7.7 us at 2500 tokens, 22.3 / 17.4 at 7800), but four where there are few
// workgroups anyway and the larger ones only take longer to end (5.2 / 5.7 at 256 tokens, 5.6 / 5.8 at 512, 6.1 / 6.0
// at 768), and four where memory bounds it (32 heads 71.5 / 78.6 at 50000, 40 heads 134.3 / 137.3 at 75600;
// below 256 MB eight: 24 heads 34.5 / 32.1 at 32760).
inline int head_max_norm_waves(int64_t rows, int heads) { return rows <= 640 || rows * heads > 1000000 ? 4 : 8; }

}  // namespace wanmi
