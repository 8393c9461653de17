// w4a16_few.hpp -- host interface of the few-row W4A16 GEMM (w4a16_few.hip),
// to which the entry points of w4a16_gemm.hip route small M.
#pragma once

#include <stdint.h>

#include "common.hpp"

namespace cfa {
namespace w4few {

// Eight 16-row tiles, the most whose sums a wave's registers hold.  Gate/up of
// the 8B target, us: M = 64 31, 65 42 (eight tiles from there), 128 43, and
// 129 68 on w4a16_gemm.hip's 256-row tiles.
constexpr int kMaxM = 128;
constexpr int kMaxSplits = 16;

// Shapes the kernels take: w4few_kernel (17 rows and more) moves the words of
// 16 word rows by 32-bit byte offsets, 64 N bytes and a line.
constexpr int kRowM = 16;
constexpr int kMaxN = 1 << 26;
inline bool takes(int M, int N, int K) {
  return M > 0 && M <= kMaxM && N > 0 && N % 128 == 0 && K > 0 && K % 128 == 0 && (M <= kRowM || N <= kMaxN);
}

// The group of k-slice sl without a division: sl / d = mulhi(2 sl, mul) >>
// shift with mul = ceil(2^(31 + shift) / d) and shift = ceil(log2 d), exact
// for every d >= 1 and sl < 2^26 (K < 2^31): mul d = 2^(31 + shift) + e with
// e < d <= 2^shift, so the product is at most sl e < 2^(26 + shift) too
// large, below the 2^(31 + shift) / d of a quotient's step (the same number
// with shift 0 and 2^32 was exact only for sl d < 2^32).
struct SliceDiv {
  uint32_t mul;
  int shift;
};
inline SliceDiv slice_div(uint32_t d) {
  int s = 0;
  while ((1ull << s) < d) ++s;
  return SliceDiv{(uint32_t)(((1ull << (31 + s)) + d - 1) / d), s};
}
CFA_HD uint32_t slice_group(uint32_t sl, SliceDiv d) {
  return (uint32_t)(((uint64_t)(2u * sl) * d.mul) >> 32) >> d.shift;
}

// Splits of K for a shape that it takes.
int splits(int M, int N, int K);

// form: how the weights are formed (0 bf16 as cfa_w4a16_dequant, 1 bf16 as
// cfa_w4a16_gemm_zp, 2 fp16).  out: 0 C [M, N], 1 SiLU-gated C [M, N / 2] (S == 1), 2 fp32 partials
// part [S, M, N].  The caller has checked shapes and 16-byte alignment.
int launch(const void *a, const uint32_t *b_quant, const void *scales, const void *zeros, int M, int N, int K,
           int group, int form, void *c, float *part, int S, int out, void *stream);

// c [MN] fp16 = the partials' sum in split order
int reduce_f16(const float *part, void *c, long long MN, int S, void *stream);

}  // namespace w4few
}  // namespace cfa
