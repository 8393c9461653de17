// w4a16_few.hip -- fused W4A16 GEMM for few rows (M <= 128): decode and the
// verify step of a few users, where the work is reading the packed weights
// once.  C [M, N] = A [M, K] . W [K, N] with bf16 or fp16 activations and the
// weight format of w4a16_gemm.hip.
//
// A work-group owns 128 columns of C and one of S k ranges.  Each pipeline
// step moves 128 k -- the packed words of its columns (8 KiB), their scale
// and zero rows and the matching columns of A -- by direct HBM -> LDS
// transfers into a ring, kStages steps ahead (all of the CU's LDS: a
// transfer from HBM takes 2-3 us here, so the bytes in flight set the rate).
// Wave (nw, kw) of the eight multiplies columns 64 nw .. and k-slice 32 kw ..
// of the step on 16 x 16 x 32 MFMAs.  Lane l reads 16 bytes of words: columns
// 4 (l % 16) .. + 3 of word row l / 16 of its slice, so that each word is
// exactly its part of one MFMA's B operand (k = 8 (l / 16) .. + 7 of one
// column): the weights are dequantised in registers, each once for all rows.
// (Column tile j of the wave is columns 4 c + j, c = 0 .. 15, which leaves
// every lane four consecutive columns of the result.)  The four k-slices'
// sums meet in LDS in wave order; with S > 1, fp32 partials go to the
// workspace and are summed in split order, so every result is reproducible.
//
// At most 16 rows take w4row_kernel instead, operands straight to registers.
// (For more rows that form was slower, gate/up at M = 63 41 us against 31:
// loads return in order, so a wave's words, from HBM, hold back its A
// operands, as many bytes again per row tile, from L2.)
//
// us per call, weights from HBM, before (256-row tiles, w4a16_gemm.hip) ->
// now, at the 8B target's gate/up / down / QKV / O shapes:
//   M = 1    60 / 34 / 21 / 18  ->  19 / 14 / 13 / 12
//   M = 63   64 / 37 / 27 / 25  ->  31 / 22 / 17 / 15
//   M = 128  68 / 40 / 28 / 25  ->  45 / 30 / 23 / 22
// Bound: the words from HBM (59 MB for gate/up: 12 us at the rate of a large
// copy), the start and the drain of a short kernel, and from M = 17 on the
// transfers of A (one copy per 128 columns, from L2).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include "abi_internal.hpp"
#include "lds_dma.hpp"
#include "silu.hpp"
#include "w4a16_few.hpp"

namespace cfa {
namespace w4few {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kBN = 128;            // columns per work-group
constexpr int kSK = 32;             // k per MFMA
constexpr int kStep = 128;          // k per pipeline step
constexpr int kWaves = 8;
constexpr int kNT = 64 * kWaves;
constexpr int kWBytes = kStep / 8 * kBN * 4;  // packed words of a step, 8 KiB
constexpr int kSBytes = 4 * 2 * kBN * 2;      // a scale and a zero row per k-slice, 2 KiB

struct Args {
  const uint16_t *A;  // [M, K]
  const uint32_t *q;  // [K / 8, N]
  const __half *s;    // [K / group, N]
  const __half *z;    // [K / group, N] or null
  uint16_t *C;        // [M, N], or [M, N / 2] with the SiLU epilogue
  float *part;        // [S, M, N] (out == kPart)
  int M, N, K, S;
  int tiles;          // column tiles
  int steps;          // pipeline steps per split
  int spg;            // k-slices of 32 per scale group
  SliceDiv group_of;  // division by spg
  int out;            // Out
};
enum Out : int { kPlain = 0, kSilu = 1, kPart = 2 };

template <int MT>
struct Cfg {
  static constexpr int kABytes = MT * 16 * kStep * 2;
  static constexpr int kStage = kABytes + kWBytes + kSBytes;
  static constexpr int kStages = std::min(10, 150 * 1024 / kStage);
  // transfers (1 KiB) of a stage, and per wave (the last ones repeat)
  static constexpr int kX = kStage / 1024;
  static constexpr int kLPI = (kX + kWaves - 1) / kWaves;
  // row tiles whose wave sums meet in the ring's LDS at a time
  static constexpr int kRT = MT == 8 ? 2 : MT;
  static_assert(kStages >= 3 && kStages * kStage >= kWaves * kRT * 4096, "LDS");
  static_assert((kStages - 1) * kLPI < 64, "vmcnt");
};

// s_waitcnt vmcnt(N) lgkmcnt(0)
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | (((N >> 4) & 3) << 14));
}

// Byte P of v as a float (v_cvt_f32_ubyte<P>, see w4a16_gemm.hip).
template <int P>
__device__ __forceinline__ float ubyte_f32(uint32_t v) {
  float r;
  asm("v_cvt_f32_ubyte%2 %0, %1" : "=v"(r) : "v"(v), "i"(P));
  return r;
}
// How the weights are formed: kBf16 bf16((nibble - z) * s), bit for bit what
// cfa_w4a16_dequant writes; kBf16Fma bf16(fma(nibble, s, -z * s)), within one
// bf16 step of it and one instruction a weight less, as w4a16_gemm.hip does;
// kF16 (fp16(nibble) - z) * s in fp16, bit for bit cfa_w4a16_dequant's.
enum Form : int { kBf16 = 0, kBf16Fma = 1, kF16 = 2 };

// Columns' scales and zero points as the dequantisation uses them.
template <int FORM>
struct Scale {
  float s, z;
  __device__ __forceinline__ void set(uint32_t sh, uint32_t zh) {
    s = __half2float(__ushort_as_half((uint16_t)sh));
    z = __half2float(__ushort_as_half((uint16_t)zh));
    if constexpr (FORM == kBf16Fma) z = -z * s;
  }
  __device__ __forceinline__ float weight(float n) const {
    return FORM == kBf16Fma ? __builtin_fmaf(n, s, z) : (n - z) * s;
  }
  template <int P>
  __device__ __forceinline__ uint32_t pair(uint32_t lo, uint32_t hi) const {
    return __builtin_bit_cast(
        uint32_t, __builtin_convertvector(f32x2{weight(ubyte_f32<P>(lo)), weight(ubyte_f32<P>(hi))}, bf16x2));
  }
  __device__ __forceinline__ bf16x8 word(uint32_t w) const {
    const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;
    return __builtin_bit_cast(bf16x8, make_uint4(pair<0>(lo, hi), pair<1>(lo, hi), pair<2>(lo, hi), pair<3>(lo, hi)));
  }
  // A operand as loaded
  static __device__ __forceinline__ bf16x8 a_op(const uint4 &a) { return __builtin_bit_cast(bf16x8, a); }
  static __device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
// fp16, each operation rounded to fp16: nibbles k and k + 4 of the word become the fp16
// pair 1024 + n (bits 0x6400 | n), 1024 is subtracted exactly, and z and s
// follow on the packed fp16 unit.  The operand then holds k in the order
// 0 4 1 5 2 6 3 7, and so does A's (a_op).
template <>
struct Scale<kF16> {
  f16x2 s, z;
  __device__ __forceinline__ void set(uint32_t sh, uint32_t zh) {
    const _Float16 sf = __builtin_bit_cast(_Float16, (uint16_t)sh), zf = __builtin_bit_cast(_Float16, (uint16_t)zh);
    s = f16x2{sf, sf};
    z = f16x2{zf, zf};
  }
  __device__ __forceinline__ uint32_t pair(uint32_t w) const {
    const f16x2 n = __builtin_bit_cast(f16x2, (w & 0x000f000fu) | 0x64006400u) -
                    f16x2{(_Float16)1024.0f, (_Float16)1024.0f};
    return __builtin_bit_cast(uint32_t, (n - z) * s);
  }
  __device__ __forceinline__ f16x8 word(uint32_t w) const {
    return __builtin_bit_cast(f16x8, make_uint4(pair(w), pair(w >> 4), pair(w >> 8), pair(w >> 12)));
  }
  static __device__ __forceinline__ f16x8 a_op(const uint4 &a) {
    return __builtin_bit_cast(f16x8, make_uint4(__builtin_amdgcn_perm(a.z, a.x, 0x05040100u),
                                                __builtin_amdgcn_perm(a.z, a.x, 0x07060302u),
                                                __builtin_amdgcn_perm(a.w, a.y, 0x05040100u),
                                                __builtin_amdgcn_perm(a.w, a.y, 0x07060302u)));
  }
  static __device__ __forceinline__ f32x4 mfma(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

template <int FORM>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (FORM == kF16)
    return __builtin_bit_cast(uint32_t, f16x2{(_Float16)a, (_Float16)b});
  else
    return silu_pk(a, b);
}

// A wave's sums of one 16 x 64 tile at row r0, column n0 (v[j][e]: row
// 4 (lane / 16) + e, column 4 (lane % 16) + j) to the output.
template <int FORM>
__device__ __forceinline__ void store_tile(const Args &a, const f32x4 (&v)[4], int r0, int n0, int split) {
  const int lane = threadIdx.x & 63, g = lane >> 4, col = lane & 15;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = r0 + 4 * g + e;
    if (a.out == kSilu) {
      // columns 0 .. 31 of a 64-column tile are gate features, 32 .. 63
      // their up columns: lane col < 8 pairs with lane col + 8
      const float p0 = __shfl_xor(v[0][e], 8, 64), p1 = __shfl_xor(v[1][e], 8, 64);
      const float p2 = __shfl_xor(v[2][e], 8, 64), p3 = __shfl_xor(v[3][e], 8, 64);
      if (row < a.M && col < 8)
        *reinterpret_cast<uint2 *>(a.C + (long long)row * (a.N / 2) + n0 / 2 + 4 * col) =
            make_uint2(silu_gate2(v[0][e], p0, v[1][e], p1), silu_gate2(v[2][e], p2, v[3][e], p3));
    } else if (row < a.M) {
      const int c0 = n0 + 4 * col;
      if (a.out == kPart)
        *reinterpret_cast<float4 *>(a.part + ((long long)split * a.M + row) * a.N + c0) =
            make_float4(v[0][e], v[1][e], v[2][e], v[3][e]);
      else
        *reinterpret_cast<uint2 *>(a.C + (long long)row * a.N + c0) =
            make_uint2(pack2<FORM>(v[0][e], v[1][e]), pack2<FORM>(v[2][e], v[3][e]));
    }
  }
}

template <int MT, int FORM>
__global__ __launch_bounds__(kNT, 2) void w4few_kernel(Args a) {
  using Cf = Cfg<MT>;
  using Sc = Scale<FORM>;
  constexpr int kS = Cf::kStages, LPI = Cf::kLPI;
  __shared__ __align__(16) uint8_t lds[kS * Cf::kStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = wave & 1, kw = wave >> 1;
  const int g = lane >> 4, col = lane & 15;
  // work-groups go to the 8 XCDs round-robin by linear index: each XCD takes
  // an eighth of the column tiles, next to each other
  const int per = (a.tiles + 7) / 8, tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if ((int)blockIdx.x / 8 >= per || tile >= a.tiles) return;
  const int n0 = tile * kBN, split = blockIdx.y;
  const int u0 = split * a.steps, nu = min(a.K / kStep, u0 + a.steps) - u0;  // this split's steps
  if (nu <= 0) return;  // (never: the host sizes the splits)

  // This wave's transfers of a stage, x = LPI wave + j: A (4 rows of 256
  // bytes, 16-byte chunk c of row r at position c ^ (r % 16)), then the words
  // (2 rows), then the scales (lanes 0-15 the scale row of k-slice 2 y, 16-31
  // its zero row, 32-63 those of slice 2 y + 1).  A and the words go from a
  // uniform base, advanced per step, and a lane's constant offset.  (Every
  // wave issues the same number, so one wait count serves all; leaving out
  // the repeats and A's rows past M was no faster.)
  const uint8_t *base[LPI];
  uint32_t voff[LPI];
#pragma unroll
  for (int j = 0; j < LPI; ++j) {
    const int x = min(LPI * wave + j, Cf::kX - 1);
    if (x < MT * 4) {
      const int row = 4 * x + (lane >> 4), c = (lane & 15) ^ (row & 15);
      base[j] = reinterpret_cast<const uint8_t *>(a.A) + (long long)u0 * (kStep * 2);
      voff[j] = ((uint32_t)min(row, a.M - 1) * (uint32_t)a.K + 8u * c) * 2u;
    } else {
      const int row = 2 * (x - MT * 4) + (lane >> 5);
      base[j] = reinterpret_cast<const uint8_t *>(a.q + n0) + (long long)u0 * (kStep / 8) * a.N * 4;
      voff[j] = ((uint32_t)row * (uint32_t)a.N + 4u * (lane & 31)) * 4u;
    }
  }
  const long long wstep = (long long)(kStep / 8) * a.N * 4;
  // the stage of step u0 + u (past the split's end its last step again)
  int iu = 0, islot = 0;
  auto issue = [&]() __attribute__((always_inline)) {
    uint8_t *st = lds + islot * Cf::kStage;
    const bool more = iu + 1 < nu;
#pragma unroll
    for (int j = 0; j < LPI; ++j) {
      const int x = min(LPI * wave + j, Cf::kX - 1);
      uint8_t *dst = st + 1024 * x;
      if (x < MT * 4 + kWBytes / 1024) {
        dma16_s(base[j], voff[j], (CFA_LDS void *)dst);
        if (more) base[j] += x < MT * 4 ? kStep * 2 : wstep;
      } else {
        const uint32_t sl = 4u * (uint32_t)(u0 + iu) + 2u * (x - MT * 4 - kWBytes / 1024) + (lane >> 5);
        const long long grp = slice_group(sl, a.group_of);
        const __half *t = (lane & 16) && a.z ? a.z : a.s;
        dma16(t + grp * a.N + n0 + 8 * (lane & 15), (CFA_LDS void *)dst);
      }
    }
    iu += more ? 1 : 0;
    islot = islot + 1 == kS ? 0 : islot + 1;
  };

  f32x4 acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // operand offsets in a stage
  const int aoff = col * (kStep * 2) + (((4 * kw + g) ^ col) << 4);
  const int woff = Cf::kABytes + (4 * kw + g) * (kBN * 4) + (64 * nw + 4 * col) * 4;
  const int soff = Cf::kABytes + kWBytes + kw * 512 + (64 * nw + 4 * col) * 2;
  const uint32_t zmask = a.z != nullptr ? 0xffffffffu : 0u;

  struct Ops {
    uint4 w;
    uint2 s, z;
    uint4 x[MT];
  };
  int slot = 0;
  auto read_ops = [&](Ops &o) __attribute__((always_inline)) {  // the next stage's
    const uint8_t *st = lds + slot * Cf::kStage;
    slot = slot + 1 == kS ? 0 : slot + 1;
    o.w = *reinterpret_cast<const uint4 *>(st + woff);
    o.s = *reinterpret_cast<const uint2 *>(st + soff);
    o.z = *reinterpret_cast<const uint2 *>(st + soff + 256);
#pragma unroll
    for (int i = 0; i < MT; ++i) o.x[i] = *reinterpret_cast<const uint4 *>(st + aoff + i * 16 * kStep * 2);
  };
  auto multiply = [&](const Ops &o) __attribute__((always_inline)) {
    const uint2 z = make_uint2(o.z.x & zmask, o.z.y & zmask);
    Sc s0, s1, s2, s3;
    s0.set(o.s.x & 0xffff, z.x & 0xffff);
    s1.set(o.s.x >> 16, z.x >> 16);
    s2.set(o.s.y & 0xffff, z.y & 0xffff);
    s3.set(o.s.y >> 16, z.y >> 16);
    const auto b0 = s0.word(o.w.x), b1 = s1.word(o.w.y), b2 = s2.word(o.w.z), b3 = s3.word(o.w.w);
    decltype(Sc::a_op(o.x[0])) xa[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) xa[i] = Sc::a_op(o.x[i]);
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i][0] = Sc::mfma(xa[i], b0, acc[i][0]);
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i][1] = Sc::mfma(xa[i], b1, acc[i][1]);
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i][2] = Sc::mfma(xa[i], b2, acc[i][2]);
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i][3] = Sc::mfma(xa[i], b3, acc[i][3]);
  };
  // Every step issues one stage's transfers (past the split's end too, to
  // slots no longer read), so that the waits always count the same.  At step
  // t, after the barrier, stage t + 1 has landed (kS - 2 later ones are in
  // flight) and every wave has read stage t into registers, which frees its
  // slot for stage t + kS; the wave reads stage t + 1's operands and
  // multiplies stage t's.
  for (int u = 0; u < kS; ++u) issue();
  wait_vm_lgkm0<(kS - 1) * LPI>();
  block_barrier();
  Ops o0, o1;
  read_ops(o0);
  auto step = [&](const Ops &cur, Ops &nxt) __attribute__((always_inline)) {
    wait_vm_lgkm0<(kS - 2) * LPI>();
    block_barrier();
    issue();
    read_ops(nxt);
    multiply(cur);
  };
  int t = 0;
  for (; t + 1 < nu; t += 2) {
    step(o0, o1);
    step(o1, o0);
  }
  if (t < nu) multiply(o0);
  wait_vm_lgkm0<0>();  // the last steps' repeat transfers have landed

  // acc[i][j][e]: row 16 i + 4 g + e, column n0 + 64 nw + 4 col + j.  Row
  // tile i of column half nw is summed over the k-slices and stored by wave
  // (nw, i % 4).
  f32x4 *red = reinterpret_cast<f32x4 *>(lds);
  constexpr int RT = Cf::kRT;
#pragma unroll
  for (int i0 = 0; i0 < MT; i0 += RT) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[((wave * RT + i) * 4 + j) * 64 + lane] = acc[i0 + i][j];
    __syncthreads();
    if (kw >= RT) continue;
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = red[((nw * RT + kw) * 4 + j) * 64 + lane];
#pragma unroll
      for (int k = 1; k < 4; ++k) v[j] += red[(((2 * k + nw) * RT + kw) * 4 + j) * 64 + lane];
    }
    store_tile<FORM>(a, v, 16 * (i0 + kw), n0 + 64 * nw, split);
  }
}

// M <= 16: a work-group owns 64 columns, its eight waves one k range each,
// and both operands go straight to registers, kRowDepth steps of 32 k ahead
// (in pairs, whose A operands share 128-byte lines).  A is so small that it
// hits the cache, and no barrier ties the waves together: gate/up at M = 1
// 18.7 us against 22.9 with the ring (59 MB of words), down 13.7 against 17.
constexpr int kRowBN = 64;
constexpr int kRowDepth = 4;
template <int FORM>
__global__ __launch_bounds__(kNT) void w4row_kernel(Args a) {
  using Sc = Scale<FORM>;
  __shared__ f32x4 red[kWaves * 4 * 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, col = lane & 15;
  const int n0 = blockIdx.x * kRowBN, split = blockIdx.y;
  const int c0 = n0 + 4 * col;  // this lane's columns c0 .. c0 + 3
  // this wave's steps: whole pairs (K % 128 == 0)
  const int pairs = a.K / (2 * kSK), parts = a.S * kWaves, p = split * kWaves + wave;
  const int t0 = 2 * (int)((long long)p * pairs / parts), t1 = 2 * (int)((long long)(p + 1) * pairs / parts);
  const uint32_t *qp = a.q + (long long)g * a.N + c0;
  const uint16_t *ap = a.A + (long long)min(col, a.M - 1) * a.K + 8 * g;
  uint4 W[kRowDepth], X[kRowDepth];
  auto issue = [&](int slot, int t) __attribute__((always_inline)) {  // (past the end: the last pair again)
    t = min(t, t1 - 2);
#pragma unroll
    for (int k = 0; k < 2; ++k) X[slot + k] = *reinterpret_cast<const uint4 *>(ap + (long long)(t + k) * kSK);
#pragma unroll
    for (int k = 0; k < 2; ++k)
      W[slot + k] = *reinterpret_cast<const uint4 *>(qp + (long long)(t + k) * (kSK / 8) * a.N);
  };
  f32x4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (t0 < t1) {
    // scales: the current group's as operands, the next one's as loaded
    Sc sc[4];
    uint2 ns, nz = make_uint2(0, 0);
    auto load_scales = [&](int grp) __attribute__((always_inline)) {
      grp = min(grp, (t1 - 1) / a.spg);
      ns = *reinterpret_cast<const uint2 *>(a.s + (long long)grp * a.N + c0);
      if (a.z) nz = *reinterpret_cast<const uint2 *>(a.z + (long long)grp * a.N + c0);
    };
    auto take_scales = [&]() __attribute__((always_inline)) {
      sc[0].set(ns.x & 0xffff, nz.x & 0xffff);
      sc[1].set(ns.x >> 16, nz.x >> 16);
      sc[2].set(ns.y & 0xffff, nz.y & 0xffff);
      sc[3].set(ns.y >> 16, nz.y >> 16);
    };
    int grp = t0 / a.spg, left = (grp + 1) * a.spg - t0;  // steps left in the group
    load_scales(grp);
#pragma unroll
    for (int d = 0; d < kRowDepth; d += 2) issue(d, t0 + d);
    take_scales();
    load_scales(grp + 1);
    for (int t = t0; t < t1; t += kRowDepth) {
#pragma unroll
      for (int d = 0; d < kRowDepth; ++d) {
        if (t + d < t1) {
          if (left == 0) {
            take_scales();
            ++grp;
            load_scales(grp + 1);
            left = a.spg;
          }
          --left;
          const uint4 w = W[d];
          const auto x = Sc::a_op(X[d]);
          acc[0] = Sc::mfma(x, sc[0].word(w.x), acc[0]);
          acc[1] = Sc::mfma(x, sc[1].word(w.y), acc[1]);
          acc[2] = Sc::mfma(x, sc[2].word(w.z), acc[2]);
          acc[3] = Sc::mfma(x, sc[3].word(w.w), acc[3]);
        }
        if (d % 2 == 1) issue(d - 1, t + d - 1 + kRowDepth);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) red[(wave * 4 + j) * 64 + lane] = acc[j];
  __syncthreads();
  if (wave != 0) return;
  f32x4 v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[j] = red[j * 64 + lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v[j] += red[(w * 4 + j) * 64 + lane];
  }
  store_tile<FORM>(a, v, 0, n0, split);
}

// C = fp16 of the sum of the split partials in split order.
__global__ __launch_bounds__(256) void w4few_reduce_f16_kernel(const float *part, uint16_t *C, long long MN,
                                                               int splits) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= MN) return;
  float4 acc = *reinterpret_cast<const float4 *>(part + i);
  for (int s = 1; s < splits; ++s) {
    const float4 v = *reinterpret_cast<const float4 *>(part + (long long)s * MN + i);
    acc.x += v.x;
    acc.y += v.y;
    acc.z += v.z;
    acc.w += v.w;
  }
  *reinterpret_cast<uint2 *>(C + i) = make_uint2(pack2<kF16>(acc.x, acc.y), pack2<kF16>(acc.z, acc.w));
}

// As many splits as fill the CUs (one work-group each), of at least 4 steps;
// w4row_kernel: enough for 192 work-groups of at least 128 k per wave
// (unsplit from N = 12288 on, where the reduction would cost more than the
// idle CUs).  At most 16 of them, as w4a16_gemm.hip takes for more rows, so
// that a workspace for more rows serves these too; past 16 the partials cost
// more than the CUs give (us at M = 1 / 64 / 128, without and with the bound:
// N = 1024, K = 14336 12.5 / 20.0 / 25.0 -> 10.9 / 17.1 / 22.4; N = 256, K =
// 65536 22.7 / 68.4 / 88.5 -> 15.5 / 36.0 / 48.5).
int splits(int M, int N, int K) {
  if (M <= kRowM) {
    int S = 1;
    while (S < kMaxSplits && N / kRowBN * S < 192 && K / (2 * S * kWaves) >= 128) S *= 2;
    return S;
  }
  const int tiles = N / kBN, steps = K / kStep;
  const int cus = abi::device_cu_count();
  const int S = std::max(1, std::min({cus / tiles, steps / 4, kMaxSplits}));
  const int per = (steps + S - 1) / S;
  return (steps + per - 1) / per;
}

}  // namespace w4few
}  // namespace cfa

int cfa::w4few::launch(const void *a, const uint32_t *b_quant, const void *scales, const void *zeros, int M,
                       int N, int K, int group, int form, void *c, float *part, int S, int out, void *stream) {
  Args g{};
  g.A = (const uint16_t *)a;
  g.q = b_quant;
  g.s = (const __half *)scales;
  g.z = (const __half *)zeros;
  g.C = (uint16_t *)c;
  g.part = part;
  g.M = M;
  g.N = N;
  g.K = K;
  g.S = S;
  g.tiles = N / kBN;
  g.steps = (K / kStep + S - 1) / S;
  g.spg = group / kSK;
  g.group_of = slice_div((uint32_t)g.spg);
  g.out = out;
  const dim3 grid((unsigned)((g.tiles + 7) / 8 * 8), (unsigned)S);
  hipStream_t st = (hipStream_t)stream;
  const dim3 rgrid((unsigned)(N / kRowBN), (unsigned)S);
#define CFA_FEW(FORM)                                                                                \
  do {                                                                                               \
    if (M <= kRowM)                                                                                  \
      CFA_LAUNCH("w4a16_gemm_few", w4row_kernel<FORM>, rgrid, dim3(kNT), 0, st, g);                    \
    else if (M <= 32)                                                                                \
      CFA_LAUNCH("w4a16_gemm_few", (w4few_kernel<2, FORM>), grid, dim3(kNT), 0, st, g);                \
    else if (M <= 64)                                                                                \
      CFA_LAUNCH("w4a16_gemm_few", (w4few_kernel<4, FORM>), grid, dim3(kNT), 0, st, g);                \
    else                                                                                             \
      CFA_LAUNCH("w4a16_gemm_few", (w4few_kernel<8, FORM>), grid, dim3(kNT), 0, st, g);                \
  } while (0)
  switch (form) {
    case kF16: CFA_FEW(kF16); break;
    case kBf16Fma: CFA_FEW(kBf16Fma); break;
    default: CFA_FEW(kBf16); break;
  }
#undef CFA_FEW
  return CFA_OK;
}

int cfa::w4few::reduce_f16(const float *part, void *c, long long MN, int S, void *stream) {
  CFA_LAUNCH("w4a16_gemm_few_reduce", w4few_reduce_f16_kernel, dim3((unsigned)((MN / 4 + 255) / 256)), dim3(256),
             0, (hipStream_t)stream, part, (uint16_t *)c, MN, S);
  return CFA_OK;
}
