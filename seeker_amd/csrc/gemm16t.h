// The wide f16 GEMM's large-tile kernel: y = W x over more than 64 columns with
// the reference's wide-GEMM arithmetic (ops/matmul.rs:433-446 ->
// mul_mm_cm.slang: weights dequantized and rounded to f16, activations rounded
// to f16, f32 accumulation).
//
// A workgroup of 4 waves (one per SIMD) covers 16 row tiles x 32 CG columns:
// wave w decodes tiles 4 w .. 4 w + 3 of its own (two pairs of 32 rows) and
// multiplies each pair by all CG groups of 32 columns, so a B fragment read
// from LDS feeds the matrix core for 64 clocks. That ratio is what the shape is
// chosen for: at half of it (8 waves of 2 tiles) the B reads of a CU need its
// whole LDS bandwidth at the matrix cores' peak rate (1 KB per 32 clocks per
// SIMD = 128 B per clock). One wave per SIMD hides nothing by itself, so the
// loop is software-pipelined by hand: while the 4 CG MFMAs of a sub-block (32
// k) run, the wave reads the next sub-block's B fragments (each into the
// register its own last use freed) and decodes the next sub-block's weights, a
// few instructions in the shadow of every MFMA.
//
// Staging: B in stages of 64 k through a ring of three LDS buffers, the weight
// words and row headers in stages of 128 k through two (they are read into
// registers at once, so two cover two stages ahead). Every load is a direct
// global -> LDS load issued unconditionally (past the last stage it repeats the
// last one into a buffer nobody reads), so the waits are exact counts.
//
// Bound by the matrix cores and the decode issue: 28672 x 4096 x 2048 columns
// 498 us (966 TFLOP/s; a library f16 product of that size reaches ~1210), 192
// columns 60 us against 69 with 8 waves of 2 tiles (k_gemm16w3_q4k) in passes
// of 192. Without the decode (timing only) 1.35x faster, without the B loads
// 1.04x.
#pragma once
#include <type_traits>

#include "sh_internal.h"
#include "sh_dma.h"
#include "sh_qkv.h"

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
struct alignas(16) u32x4 { uint32_t x, y, z, w; };

__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }

// f16(p.lo * a + c), f16(p.hi * a + c) of an f16 pair, each rounded once (see
// q4r_frag16 in gemv.hip: a masked nibble is the f16 subnormal q 2^-24).
__device__ __forceinline__ uint32_t fma_mix_pair(uint32_t p, float a, float c) {
  uint32_t r;
  asm("v_fma_mixlo_f16 %0, %1, %2, %3 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
      : "=&v"(r)
      : "v"(p), "v"(a), "v"(c));
  return r;
}

template <int N, class Fn, int I = 0>
__device__ __forceinline__ void static_for(Fn&& fn) {
  if constexpr (I < N) {
    fn(std::integral_constant<int, I>{});
    static_for<N, Fn, I + 1>(static_cast<Fn&&>(fn));
  }
}

// acc += A B with the accumulator held in AGPRs, in place. As asm: with the
// builtin the compiler rotates the loop-carried accumulators through other
// registers (172 moves per 192 MFMAs of 16x16x32). It does not see the matrix
// instruction's register hazards here, which the loop's distances cover: an
// accumulator is used again 2 CG MFMAs later, a weight fragment is complete
// before the sub-block that reads it starts (mfma_fence).
__device__ __forceinline__ void mfma_acc(f16v& acc, h8 a, h8 b) {
  asm("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// Wait states between the vector instructions that wrote a fragment and the
// MFMAs that read it.
__device__ __forceinline__ void mfma_fence() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 3" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// The weight formats. A lane serves one row of a pair of 16-row tiles: row
// lane % 16 of tile (lane / 16) % 2. The MFMA's k index is free as long as both
// operands use the same one: MFMA j of a sub-block (32 k) takes the 8-element
// groups g = 2 j and 2 j + 1 of the tile layout, group 2 j + lane / 32 in this
// lane.
//   issue  loads stage h (128 k) of a tile into LDS
//   read   a tile pair's stage into registers (w: the lane's own tile)
//   scale  the factors of sub-block mp
//   pair   f16 elements 2 i, 2 i + 1 of the lane's 8 of MFMA j

// Q4_K: a stage (half a superblock) of a tile is its 1 KB of nibble words and
// the 256 B row header (d | dmin << 16, 12 scale bytes per row).
struct Q4K {
  static constexpr int kLoads = 2;
  static constexpr uint32_t kStage = 1280, kUnit = 2;
  struct Regs {
    u32x4 q[2];
    uint32_t scw, mw;
    float d24, ndmin;
  };
  struct Scale {
    float a24, a20, nb;
  };
  static __device__ __forceinline__ void issue(const uint8_t* Wp, uint32_t tile, uint32_t nh, uint32_t h,
                                               const uint8_t* dst, int lane) {
    const uint8_t* src = Wp + ((size_t)tile * (nh / 2) + (h >> 1)) * SH_Q4K_TILE_BYTES;
    sh_dma16_snt(src + 1024 * (h & 1), 16 * lane, dst);
    sh_dma4_snt(src + 2048, 4 * lane, dst + 1024);
  }
  static __device__ __forceinline__ Regs read(const uint8_t* w, int kh, int r, uint32_t h) {
    Regs s;
    s.q[0] = *(const u32x4*)(w + 16 * (16 * kh + r));
    s.q[1] = *(const u32x4*)(w + 16 * (16 * (2 + kh) + r));
    const uint32_t dd = *(const uint32_t*)(w + 1024 + 4 * r);
    const uint32_t* sp = (const uint32_t*)(w + 1024 + 64 + 12 * r);
    const uint32_t s0 = sp[0], s1 = sp[1], s2 = sp[2];
    // the 6-bit scales and minimums of sub-blocks 4h .. 4h + 3
    const bool odd = h & 1;
    s.scw = odd ? ((s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u)) : (s0 & 0x3F3F3F3Fu);
    s.mw = odd ? (((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u)) : (s1 & 0x3F3F3F3Fu);
    s.d24 = (float)as_h2(dd).x * 16777216.0f;
    s.ndmin = -(float)as_h2(dd).y;
    return s;
  }
  static __device__ __forceinline__ Scale scale(const Regs& s, int mp) {
    Scale v;
    v.a24 = s.d24 * (float)((s.scw >> (8 * mp)) & 0xFFu);
    v.a20 = v.a24 * 0.0625f;
    v.nb = s.ndmin * (float)((s.mw >> (8 * mp)) & 0xFFu);
    return v;
  }
  static __device__ __forceinline__ uint32_t pair(const Regs& s, const Scale& v, int mp, int j, int i) {
    const uint32_t w = mp == 0 ? s.q[j].x : mp == 1 ? s.q[j].y : mp == 2 ? s.q[j].z : s.q[j].w;
    const uint32_t x = i < 2 ? w : w >> 8;
    return (i & 1) ? fma_mix_pair(x & 0x00F000F0u, v.a20, v.nb) : fma_mix_pair(x & 0x000F000Fu, v.a24, v.nb);
  }
};

// Two f16 from two f32, each rounded to nearest.
__device__ __forceinline__ uint32_t pack16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, h2{(_Float16)lo, (_Float16)hi});
}
// rf(p a + c) in f32, p an f16 half (lo / hi) of the word.
__device__ __forceinline__ float fma_mix_lo(uint32_t p, float a, float c) {
  float r;
  asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(p), "v"(a), "v"(c));
  return r;
}
__device__ __forceinline__ float fma_mix_hi(uint32_t p, float a, float c) {
  float r;
  asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(p), "v"(a), "v"(c));
  return r;
}
// hw shifted left by n (right by -n).
__device__ __forceinline__ uint32_t shl(uint32_t hw, int n) { return n >= 0 ? hw << n : hw >> -n; }

// Q5_K: 1 KB of nibble words, one high-bit word per lane of this half, the
// 256 B row header. The reference's order of f32 operations, each rounded:
// f16(rf(d1 q) - m1) with d1 = rf(d sc), m1 = rf(dmin m) (gemm16x.hip); the
// 5-bit q is assembled as an f16 subnormal (q 2^-24 or 2^-20), so one fma_mix
// gives rf(d1 q).
struct Q5K {
  static constexpr int kLoads = 3;
  static constexpr uint32_t kStage = 1536, kUnit = 2;
  struct Regs {
    u32x4 q[2];
    uint32_t hw[2], scw, mw;
    float d, dmin;
  };
  struct Scale {
    float a24, a20, m1;
  };
  static __device__ __forceinline__ void issue(const uint8_t* Wp, uint32_t tile, uint32_t nh, uint32_t h,
                                               const uint8_t* dst, int lane) {
    const uint8_t* src = Wp + ((size_t)tile * (nh / 2) + (h >> 1)) * SH_Q5K_TILE_BYTES;
    sh_dma16_snt(src + 1024 * (h & 1), 16 * lane, dst);
    sh_dma4_snt(src + 2048 + 4 * (h & 1), 8 * lane, dst + 1024);
    sh_dma4_snt(src + 2560, 4 * lane, dst + 1280);
  }
  static __device__ __forceinline__ Regs read(const uint8_t* w, int kh, int r, uint32_t h) {
    Regs s;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int at = 16 * (2 * j + kh) + r;
      s.q[j] = *(const u32x4*)(w + 16 * at);
      s.hw[j] = *(const uint32_t*)(w + 1024 + 4 * at);
    }
    const uint32_t dd = *(const uint32_t*)(w + 1280 + 4 * r);
    const uint32_t* sp = (const uint32_t*)(w + 1280 + 64 + 12 * r);
    const uint32_t s0 = sp[0], s1 = sp[1], s2 = sp[2];
    const bool odd = h & 1;
    s.scw = odd ? ((s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u)) : (s0 & 0x3F3F3F3Fu);
    s.mw = odd ? (((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u)) : (s1 & 0x3F3F3F3Fu);
    s.d = (float)as_h2(dd).x;
    s.dmin = (float)as_h2(dd).y;
    return s;
  }
  static __device__ __forceinline__ Scale scale(const Regs& s, int mp) {
    Scale v;
    const float d1 = s.d * (float)((s.scw >> (8 * mp)) & 0xFFu);
    v.a24 = d1 * 16777216.0f;
    v.a20 = d1 * 1048576.0f;
    v.m1 = s.dmin * (float)((s.mw >> (8 * mp)) & 0xFFu);
    return v;
  }
  static __device__ __forceinline__ uint32_t pair(const Regs& s, const Scale& v, int mp, int j, int i) {
    const uint32_t w = mp == 0 ? s.q[j].x : mp == 1 ? s.q[j].y : mp == 2 ? s.q[j].z : s.q[j].w;
    const uint32_t x = i < 2 ? w : w >> 8;
    const int base = (mp & 1) * 2 + (mp >> 1) * 8;  // of the sub-block's bits in the high-bit word
    const uint32_t y = shl(s.hw[j], 4 - base - (i >> 1));
    const uint32_t p = (i & 1) ? (x & 0x00F000F0u) | (y & 0x01000100u) : (x & 0x000F000Fu) | (y & 0x00100010u);
    const float a = (i & 1) ? v.a20 : v.a24;
    return pack16(fma_mix_lo(p, a, 0.f) - v.m1, fma_mix_hi(p, a, 0.f) - v.m1);
  }
};

// Q6_K: 1 KB of nibble words, two high-bit words per lane of this half, then
// 16 rows x (even scales, odd scales) of this half and the rows' f16 d.
// f16(rf(ds (q - 32))), ds = rf(d sc): the 6-bit q as an f16 subnormal, one
// fma_mix ds q - 32 ds rounds the exact product once. MFMA j's 16 k share the
// scale 2 m + j.
struct Q6K {
  static constexpr int kLoads = 4;
  static constexpr uint32_t kStage = 1792, kUnit = 2;
  struct Regs {
    u32x4 q[2];
    uint32_t hw[2][2], scw[2];
    float d;
  };
  struct Scale {
    float a24[2], a20[2], nb[2];
  };
  static __device__ __forceinline__ void issue(const uint8_t* Wp, uint32_t tile, uint32_t nh, uint32_t h,
                                               const uint8_t* dst, int lane) {
    const uint8_t* src = Wp + ((size_t)tile * (nh / 2) + (h >> 1)) * SH_Q6K_TILE_BYTES;
    const uint32_t hf = h & 1, r = lane & 15;
    sh_dma16_snt(src + 1024 * hf, 16 * lane, dst);
    sh_dma4_snt(src + 2048 + 8 * hf, 16 * lane, dst + 1024);
    sh_dma4_snt(src + 2048 + 8 * hf + 4, 16 * lane, dst + 1280);
    // lanes 0-15 the rows' even scales, 16-31 the odd ones, 32-63 the dword of d
    sh_dma4_snt(src + 3072, lane < 32 ? 16 * r + 8 * (lane >> 4) + 4 * hf : 256 + 2 * (r & 14), dst + 1536);
  }
  static __device__ __forceinline__ Regs read(const uint8_t* w, int kh, int r, uint32_t) {
    Regs s;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int at = 16 * (2 * j + kh) + r;
      s.q[j] = *(const u32x4*)(w + 16 * at);
      s.hw[j][0] = *(const uint32_t*)(w + 1024 + 4 * at);
      s.hw[j][1] = *(const uint32_t*)(w + 1280 + 4 * at);
      s.scw[j] = *(const uint32_t*)(w + 1536 + 4 * (16 * j + r));
    }
    const uint32_t dd = *(const uint32_t*)(w + 1536 + 4 * (32 + r));
    s.d = (r & 1) ? (float)as_h2(dd).y : (float)as_h2(dd).x;
    return s;
  }
  static __device__ __forceinline__ Scale scale(const Regs& s, int mp) {
    Scale v;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float ds = s.d * (float)((int32_t)(s.scw[j] << (24 - 8 * mp)) >> 24);
      v.a24[j] = ds * 16777216.0f;
      v.a20[j] = ds * 1048576.0f;
      v.nb[j] = ds * -32.0f;
    }
    return v;
  }
  static __device__ __forceinline__ uint32_t pair(const Regs& s, const Scale& v, int mp, int j, int i) {
    const uint32_t w = mp == 0 ? s.q[j].x : mp == 1 ? s.q[j].y : mp == 2 ? s.q[j].z : s.q[j].w;
    const uint32_t x = i < 2 ? w : w >> 8;
    const uint32_t y = shl(s.hw[j][mp >> 1], 4 - 8 * (mp & 1) - 2 * (i >> 1));
    const uint32_t p = (i & 1) ? (x & 0x00F000F0u) | (y & 0x03000300u) : (x & 0x000F000Fu) | (y & 0x00300030u);
    const float a = (i & 1) ? v.a20[j] : v.a24[j];
    return pack16(fma_mix_lo(p, a, v.nb[j]), fma_mix_hi(p, a, v.nb[j]));
  }
};

// Q8_0: a stage is 4 tile-blocks of 544 B (512 B of int8, the rows' f16 d).
// f16(d q): the product is exact in f32, so one f16 multiply rounds it the same.
struct Q8 {
  static constexpr int kLoads = 3;
  static constexpr uint32_t kStage = 2176, kUnit = 1;
  struct Regs {
    uint2 q[4][2];
    uint16_t d[4];
  };
  struct Scale {
    h2 d;
  };
  static __device__ __forceinline__ void issue(const uint8_t* Wp, uint32_t tile, uint32_t nh, uint32_t h,
                                               const uint8_t* dst, int lane) {
    const uint8_t* src = Wp + ((size_t)tile * nh + h) * (4 * SH_Q8_TILE_BYTES);
    sh_dma16_snt(src, 16 * lane, dst);
    sh_dma16_snt(src + 1024, 16 * lane, dst + 1024);
    if (lane < 8) sh_dma16_snt(src + 2048, 16 * lane, dst + 2048);
  }
  static __device__ __forceinline__ Regs read(const uint8_t* w, int kh, int r, uint32_t) {
    Regs s;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
      for (int j = 0; j < 2; ++j) s.q[b][j] = *(const uint2*)(w + 544 * b + 8 * (16 * (2 * j + kh) + r));
      s.d[b] = *(const uint16_t*)(w + 544 * b + 512 + 2 * r);
    }
    return s;
  }
  static __device__ __forceinline__ Scale scale(const Regs& s, int mp) {
    const _Float16 d = __builtin_bit_cast(_Float16, s.d[mp]);
    return Scale{h2{d, d}};
  }
  static __device__ __forceinline__ uint32_t pair(const Regs& s, const Scale& v, int mp, int j, int i) {
    const uint32_t w = (i < 2 ? s.q[mp][j].x : s.q[mp][j].y) ^ 0x80808080u;  // q + 128
    // f16 1024 + (q + 128) by the exponent 0x64, then the exact q
    const uint32_t p = __builtin_amdgcn_perm(0x64646464u, w, (i & 1) ? 0x04030402u : 0x04010400u);
    const h2 q = as_h2(p) - h2{(_Float16)1152.f, (_Float16)1152.f};
    return __builtin_bit_cast(uint32_t, q * v.d);
  }
};

constexpr int kTiles = 4, kWaves = 4;  // row tiles per wave, waves per workgroup
constexpr int kBStages = 3;

template <class F, int CG, int EPI>
__global__ __launch_bounds__(64 * kWaves, 1) void k_gemm16t(const uint8_t* __restrict__ Wp, uint32_t tiles, uint32_t nh,
                                                            uint32_t HS, const uint16_t* __restrict__ Bh, uint32_t ldb,
                                                            uint32_t N, uint32_t ncb, uint32_t nrb, EpiArgs ea) {
  constexpr int T = kTiles, TP = T / 2;
  constexpr int P = TP * 9;           // decode pieces per sub-block: a scale and 2 x 4 f16 pairs per tile pair
  constexpr int NBL = CG;             // one wave's B loads per 64-k stage (4 CG fragments)
  constexpr int NWL = T * F::kLoads;  // one wave's weight loads per 128-k stage
  __shared__ h8 sB[kBStages][CG * 4 * 64];  // [buffer][(column group * 4 + sub-block * 2 + MFMA) * 64 + lane]
  __shared__ __attribute__((aligned(16))) uint8_t sW[2][kWaves * T * F::kStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kh = lane >> 5, tl = (lane >> 4) & 1, r = lane & 15;
  // The column blocks of a row block run on one XCD (workgroups are dealt to
  // the 8 XCDs in turn), one after the other: the later ones find the weights
  // in its L2.
  uint32_t rb, cb;
  if (nrb >= 16) {
    const uint32_t j = blockIdx.x / 8;
    rb = j / ncb * 8 + blockIdx.x % 8;
    cb = j % ncb;
  } else {
    rb = blockIdx.x / ncb;
    cb = blockIdx.x % ncb;
  }
  if (rb >= nrb) return;  // whole workgroup: the last 8 row blocks may be fewer
  const uint32_t tile0 = (rb * kWaves + wave) * T, col0 = cb * CG * 32;
  const uint32_t ks = blockIdx.y, h0 = ks * HS, nhs = min(h0 + HS, nh) - h0, nst = 2 * nhs;

  // byte offsets of this lane's B loads within stage 0: fragment wave + 4 i is
  // sub-block wave / 2, MFMA wave % 2 of column group i
  uint32_t boff[NBL];
#pragma unroll
  for (int i = 0; i < NBL; ++i) {
    const uint32_t col = min(col0 + 32 * i + (uint32_t)(lane & 31), N - 1);
    boff[i] = (col * ldb + 32 * (wave >> 1) + 8 * (2 * (wave & 1) + kh)) * 2;
  }
  const uint16_t* bsrc = Bh + 128 * (size_t)h0;
  auto issue_b1 = [&](uint32_t s, int slot, int i) __attribute__((always_inline)) {
    sh_dma16_s(bsrc + 64 * (size_t)min(s, nst - 1), boff[i], &sB[slot][(wave + kWaves * i) * 64]);
  };
  auto issue_w1 = [&](uint32_t h, int t) __attribute__((always_inline)) {
    const uint32_t tt = min(tile0 + t, tiles - 1);  // clamp keeps loads in bounds
    F::issue(Wp, tt, nh, h0 + min(h, nhs - 1), &sW[h & 1][(wave * T + t) * F::kStage], lane);
  };

  f16v acc[TP][CG];
#pragma unroll
  for (int p = 0; p < TP; ++p)
#pragma unroll
    for (int c = 0; c < CG; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[p][c][i] = 0.f;
  typename F::Regs wr[TP];
  typename F::Scale sc[TP];
  h8 bb[2][CG];
  uint32_t a[TP][2][4], an[TP][2][4];

  auto read_w = [&](uint32_t h) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < TP; ++p)
      wr[p] = F::read(&sW[h & 1][(wave * T + 2 * p + tl) * F::kStage], kh, r, h0 + min(h, nhs - 1));
  };
  auto piece = [&](int mp, int n) __attribute__((always_inline)) {
    const int p = n / 9, i = n % 9 - 1;
    if (i < 0) sc[p] = F::scale(wr[p], mp);
    else an[p][i / 4][i % 4] = F::pair(wr[p], sc[p], mp, i / 4, i % 4);
  };
  auto take = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < TP; ++p)
#pragma unroll
      for (int i = 0; i < 8; ++i) a[p][i / 4][i % 4] = an[p][i / 4][i % 4];
  };
  // One sub-block: the MFMAs of a and bb; meanwhile bb <- next (the fragments
  // of the next sub-block) and an <- the decode of its weights (sub-block mp of
  // wr), from MFMA n0 on, and extra(n). Each MFMA is followed by its share of
  // those instructions: it keeps the matrix core for 32 clocks of which its
  // issue takes 4, and up to 6 vector instructions fit in its shadow (fma_mix
  // counts twice), where a 16x16x32 one has room for 2.
  auto sub = [&](const h8* next, auto mpc, auto n0c, auto&& extra) __attribute__((always_inline)) {
    constexpr int M = 4 * CG, mp = decltype(mpc)::value, n0 = decltype(n0c)::value;
    mfma_fence();
    static_for<M>([&](auto nc) __attribute__((always_inline)) {
      constexpr int n = decltype(nc)::value, j = n / (2 * CG), c = n / 2 % CG, p = n % 2;
      mfma_acc(acc[p][c], __builtin_bit_cast(h8, u32x4{a[p][j][0], a[p][j][1], a[p][j][2], a[p][j][3]}), bb[j][c]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (p == TP - 1) bb[j][c] = next[(c * 4 + j) * 64 + lane];
      extra(nc);
      if constexpr (n >= n0) {
        constexpr int q0 = P * (n - n0) / (M - n0), nq = P * (n + 1 - n0) / (M - n0) - q0;
        static_for<nq>([&](auto k) __attribute__((always_inline)) { piece(mp, q0 + decltype(k)::value); });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    take();
  };

  // prologue, in the order the stages issue: W(0), B(0), B(1), W(1), B(2)
#pragma unroll
  for (int t = 0; t < T; ++t) issue_w1(0, t);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
#pragma unroll
    for (int i = 0; i < NBL; ++i) issue_b1(j, j, i);
    if (j == 1)
#pragma unroll
      for (int t = 0; t < T; ++t) issue_w1(1, t);
  }
  sh_wait_vm<2 * NBL + NWL>();
  sh_lds_barrier();
  read_w(0);
#pragma unroll
  for (int c = 0; c < 2 * CG; ++c) bb[c % 2][c / 2] = sB[0][(c / 2 * 4 + c % 2) * 64 + lane];
#pragma unroll
  for (int q = 0; q < P; ++q) piece(0, q);
  take();

  int sl = 0;  // s % 3, wave-uniform
  constexpr int kLate = CG / 2;  // the weight words of a new stage come from LDS first
  for (uint32_t h = 0; h < nhs; ++h) {
    static_for<2>([&](auto parc) __attribute__((always_inline)) {
      constexpr int par = decltype(parc)::value;
      const uint32_t s = 2 * h + par;
      const int slot = __builtin_amdgcn_readfirstlane(sl), nslot = slot == 2 ? 0 : slot + 1;
      sub(&sB[slot][128], std::integral_constant<int, 2 * par + 1>{}, std::integral_constant<int, 0>{}, [](auto) {});
      // B(s + 1) landed (issued two stages ago; after it B(s + 2) and one
      // weight stage), as did W(h + 1), older; every wave has read all of stage
      // s, whose buffer stage s + 3 now refills
      sh_wait_vm<NBL + NWL>();
      sh_lds_barrier();
      if (par) read_w(h + 1);
      sub(&sB[nslot][0], std::integral_constant<int, par ? 0 : 2>{}, std::integral_constant<int, par ? kLate : 0>{},
          [&](auto nc) __attribute__((always_inline)) {
            // one load after every MFMA: B(s + 3), then W(h + 2)
            constexpr int n = decltype(nc)::value;
            if constexpr (n < NBL) issue_b1(s + 3, slot, n);
            if constexpr (par == 0 && n >= NBL && n < NBL + T) issue_w1(h + 2, n - NBL);
          });
      sl = nslot;
    });
  }
  sh_wait_vm<0>();  // no load may be in flight into LDS when the workgroup ends
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last MFMAs' results
  __builtin_amdgcn_sched_barrier(0);

  if (EPI == EPI_QKV && ea.row_base + tile0 * 16 >= ea.Dq + ea.Dkv) {
    // V rows go out with the lanes along the columns: consecutive keys of a row
    // are neighbours in the cache's transposed blocks
    if (tile0 >= tiles) return;
    QkvColDev tv[CG];
#pragma unroll
    for (int c = 0; c < CG; ++c) tv[c] = ea.tab[min(col0 + 32 * c + (lane & 31), N - 1)];
#pragma unroll
    for (int c = 0; c < CG; ++c) {
      const uint32_t col = col0 + 32 * c + (lane & 31);
      if (col >= N) continue;
      const QkvColDev t = tv[c];
#pragma unroll
      for (int p = 0; p < TP; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (tile0 + 2 * p + q / 2 >= tiles) continue;
          const f16v& a4 = acc[p][c];
          const float v[4] = {a4[4 * q], a4[4 * q + 1], a4[4 * q + 2], a4[4 * q + 3]};
          qkv_store4(ea, ea.row_base + (tile0 + 2 * p) * 16 + 8 * q + 4 * kh, v, float2{}, float2{}, t.slot, t.mseq,
                     t.kc, t.vc, nullptr);
        }
    }
    return;
  }
  // Epilogue, one column group at a time through the wave's own slice of LDS:
  // lane holds column lane % 32, rows 8 q + 4 kh + 0..3 of each pair's 32; read
  // back as 16 lanes x 4 rows of a column, so a store covers the wave's whole 64
  // rows (256 B) of 4 columns instead of 32 B of 32.
  sh_lds_barrier();  // every wave is done with the B buffers
  constexpr uint32_t kLd = 68;  // floats per column: 64 rows, padded to spread the banks
  float* st = reinterpret_cast<float*>(&sB[0][0]) + wave * 32 * kLd;
  const uint32_t er = 4 * (lane & 15), row0 = tile0 * 16 + er;
  const bool vec = ea.ldo % 4 == 0 && (uintptr_t)ea.out % 16 == 0;  // 16-byte rows
#pragma unroll
  for (int c = 0; c < CG; ++c) {
#pragma unroll
    for (int p = 0; p < TP; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f16v& v = acc[p][c];
        *(float4*)(st + (lane & 31) * kLd + 32 * p + 8 * q + 4 * kh) =
            make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
      }
    __builtin_amdgcn_wave_barrier();
    if (EPI == EPI_SWIGLU) {  // 8 lanes cover the 32 h rows of a column's 2 gate / up pairs
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t lc = 8 * i + (lane >> 3), col = col0 + 32 * c + lc, p = (lane >> 2) & 1, rr = 4 * (lane & 3);
        const float4 gt = *(const float4*)(st + lc * kLd + 32 * p + rr);
        const float4 up = *(const float4*)(st + lc * kLd + 32 * p + 16 + rr);
        if (col >= N || tile0 + 2 * p + 1 >= tiles) continue;
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        const h4 h = {(_Float16)((gt.x / (1.0f + expf(-gt.x))) * up.x), (_Float16)((gt.y / (1.0f + expf(-gt.y))) * up.y),
                      (_Float16)((gt.z / (1.0f + expf(-gt.z))) * up.z), (_Float16)((gt.w / (1.0f + expf(-gt.w))) * up.w)};
        *(uint2*)(ea.h16 + (size_t)col * ea.ldh + (tile0 / 2 + p) * 16 + rr) = __builtin_bit_cast(uint2, h);
      }
      __builtin_amdgcn_wave_barrier();
      continue;
    }
    if (EPI == EPI_QKV) {
      // q and k rows: the 8 columns' table entries, then their rotations, all in
      // flight before the first is used (one by one a group waited for 16 loads
      // in turn: 6144 x 4096 x 2048 columns 150 -> 136 us, a 2048-column pass of two
      // 8B layers 2357 -> 2315 us)
      const uint32_t i0 = (ea.row_base + row0) % ea.hd;
      QkvColDev t[8];
      float2 cs[8][2];
#pragma unroll
      for (int i = 0; i < 8; ++i) t[i] = ea.tab[min(col0 + 32 * c + 4 * i + (lane >> 4), N - 1)];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float2* rp = ea.rope + (size_t)t[i].pos * (ea.hd / 2) + i0 / 2;
        cs[i][0] = rp[0];
        cs[i][1] = rp[1];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t lc = 4 * i + (lane >> 4), col = col0 + 32 * c + lc;
        const float4 v = *(const float4*)(st + lc * kLd + er);
        if (col >= N || row0 >= tiles * 16) continue;
        const float o[4] = {v.x, v.y, v.z, v.w};
        qkv_store4(ea, ea.row_base + row0, o, cs[i][0], cs[i][1], t[i].slot, t[i].mseq, t[i].kc, t[i].vc,
                   ea.out + (size_t)col * ea.Dq);
      }
      __builtin_amdgcn_wave_barrier();
      continue;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t lc = 4 * i + (lane >> 4), col = col0 + 32 * c + lc;
      const float4 v = *(const float4*)(st + lc * kLd + er);
      if (col >= N || row0 >= tiles * 16) continue;
      float* out = ea.out + (size_t)col * ea.ldo + row0;
      if (EPI == EPI_PART) {
        *(float4*)(out + ks * ea.part_stride) = v;
      } else if (row0 + 3 < ea.rows && vec) {
        float4 o = v;
        if (EPI == EPI_ADD) {
          const float4 y = *(const float4*)out;
          o = make_float4(y.x + v.x, y.y + v.y, y.z + v.z, y.w + v.w);
        }
        *(float4*)out = o;
      } else {
        const float o[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (row0 + j < ea.rows) out[j] = EPI == EPI_ADD ? out[j] + o[j] : o[j];
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <class F, int CG, int EPI>
void launch(sh_engine* e, const QMat& w, const uint16_t* bh, uint32_t ldb, uint32_t N, const Gemm16tPlan& p,
            const EpiArgs& ea) {
  const uint32_t nrb = (w.tiles + 15) / 16;
  const dim3 grid(nrb >= 16 ? (nrb + 7) / 8 * 8 * p.ncb : nrb * p.ncb, p.KS);
  hipLaunchKernelGGL((k_gemm16t<F, CG, EPI>), grid, dim3(64 * kWaves), 0, e->stream, w.d, w.tiles, w.K / 128, p.HS, bh,
                     ldb, N, p.ncb, nrb, ea);
}

}  // namespace
