// Finishing a column's fused QKV rows: RoPE, the q rows out, the K / V cache
// writes. Shared by the GEMV epilogues (gemv.hip), the split finish and the
// large-tile wide GEMM (gemm16t.hip).
#pragma once
#include "sh_internal.h"

__device__ __forceinline__ uint16_t f2h_bits(float x) { return __builtin_bit_cast(uint16_t, (_Float16)x); }

// Slot of key kappa (0..31) inside a 32-key V block: the PV MFMA's B operand
// (probabilities) arrives with lane group g holding keys {4g..4g+3, 16+4g..16+4g+3}.
__device__ __forceinline__ uint32_t v_slot(uint32_t kappa) {
  return 8u * ((kappa & 15u) >> 2) + 4u * (kappa >> 4) + (kappa & 3u);
}

// Rows r0..r0+3 of one column's fused QKV output: q rows are roped (cs0, cs1 the
// (cos, sin) of the two pairs) into qcol, k rows roped and v rows stored as f16
// in the column's cache slot (V slot-permuted within its 32-key block).
__device__ __forceinline__ void qkv_store4(const EpiArgs& ea, uint32_t r0, const float v[4], float2 cs0, float2 cs1,
                                           uint32_t slot, uint32_t ms, uint16_t* kc, uint16_t* vc, float* qcol) {
  if (r0 < ea.Dq + ea.Dkv) {
    float o[4];
    o[0] = v[0] * cs0.x - v[1] * cs0.y;
    o[1] = v[0] * cs0.y + v[1] * cs0.x;
    o[2] = v[2] * cs1.x - v[3] * cs1.y;
    o[3] = v[2] * cs1.y + v[3] * cs1.x;
    if (r0 < ea.Dq) {
      float* q = qcol + r0;
      for (int j = 0; j < 4; ++j) q[j] = o[j];
    } else {
      const uint32_t rr = r0 - ea.Dq, kh = rr / ea.hd, i0 = rr % ea.hd;
      uint16_t* k = kc + (((size_t)ea.layer * ea.n_kv + kh) * ms + slot) * ea.hd + i0;
      for (int j = 0; j < 4; ++j) k[j] = f2h_bits(o[j]);
    }
  } else {
    const uint32_t rr = r0 - ea.Dq - ea.Dkv, kh = rr / ea.hd, i0 = rr % ea.hd;
    uint16_t* vb = vc + (((size_t)ea.layer * ea.n_kv + kh) * (ms / 32) + slot / 32) * ea.hd * 32;
    const uint32_t sl = v_slot(slot & 31);
    for (int j = 0; j < 4; ++j) vb[(size_t)(i0 + j) * 32 + sl] = f2h_bits(v[j]);
  }
}
// The same with the rotations of RoPE position pos.
__device__ __forceinline__ void qkv_store4(const EpiArgs& ea, uint32_t r0, const float v[4], int32_t pos,
                                           uint32_t slot, uint32_t ms, uint16_t* kc, uint16_t* vc, float* qcol) {
  float2 cs0 = make_float2(1.f, 0.f), cs1 = cs0;
  if (r0 < ea.Dq + ea.Dkv) {  // Dq is whole heads: row r0's pair index is the same in q and k
    const float2* rp = ea.rope + (size_t)pos * (ea.hd / 2) + (r0 % ea.hd) / 2;
    cs0 = rp[0];
    cs1 = rp[1];
  }
  qkv_store4(ea, r0, v, cs0, cs1, slot, ms, kc, vc, qcol);
}
