// Epilogues of the prefill GEMMs: the store, residual and SwiGLU forms of a
// lane's 4 consecutive features of one token row.
#pragma once
#include "common.h"
#include "kernels.h"

namespace yuear {

__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  return uint32_t(f2bf(a)) | uint32_t(f2bf(b)) << 16;
}

// SwiGLU epilogue (ar.cpp:36-51) on interleaved (gate_i, up_i) columns: the
// lane's features n .. n + 3 (n a multiple of 4) are two pairs, written as
// outputs n / 2 and n / 2 + 1 of the row with the rounding points of the
// decode GEMV's epilogue: g, u rounded to bf16, silu(g) rounded, then g * u.
__device__ __forceinline__ uint16_t swiglu_one(float gate, float up) {
  const float g = rbf(gate), u = rbf(up);
  const float act = rbf(g * (1.0f / (1.0f + expf(-g))));
  return f2bf(act * u);
}
__device__ __forceinline__ void swiglu_store(const GemmParams &p, int m, int n, const float *v) {
  uint16_t *c = p.c + size_t(m) * p.ldc + (n >> 1);
  if (n + 3 < p.n && (p.ldc & 1) == 0) {
    *reinterpret_cast<uint32_t *>(c) =
        uint32_t(swiglu_one(v[0], v[1])) | uint32_t(swiglu_one(v[2], v[3])) << 16;
  } else {
    if (n + 1 < p.n)
      c[0] = swiglu_one(v[0], v[1]);
    if (n + 3 < p.n)
      c[1] = swiglu_one(v[2], v[3]);
  }
}

// Epilogue of a lane's 4 consecutive features n .. n + 3 (n a multiple of 4)
// of token row m < p.m: the 8-byte form when all four are in range and rows
// stay 8-byte aligned, else element by element.
__device__ __forceinline__ void epilogue4(const GemmParams &p, int m, int n, const float *v) {
  if (p.residual == 2) {
    swiglu_store(p, m, n, v);
    return;
  }
  uint16_t *c = p.c + size_t(m) * p.ldc + n;
  if (n + 3 < p.n && (p.ldc & 3) == 0) {
    uint2 o;
    if (p.residual) {
      const uint2 old = *reinterpret_cast<const uint2 *>(c);
      o.x = pack_bf16x2(bf2f(uint16_t(old.x)) + rbf(v[0]), bf2f(uint16_t(old.x >> 16)) + rbf(v[1]));
      o.y = pack_bf16x2(bf2f(uint16_t(old.y)) + rbf(v[2]), bf2f(uint16_t(old.y >> 16)) + rbf(v[3]));
    } else {
      o.x = pack_bf16x2(v[0], v[1]);
      o.y = pack_bf16x2(v[2], v[3]);
    }
    *reinterpret_cast<uint2 *>(c) = o;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < p.n)
        c[e] = p.residual ? f2bf(bf2f(c[e]) + rbf(v[e])) : f2bf(v[e]);
  }
}

}  // namespace yuear
