// Query tiles of multi-query attention with head_dim 128 on gfx950 MFMA,
// shared by the causal prefill attention (prefill.hip, ar.cpp:284-291) and
// the acoustic-model attention (nar_attention.hip, nar_attention.cpp:63-218):
// fp32 scores of bf16 operands, an exp2 online softmax in fp32, P fed to P.V
// as three truncated bf16 pieces (its 24 significant bits: every product
// exact), fp32 sums, bf16(o / l).
//
//   S^T[key][query] = K[key][:] . q[query][:]            (attn_core.h rows)
//   O^T[dim][query] += V^T[dim][key] . P^T[key][query]
//
// Two forms. The key-split tile (attn_query_tile, 16 or 32 queries) has its 4
// or 8 waves split the tile's 32-key blocks and merges their (m, l, O) through
// LDS: for launches with few tiles, whose time is the longest wave's chain of
// blocks and the rate at which one CU pulls K and V (4 waves: two workgroups
// to a CU, for more tiles than CUs). The 64-query tile (attn_query_tile64) has
// its 4 waves walk the same blocks, fetched once per workgroup, one or two a
// step: for launches that fill the GPU, bound by VALU and MFMA issue.
#pragma once
#include <algorithm>
#include <type_traits>

#include "attn_core.h"
#include "common.h"

namespace yuear {
namespace attn {

struct QueryTile {
  const u32x4 *kc = nullptr;  // this kv head's K rows, row-major [slot][128]
  const u32x4 *vc = nullptr;  // its V in 32-key dim-major blocks (v_index) or as rows
  int kend = 0;               // keys [0, kend) are read
  int kv_len = 0;             // non-causal: keys [0, kv_len) are visible
  int causal_pos = -1;        // >= 0: query t sees keys <= causal_pos + t
  const uint16_t *q = nullptr;  // query 0 of the tile
  size_t q_stride = 0;          // elements between consecutive queries
  int nq = 0;                   // valid queries of the tile
  uint16_t *out = nullptr;      // output row of query 0
  size_t out_stride = 0;
  // key-split tile, non-causal: key blocks [blk0, blk1) of the tile (blk1 0:
  // all) and, when set, an unnormalised partial per query instead of out: 132
  // floats {o[128], m, l, pad} at part + query * 132 (m the largest raw score,
  // l the sum of exp2((s - m) qscale), o that of exp2((s - m) qscale) v)
  int blk0 = 0, blk1 = 0;
  float *part = nullptr;
};

// One online-softmax step of a lane's query over 8 N / 2 raw scores st (16-key
// rows of S^T, masked to -inf where not visible): updates the running maximum
// m (of the raw scores) and this lane's part l of the denominator, leaves the
// three truncated bf16 pieces of p = exp2((score - m) * qscale) in pw per 32
// keys (the top 8, next 8 and last 8 significant bits of p; each remainder is
// exact, so p is their sum), and returns the factor for the previous O. The
// difference is taken first, so the largest score's exponent is exactly 0
// whatever its size (fma(score, qscale, -round(m * qscale)) leaves it the
// rounding error of the product: past 2^32 that overflows exp2 or underflows
// every weight).
template <int N>
__device__ __forceinline__ float softmax_step(const f32x4 (&st)[N], float qscale, float &m_run,
                                              float &l_run, uint32_t (&pw)[N / 2][3][4]) {
  float mx = st[0][0];
#pragma unroll
  for (int e = 1; e < 4 * N; ++e)
    mx = fmaxf(mx, st[e >> 2][e & 3]);
  mx = max_halves(max_row_pairs(mx));
  const float m_new = fmaxf(m_run, mx);
  const float m_use = m_new == -__builtin_inff() ? 0.f : m_new;
  const float corr = __builtin_amdgcn_exp2f((m_run - m_use) * qscale);
  float ps = 0.f;
#pragma unroll
  for (int g = 0; g < N / 2; ++g)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 &s = st[2 * g + (q >> 1)];
      float p0 = __builtin_amdgcn_exp2f((s[2 * (q & 1)] - m_use) * qscale);
      float p1 = __builtin_amdgcn_exp2f((s[2 * (q & 1) + 1] - m_use) * qscale);
      ps += p0;
      ps += p1;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const uint32_t u0 = __builtin_bit_cast(uint32_t, p0);
        const uint32_t u1 = __builtin_bit_cast(uint32_t, p1);
        pw[g][k][q] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);  // hi16(u0) | hi16(u1) << 16
        p0 -= __builtin_bit_cast(float, u0 & 0xffff0000u);
        p1 -= __builtin_bit_cast(float, u1 & 0xffff0000u);
      }
    }
  l_run = l_run * corr + ps;
  m_run = m_new;
  return corr;
}
__device__ __forceinline__ u32x4 piece(const uint32_t (&w)[4]) { return u32x4{w[0], w[1], w[2], w[3]}; }

// A lane's 4 output dims from d of one query row: bf16(o / l).
__device__ __forceinline__ void store_dims(uint16_t *dst, int d, f32x4 o, float l) {
  const uint32_t lo = uint32_t(f2bf(o[0] / l)) | (uint32_t(f2bf(o[1] / l)) << 16);
  const uint32_t hi = uint32_t(f2bf(o[2] / l)) | (uint32_t(f2bf(o[3] / l)) << 16);
  *reinterpret_cast<uint2 *>(dst + d) = uint2{lo, hi};
}

typedef __attribute__((address_space(3))) void *lds_ptr_t;

// Buffers over a tile's K rows and V: reads past the last key (of V in blocks:
// past its last block) give zeros; the scores of those keys are masked. Their
// 32-bit range and offsets end at kMaxRange keys, so the key-split tile, which
// any cache may take, has a buffer per 32-key block.
constexpr int kMaxRange = (1 << 24) - kBlock;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t key_rsrc(const u32x4 *base, int first, int keys) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4 *>(base) + size_t(first) * (D / 8), 0,
                                           uint32_t(keys) * (D * 2), 0x00020000);
}

// V of a 32-key block staged as it lies in memory, 8 KiB either way.
//
// Rows ([32 keys][128 dims]): 16-byte chunk c of key R at slot c ^ 2 h(R) of
// its row, h(R) = R % 4 + 4 (R / 8 % 2). The P.V operand of dim tile dt (lane
// (i, r): dim 16 dt + i, keys 8 r + [0, 8)) is two transposing reads
// (ds_read_b64_tr_b16: in each group of 16 lanes, lane 4 a + b gives the
// address of 4 dims from 4 b of key a and lane j receives dim j of the 4
// keys), keys 8 r + a and 8 r + 4 + a; the swizzle puts the 8 keys of half a
// wave in 8 different 32-byte windows.
__device__ __forceinline__ uint32_t v_row_fetch(int lane, int q) {  // load q's lane offset in bytes
  const int R = 4 * q + (lane >> 4);
  return uint32_t(R * (D * 2) + ((lane & 15) ^ (2 * ((R & 3) + 4 * ((R >> 3) & 1)))) * 16);
}
__device__ __forceinline__ int v_row_read(int lane, int dt) {  // u32x4 slots x 2 (8-byte units)
  const int R = 8 * (lane >> 4) + ((lane >> 2) & 3);
  return R * 32 + ((dt ^ ((R & 3) + 4 * ((R >> 3) & 1))) * 4) + (lane & 3);
}
__device__ __forceinline__ u32x4 v_row_operand(const u32x4 *stage, int at) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) s16x4 *lds_s16x4;
  const u32x2 *p = reinterpret_cast<const u32x2 *>(stage) + at;
  const u32x2 lo = __builtin_bit_cast(
      u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)const_cast<u32x2 *>(p)));
  const u32x2 hi = __builtin_bit_cast(  // keys + 4
      u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)const_cast<u32x2 *>(p + 128)));
  return u32x4{lo.x, lo.y, hi.x, hi.y};
}
// Blocks (dim-major [128 dims][32 keys]): 16-byte chunk c of dim d at slot
// c ^ (d / 4) % 4 of its 64 bytes; an operand is one 16-byte read.
__device__ __forceinline__ uint32_t v_block_fetch(int lane, int q) {
  return uint32_t(q * 1024 + (lane >> 2) * 64 + ((lane & 3) ^ (lane >> 4)) * 16);
}

// ---------------------------------------------------------------------------
// Key-split tile of 16 C queries: wave w of W walks the 32-key blocks w,
// w + W, ... A block's K and V are 8 contiguous KiB each; a wave fetches them
// into an LDS stage of its own by direct-to-LDS loads of whole KiB and moves
// them to registers before it refills the stage, so the next block is in
// flight during the products and no barrier runs before the merge. Loading
// the MFMA operands straight into registers (16 rows x 64 bytes a load) left a
// CU at ~45 KB/us, more waves or not; this pulls ~80. Slot p of a stage, K:
// key p / 16, 16-byte chunk (p % 16) ^ f(key), f = the key's row of its S^T
// tile; V as above. Operand reads then go to 16 different 16-byte slots per
// group of lanes (gemm.hip).
// MI355X, 24/8 heads, us, before (4 waves, registers) -> now: 33 queries after
// 2000 keys 26.7 -> 13.9, 160 after 600 13.5 -> 8.4, 160 from 0 7.5 -> 5.3, 512
// from 0 14.1 -> 11.2, 700 after 600 (64-query tiles) 34.4 -> 27.6.

template <int C, int W>
struct TileLds {
  u32x4 kv[W][2][512];  // [wave][K | V]; the merge's O lies over it
  float m[W][C][16], l[W][C][16];
};

template <int C, bool kRows, int W>
__device__ __forceinline__ void attn_query_tile(const QueryTile &t, float qscale,
                                                TileLds<C, W> &sh) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane >> 4, i = lane & 15;
  const int nblk = t.blk1 ? t.blk1 : (t.kend + kBlock - 1) / kBlock;  // blocks [blk0, nblk)
  const int first = t.blk0 + wave;
  u32x4 *ks = sh.kv[wave][0], *vs = sh.kv[wave][1];
  auto fetch = [&](int kb) {
    const int keys = min(kBlock, t.kend - kb);
    const auto rk = key_rsrc(t.kc, kb, keys), rv = key_rsrc(t.vc, kb, kRows ? keys : kBlock);
#pragma unroll
    for (int q = 0; q < 8; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rk, (lds_ptr_t)(ks + 64 * q), 16,
          uint32_t((4 * q + r) * (D * 2) + (i ^ (4 * (q >> 1) + r)) * 16), 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 8; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rv, (lds_ptr_t)(vs + 64 * q), 16,
          kRows ? v_row_fetch(lane, q) : v_block_fetch(lane, q), 0, 0, 0);
  };
  if (first < nblk)
    fetch(first * kBlock);

  // Q^T operands: column tile c, query 16 c + i (clamped), dims 32 s + 8 r
  u32x4 qb[C][4];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int qi = min(16 * c + i, t.nq - 1);
    const u32x4 *src = reinterpret_cast<const u32x4 *>(t.q + size_t(qi) * t.q_stride);
#pragma unroll
    for (int s = 0; s < 4; ++s)
      qb[c][s] = src[4 * s + r];
  }
  float m_run[C], l_run[C];
  f32x4 o[C][8];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    m_run[c] = -__builtin_inff();
    l_run[c] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      o[c][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto block = [&](int blk, auto mask_tag) {
    constexpr bool kMask = decltype(mask_tag)::value;
    const int kb = blk * kBlock;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the block has landed
    __builtin_amdgcn_sched_barrier(0);
    u32x4 kr[8], vr[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      kr[j] = ks[key_ofs(j >> 2, i) * 16 + ((4 * (j & 3) + r) ^ i)];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      vr[dt] = kRows ? v_row_operand(vs, v_row_read(lane, dt)) : vs[64 * dt + 4 * i + (r ^ (i >> 2))];
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): it is in registers
    __builtin_amdgcn_sched_barrier(0);
    if (blk + W < nblk)
      fetch(kb + W * kBlock);
    // a score tile's four k-steps depend on each other: the chains of the
    // tiles are interleaved, and below those of the dim tiles
    f32x4 st[C][2];
#pragma unroll
    for (int c = 0; c < C; ++c)
      st[c][0] = st[c][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int T = 0; T < 2; ++T)
          st[c][T] = mfma(kr[4 * T + s], qb[c][s], st[c][T]);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if constexpr (kMask) {  // lane (query 16 c + i, r): keys kb + 8 r + 4 T + u
        const int kmax = (t.causal_pos >= 0 ? t.causal_pos + 16 * c + i : t.kv_len - 1) - kb - 8 * r;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (e > kmax)
            st[c][e >> 2][e & 3] = -__builtin_inff();
      }
      uint32_t pw[1][3][4];
      const float corr = softmax_step<2>(st[c], qscale, m_run[c], l_run[c], pw);
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
        o[c][dt] *= corr;
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
          o[c][dt] = mfma(vr[dt], piece(pw[0][k]), o[c][dt]);
    }
  };
  // blocks every query of the tile sees in full run without the mask
  const int kfull = (t.causal_pos >= 0 ? t.causal_pos + 1 : t.kv_len) / kBlock;
  int blk = first;
  for (; blk < min(kfull, nblk); blk += W)
    block(blk, std::false_type{});
  for (; blk < nblk; blk += W)
    block(blk, std::true_type{});

  // Merge the waves' partials: wave w finishes column tile w / (W / C) and C
  // of its dim tiles. A wave that saw no visible key of a query has m = -inf
  // and weight 0 (the range's first key is in wave 0's first block and
  // visible to every query, so the maximum is finite). Every load of the stages has landed;
  // past the barrier the merge may use them.
  __syncthreads();
  f32x4 *mo = reinterpret_cast<f32x4 *>(&sh.kv[0][0][0]);  // [wave][c][dt][lane]
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const float l = sum_halves(sum_row_pairs(l_run[c]));
    if (r == 0) {
      sh.m[wave][c][i] = m_run[c];
      sh.l[wave][c][i] = l;
    }
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      mo[((wave * C + c) * 8 + dt) * 64 + lane] = o[c][dt];
  }
  __syncthreads();
  const int c = wave / (W / C), d0 = (8 * C / W) * (wave % (W / C));
  float f[W], M = -__builtin_inff();
#pragma unroll
  for (int w = 0; w < W; ++w)
    M = fmaxf(M, sh.m[w][c][i]);
  float L = 0.f;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const float m = sh.m[w][c][i];
    f[w] = m == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f((m - M) * qscale);
    L += f[w] * sh.l[w][c][i];
  }
  const int qi = 16 * c + i;
  if (qi < t.nq) {
    float *pq = t.part ? t.part + size_t(qi) * 132 : nullptr;
    if (pq && d0 == 0 && r == 0) {
      pq[128] = M;
      pq[129] = L;
    }
    uint16_t *dst = t.out + size_t(qi) * t.out_stride;
#pragma unroll
    for (int dt = d0; dt < d0 + 8 * C / W; ++dt) {
      f32x4 acc = mo[(c * 8 + dt) * 64 + lane] * f[0];
#pragma unroll
      for (int w = 1; w < W; ++w)
        acc += mo[((w * C + c) * 8 + dt) * 64 + lane] * f[w];
      // lane (query, r) holds dims 16 dt + 4 r + [0, 4)
      if (pq)
        *reinterpret_cast<f32x4 *>(pq + 16 * dt + 4 * r) = acc;
      else
        store_dims(dst, 16 * dt + 4 * r, acc, L);
    }
  }
}

// ---------------------------------------------------------------------------
// 64-query tile with K/V shared through LDS: wave w owns queries 16 w + i and
// all four waves walk the same keys, N 32-key blocks per step (N = 2: one
// rescale of O and one cross-lane maximum for both). Each block's K and V are
// fetched once per workgroup (each wave loads a quarter: K pieces and V dim
// tiles 2 w, 2 w + 1 in the MFMA operand layout of load_k / load_v, which the
// operand reads then find at constant offsets; whole-KiB loads with swizzled
// reads measured 0-8% slower here) into an LDS ring of two steps, one step
// ahead; every wave reads its operands from LDS. No merge across waves.
template <int N>
struct Tile64Lds {  // N = 2: 64 KiB, two workgroups per CU; N = 1: 32 KiB, five
  u32x4 k[2][N][8][64];  // [stage][32-key block][piece][lane]
  u32x4 v[2][N][8][64];
};
template <int N>
constexpr int kTile64Waves = N == 1 ? 5 : 2;  // waves per SIMD (LDS, registers)

template <bool kRows, int N>
__device__ __forceinline__ void attn_query_tile64(const QueryTile &t, float qscale,
                                                  Tile64Lds<N> &sh) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane >> 4, i = lane & 15;
  const int nblk = t.blk1 ? t.blk1 : (t.kend + kBlock - 1) / kBlock, nkeys = nblk * kBlock;
  const int last = t.kend - 1;
  u32x4 qb[4];
  {
    const int qi = min(16 * wave + i, t.nq - 1);
    const u32x4 *src = reinterpret_cast<const u32x4 *>(t.q + size_t(qi) * t.q_stride);
#pragma unroll
    for (int s = 0; s < 4; ++s)
      qb[s] = src[4 * s + r];
  }
  const int kmax = t.causal_pos >= 0 ? t.causal_pos + 16 * wave + i : t.kv_len - 1;
  const auto rk = key_rsrc(t.kc, 0, t.kend);
  const auto rv = key_rsrc(t.vc, 0, kRows ? t.kend : (t.kend + kBlock - 1) / kBlock * kBlock);
  // this wave's quarter of the N blocks at kb0 into `stage`: K pieces 2 w,
  // 2 w + 1 (T = w / 2, s = 2 (w % 2) + {0, 1}) and V dim tiles 2 w, 2 w + 1.
  // Keys are clamped to the last visible one.
  auto fetch = [&](int kb0, int stage) {
#pragma unroll
    for (int g = 0; g < N; ++g) {
      const int kb = kb0 + kBlock * g;
      const int key = min(kb + key_ofs(wave >> 1, i), last);
      const uint32_t ko = uint32_t(key * (D / 8) + 8 * (wave & 1) + r) * 16;
      // the missing half of an odd last step: V past the range, zeros (its
      // weights are zero, and 0 * inf of another block would be NaN)
      const uint32_t vb = uint32_t(N > 1 ? min(kb, nkeys) : kb) * (D * 2);
      const uint32_t vo0 = vb + (kRows ? v_row_fetch(lane, 2 * wave)
                                       : uint32_t((32 * wave + i) * (kBlock / 8) + r) * 16);
      const uint32_t vo1 = kRows ? vb + v_row_fetch(lane, 2 * wave + 1) : vo0 + 1024;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_ptr_t)&sh.k[stage][g][2 * wave][0], 16, ko,
                                               0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lds_ptr_t)&sh.k[stage][g][2 * wave + 1][0], 16,
                                               ko + 64, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_ptr_t)&sh.v[stage][g][2 * wave][0], 16, vo0,
                                               0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lds_ptr_t)&sh.v[stage][g][2 * wave + 1][0], 16,
                                               vo1, 0, 0, 0);
    }
  };

  float m_run = -__builtin_inff(), l_run = 0.f;
  f32x4 o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
    o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int first = t.blk0 / N, steps = (nblk + N - 1) / N;  // steps [first, steps)
  fetch(N * first * kBlock, first & 1);
  __builtin_amdgcn_s_waitcnt(0);  // (a barrier waits for no load)
  __syncthreads();
  // one step of 32 N keys; kMask: the causal / key-length mask, needed only
  // from the first step with a key past the smallest kmax of the tile's queries
  auto step = [&](int x, auto mask_tag) {
    constexpr bool kMask = decltype(mask_tag)::value;
    const int stage = x & 1, kb = N * x * kBlock;
    // step x + 1 into the stage every wave finished reading before the
    // previous barrier; in flight during this step's products
    if (x + 1 < steps)  // uniform
      fetch(kb + N * kBlock, stage ^ 1);
    // 2 N independent chains of four dependent MFMAs, interleaved
    f32x4 st[2 * N];
#pragma unroll
    for (int j = 0; j < 2 * N; ++j)
      st[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int j = 0; j < 2 * N; ++j)
        st[j] = mfma(sh.k[stage][j >> 1][4 * (j & 1) + s][lane], qb[s], st[j]);
    if constexpr (kMask) {  // lane (query 16 w + i, r): keys kb + 32 g + 8 r + 4 T + u
#pragma unroll
      for (int e = 0; e < 8 * N; ++e)
        if (kb + 32 * (e >> 3) + 8 * r + (e & 7) > kmax)
          st[e >> 2][e & 3] = -__builtin_inff();
    }
    uint32_t pw[N][3][4];
    const float corr = softmax_step<2 * N>(st, qscale, m_run, l_run, pw);
    if constexpr (N == 1) {  // dim tile by dim tile: 96 registers
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        const u32x4 vr = kRows ? v_row_operand(sh.v[stage][0][0], v_row_read(lane, dt))
                               : sh.v[stage][0][dt][lane];
        o[dt] *= corr;
#pragma unroll
        for (int k = 0; k < 3; ++k)
          o[dt] = mfma(vr, piece(pw[0][k]), o[dt]);
      }
    } else {
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
        o[dt] *= corr;
    }
#pragma unroll
    for (int g = 0; g < (N == 1 ? 0 : N); ++g) {
      u32x4 vr[8];
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
        vr[dt] = kRows ? v_row_operand(sh.v[stage][g][0], v_row_read(lane, dt))
                       : sh.v[stage][g][dt][lane];
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
          o[dt] = mfma(vr[dt], piece(pw[g][k]), o[dt]);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's part of step x + 1
    __syncthreads();
  };
  const int kfull = t.causal_pos >= 0 ? t.causal_pos + 1 : t.kv_len;
  int x = first;
  for (; x < min(kfull / (N * kBlock), steps); ++x)
    step(x, std::false_type{});
  for (; x < steps; ++x)
    step(x, std::true_type{});
  // lane (query 16 w + i, r) holds dims 16 dt + 4 r + [0, 4)
  const float L = sum_halves(sum_row_pairs(l_run));
  const int qi = 16 * wave + i;
  if (qi >= t.nq)
    return;
  if (t.part) {
    float *pq = t.part + size_t(qi) * 132;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      *reinterpret_cast<f32x4 *>(pq + 16 * dt + 4 * r) = o[dt];
    if (r == 0) {
      pq[128] = m_run;
      pq[129] = L;
    }
    return;
  }
  uint16_t *dst = t.out + size_t(qi) * t.out_stride;
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
    store_dims(dst, 16 * dt + 4 * r, o[dt], L);
}

// How a launch of `heads` heads (batch included) x q_len queries over kv_len
// keys is cut: queries and waves per workgroup (64: attn_query_tile64 with
// `blocks` key blocks a step, else the key-split tile) and, where the keys may
// be dealt (non-causal), groups > 0: the steps of all tiles go to that many
// workgroups in equal contiguous runs, merged by another kernel.
struct TilePlan {
  int queries = 64, waves = 4, groups = 0;
  int blocks = 2;
  int step_blocks() const { return queries == 64 ? blocks : waves; }
};
constexpr int kMaxPieces = 16;  // workgroups that may hold parts of a dealt tile
// Workgroups for `total` steps of tiles of `steps` each: a multiple of 8, at
// most `slots`, with at least two steps a workgroup and at most kMaxPieces
// pieces a tile (and total * groups in 31 bits, which the kernels count in); 0:
// no more workgroups than tiles.
inline int deal_groups(long long total, long long steps, int slots) {
  const long long per = std::max<long long>(2, (steps - 1) / (kMaxPieces - 1) + 1);
  const long long g = std::min<long long>(slots, total / per) / 8 * 8;
  return total < (1 << 21) && g * steps > total ? int(g) : 0;
}
// By a time model in us, fitted on MI355X's 256 CUs, every form timed: 1571
// causal shapes (1-192 heads, 1-12000 queries after 0-20000 keys) and 1704 others
// (1-192 heads, 1-5000 queries x 20-24000 keys). Of the launches over 9 us the pick
// is 0.3% / 1.7% from the fastest form on average (12% / 47% at worst: few queries
// a head over caches past L2, where the order in which workgroups meet the same
// keys decides). A step of a tile costs `alone` where a workgroup has a CU to
// itself and `full` where as many as fit do (`slots` on the chip), in between in
// proportion; a further round of workgroups costs `round`. Causal tiles are of
// unequal length: the longest one's chain, or `spread` times the mean of all.
//
// Which form where: key-split tiles while 64-query tiles leave CUs idle; one
// round of 64-query tiles two blocks a step; past it, one block a step, five
// workgroups to a CU, hides more latency and shares K and V in L2 among more
// tiles (24 heads x 8 x 2500 x 8000: 4.1 ms, dealt key-split tiles, which a model
// fitted to batch 1 took, 7.1; 64 heads x 4096 causal 540 us, two blocks 563).
// Key-split tiles past one round only for up to 64 heads: more heads pull K and
// V past L2 (24 heads x 8 x 160 x 8000: 372 us, 596 key-split). Dealt: few heads
// and long caches (1 head x 1 x 20000: 99 us undealt, 19 dealt to 8 workgroups).
inline TilePlan attn_tile_plan(long long heads, int q_len, int kv_len, bool causal, bool deal) {
  struct Form {
    int queries, waves, blocks, slots;
    double launch, round, alone, full, spread;  // spread: causal
    double deal = 0, deal_full = 0, merge = 0, merge_mb = 0;  // dealt to <= 256 / more workgroups
  };
  static const Form whole[] = {
      {16, 4, 0, 512, 4.468, 1.41, 0.9603, 1.568, 0, 0.8873, 1.623, 1.925, 0.5537},
      {16, 8, 0, 256, 4.574, 8.894, 1.106, 5.091, 0, 1.692, 0, 2.057, 0.177},
      {32, 4, 0, 512, 5.886, 1.447, 1.113, 2.081, 0, 0.8195, 5.109, 2.233, 0.5655},
      {32, 8, 0, 256, 7.677, 35.84, 1.647, 1.84, 0, 2.142, 0, 3.061, 0.2742},
      {64, 4, 2, 512, 5.386, 27.74, 1.122, 1.901, 0, 2, 1.614, 1.833, 0.5814},
      {64, 4, 1, 1280, 5.319, 0.2201, 0.6365, 2.38, 0}};
  static const Form tri[] = {
      {16, 4, 0, 512, 4.499, 8.94, 1.016, 1.214, 1.218},
      {16, 8, 0, 256, 6.903, 4.535, 0.8857, 1.604, 1.296},
      {32, 4, 0, 512, 5.473, 12.35, 1.32, 1.823, 1.073},
      {32, 8, 0, 256, 7.815, 10.35, 2.116, 2.201, 1.103},
      {64, 4, 2, 512, 4.666, 9.123, 1.19, 1.601, 1.212},
      {64, 4, 1, 1280, 4.695, 0, 0.6214, 1.485, 1.353}};
  const int nb = (kv_len + kBlock - 1) / kBlock;
  TilePlan best;
  double best_t = __builtin_inf();
  auto take = [&](const Form &f, int groups, double t) {
    if (t < best_t) {
      best = TilePlan{f.queries, f.waves, groups, f.blocks};
      best_t = t;
    }
  };
  const bool far = kv_len > kMaxRange;  // past the 64-query tile's buffers
  for (const Form &f : causal ? tri : whole) {
    if (far && f.queries == 64)
      continue;
    const int blocks = f.queries == 64 ? f.blocks : f.waves, per_cu = f.slots / 256;
    const long long tiles = heads * ((q_len + f.queries - 1) / f.queries);
    const long long steps = (nb + blocks - 1) / blocks, total = tiles * steps;
    // a step where n workgroups, less than a full chip, are spread over the CUs
    auto step = [&](long long n) {
      return f.alone +
             (per_cu == 1 ? 0.0 : (f.full - f.alone) * double((n - 1) / 256) / (per_cu - 1));
    };
    if (f.queries == 64 || far || tiles <= (heads <= 64 ? 1536 : 512)) {
      const long long full = tiles / f.slots, rem = tiles % f.slots;
      const double rate = double(full) * f.full + (rem ? step(rem) : 0.0);
      if (causal) {
        const double mean = (nb - std::max(0, q_len - f.queries) / 64.0) / blocks;
        take(f, 0, f.launch + f.round * std::max(0.0, double(tiles) / f.slots - 1) +
                       std::max(step(std::min<long long>(tiles, f.slots)) * double(steps),
                                f.spread * rate * mean));
      } else {
        take(f, 0, f.launch + f.round * double(full + (rem > 0) - 1) + rate * double(steps));
      }
    }
    const int groups = deal && f.deal > 0 ? deal_groups(total, steps, f.slots) : 0;
    if (groups) {
      const double mb = double(groups + std::min<long long>(groups, tiles)) * f.queries * (132 * 4e-6);
      take(f, groups, f.launch + f.merge + f.merge_mb * mb +
                          (groups <= 256 ? f.deal : f.deal_full) *
                              double((total + groups - 1) / groups));
    }
  }
  return best;
}

}  // namespace attn
}  // namespace yuear
