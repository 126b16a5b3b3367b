// Acoustic-model attention on gfx950 MFMA: the drop-in for nar_attention()
// (native/src/nar_attention.cpp:224-270) and its custom Metal kernel
// lyra_nar_precise_attention (nar_attention.cpp:63-218).
//
// Tensors are [batch, heads, tokens, 128] bf16 (q: Hq heads, Lq tokens; k, v:
// Hkv heads, Lk tokens; query head h reads kv head h / (Hq / Hkv)); the
// output has q's shape. Arithmetic of the reference kernel: fp32 scores of
// the bf16 operands scaled by scale * log2(e) (one fp32 constant), an exp2
// online softmax in fp32, P kept in fp32 for P.V ("precise" left operand),
// fp32 sums, bf16(o / l). causal (Lq == Lk, the conditioning prefill of
// nar.cpp:176) hides the keys after each query's own position.
//
// Structure: the query tiles of attn_tile.h (shared with the causal prefill
// attention) as attn_tile_plan chooses; non-causal launches may deal the keys
// of their tiles to a full chip of workgroups, merged by a second kernel. K and
// V are read as given, V through transposing LDS reads. (Rewriting V into
// dim-major blocks first makes the 64-query tile 2-5% faster, but cost 5 us a
// call: 512 x 3512, 24 heads, 57 against 55 us; 1024 x 8000 198 against 198.)
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "attn_core.h"
#include "attn_tile.h"
#include "common.h"
#include "kernels.h"

namespace yuear {

namespace {

using attn::D;
using attn::f32x4;
using attn::kBlock;

// Tile `tile` of kQ queries of one (batch, head).
template <int kQ>
__device__ __forceinline__ attn::QueryTile nar_tile(const NarAttnParams &p, int bh, int tile) {
  const int h = bh % p.heads, b = bh / p.heads;
  const int q0 = tile * kQ;
  const int kvh = h / (p.heads / p.kv_heads);
  const size_t kvhead = size_t(b) * p.kv_heads + kvh;
  attn::QueryTile t;
  t.kc = reinterpret_cast<const u32x4 *>(p.k) + kvhead * p.kv_len * (D / 8);
  t.vc = reinterpret_cast<const u32x4 *>(p.v) + kvhead * p.kv_len * (D / 8);
  t.nq = min(kQ, p.q_len - q0);
  t.kv_len = p.kv_len;
  t.kend = p.causal ? q0 + t.nq : p.kv_len;
  t.causal_pos = p.causal ? q0 : -1;
  t.q = p.q + (size_t(bh) * p.q_len + q0) * D;
  t.q_stride = D;
  t.out = p.out + (size_t(bh) * p.q_len + q0) * D;
  t.out_stride = D;
  return t;
}

// The tiles of a workgroup. A dealt launch (p.groups > 0, non-causal): the
// steps of all tiles (W key blocks each, tile by tile, a head's tiles
// together) are cut into p.groups equal runs, one per workgroup, so the chip is
// as full at the end as at the start whatever the number of tiles: 700 x 3512,
// 24 heads (528 tiles of 32 on 512 slots) 87 -> 75 us against 64-query tiles
// over equal ranges of keys. A run's part of a tile that it does not hold whole
// leaves a partial in the workgroup's slot 2 g (the part begins within the
// tile) or 2 g + 1 (it begins the tile). Workgroup b takes run (b % 8) * groups
// / 8 + b / 8: an XCD's workgroups take neighbouring runs, whose heads share K
// and V in its L2.
template <int kQ, int W, class F>
__device__ __forceinline__ void nar_run(const NarAttnParams &p, F &&tile_fn) {
  if (p.groups == 0) {
    const int tile = p.causal ? gridDim.y - 1 - blockIdx.y : blockIdx.y;  // longest first
    tile_fn(nar_tile<kQ>(p, blockIdx.x, tile));
    return;
  }
  const int per_head = (p.q_len + kQ - 1) / kQ, nb = (p.kv_len + kBlock - 1) / kBlock;
  const int steps = (nb + W - 1) / W;  // per tile
  const int total = p.batch * p.heads * per_head * steps;  // total * groups < 2^31
  const int g = int(blockIdx.x % 8) * (p.groups / 8) + int(blockIdx.x / 8);
  const int end = total * (g + 1) / p.groups;
  for (int s = total * g / p.groups; s < end;) {
    const int tile = s / steps, x0 = s - tile * steps, x1 = min(steps, x0 + end - s);
    attn::QueryTile t = nar_tile<kQ>(p, tile / per_head, tile % per_head);
    t.blk0 = x0 * W;
    t.blk1 = min(nb, x1 * W);
    if (x1 - x0 < steps)
      t.part = p.part + size_t(2 * g + (x0 == 0)) * (kQ * 132);
    tile_fn(t);
    s += x1 - x0;
  }
}
// 16 C queries per workgroup, keys split over its waves.
template <int C, int W>
__global__ __launch_bounds__(W * 64)
__attribute__((amdgpu_waves_per_eu(2, 2))) void nar_attn_kernel(NarAttnParams p, float qscale) {
  __shared__ attn::TileLds<C, W> sh;
  nar_run<16 * C, W>(p, [&](const attn::QueryTile &t) {
    attn::attn_query_tile<C, true, W>(t, qscale, sh);
    __syncthreads();  // the merge has read the stages
  });
}
// 64 queries per workgroup, N key blocks a step.
template <int N>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(attn::kTile64Waves<N>, attn::kTile64Waves<N>))) void
nar_attn64_kernel(NarAttnParams p, float qscale) {
  __shared__ attn::Tile64Lds<N> sh;
  nar_run<64, N>(p, [&](const attn::QueryTile &t) {
    attn::attn_query_tile64<true, N>(t, qscale, sh);  // ends with its reads done
  });
}

// out[row][d] = bf16(sum_s w_s o_s[d] / sum_s w_s l_s), w_s = exp2((m_s - max m) qscale)
// over the up to kPieces partials of each query row of a tile that more than
// one workgroup holds; one thread per (row, 4 dims). All of a thread's loads
// are issued before the first use (a piece it lacks is read as its last one,
// with weight 0).
template <int kPieces>
__global__ __launch_bounds__(256) void nar_merge_kernel(NarAttnParams p, float qscale, int kq,
                                                        int steps, int per_head, int total) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const int row = int(idx / 32);
  if (row >= p.batch * p.heads * p.q_len)
    return;
  const int d4 = int(idx % 32) * 4;
  const int bh = row / p.q_len, q = row - bh * p.q_len;
  const int tile = bh * per_head + q / kq;
  // workgroup w holds step s: w * total / groups <= s
  const int w0 = ((tile * steps + 1) * p.groups + total - 1) / total - 1;
  const int w1 = ((tile + 1) * steps * p.groups + total - 1) / total - 1;
  const int n = w1 - w0;  // pieces after the first
  if (n == 0)
    return;
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  f32x2 ml[kPieces];
  f32x4 v[kPieces];
#pragma unroll
  for (int s = 0; s < kPieces; ++s) {
    const float *ps =
        p.part + (size_t(2 * (w0 + min(s, n)) + (s == 0)) * kq + q % kq) * 132;
    ml[s] = *reinterpret_cast<const f32x2 *>(ps + 128);
    v[s] = *reinterpret_cast<const f32x4 *>(ps + d4);
  }
  float M = ml[0].x;
#pragma unroll
  for (int s = 1; s < kPieces; ++s)
    M = fmaxf(M, ml[s].x);
  float L = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < kPieces; ++s) {
    const float w = s > n || ml[s].x == -__builtin_inff()
                        ? 0.f
                        : __builtin_amdgcn_exp2f((ml[s].x - M) * qscale);
    L += w * ml[s].y;
    o += w * v[s];
  }
  attn::store_dims(p.out + size_t(row) * D, d4, o, L);
}

// Keys [0, n) of each cache head (V in 32-key dim-major blocks, kv_stride slots
// apart) -> row-major [heads][n][128]; one thread
// per 8 dims of one key.
__global__ __launch_bounds__(256) void v_rows_kernel(const uint16_t *vb, int kv_stride, int heads,
                                                     int n, uint16_t *out) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long long)heads * n * (D / 8))
    return;
  const int d8 = int(idx % (D / 8)) * 8;
  const long long row = idx / (D / 8);
  const int t = int(row % n), h = int(row / n);
  const uint16_t *src = vb + size_t(h) * kv_stride * D;
  uint32_t w[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    w[j] = uint32_t(src[attn::v_index(t, d8 + 2 * j)]) |
           (uint32_t(src[attn::v_index(t, d8 + 2 * j + 1)]) << 16);
  *reinterpret_cast<u32x4 *>(out + size_t(row) * D + d8) = u32x4{w[0], w[1], w[2], w[3]};
}

}  // namespace

hipError_t launch_v_rows(const uint16_t *vb, int kv_stride, int heads, int n, uint16_t *out,
                         hipStream_t s) {
  if (heads < 1 || n < 1 || n > kv_stride)
    return hipErrorInvalidValue;
  const long long threads = (long long)heads * n * (D / 8);
  hipLaunchKernelGGL(v_rows_kernel, dim3(unsigned((threads + 255) / 256)), dim3(256), 0, s, vb,
                     kv_stride, heads, n, out);
  return hipGetLastError();
}

namespace {
attn::TilePlan nar_plan(int batch, int heads, int q_len, int kv_len, int causal, bool deal) {
  return attn::attn_tile_plan((long long)batch * heads, q_len, kv_len, causal != 0, deal);
}
size_t part_floats(const attn::TilePlan &plan) {  // two slots per workgroup
  return size_t(plan.groups) * 2 * plan.queries * 132;
}
}  // namespace

size_t nar_attention_part_floats(int batch, int heads, int q_len, int kv_len, int causal) {
  return part_floats(nar_plan(batch, heads, q_len, kv_len, causal, true));
}

size_t nar_attention_workspace_elems(int batch, int kv_heads, int kv_len) {
  return size_t(batch) * kv_heads * size_t((kv_len + kBlock - 1) / kBlock * kBlock) * D;
}

hipError_t launch_nar_attention(NarAttnParams p, hipStream_t s) {
  if (p.batch < 1 || p.heads < 1 || p.kv_heads < 1 || p.heads % p.kv_heads || p.q_len < 1 ||
      p.kv_len < 1 || (p.causal && p.q_len != p.kv_len) || !p.q || !p.k || !p.v || !p.out)
    return hipErrorInvalidValue;
  // scale * log2(e) as in the reference kernel (nar_attention.cpp:95)
  const float qscale = 0.08838834764831845f * 1.4426950408889634f;
  attn::TilePlan plan = nar_plan(p.batch, p.heads, p.q_len, p.kv_len, p.causal, true);
  if (plan.groups && (!p.part || p.part_floats < part_floats(plan)))
    plan = nar_plan(p.batch, p.heads, p.q_len, p.kv_len, p.causal, false);
  p.groups = plan.groups;
  const int heads = p.batch * p.heads, per_head = (p.q_len + plan.queries - 1) / plan.queries;
  const dim3 grid = plan.groups ? dim3(plan.groups) : dim3(heads, per_head);
  const dim3 threads(64 * plan.waves);
  if (plan.queries == 16 && plan.waves == 4)
    hipLaunchKernelGGL((nar_attn_kernel<1, 4>), grid, threads, 0, s, p, qscale);
  else if (plan.queries == 16)
    hipLaunchKernelGGL((nar_attn_kernel<1, 8>), grid, threads, 0, s, p, qscale);
  else if (plan.queries == 32 && plan.waves == 4)
    hipLaunchKernelGGL((nar_attn_kernel<2, 4>), grid, threads, 0, s, p, qscale);
  else if (plan.queries == 32)
    hipLaunchKernelGGL((nar_attn_kernel<2, 8>), grid, threads, 0, s, p, qscale);
  else if (plan.blocks == 1)
    hipLaunchKernelGGL(nar_attn64_kernel<1>, grid, threads, 0, s, p, qscale);
  else
    hipLaunchKernelGGL(nar_attn64_kernel<2>, grid, threads, 0, s, p, qscale);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || !plan.groups)
    return e;
  const int nb = (p.kv_len + kBlock - 1) / kBlock;
  const int steps = (nb + plan.step_blocks() - 1) / plan.step_blocks();
  const int total = heads * per_head * steps;
  const int pieces = (steps - 1) / (total / plan.groups) + 2;  // at most
  const dim3 mgrid(unsigned(((long long)heads * p.q_len * 32 + 255) / 256));
  auto merge = pieces <= 2   ? nar_merge_kernel<2>
               : pieces <= 4 ? nar_merge_kernel<4>
               : pieces <= 8 ? nar_merge_kernel<8>
                             : nar_merge_kernel<attn::kMaxPieces>;
  hipLaunchKernelGGL(merge, mgrid, dim3(256), 0, s, p, qscale, plan.queries, steps, per_head,
                     total);
  return hipGetLastError();
}

}  // namespace yuear
