// Prefill projections for few tokens on gfx950 MFMA: C = A . W^T with the
// epilogues of gemm.hip (store, residual, SwiGLU; native/src/ar.cpp:20-51,
// 292-298), for shapes whose output is one round of tiles on the GPU.
//
// Bound: the bytes that a CU pulls from its L2, and the weights from HBM. With
// one tile per CU nothing but more bytes in flight shortens the K loop, and a
// 128 x 128 tile leaves most CUs idle at a few hundred tokens. So the output
// is cut into up to one tile per CU, as square as it goes (a tile of BM x BN
// reads (BM + BN) K values), and the waves of a workgroup split K: each wave
// has a K range of its own, a ring of its own in LDS filled by direct-to-LDS
// loads, and the whole tile's accumulators. No barrier runs in the K loop, no
// partial sum leaves the workgroup: the waves' tiles are added through LDS, in
// wave order, before the epilogue. A load instruction moves 8 rows x 128 bytes
// (whole cache lines): the same kernel reading MFMA fragments straight into
// registers (16 rows x 64 bytes a load) pulled a third of the bytes per second.
//
// Ring depth 1 is enough with 8 waves, and with 4 waves of a large tile: a
// wave's fragments go to registers before its stage is refilled, so a stage is
// in flight while its MFMAs run.
//
// Measured on MI355X with cold weights, us per launch, against the best of the
// 128-wide tiles (one pass / K split over workgroups and a reduce kernel):
//   tokens  5120x3072         3072x3072         16384x3072 SwiGLU  3072x8192
//     16    10.0 (41 / 15)     7.3 (41 / 12)    21.8 (47 / 28)     13.1 (99 / 18)
//    130    15.7 (42 / 26)    12.1 (42 / 24)    36   (48)          23.5 (98 / 29)
//    301    24.9 (43 / 35)    15.9 (43 / 26)    -                  30.7 (100 / 39)
//    700    35.3 (45)         25.4 (44 / 38)    -                  50.1 (102 / 56)
#include "common.h"
#include "gemm_epilogue.h"
#include "kernels.h"

namespace yuear {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *lds_ptr_t;

constexpr int kBK = 64;  // K per step: 128 bytes of a row

// The kernel's only LDS object, so that the compiler does not wait for the
// loads in flight before it reads a landed stage (see gemm.hip).
extern __shared__ __attribute__((aligned(1024))) char ksplit_ring[];

// vmcnt(N): at most N of this wave's vector memory operations in flight.
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N < 64, "vmcnt has 6 bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const void *base, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0,
                                           uint32_t(bytes > 0xffffffffu ? 0xffffffffu : bytes),
                                           0x00020000);
}

// MT x NB tiles of 16 tokens x 16 features per workgroup of W waves, each with
// DEPTH stages of (16 NB + 16 MT) rows x 128 bytes: W rows, then A rows, chunk
// kc of row R at slot kc ^ ((R >> 1) & 7) as in gemm.hip (no bank conflicts).
// MFMA layouts as in gemm_tile16 there: lane l holds token l % 16, features
// 4 (l / 16) + [0, 4) of a 16 x 16 tile.
template <int MT, int NB, int W, int DEPTH>
__device__ __forceinline__ void ksplit_tile(const GemmParams &p, int tiles_m, int tiles) {
  constexpr int BM = 16 * MT, BN = 16 * NB;
  constexpr int L = (BM + BN) / 8, STAGE = L * 1024;  // 1 KiB loads per stage
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // XCD x (workgroups are dispatched round-robin) takes a contiguous range of
  // tiles, the token tiles of one weight block next to each other: each weight
  // byte is fetched from HBM into one L2 only
  const int per_xcd = int(gridDim.x) >> 3;
  const int t = int(blockIdx.x & 7) * per_xcd + int(blockIdx.x >> 3);
  if (t >= tiles)
    return;
  const int m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;
  const int steps = p.k / kBK;
  const int beg = steps * wave / W, end = steps * (wave + 1) / W;
  const auto ra = rows_rsrc(p.a + size_t(m0) * p.lda, size_t(p.m - m0) * p.lda * 2);
  const auto rw = rows_rsrc(p.w + size_t(n0) * p.k, size_t(p.n - n0) * p.k * 2);
  char *ring = ksplit_ring + wave * (DEPTH * STAGE);
  // lane l of load q: row 8 q + l / 8, chunk (l % 8) ^ f(row). All of a load's
  // offset is in the vector part, which the buffer's range check covers
  uint32_t ga[2], gw[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    const int kc = (lane & 7) ^ (lane >> 4) ^ (4 * o);
    ga[o] = uint32_t((8 * o + (lane >> 3)) * p.lda + kc * 8) * 2;
    gw[o] = uint32_t((8 * o + (lane >> 3)) * p.k + kc * 8) * 2;
  }
  auto dma = [&](int slot, int s) {
    char *stage = ring + slot * STAGE;
#pragma unroll
    for (int q = 0; q < L; ++q) {
      const int rows16 = q < 2 * NB ? q >> 1 : (q >> 1) - NB;
      const uint32_t off = uint32_t(rows16 * 16 * (q < 2 * NB ? p.k : p.lda) + s * kBK) * 2;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(q < 2 * NB ? rw : ra, (lds_ptr_t)(stage + q * 1024),
                                               16, (q < 2 * NB ? gw[q & 1] : ga[q & 1]) + off, 0, 0,
                                               0);
    }
  };

  f32x4 acc[NB][MT];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int a = 0; a < MT; ++a)
      acc[b][a] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int i16 = lane & 15, q4 = lane >> 4;
  const int f = (lane >> 1) & 7, row = i16 * 128;
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (beg + d < end)
      dma(d, beg + d);
  for (int s = beg, slot = 0; s < end; ++s) {
    if (DEPTH > 1 && s + DEPTH <= end)
      wait_loads<(DEPTH - 1) * L>();
    else
      wait_loads<0>();
    __builtin_amdgcn_sched_barrier(0);
    const char *stage = ring + slot * STAGE;
    bf16x8 wf[2][NB], af[2][MT];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int co = row + (((4 * h + q4) ^ f) * 16);
#pragma unroll
      for (int b = 0; b < NB; ++b)
        wf[h][b] = *reinterpret_cast<const bf16x8 *>(stage + b * 2048 + co);
#pragma unroll
      for (int a = 0; a < MT; ++a)
        af[h][a] = *reinterpret_cast<const bf16x8 *>(stage + (NB + a) * 2048 + co);
    }
    // the stage is in registers (lgkmcnt(0)) before its refill is issued
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_sched_barrier(0);
    if (s + DEPTH < end)
      dma(slot, s + DEPTH);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int a = 0; a < MT; ++a)
          acc[b][a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][b], af[h][a], acc[b][a], 0, 0, 0);
    slot = slot + 1 == DEPTH ? 0 : slot + 1;
  }
  // every load has landed (the last step waits for all); past the barrier the
  // rings are free for the sums

  // Sum over the waves, RP rows of tiles at a time, RP as many as the rings
  // hold. A thread takes 4 consecutive features of a token, neighbours in a
  // wave the next ones of the same token (whole lines of C). The quad of token
  // i, feature quad r of tile (a, b) lies at i ^ (r + 4 b) % 16 of the tile's
  // r-th quarter, so that both the writes (16 tokens of one quad) and the
  // reads (16 quads of one token) go to 16 different 16-byte slots.
  f32x4 *red = reinterpret_cast<f32x4 *>(ksplit_ring);
  constexpr int kFit = W * DEPTH * STAGE / (W * NB * 1024);
  constexpr int RP = MT < kFit ? MT : kFit;
  static_assert(RP >= 1, "a row of tiles of every wave fits in the rings");
#pragma unroll
  for (int a0 = 0; a0 < MT; a0 += RP) {
    __syncthreads();
#pragma unroll
    for (int a = a0; a < (a0 + RP < MT ? a0 + RP : MT); ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        red[((wave * RP + a - a0) * NB + b) * 64 + (i16 ^ ((q4 + 4 * b) & 15)) + 16 * q4] = acc[b][a];
    __syncthreads();
    const int rows = (MT - a0 < RP ? MT - a0 : RP) * 16;
    for (int x = threadIdx.x; x < rows * (4 * NB); x += W * 64) {
      const int mr = x / (4 * NB), nq = x % (4 * NB), b = nq >> 2, r = nq & 3;
      const f32x4 *src =
          red + ((mr >> 4) * NB + b) * 64 + ((mr & 15) ^ ((r + 4 * b) & 15)) + 16 * r;
      f32x4 v = src[0];
#pragma unroll
      for (int w = 1; w < W; ++w)
        v += src[w * RP * NB * 64];
      const int m = m0 + 16 * a0 + mr;
      if (m < p.m) {
        const float o[4] = {v.x, v.y, v.z, v.w};
        epilogue4(p, m, n0 + 4 * nq, o);
      }
    }
  }
}

// Tile shapes: MT, NB, W, DEPTH. Concrete kernels over a device template (a
// template kernel instantiated from host code gets no launch stub here).
#define YUEAR_KSPLIT_SHAPES(X)                                                               \
  X(1, 1, 8, 2) X(1, 2, 8, 2) X(1, 4, 8, 1) X(2, 2, 8, 1) X(3, 2, 8, 1) X(2, 4, 8, 1)         \
  X(3, 4, 8, 1) X(4, 4, 8, 1) X(5, 4, 8, 1) X(6, 4, 8, 1) X(4, 6, 8, 1) X(8, 4, 4, 1)         \
  X(6, 6, 4, 1) X(6, 8, 4, 1) X(8, 6, 4, 1) X(8, 8, 4, 1)
#define YUEAR_KSPLIT_KERNEL(MT, NB, W, DEPTH)                                                \
  __global__ __launch_bounds__(W * 64) void gemm_ksplit_##MT##x##NB(GemmParams p, int tiles_m, \
                                                                    int tiles) {            \
    ksplit_tile<MT, NB, W, DEPTH>(p, tiles_m, tiles);                                        \
  }
YUEAR_KSPLIT_SHAPES(YUEAR_KSPLIT_KERNEL)
#undef YUEAR_KSPLIT_KERNEL

struct KsplitShape {
  int mt, nb, waves, depth;
  void (*kernel)(GemmParams, int, int);
  int lds() const { return waves * depth * (mt + nb) * 2048; }
};
#define YUEAR_KSPLIT_ENTRY(MT, NB, W, DEPTH) {MT, NB, W, DEPTH, gemm_ksplit_##MT##x##NB},
const KsplitShape kShapes[] = {YUEAR_KSPLIT_SHAPES(YUEAR_KSPLIT_ENTRY)};
#undef YUEAR_KSPLIT_ENTRY
constexpr int kNumShapes = int(sizeof(kShapes) / sizeof(kShapes[0]));

}  // namespace

// The shapes that do the GEMM in one round (a workgroup per CU, two where two
// rings fit in its 160 KiB of LDS), and among them the one of least time: a CU
// reads its tiles' rows at 86 KB/us and spends 0.17 us per 16 x 16 tile on the
// sums and the epilogue. Fitted to every shape at 9-2048 tokens and the
// projections of both decoder widths on MI355X with cold weights: the pick is
// within 0.8% of the fastest on average, within 14% always. Past one round the
// 128-wide tiles read fewer bytes per product: gate/up at 301 tokens 61 us in
// two rounds, 56 with 256 x 128 tiles. Within one round they win at short K, whose
// sums over the waves cost more than the products (700 x 4096 x 256: 9.4 us, 8.6
// with 128 x 128 tiles): *us is the estimate that gemm_pick compares, fitted with
// theirs.
int gemm_ksplit_choice(int m, int n, int k, int cus, double *us) {
  int best = -1;
  double best_t = 0;
  for (int i = 0; i < kNumShapes; ++i) {
    const KsplitShape &s = kShapes[i];
    const int bm = 16 * s.mt, bn = 16 * s.nb;
    const long long tiles = (long long)((m + bm - 1) / bm) * ((n + bn - 1) / bn);
    const int per_cu = s.lds() <= 80 * 1024 ? 2 : 1;
    if (tiles > (long long)cus * per_cu)
      continue;
    const double kb = double(bm + bn) * k * 2e-3;  // KB of rows a tile reads
    const int rounds = tiles > cus ? 2 : 1;
    const double t = rounds * (kb / 86.0 + 0.17 * s.mt * s.nb);
    if (best < 0 || t < best_t) {
      best = i;
      best_t = t;
      *us = 1.215 + rounds * (kb / 74.7 + 0.1482 * s.mt * s.nb + 0.7085);
    }
  }
  return best;
}

hipError_t launch_gemm_ksplit(const GemmParams &p, int shape, hipStream_t st) {
  if (p.m < 1 || p.n < 1 || p.k < kBK || p.k % kBK || p.lda < p.k || p.lda % 8 || !p.a || !p.w ||
      !p.c || p.residual < 0 || p.residual > 2 || (p.residual == 2 && p.n % 2) ||
      p.ldc < (p.residual == 2 ? p.n / 2 : p.n) || shape < 0 || shape >= kNumShapes)
    return hipErrorInvalidValue;
  const KsplitShape &s = kShapes[shape];
  const int tiles_m = (p.m + 16 * s.mt - 1) / (16 * s.mt);
  const int tiles = tiles_m * ((p.n + 16 * s.nb - 1) / (16 * s.nb));
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(s.kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, s.lds());
  if (e != hipSuccess)
    return e;
  hipLaunchKernelGGL(s.kernel, dim3((tiles + 7) / 8 * 8), dim3(s.waves * 64), s.lds(), st, p,
                     tiles_m, tiles);
  return hipGetLastError();
}

}  // namespace yuear
