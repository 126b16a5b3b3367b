// Batched decode projections (3..8 independent rows) on MFMA, gfx950.
//
// y[b, r] = x[b, :] . W[row(r), :] with fp32 accumulation and one bf16
// rounding (native/src/ar.cpp:20-29), for the batched-sequence decode where
// a VALU GEMV would do 8 dot products per weight element. The weight stream
// is still read exactly once: the work is HBM-bound, v_mfma_f32_16x16x32_bf16
// only keeps the arithmetic off the VALU.
//
// Workgroup: T tiles of 8 consecutive weight rows; KW waves per tile split K,
// each in steps of 64 k. One MFMA takes 8 rows x 64 k: A row i and i + 8 are the
// two 32-k halves of weight row i (lane l: row l % 8, half l / 8 % 2, k 8 (l /
// 16) + [0, 8): 8 whole 128-byte lines a load), B column j and j + 8 the same
// halves of batch row j (zero beyond the batch), so the first and the last 8 x 8
// of D hold the halves' sums and the rest is not used. Tiles of 8 rows, not 16:
// 2048 rows x 6144 k made 128 workgroups and left half of the CUs idle (11.4 ->
// 6.9 us with 6 rows of activations).
//
// Bound by the latency of one round (launch, activations, weights, sums) and,
// from about 32 MB on, by HBM. The activations are staged in LDS once per
// workgroup, with the RMSNorm prologue (ar.cpp:30-35) or layer 0's gather done on
// the way while the weights are in flight: a row kernel before this one cost 3.5
// to 4.5 us and a launch. Its VALU work is per workgroup, so a workgroup is given
// as many tiles as leave one for each CU (or two, or a loop over tile sets with
// the next set's weights loaded as this one's are consumed); see launch_k. Each
// thread first loads its 16-byte activation chunk of every row, then all weight
// loads of its wave (non-temporal), so the staging waits only for the former
// (the vector-memory counter drains in issue order). The waves' sums are added
// through LDS in wave order, then the epilogue (store / residual / SwiGLU) runs
// one thread per (row, column).
// MI355X, us, 6 rows, before -> now (row kernel included): 4096 x 2048 normed
// 7.2 -> 6.0, 2048 x 2048 5.1 -> 4.4, 12288 x 2048 SwiGLU 13.4 -> 11.2; 5120 x
// 3072 14.0 -> 9.1, 16384 x 3072 SwiGLU 24.9 -> 18.7, 3072 x 8192 14.0 -> 12.0.
#include "common.h"
#include "kernels.h"

namespace yuear {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// Rows prepared in a buffer of their own (grid = batch rows, 256 threads), where
// the caller gives one: y may then overlap x (workgroups read x while others
// write y), and normed rows of more than 3072 are faster so (gemv_mfma_staged).
// Gather from the embedding (copy-out to x_out) and/or RMSNorm with the rounding
// points of ar.cpp:30-35, written to p.stage.
__global__ __launch_bounds__(256) void stage_rows_kernel(GemvParams p) {
  __shared__ float red[4];
  constexpr int kMaxChunks = 4;  // k <= 8192
  const int b = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nch = p.k >> 3;
  const uint16_t *src;
  if (p.embed) {
    const int t = min(max(p.tokens[b], 0), p.embed_rows - 1);
    src = p.embed + size_t(t) * p.k;
  } else {
    src = p.x + size_t(b) * p.x_stride;
  }
  const u32x4 *s4 = reinterpret_cast<const u32x4 *>(src);
  const u32x4 *g4 = reinterpret_cast<const u32x4 *>(p.norm_w ? p.norm_w : src);
  u32x4 *dst = reinterpret_cast<u32x4 *>(p.stage + size_t(b) * p.k);
  // one round of loads: this thread's chunks c = t + 256 i and their gains
  u32x4 v[kMaxChunks], g[kMaxChunks];
#pragma unroll
  for (int i = 0; i < kMaxChunks; ++i) {
    const int c = min(int(threadIdx.x) + 256 * i, nch - 1);
    v[i] = s4[c];
    g[i] = g4[c];
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < kMaxChunks; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c >= nch)
      continue;
    if (p.x_out)
      reinterpret_cast<u32x4 *>(p.x_out + size_t(b) * p.x_stride)[c] = v[i];
    const uint32_t w4[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float lo = bflo(w4[q]), hi = bfhi(w4[q]);
      ss += lo * lo;
      ss += hi * hi;
    }
  }
  if (!p.norm_w) {
#pragma unroll
    for (int i = 0; i < kMaxChunks; ++i) {
      const int c = threadIdx.x + 256 * i;
      if (c < nch)
        dst[c] = v[i];
    }
    return;
  }
  ss = wave_sum(ss);
  if (lane == 0)
    red[wave] = ss;
  __syncthreads();
  const float total = (red[0] + red[1]) + (red[2] + red[3]);
  const float scale = rbf(1.0f / __builtin_sqrtf(total / float(p.k) + p.eps));
#pragma unroll
  for (int i = 0; i < kMaxChunks; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c >= nch)
      continue;
    const uint32_t vi[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
    const uint32_t gi[4] = {g[i].x, g[i].y, g[i].z, g[i].w};
    uint32_t o[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t lo = f2bf(rbf(bflo(vi[q]) * scale) * bflo(gi[q]));
      const uint32_t hi = f2bf(rbf(bfhi(vi[q]) * scale) * bfhi(gi[q]));
      o[q] = lo | (hi << 16);
    }
    dst[c] = u32x4{o[0], o[1], o[2], o[3]};
  }
}

// K = KW * STEPS * 64; T tiles of 8 rows per workgroup.
template <int KW, int STEPS, int T>
struct Shape {
  static constexpr int K = KW * STEPS * 64;
  static constexpr int NT = KW * T * 64;
  static constexpr int NCH = K / 8;     // 16-byte chunks per activation row
  static constexpr int G = NT / NCH;    // rows staged at a time
  static constexpr int WG = NCH / 64;   // waves per staged row
  static_assert(NT <= 1024 && G >= 1 && NCH % 64 == 0, "one activation chunk per thread");
  static size_t lds_bytes(int batch) {
    return (size_t(batch) * NCH + (batch - 1) / 4 * 8 + 4) * 16 + KW * T * 512 + 8 * WG * 4;
  }
};

// The widest rows that a workgroup gathers and normalises itself.
constexpr int kMaxOwnRows = 3072;

// LOOP: a workgroup walks the sets of T tiles blockIdx + i gridDim.
template <int KW, int STEPS, int T, bool LOOP, int EPI>
__global__ __launch_bounds__(KW * T * 64) void gemv_mfma_kernel(GemvParams p) {
  extern __shared__ u32x4 lds[];
  using S = Shape<KW, STEPS, T>;
  constexpr int K = S::K, NCH = S::NCH, G = S::G, R = (8 + G - 1) / G;
  constexpr bool kPlain = K > kMaxOwnRows;  // x is prepared: no gather, no norm
  const int B = p.batch;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float *red = reinterpret_cast<float *>(lds + B * NCH + (B - 1) / 4 * 8 + 4);  // [wave][slice][8][8]
  float *ssq = red + KW * T * 128;                                             // [8][WG]

  // 1. this thread's chunk c of the rows grp, grp + G, ... first
  const int grp = wave / S::WG, c = int(threadIdx.x) - grp * NCH;
  u32x4 xr[R], gain;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int b = grp + G * i;
    if (grp < G && b < B) {
      const uint16_t *src = !kPlain && p.embed
                                ? p.embed + size_t(min(max(p.tokens[b], 0), p.embed_rows - 1)) * K
                                : p.x + size_t(b) * p.x_stride;
      xr[i] = reinterpret_cast<const u32x4 *>(src)[c];
    }
  }
  if (!kPlain && p.norm_w && grp < G)
    gain = reinterpret_cast<const u32x4 *>(p.norm_w)[c];
  // keep these loads ahead of the weight stream (the scheduler may otherwise
  // sink some below it, and the staging would then wait for every weight)
  __builtin_amdgcn_sched_barrier(0);

  // 2. this wave's weight stream: row n0 + l % 8 (clamped; mapped for the
  // lm_head phases), k = 64 (kw STEPS + s) + 32 (l / 8 % 2) + 8 (l / 16); from
  // the tiled copy when there is one (the 16-byte piece of (row, 32 k) sits at
  // ((row / 16) (K / 32) + k / 32) 64 + row % 16 + 16 (l / 16))
  const int kw = wave % KW, half = (lane >> 3) & 1;
  const int step = p.w_tiled ? 128 : 8;
  auto weights = [&](int set) {
    const int lr = min((set * T + wave / KW) * 8 + (lane & 7), p.n - 1);
    const int row = lr < p.seg0_len ? p.seg0_start + lr : p.seg1_start + (lr - p.seg0_len);
    return p.w_tiled ? reinterpret_cast<const u32x4 *>(p.w_tiled) +
                           (size_t(row >> 4) * (K / 32) + kw * STEPS * 2 + half) * 64 + (row & 15) +
                           16 * (lane >> 4)
                     : reinterpret_cast<const u32x4 *>(p.w + size_t(row) * K) + kw * STEPS * 8 +
                           4 * half + (lane >> 4);
  };
  u32x4 a[STEPS];
  {
    const u32x4 *w = weights(blockIdx.x);
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
      a[s] = __builtin_nontemporal_load(w + step * s);
  }

  // 3. gather copy-out, RMSNorm, staging
  if (!kPlain && p.x_out && blockIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (grp < G && grp + G * i < B)
        reinterpret_cast<u32x4 *>(p.x_out + size_t(grp + G * i) * p.x_stride)[c] = xr[i];
  }
  if (!kPlain && p.norm_w) {
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (grp < G && grp + G * i < B) {
        const uint32_t w4[4] = {xr[i].x, xr[i].y, xr[i].z, xr[i].w};
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float lo = bflo(w4[q]), hi = bfhi(w4[q]);
          ss += lo * lo;
          ss += hi * hi;
        }
        ss = wave_sum(ss);
        if (lane == 0)
          ssq[(grp + G * i) * S::WG + wave % S::WG] = ss;
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (grp < G && grp + G * i < B) {
        float total = 0.f;
#pragma unroll
        for (int w = 0; w < S::WG; ++w)
          total += ssq[(grp + G * i) * S::WG + w];
        const float scale = rbf(1.0f / __builtin_sqrtf(total / float(K) + p.eps));
        const uint32_t vi[4] = {xr[i].x, xr[i].y, xr[i].z, xr[i].w};
        const uint32_t gi[4] = {gain.x, gain.y, gain.z, gain.w};
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t lo = f2bf(rbf(bflo(vi[q]) * scale) * bflo(gi[q]));
          const uint32_t hi = f2bf(rbf(bfhi(vi[q]) * scale) * bfhi(gi[q]));
          o[q] = lo | (hi << 16);
        }
        xr[i] = u32x4{o[0], o[1], o[2], o[3]};
      }
  }
  // row b starts at chunk b NCH + b % 4 + 8 (b / 4): of the 16 lanes an operand
  // read is served in at a time, at most two pairs share a 16-byte slot of the 64
  // banks. (Rows two chunks apart, without conflicts: the same to 0.1 us, but k
  // 8192, at its register limit, 11.8 -> 13.0 us.)
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int b = grp + G * i;
    if (grp < G && b < B)
      lds[b * NCH + (b & 3) + 8 * (b >> 2) + c] = xr[i];
  }
  __syncthreads();

  // 4. MFMA over this wave's K slice; of D's 16 x 16 the (first 8 rows, first 8
  // columns) hold the first halves' sums and the last 8 x 8 the second's
  const int j = lane & 7;
  const bool live = j < B;
  const int jb = min(j, B - 1);
  const u32x4 *xrow = lds + jb * NCH + (jb & 3) + 8 * (jb >> 2) + kw * STEPS * 8 +
                      4 * ((lane >> 3) & 1) + (lane >> 4);
  const int sets = (p.n + 8 * T - 1) / (8 * T);
  for (int set = blockIdx.x;; set += gridDim.x) {
    const bool more = LOOP && set + int(gridDim.x) < sets;  // uniform
    const u32x4 *next = weights(more ? set + int(gridDim.x) : set);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const u32x4 bv = live ? xrow[8 * s] : u32x4{0u, 0u, 0u, 0u};
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[s]), as_bf16x8(bv), acc, 0, 0, 0);
      if (more)
        a[s] = __builtin_nontemporal_load(next + step * s);
    }

    // 5. sum the waves' halves (wave order), epilogue per (row, column)
    if ((lane >> 5) == ((lane >> 3) & 1)) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        red[wave * 128 + (lane >> 5) * 64 + (4 * ((lane >> 4) & 1) + t) * 8 + j] = acc[t];
    }
    __syncthreads();
    if (wave < T) {
      const int i = lane >> 3, row = (set * T + wave) * 8 + i;  // column j
      float y = 0.f, y1 = 0.f;
#pragma unroll
      for (int w = 0; w < 2 * KW; ++w)
        y += red[wave * KW * 128 + w * 64 + lane];
      if constexpr (EPI == kEpiSwiGLU)
        y1 = __shfl_down(y, 8);
      if (j < B && row < p.n) {
        uint16_t *yb = p.y + size_t(j) * p.y_stride;
        if constexpr (EPI == kEpiSwiGLU) {
          if ((i & 1) == 0) {  // rows (2m, 2m + 1) = (gate_m, up_m)
            const float g = rbf(y), u = rbf(y1);
            const float act = rbf(g * (1.0f / (1.0f + expf(-g))));
            yb[row >> 1] = f2bf(act * u);
          }
        } else if constexpr (EPI == kEpiResidual) {
          yb[row] = f2bf(bf2f(yb[row]) + rbf(y));
        } else {
          yb[row] = f2bf(y);
        }
      }
    }
    if (!more)
      break;
    __syncthreads();  // the sums are read
  }
  if (p.advance && blockIdx.x == 0 && threadIdx.x < p.batch)
    p.advance[threadIdx.x] += 1;
}

constexpr int kLoopGroups = 512;  // two workgroups of 8 waves per CU

template <int KW, int STEPS, int T, bool LOOP, int EPI>
hipError_t launch_epi(const GemvParams &p, hipStream_t s) {
  const size_t lds = Shape<KW, STEPS, T>::lds_bytes(p.batch);
  auto kern = gemv_mfma_kernel<KW, STEPS, T, LOOP, EPI>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
  if (e != hipSuccess)
    return e;
  int grid = (p.n + 8 * T - 1) / (8 * T);
  if (LOOP) {  // equal numbers of sets
    const int rounds = (grid + kLoopGroups - 1) / kLoopGroups;
    grid = (grid + rounds - 1) / rounds;
  }
  hipLaunchKernelGGL(kern, dim3(grid), dim3(KW * T * 64), lds, s, p);
  return hipGetLastError();
}

template <int KW, int STEPS, int T, bool LOOP = false>
hipError_t launch_shape(const GemvParams &p, hipStream_t s) {
  switch (p.epilogue) {
  case kEpiStore: return launch_epi<KW, STEPS, T, LOOP, kEpiStore>(p, s);
  case kEpiResidual: return launch_epi<KW, STEPS, T, LOOP, kEpiResidual>(p, s);
  case kEpiSwiGLU: return launch_epi<KW, STEPS, T, LOOP, kEpiSwiGLU>(p, s);
  }
  return hipErrorInvalidValue;
}

// Tiles per workgroup: the fewest that leave at most one workgroup per CU (256),
// so each CU stages and normalises the activations once and all CUs have a part
// of the weights. Beyond: a loop over sets of two tiles (16384 x 3072, 6 rows:
// 18.7 us; sets of four in two rounds 21.3), or, where three tiles' 12 waves fit
// a CU twice, one round of those (12288 x 2048: 11.2 us, the loop 12.4). Normed
// rows take the threads of another tile even so (4096 x 2048, 8 rows: 8.7 us with
// one tile, 6.7 with two; 1024 x 3072 10.1 with two, 9.2 with three). K of 6144
// and more is a single workgroup per CU: 16 waves on one tile, or on two (its rows
// are always prepared, so its 128 registers a lane hold the weights of 16 steps:
// 101, where the gather and norm code made it spill 12-29 of them).
hipError_t launch_k(const GemvParams &p, hipStream_t s) {
  const int tiles = (p.n + 7) / 8;
  // rows of one tile a workgroup; two tiles are one workgroup, which has read all of
  // x before it writes: up to 16 outputs may lie over x
  const bool norm = p.norm_w != nullptr, single = tiles <= 256 && tiles != 2;
  switch (p.k) {
  case 2048:
    return single && !norm ? launch_shape<4, 8, 1>(p, s)
           : tiles <= 512  ? launch_shape<4, 8, 2>(p, s)
           : tiles <= 768  ? launch_shape<4, 8, 3>(p, s)
           : tiles <= 1024 ? launch_shape<4, 8, 4>(p, s)
           : tiles <= 1536 ? launch_shape<4, 8, 3>(p, s)
                           : launch_shape<4, 8, 2, true>(p, s);
  case 3072:
    return tiles <= 512 && !norm ? launch_shape<4, 12, 2>(p, s)
           : tiles <= 768        ? launch_shape<4, 12, 3>(p, s)
           : tiles <= 1024       ? launch_shape<4, 12, 4>(p, s)
                                 : launch_shape<4, 12, 2, true>(p, s);
  case 6144:
    return single ? launch_shape<16, 6, 1>(p, s) : launch_shape<8, 12, 2>(p, s);
  case 8192:
    return single ? launch_shape<16, 8, 1>(p, s) : launch_shape<8, 16, 2>(p, s);
  }
  return hipErrorInvalidValue;
}

__global__ __launch_bounds__(256) void tile_rows_kernel(const uint16_t *w, int n, int k,
                                                        uint16_t *out, size_t total) {
  const size_t o = size_t(blockIdx.x) * 256 + threadIdx.x;  // 16-byte piece of out
  if (o >= total)
    return;
  const int l = int(o & 63);
  const size_t blk = o >> 6;
  const int ks = k / 32;
  const size_t t = blk / ks;
  const int s = int(blk % ks);
  const size_t row = t * 16 + (l & 15);
  u32x4 v = u32x4{0u, 0u, 0u, 0u};
  if (row < size_t(n))
    v = reinterpret_cast<const u32x4 *>(w + row * k + 32 * s + 8 * (l >> 4))[0];
  reinterpret_cast<u32x4 *>(out)[o] = v;
}

}  // namespace

hipError_t launch_tile_rows(const uint16_t *w, int n, int k, uint16_t *out, hipStream_t s) {
  if (n < 1 || k < 32 || k % 32)
    return hipErrorInvalidValue;
  const size_t total = size_t((n + 15) / 16) * (k / 32) * 64;
  hipLaunchKernelGGL(tile_rows_kernel, dim3(unsigned((total + 255) / 256)), dim3(256), 0, s, w, n,
                     k, out, total);
  return hipGetLastError();
}

bool gemv_mfma_supported(const GemvParams &p) {
  return p.batch >= 3 && p.batch <= 8 && (p.x_stride % 8 == 0 || p.embed) &&
         (p.k == 3072 || p.k == 8192 || p.k == 2048 || p.k == 6144) &&
         (p.epilogue != kEpiSwiGLU || p.n % 2 == 0);
}

// Every workgroup would repeat the norm of 6144 or 8192 wide rows while its only
// tiles wait (3072 x 8192, 8 rows: 25 us, 16 with the row kernel before it).
bool gemv_mfma_staged(const GemvParams &p) {
  return gemv_mfma_supported(p) && (p.norm_w || p.embed || p.x_out) && p.k > kMaxOwnRows;
}

hipError_t launch_gemv_mfma(const GemvParams &p, hipStream_t s) {
  if (!gemv_mfma_supported(p) || p.n < 1 || (gemv_mfma_staged(p) && !p.stage))
    return hipErrorInvalidValue;
  if (!p.stage || (!p.norm_w && !p.embed && !p.x_out))
    return launch_k(p, s);
  hipLaunchKernelGGL(stage_rows_kernel, dim3(p.batch), dim3(256), 0, s, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return e;
  GemvParams q = p;
  q.x = p.stage;
  q.x_stride = p.k;
  q.norm_w = nullptr;
  q.embed = nullptr;
  q.x_out = nullptr;
  return launch_k(q, s);
}

}  // namespace yuear
