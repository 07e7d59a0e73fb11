// Loss head of the U-Net train step, fused: fp32 log-softmax over the class logits of every voxel, the
// (optionally class-weighted) cross-entropy sum with its normaliser, and the soft-Dice sums per (sample, class)
// in ONE pass over the logits; the backward is one more pass. This is the block ScaFFold/utils/trainer.py:634-663
// builds from torch ops (log_softmax -> nll_loss(reduction="none").sum() / normaliser, ScaFFold/utils/losses.py:
// 119-214; exp -> Dice sums -> (2I + eps) / (P + T + eps), ScaFFold/utils/dice_score.py:101-136; loss =
// CE + 1 - mean foreground Dice, trainer.py:331-333,660-663). It is bandwidth-bound: 22 B of bf16 logits and an
// 8-byte label per voxel at 11 classes.
//
// No atomics: every workgroup leaves its partial sums in its own slot and one workgroup adds the slots in a
// fixed order (the reference avoids the atomic fused reduction for the same reason, losses.py:156-160).
#include "loss.hpp"

namespace sfh {
namespace {

constexpr int kBlock = 256;

template <typename T> __device__ __forceinline__ float ld(const T* p) { return to_float(*p); }

__device__ __forceinline__ float wave_sum_all(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;  // lane 0 holds the sum
}

// The same total, pair by pair, in lane 63 and on the vector pipe alone: halves and rows of 16 lanes traded, then shifts of 8, 4, 2 and 1
// within the rows. The 3 C + 2 totals of a workgroup made 228 trips through the LDS pipe as shuffles.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum_last(float v) {
  const auto half = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(half[0]) + __uint_as_float(half[1]);
  const auto row = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(row[0]) + __uint_as_float(row[1]);
  v = dpp_add<0x118>(v);
  v = dpp_add<0x114>(v);
  v = dpp_add<0x112>(v);
  return dpp_add<0x111>(v);
}

// Voxels a thread works on between two barriers: as many as keep a tile's logits within 32 KiB of LDS, so that four
// workgroups fit a CU and a workgroup's trips to memory are one or two, not one per 256 voxels. bf16 in a trace, before and now: partial
// sums of 11 classes of 64x128x128 25 -> 18.9 us (54 MB; the totals' trips through the LDS pipe were 6 us of it), of 6 classes of
// 128-cube 36 -> 18.9, of 11 classes of 32-cube 11.7 -> 6.3, of 17 of 32x64x64 27.7 -> 14.1; backward 23 -> 18.4, 38 -> 21.2, 5.2 -> 4.9, 11.0 -> 10.2.
template <typename T, int CMAX> constexpr int kVoxels = 32768 / (kBlock * CMAX * (int)sizeof(T)) >= 4   ? 4
                                                        : 32768 / (kBlock * CMAX * (int)sizeof(T)) >= 2 ? 2
                                                                                                        : 1;

// The kernels are built for up to CMAX classes; a class below the smallest count that CMAX is taken for needs no question.
template <int CMAX>
__device__ __forceinline__ bool has_class(int c, int C) {
  constexpr int kFewest = CMAX == 32 ? 17 : CMAX == 16 ? 13 : CMAX == 4 ? 2 : CMAX - 1;
  return c < kFewest || c < C;
}

// A tile's logits are one contiguous byte range whatever the class count (11 classes: 22-byte rows): it moves between
// global memory and LDS in 16-byte pieces when the range starts on a 16-byte boundary (`vec`), element by element else.
template <typename T>
__device__ __forceinline__ void tile_in(T* tile, const T* __restrict__ src, int nelem, bool vec) {
  const int tid = threadIdx.x;
  if (vec) {
    constexpr int E = 16 / (int)sizeof(T), U = 8;  // pieces of a thread in flight
    const int npiece = nelem / E;
    for (int i0 = tid; i0 < npiece; i0 += U * kBlock) {
      uint4 piece[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int i = i0 + k * kBlock;
        piece[k] = reinterpret_cast<const uint4*>(src)[i < npiece ? i : npiece - 1];
      }
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int i = i0 + k * kBlock;
        if (i < npiece) reinterpret_cast<uint4*>(tile)[i] = piece[k];
      }
    }
    for (int i = npiece * E + tid; i < nelem; i += kBlock) tile[i] = src[i];
  } else {
    for (int i = tid; i < nelem; i += kBlock) tile[i] = src[i];
  }
}
template <typename T>
__device__ __forceinline__ void tile_out(T* __restrict__ dst, const T* tile, int nelem, bool vec) {
  const int tid = threadIdx.x;
  if (vec) {
    constexpr int E = 16 / (int)sizeof(T);
    const int npiece = nelem / E;
    for (int i = tid; i < npiece; i += kBlock) reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(tile)[i];
    for (int i = npiece * E + tid; i < nelem; i += kBlock) dst[i] = tile[i];
  } else {
    for (int i = tid; i < nelem; i += kBlock) dst[i] = tile[i];
  }
}

// The labels of a thread's voxels of one tile, asked for before the tile's logits are waited for.  A label outside
// [0, C) (an ignored voxel) becomes -1.
template <int VOX>
__device__ __forceinline__ void labels_in(int (&y)[VOX], const int64_t* __restrict__ lab, int nv, int C) {
  int64_t raw[VOX];
#pragma unroll
  for (int u = 0; u < VOX; ++u) {
    const int i = (int)threadIdx.x + u * kBlock;
    raw[u] = lab[i < nv ? i : nv - 1];
  }
#pragma unroll
  for (int u = 0; u < VOX; ++u) y[u] = raw[u] >= 0 && raw[u] < C ? (int)raw[u] : -1;
}

// Quantities per sample: inter[c], psum[c], tsum[c] (3 * C), then the two launch-wide ones: ce_sum, normaliser.
template <typename T, int CMAX>
__global__ void __launch_bounds__(kBlock) ce_dice_partial(const T* __restrict__ logits, const int64_t* __restrict__ labels,
                                                          const float* __restrict__ cw, float* __restrict__ part, int64_t S, int C,
                                                          int nsplit, int64_t per_split, int vec) {
  extern __shared__ __align__(16) char smem_raw[];
  T* tile = reinterpret_cast<T*>(smem_raw);  // kVoxels * kBlock voxels x C logits
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = blockIdx.y, split = blockIdx.x;
  const T* src = logits + (int64_t)n * S * C;
  const int64_t* lab = labels + (int64_t)n * S;
  constexpr int VOX = kVoxels<T, CMAX>;
  float inter[CMAX], psum[CMAX], ce = 0.f, norm = 0.f;
  int tsum[CMAX];  // voxels of a class: whole numbers
#pragma unroll
  for (int c = 0; c < CMAX; ++c) {
    inter[c] = psum[c] = 0.f;
    tsum[c] = 0;
  }
  const int64_t begin = (int64_t)split * per_split;
  int64_t end = begin + per_split;
  if (end > S) end = S;
  for (int64_t v0 = begin; v0 < end; v0 += VOX * kBlock) {
    const int nv = (int)((end - v0) < VOX * kBlock ? (end - v0) : VOX * kBlock);
    int label[VOX];
    labels_in<VOX>(label, lab + v0, nv, C);
    __syncthreads();
    tile_in<T>(tile, src + v0 * C, nv * C, vec != 0);
    __syncthreads();
#pragma unroll 1
    for (int u = 0; u < VOX; ++u) {
      const int at = tid + u * kBlock;
      if (at >= nv) break;
      const T* row = tile + at * C;
      float x[CMAX];
      float m = -INFINITY;
#pragma unroll
      for (int c = 0; c < CMAX; ++c) {
        x[c] = has_class<CMAX>(c, C) ? to_float(row[c]) : -INFINITY;
        m = fmaxf(m, x[c]);
      }
      float s = 0.f;
#pragma unroll
      for (int c = 0; c < CMAX; ++c) {
        x[c] = has_class<CMAX>(c, C) ? expf(x[c] - m) : 0.f;  // x now holds exp(logit - max)
        s += x[c];
      }
      const float inv = 1.f / s, logs = logf(s);
      int y = label[0];
#pragma unroll
      for (int k = 1; k < VOX; ++k) y = u == k ? label[k] : y;
#pragma unroll
      for (int c = 0; c < CMAX; ++c) {
        const float p = x[c] * inv;
        const bool hit = c == y;
        psum[c] += p;
        inter[c] += hit ? p : 0.f;
        tsum[c] += hit ? 1 : 0;
      }
      if (y >= 0) {
        const float w = cw != nullptr ? cw[y] : 1.f;
        // -log p_y = log(sum) - (logit_y - max)
        ce += w * (logs - (to_float(row[y]) - m));
        norm += w;
      }
    }
  }
  // workgroup totals: every quantity through the wavefront tree, the wave totals parked in LDS, then one thread per
  // quantity adds the four wave totals in order (one barrier for all 3 C + 2 quantities)
  float* dst = part + ((int64_t)n * nsplit + split) * (3 * C + 2);
  __syncthreads();  // the tile is consumed: its LDS holds the wave totals now
  float* wave_tot = reinterpret_cast<float*>(smem_raw);  // [4][3 * CMAX + 2]
  constexpr int Q = 3 * CMAX + 2;
  auto park = [&](float v, int slot) {
    v = wave_sum_last(v);
    if (lane == 63) wave_tot[wave * Q + slot] = v;
  };
#pragma unroll
  for (int c = 0; c < CMAX; ++c) {
    park(inter[c], c);
    park(psum[c], CMAX + c);
    park((float)tsum[c], 2 * CMAX + c);
  }
  park(ce, 3 * CMAX);
  park(norm, 3 * CMAX + 1);
  __syncthreads();
  if (tid < Q) {
    const int q = tid < 3 * CMAX ? tid / CMAX : 3, c = tid < 3 * CMAX ? tid % CMAX : tid - 3 * CMAX;
    if (q == 3 || c < C) {
      const float t = (wave_tot[tid] + wave_tot[Q + tid]) + (wave_tot[2 * Q + tid] + wave_tot[3 * Q + tid]);
      dst[q == 3 ? 3 * C + c : q * C + c] = t;
    }
  }
}

// Slots lane, lane + 64, ... of a quantity (stride `q` floats between slots), added in that order with sixteen loads in
// flight at a time (one slot per trip to memory made a launch of 1024 slots sixteen trips long).
__device__ __forceinline__ float lane_slots_sum(const float* __restrict__ src, int slots, int q, int lane) {
  float s = 0.f;
  int sp = lane;
  for (; sp + 15 * 64 < slots; sp += 16 * 64) {
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = src[(int64_t)(sp + 64 * k) * q];
#pragma unroll
    for (int k = 0; k < 16; ++k) s += v[k];
  }
  for (; sp < slots; sp += 64) s += src[(int64_t)sp * q];
  return s;
}

// One 64-lane workgroup per quantity: lane l adds slots l, l + 64, ... and the lane totals meet in a fixed tree.
// stats: inter[N][C] | psum[N][C] | tsum[N][C] | ce_sum | normaliser
__global__ void __launch_bounds__(64) ce_dice_sum(const float* __restrict__ part, float* __restrict__ stats, int N, int C, int nsplit,
                                                  int unweighted, float count) {
  const int Q = 3 * C + 2;
  const int b = blockIdx.x, lane = threadIdx.x;
  float s = 0.f;
  int dst;
  if (b < N * 3 * C) {
    const int n = b / (3 * C), q = b - n * 3 * C;
    s = lane_slots_sum(part + (int64_t)n * nsplit * Q + q, nsplit, Q, lane);
    dst = (q / C) * N * C + n * C + q % C;
  } else {
    const int q = 3 * C + (b - N * 3 * C);  // ce_sum or normaliser, over all samples
    s = lane_slots_sum(part + q, N * nsplit, Q, lane);
    dst = b;
  }
  s = wave_sum_all(s);
  if (lane == 0) {
    if (b == N * 3 * C + 1 && unweighted) s = count;  // the normaliser of the unweighted mean is the voxel count
    stats[dst] = s;
  }
}

// The loss from the totals, by one wavefront: one lane per (sample, foreground class) pass; the Dice terms meet in the fixed tree.
__device__ __forceinline__ void loss_from_totals(const float* stats, float* __restrict__ loss, int N, int C, float eps) {
  const float* inter = stats;
  const float* psum = stats + N * C;
  const float* tsum = stats + 2 * N * C;
  // (asked for now: thread 0 needs them after the tree)
  const float ce_sum = stats[N * 3 * C], normaliser = stats[N * 3 * C + 1];
  float dice = 0.f;
  for (int i = threadIdx.x; i < N * C; i += 64) {
    const int c = i % C;
    if (c >= 1) {
      const float two_i = 2.f * inter[i];
      float sets = psum[i] + tsum[i];
      if (sets == 0.f) sets = two_i;
      dice += (two_i + eps) / (sets + eps);
    }
  }
  dice = wave_sum_all(dice);
  if (threadIdx.x == 0) {
    dice /= (float)(N * (C - 1));
    const float ce = ce_sum / fmaxf(normaliser, 1.1920929e-07f);
    loss[0] = ce + (1.f - dice);
  }
}

__global__ void __launch_bounds__(64) ce_dice_scalar(const float* __restrict__ stats, float* __restrict__ loss, int N, int C, float eps) {
  loss_from_totals(stats, loss, N, C, eps);
}

// Both of the above as one workgroup, for up to kTotalSamples samples and kTotalSlotsMax slots. A wavefront reads a slot's
// quantities side by side and takes every sixteenth slot, all of them in flight; the sums are those of ce_dice_sum, bit for
// bit. What bounds it is a launch and the trip of one CU: 128 slots of 35 quantities 2.9 us (the two launches 3.9 and 1.6 and the gap
// between them). With more slots, in rounds, 512 of 53 were level with the two and 1024 of 35 twice as slow.
constexpr int kTotal = 1024, kTotalWaves = kTotal / 64, kTotalSamples = 4, kTotalQ = 3 * 32 + 2, kTotalSlots = 16, kTotalSlotsMax = 256;
static_assert(kTotalSlots * kTotalWaves >= kTotalSlotsMax, "a wavefront's slots are read at once");
__global__ void __launch_bounds__(kTotal) ce_dice_total(const float* __restrict__ part, float* __restrict__ stats, float* __restrict__ loss,
                                                        int N, int C, int nsplit, int unweighted, float count, float eps) {
  __shared__ float wave_tot[kTotalWaves][kTotalQ];
  __shared__ float tot[kTotalSamples * 3 * 32 + 2];
  const int Q = 3 * C + 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int n = 0; n < N; ++n) {
    // the last two quantities run over the slots of all samples, beside the first sample's own
    for (int q = lane; q < (n == 0 ? Q : 3 * C); q += 64) {
      const bool wide = q >= 3 * C;
      const int slots = wide ? N * nsplit : nsplit;
      const float* src = part + (wide ? 0 : (int64_t)n * nsplit * Q) + q;
      float v[kTotalSlots];
#pragma unroll
      for (int k = 0; k < kTotalSlots; ++k) {
        const int at = wave + k * kTotalWaves;
        v[k] = src[(int64_t)(at < slots ? at : 0) * Q];
      }
#pragma unroll
      for (int k = 0; k < kTotalSlots; ++k) v[k] = wave + k * kTotalWaves < slots ? v[k] : 0.f;
      // slots 64 apart one after the other, then those 32 and 16 apart: the order of ce_dice_sum's lanes and of its tree
      float lane_sum[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) lane_sum[j] = ((v[j] + v[4 + j]) + v[8 + j]) + v[12 + j];
      wave_tot[wave][q] = (lane_sum[0] + lane_sum[2]) + (lane_sum[1] + lane_sum[3]);
    }
    __syncthreads();
    if (tid < (n == 0 ? Q : 3 * C)) {
      float v[kTotalWaves];
#pragma unroll
      for (int w = 0; w < kTotalWaves; ++w) v[w] = wave_tot[w][tid];
#pragma unroll
      for (int h = kTotalWaves / 2; h > 0; h >>= 1)
#pragma unroll
        for (int w = 0; w < h; ++w) v[w] += v[w + h];
      const int dst = tid < 3 * C ? (tid / C) * N * C + n * C + tid % C : N * 3 * C + tid - 3 * C;
      if (tid == 3 * C + 1 && unweighted) v[0] = count;  // the normaliser of the unweighted mean is the voxel count
      tot[dst] = v[0];
      stats[dst] = v[0];
    }
    __syncthreads();
  }
  if (wave == 0) loss_from_totals(tot, loss, N, C, eps);
}

// dlogits[v][j] = gl * ( w_y / normaliser * (p_j - [j == y])  +  p_j * (g_j - sum_c g_c p_c) ),
// g_c = -(1 / (N (C-1))) * d dice_c / d p_c = -(1 / (N (C-1))) * ([c == y] * 2 / den_c - (2 I_c + eps) / den_c^2), g_0 = 0.
template <typename T, int CMAX>
__global__ void __launch_bounds__(kBlock) ce_dice_backward(const T* __restrict__ logits, const int64_t* __restrict__ labels,
                                                           const float* __restrict__ cw, const float* __restrict__ stats,
                                                           const float* __restrict__ grad_loss, T* __restrict__ dlogits, int64_t S,
                                                           int N, int C, float eps, int64_t per_split, int vec) {
  extern __shared__ __align__(16) char smem_raw[];
  T* tile = reinterpret_cast<T*>(smem_raw);
  __shared__ float ca[CMAX], cb[CMAX];
  const int tid = threadIdx.x;
  const int n = blockIdx.y, split = blockIdx.x;
  const float gl = grad_loss[0];
  if (tid < CMAX) {
    float a = 0.f, b = 0.f;
    if (tid >= 1 && tid < C) {
      const float two_i = 2.f * stats[n * C + tid];
      float sets = stats[N * C + n * C + tid] + stats[2 * N * C + n * C + tid];
      if (sets == 0.f) sets = two_i;
      const float den = sets + eps, k = -gl / (float)(N * (C - 1));
      a = k * 2.f / den;
      b = k * (two_i + eps) / (den * den);
    }
    ca[tid] = a;
    cb[tid] = b;
  }
  const float ce_scale = gl / fmaxf(stats[N * 3 * C + 1], 1.1920929e-07f);
  const T* src = logits + (int64_t)n * S * C;
  T* dst = dlogits + (int64_t)n * S * C;
  const int64_t* lab = labels + (int64_t)n * S;
  const int64_t begin = (int64_t)split * per_split;
  int64_t end = begin + per_split;
  if (end > S) end = S;
  constexpr int VOX = kVoxels<T, CMAX>;
  for (int64_t v0 = begin; v0 < end; v0 += VOX * kBlock) {
    const int nv = (int)((end - v0) < VOX * kBlock ? (end - v0) : VOX * kBlock);
    int label[VOX];
    labels_in<VOX>(label, lab + v0, nv, C);
    __syncthreads();
    tile_in<T>(tile, src + v0 * C, nv * C, vec != 0);
    __syncthreads();
#pragma unroll 1
    for (int u = 0; u < VOX; ++u) {
      const int at = tid + u * kBlock;
      if (at >= nv) break;
      T* row = tile + at * C;
      float p[CMAX];
      float m = -INFINITY;
#pragma unroll
      for (int c = 0; c < CMAX; ++c) {
        p[c] = has_class<CMAX>(c, C) ? to_float(row[c]) : -INFINITY;
        m = fmaxf(m, p[c]);
      }
      float s = 0.f;
#pragma unroll
      for (int c = 0; c < CMAX; ++c) {
        p[c] = has_class<CMAX>(c, C) ? expf(p[c] - m) : 0.f;
        s += p[c];
      }
      const float inv = 1.f / s;
      int y = label[0];
#pragma unroll
      for (int k = 1; k < VOX; ++k) y = u == k ? label[k] : y;
      float g[CMAX], dot = 0.f, wy = 0.f;
#pragma unroll
      for (int c = 0; c < CMAX; ++c) {
        p[c] *= inv;
        const bool hit = c == y;
        g[c] = (hit ? ca[c] : 0.f) - cb[c];
        dot = fmaf(g[c], p[c], dot);
        if (hit) wy = cw != nullptr ? cw[c] : 1.f;
      }
      const float cs = ce_scale * wy;
#pragma unroll
      for (int c = 0; c < CMAX; ++c) {
        if (has_class<CMAX>(c, C)) {
#pragma clang fp contract(off)  // p_j - [j == y] of the rounded p_j, for a class that needs no question as for one that does
          const bool hit = c == y;
          const float d = fmaf(p[c], g[c] - dot, cs * (p[c] - (hit ? 1.f : 0.f)));
          row[c] = elem<T>::from_float(d);
        }
      }
    }
    __syncthreads();
    tile_out<T>(dst + v0 * C, tile, nv * C, vec != 0);
  }
}

struct LossPlan { int nsplit; int64_t per_split; };

LossPlan loss_plan(const sfh_loss_desc& p) {
  LossPlan pl;
  int64_t want = cdiv(4 * kComputeUnits, p.n);
  const int64_t tiles = cdiv(p.spatial, kBlock);
  if (want > tiles) want = tiles;
  if (want < 1) want = 1;
  pl.per_split = cdiv(tiles, want) * kBlock;
  pl.nsplit = (int)cdiv(p.spatial, pl.per_split);
  return pl;
}

// Every tile starts kBlock * classes elements after the previous one and every sample spatial * classes elements after
// the previous one: all tiles start on 16-byte boundaries when those two strides and the base pointers do.
template <typename T>
int tiles_on_16_bytes(const sfh_loss_desc& p, const void* a, const void* b) {
  const bool ok = (reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(b) & 15) == 0 &&
                  ((size_t)kBlock * p.classes * sizeof(T)) % 16 == 0 && (p.n == 1 || ((size_t)p.spatial * p.classes * sizeof(T)) % 16 == 0);
  return ok ? 1 : 0;
}

template <typename T, int CMAX>
int fwd_typed(const sfh_loss_desc& p, const void* logits, const int64_t* labels, const float* cw, float* loss, float* stats,
              float* ws, hipStream_t st) {
  const LossPlan pl = loss_plan(p);
  size_t lds = (size_t)kVoxels<T, CMAX> * kBlock * p.classes * sizeof(T);
  if (lds < 4 * (3 * CMAX + 2) * sizeof(float)) lds = 4 * (3 * CMAX + 2) * sizeof(float);  // the fold at the end reuses the tile
  hipLaunchKernelGGL((ce_dice_partial<T, CMAX>), dim3(pl.nsplit, p.n), dim3(kBlock), lds, st, (const T*)logits, labels, cw, ws,
                     p.spatial, p.classes, pl.nsplit, pl.per_split, tiles_on_16_bytes<T>(p, logits, nullptr));
  if (int rc = check_launch("ce_dice_partial")) return rc;
  if (p.n <= kTotalSamples && (int64_t)p.n * pl.nsplit <= kTotalSlotsMax) {
    hipLaunchKernelGGL(ce_dice_total, dim3(1), dim3(kTotal), 0, st, ws, stats, loss, p.n, p.classes, pl.nsplit, cw == nullptr ? 1 : 0,
                       (float)p.n * (float)p.spatial, p.eps);
    return check_launch("ce_dice_total");
  }
  hipLaunchKernelGGL(ce_dice_sum, dim3(p.n * 3 * p.classes + 2), dim3(64), 0, st, ws, stats, p.n, p.classes, pl.nsplit,
                     cw == nullptr ? 1 : 0, (float)p.n * (float)p.spatial);
  if (int rc = check_launch("ce_dice_sum")) return rc;
  hipLaunchKernelGGL(ce_dice_scalar, dim3(1), dim3(64), 0, st, stats, loss, p.n, p.classes, p.eps);
  return check_launch("ce_dice_scalar");
}

template <typename T, int CMAX>
int bwd_typed(const sfh_loss_desc& p, const void* logits, const int64_t* labels, const float* cw, const float* stats,
              const float* grad_loss, void* dlogits, hipStream_t st) {
  const LossPlan pl = loss_plan(p);
  const size_t lds = (size_t)kVoxels<T, CMAX> * kBlock * p.classes * sizeof(T);
  hipLaunchKernelGGL((ce_dice_backward<T, CMAX>), dim3(pl.nsplit, p.n), dim3(kBlock), lds, st, (const T*)logits, labels, cw, stats,
                     grad_loss, (T*)dlogits, p.spatial, p.n, p.classes, p.eps, pl.per_split, tiles_on_16_bytes<T>(p, logits, dlogits));
  return check_launch("ce_dice_backward");
}

}  // namespace

bool loss_supported(const sfh_loss_desc& p) {
  return p.n >= 1 && p.classes >= 2 && p.classes <= 32 && p.spatial >= 1 && (int64_t)p.n * cdiv(p.spatial, kBlock) < 0x7fffffffLL;
}

size_t loss_workspace_bytes(const sfh_loss_desc& p) {
  return (size_t)p.n * loss_plan(p).nsplit * (3 * p.classes + 2) * sizeof(float);
}

// Class counts in steps of two up to 12: a voxel's arithmetic is per class slot, so 6 classes in 12 slots cost as much as 12.
#define SFH_LOSS_CLASSES(cmax, fn, ...)                         \
  if (p.classes <= cmax) {                                      \
    if (dtype == SFH_BF16) return fn<bf16_t, cmax>(__VA_ARGS__); \
    if (dtype == SFH_FP16) return fn<fp16_t, cmax>(__VA_ARGS__); \
    return fn<float, cmax>(__VA_ARGS__);                        \
  }
#define SFH_LOSS_DISPATCH(fn, ...)        \
  SFH_LOSS_CLASSES(4, fn, __VA_ARGS__)    \
  SFH_LOSS_CLASSES(6, fn, __VA_ARGS__)    \
  SFH_LOSS_CLASSES(8, fn, __VA_ARGS__)    \
  SFH_LOSS_CLASSES(10, fn, __VA_ARGS__)   \
  SFH_LOSS_CLASSES(12, fn, __VA_ARGS__)   \
  SFH_LOSS_CLASSES(16, fn, __VA_ARGS__)   \
  SFH_LOSS_CLASSES(32, fn, __VA_ARGS__)   \
  return fail(SFH_ERR_UNSUPPORTED, "ce_dice: %d classes", p.classes);

int loss_forward(const sfh_loss_desc& p, int dtype, const void* logits, const int64_t* labels, const float* cw, float* loss,
                 float* stats, void* ws, hipStream_t st) {
  SFH_LOSS_DISPATCH(fwd_typed, p, logits, labels, cw, loss, stats, (float*)ws, st)
}

int loss_backward(const sfh_loss_desc& p, int dtype, const void* logits, const int64_t* labels, const float* cw, const float* stats,
                  const float* grad_loss, void* dlogits, hipStream_t st) {
  SFH_LOSS_DISPATCH(bwd_typed, p, logits, labels, cw, stats, grad_loss, dlogits, st)
}

}  // namespace sfh
