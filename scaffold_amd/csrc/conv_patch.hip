// MFMA kernels for 2x2x2, stride-2, unpadded convolutions between a BIG and a SMALL volume: the U-Net's
// transposed up-convolution (triton_conv3d/transposed.py:135-319), its data gradient (a stride-2
// convolution, transposed.py:1073) and its weight gradient (transposed.py:1113).
//
// Windows do not overlap, so there is no halo and nothing to reuse between neighbouring voxels: the
// three kernels are HBM-bound GEMMs with M = small voxels. The gather and the scatter keep their weights
// in registers and turn voxel tiles through LDS; their general forms take both MFMA operands straight from
// global memory (a lane's fragment is 8 consecutive channels of one voxel, one 16-byte load; the weight is
// pre-packed in fragment order and stays in L1/L2). The weight gradient
// contracts over voxels, so both operands must be transposed: tiles are staged in LDS in their natural
// [voxel][channel] layout and read with ds_read_b64_tr_b16, which hands each lane four consecutive
// voxels of one channel.
#include "conv_patch.hpp"
#include <type_traits>
#include "mma.hpp"
#include "reduce.hpp"

namespace sfh {
namespace {

constexpr int kTaps = 8;

struct Voxel { int nn, d, h, w; };

__host__ __device__ __forceinline__ Voxel decode_small(const PatchArgs& a, int64_t v) {
  Voxel r;
  if (v <= 0x7fffffffLL) {  // 32-bit arithmetic when it fits
    uint32_t t = (uint32_t)v;
    r.w = (int)(t % (uint32_t)a.sw); t /= (uint32_t)a.sw;
    r.h = (int)(t % (uint32_t)a.sh); t /= (uint32_t)a.sh;
    r.d = (int)(t % (uint32_t)a.sd);
    r.nn = (int)(t / (uint32_t)a.sd);
    return r;
  }
  r.w = (int)(v % a.sw);
  int64_t t = v / a.sw;
  r.h = (int)(t % a.sh);
  t /= a.sh;
  r.d = (int)(t % a.sd);
  r.nn = (int)(t / a.sd);
  return r;
}

__host__ __device__ __forceinline__ int64_t big_index(const PatchArgs& a, const Voxel& v, int tap) {
  return (((int64_t)v.nn * a.bd + 2 * v.d + (tap >> 2)) * a.bh + 2 * v.h + ((tap >> 1) & 1)) * a.bw + 2 * v.w + (tap & 1);
}

// A voxel that moves on by the same number of voxels every time (decoding it anew costs three divisions: at two wavefronts a
// SIMD some 1200 cycles a round, which bounded the weight gradient). `at`: its patch's first big voxel.
struct VoxelStep { int w, h, d; int64_t at, carry_w, carry_h, carry_d; };
VoxelStep voxel_step(const PatchArgs& a, int64_t voxels) {
  const Voxel s = decode_small(a, voxels);
  VoxelStep r;
  r.w = s.w; r.h = s.h; r.d = s.d;
  r.at = big_index(a, s, 0);
  r.carry_w = 2 * ((int64_t)a.bw - a.sw);
  r.carry_h = 2 * ((int64_t)a.bh - a.sh) * a.bw;
  r.carry_d = ((int64_t)a.bd - 2 * a.sd) * a.bh * a.bw;
  return r;
}
struct VoxelWalk {
  int w, h, d;
  int64_t at;
  __device__ __forceinline__ void start(const PatchArgs& a, int64_t v) {
    const Voxel s = decode_small(a, v);
    w = s.w; h = s.h; d = s.d;
    at = big_index(a, s, 0);
  }
  __device__ __forceinline__ void advance(const PatchArgs& a, const VoxelStep& s) {
    at += s.at;
    w += s.w; h += s.h; d += s.d;
    if (w >= a.sw) { w -= a.sw; ++h; at += s.carry_w; }
    if (h >= a.sh) { h -= a.sh; ++d; at += s.carry_h; }
    if (d >= a.sd) { d -= a.sd; at += s.carry_d; }
  }
};

// ---- gather: stride-2 convolution --------------------------------------------------------------
// The kept form. A wavefront owns one block of 32 small channels and KEEPS its weights in registers -- all eight taps of cbig
// channels, those of a depth tap (KH = 2) or of a row of the patch (KH = 4) -- while its workgroup walks tiles of 32 * VS
// voxels: the tile's patches are fetched in whole rows (2 * cbig contiguous channels) one tile ahead, laid into LDS as
// [8-channel piece][voxel] and read from there by the wavefronts of every block, so the big tensor is read once per NBW blocks.
// The KH parts of a block meet in LDS in their order. Like the scatter's general form, this one's was bound by the address path.
// grid = groups of tiles (in eights, one per XCD) x groups of NBW blocks.
// PACKED: `w` is in fragment order; else dense [csmall][tap][cbig], laid out block by block like a tile.
template <int CB>
struct GatherKept {
  static constexpr int KH = CB <= 64 ? 1 : CB / 64;  // parts of the reduction
  static constexpr int NBW = CB == 32 || CB == 256 ? 2 : 4;  // blocks of 32 small channels per workgroup
  static constexpr int VS = CB == 32 ? 2 : 1;        // 32-voxel parts of a tile
  static constexpr int UNITS = NBW * VS, THREADS = 64 * KH * UNITS;
  static constexpr int V = 32 * VS;
  static constexpr int ROW = CB / 4;                 // 16-byte pieces of the two big voxels along W
  static constexpr int PIECES = 4 * ROW;
  static constexpr int KSW = CB / 2 / KH;            // k-steps of a wavefront
  static constexpr int PLANE = V * 16 + (ROW >= 16 ? 16 : 32);  // writes of a voxel's pieces fall into different banks
  static constexpr int VOX = ROW * V / THREADS;      // voxels a thread fetches for, four rows each
  static constexpr int WPER = PIECES * 32 / THREADS; // pieces of a weight block a thread moves
  static constexpr int BUFS = KH == 4 ? 1 : 2;       // tiles in LDS (the barrier in front of the parts' sum also frees the one)
};

template <typename T, int CB, bool PACKED>
__global__ void __launch_bounds__(GatherKept<CB>::THREADS, 2)
patch_gather_kept_kernel(PatchArgs a, const T* __restrict__ big, const T* __restrict__ w, const T* __restrict__ bias,
                         T* __restrict__ small, int64_t total, int groups) {
  using C = GatherKept<CB>;
  __shared__ __attribute__((aligned(16))) char lds[C::BUFS][C::PIECES * C::PLANE];
  __shared__ float s_part[C::KH == 1 ? 1 : (C::KH - 1) * C::UNITS * 16 * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kg = lane >> 5;
  const int ncol = a.csmall / (32 * C::NBW);
  const int slot = blockIdx.x / kXcds;
  const int group = slot / ncol * kXcds + blockIdx.x % kXcds;
  if (group >= groups) return;
  const int kpart = wave / C::UNITS, unit = wave % C::UNITS;  // unit: (voxel part, block)
  const int part = unit / C::NBW;
  const int blk0 = slot % ncol * C::NBW, blk = blk0 + unit % C::NBW;
  const int64_t tiles = (total + C::V - 1) / C::V;
  uint4 next[C::VOX][4];
  auto fetch = [&](int64_t tile) {
#pragma unroll
    for (int i = 0; i < C::VOX; ++i) {
      const int64_t v = tile * C::V + (i * C::THREADS + tid) / C::ROW;
      const T* src = big + big_index(a, decode_small(a, v < total ? v : total - 1), 0) * CB + tid % C::ROW * 8;
#pragma unroll
      for (int r = 0; r < 4; ++r) next[i][r] = load16(src + ((int64_t)(r >> 1) * a.bh + (r & 1)) * a.bw * CB);
    }
  };
  fetch(group);
  uint4 wf[C::KSW];
  if constexpr (PACKED) {
#pragma unroll
    for (int i = 0; i < C::KSW; ++i) {
      const int k = kpart * C::KSW + i, tap = k / (CB / 16), c16 = k % (CB / 16);
      wf[i] = load16(w + (((((int64_t)blk * (CB / 32) + (c16 >> 1)) * kTaps + tap) * 2 + (c16 & 1)) * 64 + lane) * 8);
    }
  } else {
    uint4 raw[C::WPER];
    auto fetch_block = [&](int b) {
#pragma unroll
      for (int i = 0; i < C::WPER; ++i) raw[i] = load16(w + ((int64_t)(blk0 + b) * 32 * C::PIECES + i * C::THREADS + tid) * 8);
    };
    fetch_block(0);
#pragma unroll
    for (int b = 0; b < C::NBW; ++b) {
      char* buf = lds[b % C::BUFS];
#pragma unroll
      for (int i = 0; i < C::WPER; ++i) {
        const int q = i * C::THREADS + tid;
        *reinterpret_cast<uint4*>(buf + q % C::PIECES * C::PLANE + q / C::PIECES * 16) = raw[i];
      }
      if (b + 1 < C::NBW) fetch_block(b + 1);
      __syncthreads();
      if (unit % C::NBW == b) {
#pragma unroll
        for (int i = 0; i < C::KSW; ++i)
          wf[i] = *reinterpret_cast<const uint4*>(buf + (2 * (kpart * C::KSW + i) + kg) * C::PLANE + (lane & 31) * 16);
      }
      if constexpr (C::BUFS == 1) __syncthreads();
    }
  }
  // with 32 fragments of weights a lane has no registers left for its bias values: they wait in LDS (held, they spilled 8)
  constexpr bool kBiasInLds = C::KH == 4;
  __shared__ float s_bias[kBiasInLds ? 32 * C::NBW : 1];
  float add[16];
  if constexpr (kBiasInLds) {
    if (tid < 32 * C::NBW) s_bias[tid] = bias != nullptr ? to_float(bias[blk0 * 32 + tid]) : 0.f;
  } else {
    load_block_bias<T>(bias, blk * 32, kg, add);
  }
  int phase = 0;
  for (int64_t t = group; t < tiles; t += groups, phase ^= C::BUFS - 1) {
    char* tile = lds[phase];
#pragma unroll
    for (int i = 0; i < C::VOX; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<uint4*>(tile + (r * C::ROW + tid % C::ROW) * C::PLANE + (i * C::THREADS + tid) / C::ROW * 16) = next[i][r];
    __syncthreads();  // with two buffers the other one was read before the barrier of the tile behind it
    fetch(t + groups < tiles ? t + groups : t);
    f32x16_t acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int i = 0; i < C::KSW; ++i) {
      const int k = kpart * C::KSW + i;
      acc = Mma32<T>::run(wf[i], *reinterpret_cast<const uint4*>(tile + (2 * k + kg) * C::PLANE + (part * 32 + (lane & 31)) * 16), acc);
    }
    if constexpr (C::KH > 1) {
      if (kpart > 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s_part[(((kpart - 1) * C::UNITS + unit) * 16 + r) * 64 + lane] = acc[r];
      }
      __syncthreads();
      if (kpart == 0) {
#pragma unroll
        for (int p = 0; p < C::KH - 1; ++p)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[r] += s_part[((p * C::UNITS + unit) * 16 + r) * 64 + lane];
      }
    }
    if (kpart == 0) {
      const int64_t v = t * C::V + part * 32 + (lane & 31);
      const bool valid = v < total;
      if constexpr (kBiasInLds) {
#pragma unroll
        for (int r = 0; r < 16; ++r) add[r] = s_bias[unit % C::NBW * 32 + 8 * (r / 4) + 4 * kg + r % 4];
      }
      store_block_plus<T>(acc, small + (valid ? v : total - 1) * a.csmall + blk * 32, add, kg, valid);
    }
  }
}

// The general form. A wavefront owns 32 small voxels x NB blocks of 32 produced channels. grid = (voxel tiles of 128, groups of NB blocks).
template <typename T, int NB>
__global__ void __launch_bounds__(256) patch_gather_kernel(PatchArgs a, const T* __restrict__ big, const T* __restrict__ packed,
                                                           const T* __restrict__ bias, T* __restrict__ small, int64_t total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kg = lane >> 5;
  const int64_t v = (int64_t)blockIdx.x * 128 + wave * 32 + (lane & 31);
  const bool valid = v < total;
  const Voxel vx = decode_small(a, valid ? v : total - 1);
  const int nchunks = a.cbig / 32;
  const int blk0 = blockIdx.y * NB;
  f32x16_t acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
  for (int tap = 0; tap < kTaps; ++tap) {
    const T* src = big + big_index(a, vx, tap) * a.cbig + kg * 8;
    for (int cc = 0; cc < nchunks; ++cc) {
      uint4 bf[2], wf[2][NB];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        bf[ks] = load16(src + cc * 32 + ks * 16);
#pragma unroll
        for (int b = 0; b < NB; ++b)
          wf[ks][b] = load16(packed + (((((int64_t)(blk0 + b) * nchunks + cc) * kTaps + tap) * 2 + ks) * 64 + lane) * 8);
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = Mma32<T>::run(wf[ks][b], bf[ks], acc[b]);
    }
  }
  const int64_t vs = valid ? v : total - 1;
#pragma unroll
  for (int b = 0; b < NB; ++b) store_block<T>(acc[b], small + vs * a.csmall + (blk0 + b) * 32, bias, (blk0 + b) * 32, kg, valid);
}

// The same for launches that would leave most of the chip idle (the U-Net's deepest levels: a few hundred voxels, hundreds
// of channels, where one wavefront's chain of dependent loads sets the time). A workgroup owns 32 small voxels x one block of
// 32 produced channels; its four wavefronts take two taps each, keep the loads of four chunks in flight, and their partial
// blocks are added in wavefront order through LDS. grid = (voxel tiles of 32, csmall / 32).
template <typename T>
__global__ void __launch_bounds__(256) patch_gather_deep_kernel(PatchArgs a, const T* __restrict__ big, const T* __restrict__ packed,
                                                                const T* __restrict__ bias, T* __restrict__ small, int64_t total) {
  __shared__ float part[3][16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kg = lane >> 5;
  const int64_t v = (int64_t)blockIdx.x * 32 + (lane & 31);
  const bool valid = v < total;
  const int64_t vs = valid ? v : total - 1;
  const Voxel vx = decode_small(a, vs);
  const int nchunks = a.cbig / 32;
  const int blk = blockIdx.y;
  f32x16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  for (int tap = 2 * wave; tap < 2 * wave + 2; ++tap) {
    const T* src = big + big_index(a, vx, tap) * a.cbig + kg * 8;
    const T* wsrc = packed + ((((int64_t)blk * nchunks) * kTaps + tap) * 2 * 64 + lane) * 8;
    const int64_t wstep = (int64_t)kTaps * 2 * 64 * 8;  // elements between the fragments of consecutive chunks
    // U chunks per step: all their loads are issued before the first MFMA
    auto step = [&](int cc, auto width) {
      constexpr int U = decltype(width)::value;
      uint4 bf[U][2], wf[U][2];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          bf[u][ks] = load16(src + (cc + u) * 32 + ks * 16);
          wf[u][ks] = load16(wsrc + (cc + u) * wstep + ks * 64 * 8);
        }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) acc = Mma32<T>::run(wf[u][ks], bf[u][ks], acc);
    };
    int cc = 0;
    for (; cc + 4 <= nchunks; cc += 4) step(cc, std::integral_constant<int, 4>{});
    for (; cc < nchunks; ++cc) step(cc, std::integral_constant<int, 1>{});
  }
  if (wave > 0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave - 1][r][lane] = acc[r];
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] += part[w][r][lane];
    store_block<T>(acc, small + vs * a.csmall + blk * 32, bias, blk * 32, kg, valid);
  }
}

// ---- scatter: transposed convolution -----------------------------------------------------------
// Zeroes the two faces of `face_pieces` 16-byte pieces around a depth slab's interior `big` of `big_elems` elements,
// spread over the `nthreads` threads of the launch.
template <typename T>
__device__ __forceinline__ void zero_faces(T* big, int64_t face_pieces, int64_t big_elems, int64_t me, int64_t nthreads) {
  uint4* lo = reinterpret_cast<uint4*>(big) - face_pieces;
  uint4* hi = reinterpret_cast<uint4*>(big + big_elems);
  for (int64_t p = me; p < face_pieces; p += nthreads) {
    lo[p] = make_uint4(0, 0, 0, 0);
    hi[p] = make_uint4(0, 0, 0, 0);
  }
}

// Voxels of the big volume that are under no tap, per sample: planes, rows and columns at the end of its extents.
struct Tails { int64_t planes, rows, columns; };
__host__ __device__ __forceinline__ Tails tails_of(const PatchArgs& a) {
  return Tails{(int64_t)(a.bd - 2 * a.sd) * a.bh * a.bw, (int64_t)2 * a.sd * (a.bh - 2 * a.sh) * a.bw,
               (int64_t)4 * a.sd * a.sh * (a.bw - 2 * a.sw)};
}
// Zeroes them (the padding of an upsampled tensor to an odd level's extents), spread over the launch's threads.  The padding alone was
// a fill and a copy of the whole tensor: 32 channels of 43x124x47 17.6 us, and 8.6 for the copy its backward made.
template <typename T>
__device__ __forceinline__ void zero_tails(const PatchArgs& a, T* big, uint32_t me, uint32_t nthreads) {
  const Tails t = tails_of(a);
  const uint32_t planes = (uint32_t)t.planes, rows = (uint32_t)t.rows, all = (uint32_t)(t.planes + t.rows + t.columns);
  const uint32_t per = (uint32_t)a.cbig / 8, pieces = all * per * (uint32_t)a.n;  // (below 2^31: launch_scatter)
  const uint32_t tail_h = (uint32_t)(a.bh - 2 * a.sh) * a.bw, tail_w = (uint32_t)(a.bw - 2 * a.sw);
  for (uint32_t p = me; p < pieces; p += nthreads) {
    const uint32_t v = p / per;
    uint32_t r = v % all;
    int64_t at = (int64_t)(v / all) * a.bd * a.bh * a.bw;
    if (r < planes) {
      at += (int64_t)2 * a.sd * a.bh * a.bw + r;
    } else if (r - planes < rows) {
      r -= planes;
      at += ((int64_t)(r / tail_h) * a.bh + 2 * a.sh) * a.bw + r % tail_h;
    } else {
      r -= planes + rows;
      const uint32_t line = r / tail_w, d = line / (2 * a.sh), h = line % (2 * a.sh);
      at += ((int64_t)d * a.bh + h) * a.bw + 2 * a.sw + r % tail_w;
    }
    reinterpret_cast<uint4*>(big + at * a.cbig)[p % per] = make_uint4(0, 0, 0, 0);
  }
}

// Columns (tap, block of 32 big channels) of the 2 x 2 x 2 patch are numbered as they lie in memory: blocks, then the taps.
// A workgroup owns 4 * C neighbouring columns, a wavefront C of them, whose weights it KEEPS in registers (csmall = 16 * KS
// channels: 4 * C * KS registers a lane) while the workgroup walks tiles of 32 voxels: a tile is fetched in whole lines one
// tile ahead, laid into LDS as [8-channel piece][voxel] and read from there by all four wavefronts; the results leave in
// runs of 64 * C bytes per voxel (whole lines for C = 2).
// What bounds the general form is the CU's address path: a fragment straight from memory is 32 lines of 32 bytes each,
// and a wavefront of it fetched its weights and its tile for two taps only.
// grid = groups of tiles (in eights, one per XCD) x (cbig / 16 / C) groups of columns, those of a tile on one XCD.
// PACKED: `w` is in fragment order; else dense [csmall][tap][cbig], turned through LDS once per wavefront.
template <typename T, int KS, int C, bool PACKED>
__global__ void __launch_bounds__(256, 2) patch_scatter_kernel(PatchArgs a, const T* __restrict__ small, const T* __restrict__ w,
                                                               const T* __restrict__ bias, T* __restrict__ big, int64_t total,
                                                               int groups, int64_t face_pieces, int64_t big_elems) {
  constexpr int PIECES = 2 * KS;                        // 16-byte pieces of a voxel
  constexpr int PLANE = 512 + (PIECES >= 16 ? 16 : 32);  // bytes; writes of a voxel's pieces fall into different banks
  constexpr int PER = PIECES * 32 / 256;                // pieces a thread moves per tile
  constexpr int kTurn = 4;                              // k-steps of a weight column turned at a time
  constexpr int kLds = 2 * PIECES * PLANE > 4 * kTurn * 1024 || PACKED ? 2 * PIECES * PLANE : 4 * kTurn * 1024;
  constexpr int kOutRow = 64 * C + 16;                  // LDS bytes of a voxel's run of 64 * C bytes
  constexpr int kLanes = 4 * C;                         // lanes that store one such run
  __shared__ __attribute__((aligned(16))) char lds[kLds];
  __shared__ __attribute__((aligned(16))) char s_out[4][32 * kOutRow];
  if (face_pieces > 0)
    zero_faces(big, face_pieces, big_elems, (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256);
  if (a.bd != 2 * a.sd || a.bh != 2 * a.sh || a.bw != 2 * a.sw) zero_tails(a, big, blockIdx.x * 256 + threadIdx.x, gridDim.x * 256);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kg = lane >> 5;
  const int nblk = a.cbig / 32;
  const int ncol = 2 * nblk / C;
  const int slot = blockIdx.x / kXcds;
  const int group = slot / ncol * kXcds + blockIdx.x % kXcds;
  if (group >= groups) return;
  const int c0 = slot % ncol * 4 * C + C * wave;  // this wavefront's first column
  const int64_t tiles = (total + 31) / 32, pieces = total * PIECES;
  char* out = s_out[wave];
  uint4 next[PER];
  auto fetch = [&](int64_t tile) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      int64_t q = tile * (32 * PIECES) + i * 256 + tid;
      next[i] = load16(small + (q < pieces ? q : pieces - 1) * 8);
    }
  };
  fetch(group);
  int blk[C];
  uint4 wf[C][KS];
  float add[C][16];
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int tap = (c0 + j) / nblk;
    blk[j] = (c0 + j) % nblk;
    if constexpr (PACKED) {
#pragma unroll
      for (int k = 0; k < KS; ++k)
        wf[j][k] = load16(w + (((((int64_t)blk[j] * (KS / 2) + (k >> 1)) * kTaps + tap) * 2 + (k & 1)) * 64 + lane) * 8);
    } else {
      T* mine = reinterpret_cast<T*>(lds) + wave * (kTurn * 512);
      const T* src = w + ((int64_t)(lane >> 2) * kTaps + tap) * a.cbig + blk[j] * 32 + (lane & 3) * 8;
#pragma unroll
      for (int k0 = 0; k0 < KS; k0 += kTurn) {
        uint4 raw[kTurn];
#pragma unroll
        for (int k = 0; k < kTurn; ++k) raw[k] = load16(src + (int64_t)(k0 + k) * 16 * kTaps * a.cbig);
        __syncthreads();  // the previous k-steps have been read
#pragma unroll
        for (int k = 0; k < kTurn; ++k) *reinterpret_cast<uint4*>(mine + k * 512 + lane * 8) = raw[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kTurn; ++k) wf[j][k0 + k] = tr_fragment<T>(mine + k * 512, 32, lane);
      }
    }
    load_block_bias<T>(bias, blk[j] * 32, kg, add[j]);
  }
  if constexpr (!PACKED) __syncthreads();
  const int run0 = c0 % (2 * nblk) * 32;  // from the first of the two big voxels along W
  int phase = 0;
  for (int64_t t = group; t < tiles; t += groups, phase ^= 1) {
    char* tile = lds + phase * (PIECES * PLANE);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int q = i * 256 + tid;
      *reinterpret_cast<uint4*>(tile + (q % PIECES) * PLANE + (q / PIECES) * 16) = next[i];
    }
    __syncthreads();  // the other half was read before the barrier of the tile behind it
    fetch(t + groups < tiles ? t + groups : t);
    f32x16_t acc[C];
#pragma unroll
    for (int j = 0; j < C; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const uint4 f = *reinterpret_cast<const uint4*>(tile + (2 * k + kg) * PLANE + (lane & 31) * 16);
#pragma unroll
      for (int j = 0; j < C; ++j) acc[j] = Mma32<T>::run(wf[j][k], f, acc[j]);
    }
    // the columns of a voxel are contiguous: turned through LDS so that neighbouring lanes store one run
#pragma unroll
    for (int j = 0; j < C; ++j) {
      uint32_t run[4][2];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        run[g][0] = Mma32<T>::pack2(acc[j][4 * g] + add[j][4 * g], acc[j][4 * g + 1] + add[j][4 * g + 1]);
        run[g][1] = Mma32<T>::pack2(acc[j][4 * g + 2] + add[j][4 * g + 2], acc[j][4 * g + 3] + add[j][4 * g + 3]);
      }
      uint4 piece[2];
      trade_channel_runs(run, piece);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *reinterpret_cast<uint4*>(out + (lane & 31) * kOutRow + j * 64 + h * 32 + kg * 16) = piece[h];
    }
    const int64_t v = t * 32 + (lane & 31);
    const Voxel vx = decode_small(a, v < total ? v : total - 1);
    const int at = (int)big_index(a, vx, c0 / nblk & 6);
    const int left = (int)(total - t * 32 < 32 ? total - t * 32 : 32);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < kLanes / 2; ++i) {
      const int row = (i * 64 + lane) / kLanes;
      const uint4 piece = *reinterpret_cast<const uint4*>(out + row * kOutRow + (lane % kLanes) * 16);
      const int64_t vox = __shfl(at, row);
      if (row < left) *reinterpret_cast<uint4*>(big + vox * a.cbig + run0 + (lane % kLanes) * 8) = piece;
    }
  }
}

// The general form, for reduction widths whose weights do not fit in registers and for the smallest volumes.
// A wavefront owns 32 small voxels x one block of 32 big channels x TS of the 8 taps.
// grid = (voxel tiles of 128, cbig / 32, 8 / TS). TS = 8 reads the small tensor once; TS = 1 and 2 are for launches that
// would otherwise leave most of the chip idle or give a CU a single long chain of dependent loads (the deeper levels):
// more workgroups, each with a shorter chain, and the loads of several k-steps in flight per lane.
// `face_pieces` > 0: `big` is the interior of a depth slab whose two faces of that many 16-byte pieces (in front of it and
// behind its `big_elems` elements) the launch zeroes as well, spread over all its threads.
template <typename T, int TS>
__global__ void __launch_bounds__(256) patch_scatter_any_kernel(PatchArgs a, const T* __restrict__ small, const T* __restrict__ packed,
                                                            const T* __restrict__ bias, T* __restrict__ big, int64_t total,
                                                            int64_t face_pieces, int64_t big_elems) {
  if (face_pieces > 0) {
    const int64_t nthreads = (int64_t)gridDim.x * gridDim.y * gridDim.z * 256;
    zero_faces(big, face_pieces, big_elems, (((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * 256 + threadIdx.x,
               nthreads);
  }
  if (a.bd != 2 * a.sd || a.bh != 2 * a.sh || a.bw != 2 * a.sw)
    zero_tails(a, big, ((blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * 256 + threadIdx.x,
               gridDim.x * gridDim.y * gridDim.z * 256);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kg = lane >> 5;
  const int64_t v = (int64_t)blockIdx.x * 128 + wave * 32 + (lane & 31);
  const bool valid = v < total;
  const int64_t vc = valid ? v : total - 1;
  const int nchunks = a.csmall / 32;
  const int blk = blockIdx.y;
  const int tap0 = blockIdx.z * TS;
  f32x16_t acc[TS];
#pragma unroll
  for (int t = 0; t < TS; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
  const T* src = small + vc * a.csmall + kg * 8;
  // U half-chunks (k-steps of 16 channels) per step: all their loads are issued before the first MFMA
  auto step = [&](int k, auto width) {
    constexpr int U = decltype(width)::value;
    uint4 sf[U], wf[U][TS];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int cc = (k + u) >> 1, ks = (k + u) & 1;
      sf[u] = load16(src + cc * 32 + ks * 16);
#pragma unroll
      for (int t = 0; t < TS; ++t)
        wf[u][t] = load16(packed + (((((int64_t)blk * nchunks + cc) * kTaps + tap0 + t) * 2 + ks) * 64 + lane) * 8);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < TS; ++t) acc[t] = Mma32<T>::run(wf[u][t], sf[u], acc[t]);
  };
  int k = 0;
  if constexpr (TS == 1)
    for (; k + 8 <= 2 * nchunks; k += 8) step(k, std::integral_constant<int, 8>{});
  if constexpr (TS == 2)
    for (; k + 4 <= 2 * nchunks; k += 4) step(k, std::integral_constant<int, 4>{});
  if constexpr (TS == 4)
    for (; k + 2 <= 2 * nchunks; k += 2) step(k, std::integral_constant<int, 2>{});
  for (; k < 2 * nchunks; ++k) step(k, std::integral_constant<int, 1>{});
  const Voxel vx = decode_small(a, vc);
#pragma unroll
  for (int t = 0; t < TS; ++t)
    store_block<T>(acc[t], big + big_index(a, vx, tap0 + t) * a.cbig + blk * 32, bias, blk * 32, kg, valid);
}

// ---- reduce: weight gradient -------------------------------------------------------------------
constexpr int kVx = 32;             // voxels staged per round (two k-steps of 16)
constexpr int kSmallTile = 64;      // small channels per workgroup (two row blocks)

// A workgroup accumulates 64 small channels x 8 taps x 32 big channels over a range of voxels; its two halves of four wavefronts
// take the rounds of 32 voxels in turn (wavefront w of a half: taps 2w and 2w + 1 for both row blocks) and meet in LDS at the
// end, half 0 plus half 1, so that twice the wavefronts load without a second fp32 slice in memory. A round's products are summed by
// the matrix unit from zero and added to the running sums by the vector unit: half of the roundings of a chain through the matrix
// unit, and no second set of sums to hold -- one per parity of k-step spilled 6 registers in the form with BIAS. Relative error of the
// fp32 gradient against 64 bits, e-7, sums of the even and odd k-steps -> rounds: 64 -> 32 at 32x64x64 1.31 -> 1.29, 128 -> 64 at 32^3 1.17 ->
// 1.14, at 48x40x56 1.48 -> 1.37, 512 -> 256 at 12x10x14 0.90 -> 0.86. A round's operands are
// requested two rounds ahead and laid into the two phases of LDS in turn; a channel block's rows of 64 bytes
// lie dense, which neither the 16-byte writes nor the transposing reads meet a bank conflict on.
// grid: `by_xcd` ? eight-fold splits x tiles, the tiles of a range of voxels on one XCD (its lines come from HBM once; spread
// over the XCDs 128 -> 64 at 48x40x56 took 84 us instead of 38) : tiles x splits.
// BIAS: the workgroups of the first small-channel tile also add up the big tensor itself over the voxels -- the bias
// gradient of the transposed convolution whose weight gradient this is (every big voxel is a tap of exactly one small
// voxel there) -- as one more MFMA row block of ones, sixteen voxels at a time from zero and on in 64 bits (four additions a round;
// error over the sum of magnitudes with a chain of matrix steps and of slices -> with this and the slices' tree, e-9: 64 -> 32 at 64^3
// 0.10 -> 0.07, at 32x64x64 0.14 -> 0.10, 512 -> 256 at 12x10x14 0.66 -> 0.42): bias_part[split][cb], in a fixed order.
template <typename T, bool BIAS, int HALVES>
__global__ void __launch_bounds__(256 * HALVES, 2)
patch_reduce_kernel(PatchArgs a, const T* __restrict__ small, const T* __restrict__ big, float* __restrict__ part, int64_t total,
                    int64_t per_split, int splits, int by_xcd, VoxelStep step, float* __restrict__ bias_part) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int D = 2;                           // rounds requested ahead
  constexpr int kBlock = kVx * 32;               // elements of one [voxel][32 channels] block
  constexpr int kRound = (2 + kTaps) * kBlock;   // two blocks of the small tensor, one per tap of the big
  constexpr int kTurn = HALVES * kVx;            // voxels of a round of every half
  __shared__ __attribute__((aligned(16))) T lds[2][HALVES][kRound];
  const int nz = a.cbig / 32, tiles = a.csmall / kSmallTile * nz;
  const int slot = blockIdx.x / kXcds;
  const int split = by_xcd ? slot / tiles * kXcds + (int)(blockIdx.x % kXcds) : (int)blockIdx.x / tiles;
  const int tile = (by_xcd ? slot : (int)blockIdx.x) % tiles;
  if (split >= splits) return;
  const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  const int cs0 = tile / nz * kSmallTile, cb0 = tile % nz * 32;
  const int64_t begin = (int64_t)split * per_split;
  int64_t end = begin + per_split;
  if (end > total) end = total;
  f32x16_t acc[2][2], none;
#pragma unroll
  for (int r = 0; r < 16; ++r) none[r] = acc[0][0][r] = acc[0][1][r] = acc[1][0][r] = acc[1][1][r] = 0.f;
  double bsum = 0.;
  const bool sums_big = BIAS && cs0 == 0;
  const uint32_t one2 = sizeof(T) == 2 && std::is_same<T, bf16_t>::value ? 0x3f803f80u : 0x3c003c00u;  // two ones of T
  const uint4 ones = make_uint4(one2, one2, one2, one2);
  const int s_vox = tid >> 3, s_piece = tid & 7;          // small tile: 32 voxels x 8 pieces of 16 bytes
  const int b_vox = (tid >> 2) & 31, b_piece = tid & 3;   // big tiles: 4 taps (tid/128, +2, +4, +6) of one voxel
  const int b_tap0 = tid >> 7;
  const uint4 zero = make_uint4(0, 0, 0, 0);
  VoxelWalk walk;
  walk.start(a, begin + half * kVx + b_vox);
  int64_t tap_at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) tap_at[i] = big_index(a, Voxel{0, 0, 0, 0}, b_tap0 + 2 * i);
  struct Round { uint4 s, b[4]; } ahead[D];
  auto fetch = [&](Round& o, int64_t v0) {
    o.s = zero;
    if (v0 + s_vox < end) o.s = load16(small + (v0 + s_vox) * a.csmall + cs0 + s_piece * 8);
    if (v0 + b_vox < end) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o.b[i] = load16(big + (walk.at + tap_at[i]) * a.cbig + cb0 + b_piece * 8);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) o.b[i] = zero;
    }
    walk.advance(a, step);
  };
#pragma unroll
  for (int u = 0; u < D; ++u) fetch(ahead[u], begin + u * kTurn + half * kVx);
  for (int64_t v0 = begin; v0 < end; v0 += D * kTurn) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      const int64_t v = v0 + u * kTurn;
      if (u > 0 && v >= end) break;
      T* s_tile = lds[u & 1][half];
      T* b_tile = s_tile + 2 * kBlock;
      *reinterpret_cast<uint4*>(s_tile + (s_piece >> 2) * kBlock + s_vox * 32 + (s_piece & 3) * 8) = ahead[u].s;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<uint4*>(b_tile + (b_tap0 + 2 * i) * kBlock + b_vox * 32 + b_piece * 8) = ahead[u].b[i];
      __syncthreads();  // the other phase was read before the barrier of the round behind it
      fetch(ahead[u], v + D * kTurn + half * kVx);
      uint4 af[2][2], bf[2][2];  // [block or tap][k-step]
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int i = 0; i < 2; ++i) af[i][ks] = tr_fragment<T>(s_tile + i * kBlock + ks * 16 * 32, 32, lane);
#pragma unroll
        for (int j = 0; j < 2; ++j) bf[j][ks] = tr_fragment<T>(b_tile + (2 * wave + j) * kBlock + ks * 16 * 32, 32, lane);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const f32x16_t sum = Mma32<T>::run(af[i][1], bf[j][1], Mma32<T>::run(af[i][0], bf[j][0], none));
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] += sum[r];
        }
      if constexpr (BIAS) {
        if (sums_big) {  // every row of the block is the column sum of 16 voxels
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) bsum += (double)Mma32<T>::run(ones, bf[j][ks], none)[0];
        }
      }
    }
  }
  // part[split][cs][tap][cb]: a lane holds column cb = lane % 32 and 16 rows of its block
  float* dst = part + (int64_t)split * a.csmall * kTaps * a.cbig + ((int64_t)cs0 * kTaps + 2 * wave) * a.cbig + cb0 + (lane & 31);
  const int kg = lane >> 5;
  auto store = [&](const f32x16_t& sum, int i, int j) {
#pragma unroll
    for (int r = 0; r < 16; ++r) dst[((int64_t)(i * 32 + 8 * (r >> 2) + 4 * kg + (r & 3)) * kTaps + j) * a.cbig] = sum[r];
  };
  double* sums = reinterpret_cast<double*>(lds);  // [half][tap pair][channel]
  if constexpr (HALVES == 1) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) store(acc[i][j], i, j);
    if constexpr (BIAS) __syncthreads();
  } else {
    // half h keeps row block h and hands the other one over
    float4* hand = reinterpret_cast<float4*>(lds);
    sums += 32 * 256;
    auto give = [&](const f32x16_t (&sum)[2]) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          hand[((half * 2 + j) * 4 + g) * 256 + tid] = make_float4(sum[j][4 * g], sum[j][4 * g + 1], sum[j][4 * g + 2], sum[j][4 * g + 3]);
    };
    auto take = [&](f32x16_t (&sum)[2], int i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4 o = hand[(((i ^ 1) * 2 + j) * 4 + g) * 256 + tid];
          sum[j][4 * g] += o.x; sum[j][4 * g + 1] += o.y; sum[j][4 * g + 2] += o.z; sum[j][4 * g + 3] += o.w;
        }
        store(sum[j], i, j);
      }
    };
    __syncthreads();
    if (half == 0) give(acc[1]);
    else give(acc[0]);
    __syncthreads();
    if (half == 0) take(acc[0], 0);
    else take(acc[1], 1);
  }
  if constexpr (BIAS) {  // the sums of the wavefronts (tap pairs, halves) in that order: one row of channels per split
    sums[(half * 4 + wave) * 32 + (lane & 31)] = bsum;
    __syncthreads();
    if (sums_big && threadIdx.x < 32) {
      double sum = 0.;
#pragma unroll
      for (int t = 0; t < 4 * HALVES; ++t) sum += sums[t * 32 + threadIdx.x];
      bias_part[(int64_t)split * a.cbig + cb0 + threadIdx.x] = (float)sum;
    }
  }
#endif
}

int64_t small_voxels(const PatchArgs& a) { return (int64_t)a.n * a.sd * a.sh * a.sw; }

// Produced-channel blocks per wavefront: as many as keep at least two wavefronts per SIMD busy.
int gather_blocks(const PatchArgs& a) {
  const int nblk = a.csmall / 32;
  const int64_t wave_tiles = cdiv(small_voxels(a), 32);
  int nb = 8;
  while (nb > 1 && (nblk % nb != 0 || wave_tiles * (nblk / nb) < 2048)) nb >>= 1;
  return nb;
}

// The kept form takes the channel counts it has tiles for once there are a few dozen tiles; below that the chain of one
// workgroup's tile is longer than the deep kernel's. Before -> kept, packed weight, us: 64 -> 32 at 64^3 34 -> 26, at 32x64x64
// 19 -> 15, at 16^3 3.3 -> 4.2; 128 -> 64 at 64^3 108 -> 65, at 32^3 15.1 -> 11.2, at 16x32x32 11.8 -> 7.3, at 8^3 3.7 -> 4.8;
// 256 -> 128 at 32^3 38 -> 25, at 8x16x16 6.9 -> 6.7, at 5x7x9 (two samples) 4.8 -> 6.7; 512 -> 256 at 16^3 38 -> 22.
bool gather_kept(const PatchArgs& a) {
  if (small_voxels(a) * a.cbig < (1 << 18)) return false;
  return a.cbig == 32 || a.cbig == 256 ? a.csmall % 64 == 0 : (a.cbig == 64 || a.cbig == 128) && a.csmall % 128 == 0;
}

template <typename T, int CB>
int launch_gather_kept(const PatchArgs& a, const void* big, const void* w, bool dense, const void* bias, void* small, hipStream_t st) {
  using C = GatherKept<CB>;
  const int64_t total = small_voxels(a), tiles = cdiv(total, C::V);
  const int ncol = a.csmall / (32 * C::NBW);
  int64_t groups = cdiv((C::KH == 1 ? 2 : 1) * kComputeUnits, ncol);  // what LDS lets be resident
  if (groups > tiles) groups = tiles;
  const dim3 grid((unsigned)(cdiv(groups, kXcds) * kXcds * ncol));
  if constexpr (CB != 256) {
    if (dense) {
      hipLaunchKernelGGL((patch_gather_kept_kernel<T, CB, false>), grid, dim3(C::THREADS), 0, st, a, (const T*)big, (const T*)w,
                         (const T*)bias, (T*)small, total, (int)groups);
      return check_launch("patch_gather_kept_kernel");
    }
  }
  hipLaunchKernelGGL((patch_gather_kept_kernel<T, CB, true>), grid, dim3(C::THREADS), 0, st, a, (const T*)big, (const T*)w,
                     (const T*)bias, (T*)small, total, (int)groups);
  return check_launch("patch_gather_kept_kernel");
}

template <typename T>
int launch_gather(const PatchArgs& a, const void* big, const void* w, bool dense, const void* bias, void* small, hipStream_t st) {
  if (dense && !patch_gather_reads_dense(a)) return fail(SFH_ERR_INVALID, "conv3d fwd: this problem reads a packed weight");
  if (gather_kept(a)) {
    if (a.cbig == 32) return launch_gather_kept<T, 32>(a, big, w, dense, bias, small, st);
    if (a.cbig == 64) return launch_gather_kept<T, 64>(a, big, w, dense, bias, small, st);
    if (a.cbig == 128) return launch_gather_kept<T, 128>(a, big, w, dense, bias, small, st);
    return launch_gather_kept<T, 256>(a, big, w, dense, bias, small, st);
  }
  const int64_t total = small_voxels(a);
  const int nb = gather_blocks(a);
  const dim3 grid((unsigned)cdiv(total, 128), (unsigned)(a.csmall / 32 / nb));
  if (nb == 1 && (int64_t)grid.x * grid.y < kComputeUnits) {  // under one workgroup per CU (no gain measured above that)
    hipLaunchKernelGGL((patch_gather_deep_kernel<T>), dim3((unsigned)cdiv(total, 32), (unsigned)(a.csmall / 32)), dim3(256), 0, st, a,
                       (const T*)big, (const T*)w, (const T*)bias, (T*)small, total);
    return check_launch("patch_gather_deep_kernel");
  }
#define SFH_PATCH_GATHER(NB)                                                                                              \
  hipLaunchKernelGGL((patch_gather_kernel<T, NB>), grid, dim3(256), 0, st, a, (const T*)big, (const T*)w, (const T*)bias, \
                     (T*)small, total)
  if (nb == 8) SFH_PATCH_GATHER(8);
  else if (nb == 4) SFH_PATCH_GATHER(4);
  else if (nb == 2) SFH_PATCH_GATHER(2);
  else SFH_PATCH_GATHER(1);
#undef SFH_PATCH_GATHER
  return check_launch("patch_gather_kernel");
}

template <typename T, int KS, int C>
int launch_scatter_kept(const PatchArgs& a, const void* small, const void* w, bool dense, const void* bias, void* big, hipStream_t st,
                        int64_t face_pieces, int64_t big_elems) {
  const int64_t total = small_voxels(a), tiles = cdiv(total, 32);
  const int ncol = 2 * (a.cbig / 32) / C;
  // two workgroups per CU are what the registers allow (three and four: 5 to 20 % slower, the weights are fetched more often)
  int64_t groups = cdiv(2 * kComputeUnits, ncol);
  if (groups > tiles) groups = tiles;
  const dim3 grid((unsigned)(cdiv(groups, kXcds) * kXcds * ncol));
  if (dense)
    hipLaunchKernelGGL((patch_scatter_kernel<T, KS, C, false>), grid, dim3(256), 0, st, a, (const T*)small, (const T*)w, (const T*)bias,
                       (T*)big, total, (int)groups, face_pieces, big_elems);
  else
    hipLaunchKernelGGL((patch_scatter_kernel<T, KS, C, true>), grid, dim3(256), 0, st, a, (const T*)small, (const T*)w, (const T*)bias,
                       (T*)big, total, (int)groups, face_pieces, big_elems);
  return check_launch("patch_scatter_kernel");
}

template <typename T>
int launch_scatter(const PatchArgs& a, const void* small, const void* w, bool dense, const void* bias, void* big, hipStream_t st,
                   int64_t halo_elems) {
  const int64_t total = small_voxels(a);
  const int64_t big_elems = (int64_t)a.n * a.bd * a.bh * a.bw * a.cbig;
  if (halo_elems > 0 && (a.n != 1 || (reinterpret_cast<uintptr_t>(big) & 15) != 0 || (big_elems * (int64_t)sizeof(T)) % 16 != 0 ||
                         (halo_elems * (int64_t)sizeof(T)) % 16 != 0))
    return fail(SFH_ERR_UNSUPPORTED, "convT3d fwd: a slab output needs one sample and 16-byte aligned faces");
  const Tails tails = tails_of(a);
  if ((tails.planes + tails.rows + tails.columns) * a.n >= (1ll << 31) / (a.cbig / 8) ||
      (tails.planes + tails.rows + tails.columns > 0 && cdiv(total, 128) * (a.cbig / 32) * kTaps * 256 >= (1ll << 31)))
    return fail(SFH_ERR_UNSUPPORTED, "convT3d fwd: the padding has 2^31 pieces of 16 bytes or more");
  const int64_t face_pieces = halo_elems > 0 ? halo_elems * (int64_t)sizeof(T) / 16 : 0;
  // Weights of one (512 channels) or two columns fit in a wavefront's registers: the kept form. General form ->
  // kept form, packed weight, us: 128 -> 64 at 64^3 120 -> 74, at 32^3 20.7 -> 12.3, at 16x32x32 12 -> 8.5; 64 -> 32 at 64^3 47 -> 28,
  // at 32x64x64 25 -> 17; 256 -> 128 at 32^3 48 -> 26, at 8x16x16 7.8 -> 5.9; 512 -> 256 at 16^3 29 -> 15, at 4x8x8 7.2 -> 4.8.
  // With the weight packed, a launch of few short reductions stays with the general one, whose wavefronts have one tap each and no turn
  // through LDS: 64 -> 32 at 10^3 4.2 kept, 3.9 general, at 16^3 4.4 and 4.3, 128 -> 64 at 4^3 4.3 and 4.0, 256 -> 128 at 4^3 5.3 and 4.8; from the
  // line on the kept one is as fast or faster (128 -> 64 at 10^3 4.5 both, 64 -> 32 at 16x41x7 4.4 and 4.9).
  const int64_t reductions = cdiv(total, 32) * (a.cbig / 32) * a.csmall;
  if (patch_scatter_reads_dense(a) && (dense || reductions > 64 * 128)) {
    if (a.csmall == 64) return launch_scatter_kept<T, 4, 2>(a, small, w, dense, bias, big, st, face_pieces, big_elems);
    if (a.csmall == 128) return launch_scatter_kept<T, 8, 2>(a, small, w, dense, bias, big, st, face_pieces, big_elems);
    if (a.csmall == 256) return launch_scatter_kept<T, 16, 2>(a, small, w, dense, bias, big, st, face_pieces, big_elems);
    return launch_scatter_kept<T, 32, 1>(a, small, w, dense, bias, big, st, face_pieces, big_elems);
  }
  if (dense) return fail(SFH_ERR_INVALID, "convT3d fwd: this problem reads a packed weight");
  dim3 grid((unsigned)cdiv(total, 128), (unsigned)(a.cbig / 32));
  const int64_t wgs = (int64_t)grid.x * grid.y;
  if (wgs < kComputeUnits) {  // under one workgroup per CU: one tap per workgroup
    grid.z = kTaps;
    hipLaunchKernelGGL((patch_scatter_any_kernel<T, 1>), grid, dim3(256), 0, st, a, (const T*)small, (const T*)w, (const T*)bias,
                       (T*)big, total, face_pieces, big_elems);
  } else if (wgs < 4 * kComputeUnits) {  // under four per CU: two taps (the big voxels next to each other along W)
    grid.z = kTaps / 2;
    hipLaunchKernelGGL((patch_scatter_any_kernel<T, 2>), grid, dim3(256), 0, st, a, (const T*)small, (const T*)w, (const T*)bias,
                       (T*)big, total, face_pieces, big_elems);
  } else {
    // four taps (one big depth plane of the 2 x 2 x 2 patch) per workgroup: eight taps need 295 registers a lane, i.e. one
    // wavefront per SIMD walking four dependent trips to memory each (31 us at 64 -> 32 on 32 x 64 x 64); with half the
    // accumulators three wavefronts share a SIMD, and the small tensor read twice costs less than that gains
    grid.z = 2;
    hipLaunchKernelGGL((patch_scatter_any_kernel<T, 4>), grid, dim3(256), 0, st, a, (const T*)small, (const T*)w, (const T*)bias,
                       (T*)big, total, face_pieces, big_elems);
  }
  return check_launch("patch_scatter_any_kernel");
}

struct ReducePlan { int halves; int splits; int64_t per_split; };

// Splits of the voxels: up to one workgroup per CU, and fewer where the slices (written, then read by the sum) cost more than
// the shorter ranges gain. 0.7 us is a round of both halves, 0.6 us a megabyte of slices, fitted to sweeps of 1 to 256 splits over
// 17 problems (best plan within 5 % on each). Two workgroups of four wavefronts per CU, a slice each -> this, us with the sum: 128 -> 64
// at 64^3 120 -> 113, at 32^3 25 -> 21.5, at 48x40x56 84 -> 39; 64 -> 32 at 64^3 36 -> 34.6; 256 -> 128 at 32^3 49 -> 41, at 8x16x16 23 -> 15;
// 512 -> 256 at 4x8x8 24 -> 14. Eight at a time: a range of voxels per XCD.
// Where the rounds of all tiles do not give every CU one, a workgroup has one half: its start, and the two halves' meeting in LDS, cost
// more than the longer range. 0.65 us is a round then, 0.3 a megabyte of slices, 0.07 each of a few slices or 1.2 the grouped sum of many.
// us, workgroups of two halves under their own plan -> of one: 64 -> 32 at 4^3 7.7 -> 6.8, at 12^3 10.8 -> 8.9, at 10x8x39 10.9 -> 9.4,
// 128 -> 64 at 8^3 8.9 -> 8.3, 256 -> 128 at 5x8x4 9.6 -> 9.1; from the line on two are better: 64 -> 32 at 24^3 (432 rounds) 13.2 one, 12.6 two,
// 256 -> 128 at 8x16x16 (1024) 15.8 and 14.6.
ReducePlan reduce_plan(const PatchArgs& a) {
  const int64_t total = small_voxels(a);
  const int64_t tiles = (int64_t)(a.csmall / kSmallTile) * (a.cbig / 32);
  const int64_t rounds = cdiv(total, kVx);
  const double slice_mb = 4e-6 * kTaps * a.csmall * a.cbig;
  int64_t best = 1;
  double best_us = 1e30;
  ReducePlan p;
  p.halves = rounds * tiles < kComputeUnits ? 1 : 2;
  if (p.halves == 1) {
    for (int64_t s = 1; s <= rounds; ++s) {
      const double us = 0.65 * (double)cdiv(rounds, s) + 0.3 * slice_mb * (double)s + (s < 32 ? 0.07 * (double)s : 1.2);
      if (us < best_us) { best_us = us; best = s; }
    }
  } else {
    // two ranges at least past four rounds: one of eight rounds rounds a sum more often than eight slices of one do (512 -> 256 at
    // 4x8x8 0.56e-7 in one range, 0.55 in two; 13.0 -> 13.9 us)
    const int64_t least = rounds > 4 && 2 * tiles <= kComputeUnits ? 2 : 1;
    for (int64_t s = least; s <= rounds && (s <= least || s * tiles <= kComputeUnits); s = s < 8 ? 2 * s : s + 8) {
      const double us = 0.7 * (double)(cdiv(s * tiles, kComputeUnits) * cdiv(cdiv(rounds, s), 2)) + 0.6 * slice_mb * (double)s;
      if (us < best_us) { best_us = us; best = s; }
    }
  }
  p.per_split = cdiv(rounds, best) * kVx;
  p.splits = (int)cdiv(total, p.per_split);
  return p;
}

template <typename T>
int launch_reduce(const PatchArgs& a, const void* small, const void* big, void* g, int g_dtype, void* ws, hipStream_t st, void* gb) {
  const ReducePlan p = reduce_plan(a);
  const int64_t total = small_voxels(a);
  const int64_t tiles = (int64_t)(a.csmall / kSmallTile) * (a.cbig / 32);
  const int by_xcd = p.splits > 4;
  const dim3 grid((unsigned)((by_xcd ? cdiv(p.splits, kXcds) * kXcds : p.splits) * tiles));
  const int64_t nelem = (int64_t)a.csmall * kTaps * a.cbig;
  const VoxelStep step = voxel_step(a, p.halves * kVx);
  float* bias_part = (float*)ws + (int64_t)p.splits * nelem;  // behind the weight slices
#define SFH_PATCH_REDUCE(BIAS, HALVES)                                                                                           \
  hipLaunchKernelGGL((patch_reduce_kernel<T, BIAS, HALVES>), grid, dim3(256 * HALVES), 0, st, a, (const T*)small, (const T*)big, \
                     (float*)ws, total, p.per_split, p.splits, by_xcd, step, bias_part)
  if (gb != nullptr) {
    if (p.halves == 2) SFH_PATCH_REDUCE(true, 2);
    else SFH_PATCH_REDUCE(true, 1);
  } else {
    if (p.halves == 2) SFH_PATCH_REDUCE(false, 2);
    else SFH_PATCH_REDUCE(false, 1);
  }
#undef SFH_PATCH_REDUCE
  if (int rc = check_launch("patch_reduce_kernel")) return rc;
  if (gb == nullptr) return sum_slices(g_dtype, (const float*)ws, g, nelem, p.splits, st);
  // both sums in one launch
  return sum_slices_two(g_dtype, (const float*)ws, g, nelem, p.splits, bias_part, gb, a.cbig, p.splits, st);
}

bool geometry_ok(const PatchArgs& a, int dtype) {
  if (dtype != SFH_BF16 && dtype != SFH_FP16) return false;
  if (a.n < 1 || a.sd < 1 || a.sh < 1 || a.sw < 1) return false;
  if (a.bd < 2 * a.sd || a.bh < 2 * a.sh || a.bw < 2 * a.sw) return false;
  if (cdiv(small_voxels(a), 128) > 0x7fffffffLL) return false;
  return true;
}

}  // namespace

bool patch_supported(const PatchArgs& a, int dtype) {
  return geometry_ok(a, dtype) && a.cbig % 32 == 0 && a.csmall % 32 == 0 && a.cbig / 32 <= 65535 && a.csmall / 32 <= 65535;
}

bool patch_reduce_supported(const PatchArgs& a, int dtype) {
  return geometry_ok(a, dtype) && a.cbig % 32 == 0 && a.csmall % kSmallTile == 0 && a.cbig / 32 <= 65535 &&
         a.csmall / kSmallTile <= 65535;
}

int patch_gather(const PatchArgs& a, int dtype, const void* big, const void* w, bool dense, const void* bias, void* small,
                 hipStream_t st) {
  if (dtype == SFH_BF16) return launch_gather<bf16_t>(a, big, w, dense, bias, small, st);
  return launch_gather<fp16_t>(a, big, w, dense, bias, small, st);
}

// (256 channels: the registers of the weights and of the layout pass together spill, 33 us against 22 + a packing at 16^3)
bool patch_gather_reads_dense(const PatchArgs& a) { return gather_kept(a) && a.cbig != 256; }
// (the kept form numbers big voxels in 32 bits)
bool patch_scatter_reads_dense(const PatchArgs& a) {
  return (a.csmall == 64 || a.csmall == 128 || a.csmall == 256 || a.csmall == 512) &&
         (int64_t)a.n * a.bd * a.bh * a.bw <= 0x7fffffffLL;
}

int patch_scatter(const PatchArgs& a, int dtype, const void* small, const void* w, bool dense, const void* bias, void* big,
                  hipStream_t st, int64_t halo_elems) {
  if (dtype == SFH_BF16) return launch_scatter<bf16_t>(a, small, w, dense, bias, big, st, halo_elems);
  return launch_scatter<fp16_t>(a, small, w, dense, bias, big, st, halo_elems);
}

int patch_reduce_splits(const PatchArgs& a) { return reduce_plan(a).splits; }

size_t patch_reduce_workspace_bytes(const PatchArgs& a, bool with_bias) {
  const size_t splits = (size_t)reduce_plan(a).splits;
  return splits * a.csmall * kTaps * a.cbig * sizeof(float) + (with_bias ? splits * a.cbig * sizeof(float) : 0);
}

int patch_reduce(const PatchArgs& a, int dtype, const void* small, const void* big, void* g, int g_dtype, void* ws, hipStream_t st,
                 void* gb) {
  if (dtype == SFH_BF16) return launch_reduce<bf16_t>(a, small, big, g, g_dtype, ws, st, gb);
  return launch_reduce<fp16_t>(a, small, big, g, g_dtype, ws, st, gb);
}

}  // namespace sfh
