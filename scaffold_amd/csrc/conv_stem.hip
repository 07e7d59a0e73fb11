// The network's first convolution (3x3x3, stride 1, 1 to 4 input channels, 32 or 64 output channels) on the matrix cores:
// forward (with GroupNorm records) and weight gradient, 16-bit types.  Same contract as the other convolution kernels
// (triton_conv3d/gather_gemm.py:1187, reduce_gemm.py:1177).
//
// Bound: HBM, by the wide tensor (output or output gradient), once something feeds the matrix cores fast enough.  What
// feeds them here is a brick of 8-byte CELLS in LDS: a cell is the four 16-bit values that one tap contributes to the
// contraction, so an operand fragment (8 values of the contraction per lane) is two 8-byte LDS reads and no packing:
//   2..4 channels: the cell of a voxel is its channels, padded to four with zeros; 27 taps (kd, kh, kw);
//   1 channel:     the cell of a position is the values at w, w + 1, w + 2 and a zero; 9 taps (kd, kh).
// Padding is zeros that take part as zeros, as in the other matrix-core kernels.
// The weight is staged in the same cells once per workgroup and held in registers; a workgroup walks several tiles and has
// the next tile's voxels in flight while it works on the current one.
//
// Measured (bf16, us per launch; "floor" = the wide tensor once at the rate of a large copy, 5.2 TB/s):
//   forward + GroupNorm records: 3 -> 64 on 128^3 83 (floor 52), 3 -> 32 on 64^3 14, 1 -> 32 on 64 x 128 x 128 21.5 (13);
//   weight gradient + slice sum: 71, 16 and 23.5.
// Before: 3 channels had no matrix-core form (11 350 + 60 400 us on 128^3 through the direct kernels), and the one-channel
// kernels gathered every value of an operand by itself (31.7 and 25.8 us on 64 x 128 x 128; 28 us for a 32^3 weight
// gradient cut into 16 workgroups of 2048 voxels, now 128 of one tile: 15).
#include "conv_stem.hpp"
#include "mma.hpp"
#include "reduce.hpp"

namespace sfh {

namespace {

constexpr int kBlock = 256;

template <int CT> struct StemCells {
  static constexpr int kTaps = CT == 1 ? 9 : 27;
  static constexpr int kValues = CT == 1 ? 3 : CT;           // values of a cell that are not padding
  static constexpr int kSteps = (kTaps * 4 + 15) / 16;       // MFMA k-steps of the contraction: 3 or 7
  static constexpr int kTapCells = kSteps * 4;               // taps, padded to whole k-steps
  static constexpr int width(int tw) { return CT == 1 ? tw : tw + 2; }
};

// Brick cell of tap t relative to the cell of the output voxel's own position.
template <int CT, int BH, int BW>
__device__ __forceinline__ int tap_cell(int t) {
  return CT == 1 ? ((t / 3) * BH + t % 3) * BW : ((t / 9) * BH + (t / 3) % 3) * BW + t % 3;
}

struct StemTiles { int d, h, w; };  // tiles along each axis of a sample

// The voxels of one tile's brick on their way from memory to LDS: issued with load(), written with store().  Loads are
// unconditional from a clamped offset (a load under a branch would wait for the one before it), values outside the
// tensor become zeros when they are written.
template <int CT, int TD, int TH, int TW>
struct BrickFetch {
  using Cells = StemCells<CT>;
  static constexpr int kBD = TD + 2, kBH = TH + 2, kBW = Cells::width(TW), kCells = kBD * kBH * kBW;
  static constexpr int kRounds = (kCells + kBlock - 1) / kBlock;
  int rel[kRounds], at[kRounds];  // element offset and (d, h, w) of this thread's cells relative to the brick's corner
  uint16_t v[kRounds][Cells::kValues];
  uint32_t in;

  __device__ __forceinline__ void init(const StemArgs& a, int tid) {
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
      const int i = tid + k * kBlock;
      const int bw = i % kBW, bh = (i / kBW) % kBH, bd = i / (kBW * kBH);
      rel[k] = ((bd * a.th + bh) * a.tw + bw) * CT;
      at[k] = bd << 16 | bh << 8 | bw;
    }
  }
  // corner (id0, ih0, iw0) of the brick in the sample `xs`
  __device__ __forceinline__ void load(const StemArgs& a, const uint16_t* __restrict__ xs, int id0, int ih0, int iw0, int tid) {
    const int base = ((id0 * a.th + ih0) * a.tw + iw0) * CT;
    in = 0;
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
      const int id = id0 + (at[k] >> 16), ih = ih0 + (at[k] >> 8 & 255), iw = iw0 + (at[k] & 255);
      const bool row = tid + k * kBlock < kCells && (unsigned)id < (unsigned)a.td && (unsigned)ih < (unsigned)a.th;
#pragma unroll
      for (int e = 0; e < Cells::kValues; ++e) {
        const bool ok = row && (unsigned)(CT == 1 ? iw + e : iw) < (unsigned)a.tw;
        v[k][e] = xs[ok ? base + rel[k] + e : 0];
        in |= ok ? 1u << (k * Cells::kValues + e) : 0u;
      }
    }
  }
  __device__ __forceinline__ void store(uint2* cells, int tid) const {
    static_assert(kRounds * Cells::kValues <= 32, "one validity bit per value");
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
      uint32_t u[4] = {0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < Cells::kValues; ++e) u[e] = (in >> (k * Cells::kValues + e) & 1) ? v[k][e] : 0u;
      if (tid + k * kBlock < kCells) cells[tid + k * kBlock] = make_uint2(u[0] | u[1] << 16, u[2] | u[3] << 16);
    }
  }
};

struct TileAt { int d0, h0, w0; };
template <int TD, int TH, int TW>
__device__ __forceinline__ TileAt tile_at(int tile, const StemTiles& t) {
  TileAt r;
  r.w0 = (tile % t.w) * TW; tile /= t.w;
  r.h0 = (tile % t.h) * TH;
  r.d0 = (tile / t.h) * TD;
  return r;
}

// ---- forward ------------------------------------------------------------------------------------------------------------
constexpr int kFD = 4, kFH = 4, kFW = 32;  // a wavefront owns one plane of the tile: four runs of 32 voxels

// grid = (workgroups of a sample, samples); a workgroup takes `per` neighbouring tiles. Result blocks: rows = 32 output
// channels (the weight), columns = 32 voxels of a row.
template <typename T, int CT, int NC>
__global__ void __launch_bounds__(kBlock, NC == 1 && CT < 3 ? 3 : 2) stem_fwd_cells_kernel(StemArgs a, const T* __restrict__ x, const T* __restrict__ wt,
                                                                const T* __restrict__ bias, T* __restrict__ out, StemTiles tiles,
                                                                int per, GnPartialOut gn) {
  using Cells = StemCells<CT>;
  using Fetch = BrickFetch<CT, kFD, kFH, kFW>;
  constexpr int kWeightCells = NC * 32 * Cells::kTapCells;
  constexpr int kZeroCell = Fetch::kCells;  // what the taps that pad the last k-step read: NaN times a zero weight is NaN
  __shared__ __attribute__((aligned(16))) uint2 cells[kWeightCells > kZeroCell + 1 ? kWeightCells : kZeroCell + 1];
  __shared__ __attribute__((aligned(16))) float bias_of[NC * 32];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 31, kg = lane >> 5;
  const int ntiles = tiles.d * tiles.h * tiles.w;
  const int begin = blockIdx.x * per, end = begin + per < ntiles ? begin + per : ntiles;
  const uint16_t* xs = reinterpret_cast<const uint16_t*>(x) + (int64_t)blockIdx.y * a.td * a.th * a.tw * CT;
  T* ys = out + (int64_t)blockIdx.y * a.od * a.oh * a.ow * a.cw;
  Fetch fetch;
  fetch.init(a, tid);
  TileAt t = tile_at<kFD, kFH, kFW>(begin, tiles);
  fetch.load(a, xs, t.d0 - a.pd, t.h0 - a.ph, t.w0 - a.pw, tid);
  // the weight as cells [channel][tap], beside the first tile's voxels
#pragma unroll
  for (int k = 0; k < (kWeightCells + kBlock - 1) / kBlock; ++k) {
    const int i = tid + k * kBlock < kWeightCells ? tid + k * kBlock : kWeightCells - 1;
    const int c = i / Cells::kTapCells, tap = i % Cells::kTapCells;
    uint32_t u[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < Cells::kValues; ++e) {
      const int tc = tap < Cells::kTaps ? tap : 0;
      const int64_t off = CT == 1 ? (tc / 3) * a.ws_kd + (tc % 3) * a.ws_kh + e * a.ws_kw
                                  : (tc / 9) * a.ws_kd + ((tc / 3) % 3) * a.ws_kh + (tc % 3) * a.ws_kw + e * a.ws_thin;
      const uint32_t bits = reinterpret_cast<const uint16_t*>(wt)[(int64_t)c * a.ws_wide + off];
      u[e] = tap < Cells::kTaps ? bits : 0u;
    }
    cells[i] = make_uint2(u[0] | u[1] << 16, u[2] | u[3] << 16);
  }
  if (tid < NC * 32) bias_of[tid] = bias != nullptr ? to_float(bias[tid]) : 0.f;
  __syncthreads();
  uint4 wf[NC][Cells::kSteps];
#pragma unroll
  for (int cc = 0; cc < NC; ++cc)
#pragma unroll
    for (int ks = 0; ks < Cells::kSteps; ++ks)
      wf[cc][ks] = *reinterpret_cast<const uint4*>(cells + (cc * 32 + col) * Cells::kTapCells + ks * 4 + kg * 2);
  RunSums gn_sums[NC];  // GroupNorm statistics of the rounded output, when the caller wants them
#pragma unroll
  for (int cc = 0; cc < NC; ++cc) gn_sums[cc].clear();
  for (int tile = begin; tile < end; ++tile) {
    __syncthreads();  // the previous tile (at first: the weight) is read
    fetch.store(cells, tid);
    if (tid == 0) cells[kZeroCell] = make_uint2(0, 0);
    __syncthreads();
    const TileAt now = t;
    if (tile + 1 < end) {
      t = tile_at<kFD, kFH, kFW>(tile + 1, tiles);
      fetch.load(a, xs, t.d0 - a.pd, t.h0 - a.ph, t.w0 - a.pw, tid);
    }
    const int od = now.d0 + wave, ow = now.w0 + col;
#pragma unroll 1
    for (int i = 0; i < kFH; ++i) {
      const int oh = now.h0 + i;
      const int base = (wave * Fetch::kBH + i) * Fetch::kBW + col;
      uint4 xf[Cells::kSteps];
#pragma unroll
      for (int ks = 0; ks < Cells::kSteps; ++ks) {
        uint2 c[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int t0 = ks * 4 + e, t1 = t0 + 2;  // this lane's tap for k-half 0 and 1
          constexpr int last = Cells::kTaps - 1;
          const int o0 = tap_cell<CT, Fetch::kBH, Fetch::kBW>(t0 <= last ? t0 : last);
          const int o1 = tap_cell<CT, Fetch::kBH, Fetch::kBW>(t1 <= last ? t1 : last);
          int at = base + (kg ? o1 : o0);
          if (t1 > last) at = (t0 > last || kg) ? kZeroCell : at;
          c[e] = cells[at];
        }
        xf[ks] = make_uint4(c[0].x, c[0].y, c[1].x, c[1].y);
      }
      const bool valid = od < a.od && oh < a.oh && ow < a.ow;
      T* dst = ys + (valid ? ((int64_t)(od * a.oh + oh) * a.ow + ow) * a.cw : 0);
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        f32x16_t acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < Cells::kSteps; ++ks) acc = Mma32<T>::run(wf[cc][ks], xf[ks], acc);
        float add[16];
#pragma unroll
        for (int g = 0; g < 4; ++g) *reinterpret_cast<float4*>(add + 4 * g) = *reinterpret_cast<const float4*>(bias_of + cc * 32 + 8 * g + 4 * kg);
        store_block_plus<T>(acc, dst + cc * 32, add, kg, valid, gn_sums[cc], gn.part != nullptr, tile == begin && i == 0);
      }
    }
  }
  if (gn.part != nullptr) {
    __syncthreads();  // every wave is done reading the brick: the LDS is free
    static_assert(sizeof(cells) >= gn_partials_lds_floats(kBlock / 64, NC) * sizeof(float), "room for the wavefronts' sums");
    write_group_partials<kBlock / 64, NC>(gn_sums, reinterpret_cast<float*>(cells), gn, blockIdx.y, blockIdx.x, 0, tid);
  }
}

// ---- weight gradient ----------------------------------------------------------------------------------------------------
constexpr int kGD = 2, kGH = 4, kGW = 32;  // a wavefront owns two rows of 32 voxels: four k-steps of 16
constexpr int kGVox = kGD * kGH * kGW;

typedef short stem_v4s __attribute__((__vector_size__(4 * sizeof(short))));
__device__ __forceinline__ uint2 read_tr(const void* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) stem_v4s*)(p)));
#else
  return make_uint2(0, 0);
#endif
}

// The first `count` (clamped to 0 .. 2) of the two 16-bit values of u, the others zero.
__device__ __forceinline__ uint32_t first_halves(uint32_t u, int count) { return count >= 2 ? u : count == 1 ? u & 0xffffu : 0u; }

// G[c][tap][e] = sum_v gy[v][c] * cell(v (+) tap)[e] with the voxels as the contraction.  A tile may reach past the output:
// its voxels there have no gradient, but the cells their taps name can lie inside the tensor, and 0 x infinity is not 0.
// With CUT (an output that is not whole tiles) such rows are skipped, and in a tile that ends inside a row the values of
// voxels past the end are cleared in the operand (the cells themselves are shared with voxels that count).  Both operands lie in LDS as in
// memory (gradient rows of CW channels, brick cells) and are turned by the transposing read: of the 16 lanes that share
// one, lane m names the 8 bytes of (voxel m / 4, chunk m % 4) and gets value m % 4 of chunk m / 4 for four voxels.  For
// the brick a chunk is a cell, so the 32 columns of a result block are eight taps of four values each.
template <typename T, int CT, int NC, bool CUT>
__global__ void __launch_bounds__(kBlock, 2) stem_wgrad_cells_kernel(StemArgs a, const T* __restrict__ x, const T* __restrict__ gy,
                                                                     float* __restrict__ part, StemTiles tiles, int ntiles, int per) {
  using Cells = StemCells<CT>;
  using Fetch = BrickFetch<CT, kGD, kGH, kGW>;
  constexpr int CW = NC * 32, NB = (Cells::kTaps + 7) / 8;
  constexpr int kRow = CW + 8;                              // LDS row of a voxel's gradient: off the 128-byte period
  constexpr int kPieces = kGVox * CW / 8 / kBlock;          // 16-byte pieces of the tile's gradient per thread
  __shared__ __attribute__((aligned(16))) uint2 cells[Fetch::kCells];
  __shared__ __attribute__((aligned(16))) uint16_t grows[kGVox * kRow];
  static_assert(sizeof(grows) >= 4 * 32 * 33 * sizeof(float), "the fold at the end reuses the gradient rows");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, kg = lane >> 5;
  const int grp = lane >> 4, m = lane & 15;
  const int begin = blockIdx.x * per, end = begin + per < ntiles ? begin + per : ntiles;
  const int per_sample = tiles.d * tiles.h * tiles.w;
  // this lane's addresses for the transposing reads, relative to a k-step's first voxel
  const int g_at = ((grp >> 1) * 8 + (m >> 2)) * kRow + (grp & 1) * 16 + 4 * (m & 3);
  int c_at[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int tap = b * 8 + (grp & 1) * 4 + (m & 3);
    c_at[b] = tap_cell<CT, Fetch::kBH, Fetch::kBW>(tap < Cells::kTaps ? tap : Cells::kTaps - 1) + (grp >> 1) * 8 + (m >> 2);
  }
  f32x16_t acc[NC][NB];
#pragma unroll
  for (int cc = 0; cc < NC; ++cc)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[cc][b][r] = 0.f;
  Fetch fetch;
  fetch.init(a, tid);
  uint4 gv[kPieces];
  uint32_t gin = 0;
  TileAt t{};  // the tile in flight
  auto fetch_tile = [&](int tile) {
    const int n = tile / per_sample;
    t = tile_at<kGD, kGH, kGW>(tile - n * per_sample, tiles);
    fetch.load(a, reinterpret_cast<const uint16_t*>(x) + (int64_t)n * a.td * a.th * a.tw * CT, t.d0 - a.pd, t.h0 - a.ph, t.w0 - a.pw, tid);
    const T* gs = gy + (int64_t)n * a.od * a.oh * a.ow * CW;
    gin = 0;
#pragma unroll
    for (int k = 0; k < kPieces; ++k) {
      const int i = tid + k * kBlock, v = i / (CW / 8), p = i % (CW / 8);
      const int od = t.d0 + v / (kGH * kGW), oh = t.h0 + v / kGW % kGH, ow = t.w0 + v % kGW;
      const bool in = od < a.od && oh < a.oh && ow < a.ow;
      gv[k] = *reinterpret_cast<const uint4*>(gs + (in ? ((int64_t)(od * a.oh + oh) * a.ow + ow) * CW + p * 8 : 0));
      gin |= in ? 1u << k : 0u;
    }
  };
  if (begin < end) fetch_tile(begin);
  for (int tile = begin; tile < end; ++tile) {
    __syncthreads();  // the previous tile is read
    fetch.store(cells, tid);
#pragma unroll
    for (int k = 0; k < kPieces; ++k) {
      const int i = tid + k * kBlock, v = i / (CW / 8), p = i % (CW / 8);
      *reinterpret_cast<uint4*>(grows + v * kRow + p * 8) = (gin >> k & 1) ? gv[k] : make_uint4(0, 0, 0, 0);
    }
    __syncthreads();
    const TileAt now = t;
    if (tile + 1 < end) fetch_tile(tile + 1);
    const bool cut = now.w0 + kGW > a.ow;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int row = wave * 2 + (s >> 1), w0 = (s & 1) * 16;
      if (CUT && (now.d0 + row / kGH >= a.od || now.h0 + row % kGH >= a.oh || now.w0 + w0 >= a.ow)) continue;
      const int count = a.ow - (now.w0 + w0 + kg * 8);  // voxels of this lane's eight that the output has
      const uint16_t* gp = grows + (row * kGW + w0) * kRow + g_at;
      const uint2* cp = cells + ((row / kGH) * Fetch::kBH + row % kGH) * Fetch::kBW + w0;
      uint4 gf[NC];
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        const uint2 lo = read_tr(gp + cc * 32), hi = read_tr(gp + cc * 32 + 4 * kRow);
        gf[cc] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const uint2 lo = read_tr(cp + c_at[b]), hi = read_tr(cp + c_at[b] + 4);
        uint4 xf = make_uint4(lo.x, lo.y, hi.x, hi.y);
        if (CUT && cut) xf = make_uint4(first_halves(xf.x, count), first_halves(xf.y, count - 2), first_halves(xf.z, count - 4), first_halves(xf.w, count - 6));
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) acc[cc][b] = Mma32<T>::run(gf[cc], xf, acc[cc][b]);
      }
    }
  }
  // the four wavefronts' blocks, folded in wavefront order, become the workgroup's slice [channel][27][CT]
  float* fold = reinterpret_cast<float*>(grows);
  float* dst = part + (int64_t)blockIdx.x * 27 * CT * CW;
#pragma unroll
  for (int cc = 0; cc < NC; ++cc)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      __syncthreads();
#pragma unroll
      for (int r = 0; r < 16; ++r) fold[(wave * 32 + 8 * (r / 4) + 4 * kg + r % 4) * 33 + col] = acc[cc][b][r];
      __syncthreads();
      for (int i = tid; i < 32 * 32; i += kBlock) {
        const int c = i >> 5, j = i & 31, tap = b * 8 + (j >> 2), e = j & 3;
        float sum = fold[c * 33 + j];
#pragma unroll
        for (int w = 1; w < 4; ++w) sum += fold[(w * 32 + c) * 33 + j];
        if (tap < Cells::kTaps && e < Cells::kValues) dst[(cc * 32 + c) * 27 * CT + tap * Cells::kValues + e] = sum;
      }
    }
}

StemTiles stem_tiles(const StemArgs& a, int td, int th, int tw) {
  return StemTiles{(int)cdiv(a.od, td), (int)cdiv(a.oh, th), (int)cdiv(a.ow, tw)};
}

struct StemPlan { StemTiles tiles; int per, wgs; };

// Two workgroups per CU: what the registers of the 64-channel forms allow at once (3 and 4 per CU measured 5-20 % slower:
// the prologue is paid more often), and at most 512 GroupNorm records, which the normalisation folds without a launch of
// its own.
StemPlan fwd_plan(const StemArgs& a) {
  StemPlan p;
  p.tiles = stem_tiles(a, kFD, kFH, kFW);
  const int64_t nt = (int64_t)p.tiles.d * p.tiles.h * p.tiles.w;
  int64_t most = kComputeUnits * 2 / a.n;
  if (most < 64) most = 64;
  p.per = (int)cdiv(nt, most);
  p.wgs = (int)cdiv(nt, p.per);
  return p;
}

// Down to one tile per workgroup: a small volume is all latency, and its slices are small.
StemPlan wgrad_plan(const StemArgs& a) {
  StemPlan p;
  p.tiles = stem_tiles(a, kGD, kGH, kGW);
  const int64_t nt = (int64_t)a.n * p.tiles.d * p.tiles.h * p.tiles.w;
  p.per = (int)cdiv(nt, kComputeUnits * 2);
  p.wgs = (int)cdiv(nt, p.per);
  return p;
}

template <typename T, int CT>
int launch_fwd(const StemArgs& a, const void* x, const void* w, const void* bias, void* y, hipStream_t st, const GnPartialOut& gn) {
  const StemPlan p = fwd_plan(a);
  const dim3 grid(p.wgs, a.n);
  if (a.cw == 32) hipLaunchKernelGGL((stem_fwd_cells_kernel<T, CT, 1>), grid, dim3(kBlock), 0, st, a, (const T*)x, (const T*)w, (const T*)bias, (T*)y, p.tiles, p.per, gn);
  else hipLaunchKernelGGL((stem_fwd_cells_kernel<T, CT, 2>), grid, dim3(kBlock), 0, st, a, (const T*)x, (const T*)w, (const T*)bias, (T*)y, p.tiles, p.per, gn);
  return check_launch("stem_fwd_cells_kernel");
}

template <typename T, int CT>
int launch_wgrad(const StemArgs& a, const void* x, const void* gy, void* gw, int gw_dtype, void* ws, hipStream_t st) {
  const StemPlan p = wgrad_plan(a);
  const int ntiles = a.n * p.tiles.d * p.tiles.h * p.tiles.w;
  // Whole tiles need no look at the output's ends, which costs up to 6 % (kernel and slice sum without / with it, us: 1 -> 32
  // channels on 64 x 128 x 128 22.0 / 23.5; two samples of 3 -> 32 on 44 x 60 x 75, which need it, 20.2 / 21.2).
  const bool cut = a.od % kGD != 0 || a.oh % kGH != 0 || a.ow % kGW != 0;
#define SFH_STEM_WGRAD(NC, CUT)                                                                                                     \
  hipLaunchKernelGGL((stem_wgrad_cells_kernel<T, CT, NC, CUT>), dim3(p.wgs), dim3(kBlock), 0, st, a, (const T*)x, (const T*)gy,     \
                     (float*)ws, p.tiles, ntiles, p.per)
  if (a.cw == 32) {
    if (cut) SFH_STEM_WGRAD(1, true);
    else SFH_STEM_WGRAD(1, false);
  } else {
    if (cut) SFH_STEM_WGRAD(2, true);
    else SFH_STEM_WGRAD(2, false);
  }
#undef SFH_STEM_WGRAD
  if (int rc = check_launch("stem_wgrad_cells_kernel")) return rc;
  return sum_slices(gw_dtype, (const float*)ws, gw, (int64_t)27 * CT * a.cw, p.wgs, st);
}

#define SFH_STEM_BY_CHANNELS(fn, T, ...)          \
  switch (a.ct) {                                 \
    case 1: return fn<T, 1>(__VA_ARGS__);         \
    case 2: return fn<T, 2>(__VA_ARGS__);         \
    case 3: return fn<T, 3>(__VA_ARGS__);         \
    default: return fn<T, 4>(__VA_ARGS__);        \
  }

template <typename T>
int fwd_of(const StemArgs& a, const void* x, const void* w, const void* bias, void* y, hipStream_t st, const GnPartialOut& gn) {
  SFH_STEM_BY_CHANNELS(launch_fwd, T, a, x, w, bias, y, st, gn)
}
template <typename T>
int wgrad_of(const StemArgs& a, const void* x, const void* gy, void* gw, int gw_dtype, void* ws, hipStream_t st) {
  SFH_STEM_BY_CHANNELS(launch_wgrad, T, a, x, gy, gw, gw_dtype, ws, st)
}

}  // namespace

bool stem_supported(const StemArgs& a, int dtype) {
  if (dtype != SFH_BF16 && dtype != SFH_FP16) return false;
  if (a.n < 1 || a.n > 65535 || a.ct < 1 || a.ct > 4 || (a.cw != 32 && a.cw != 64)) return false;
  if (a.pd > 2 || a.ph > 2 || a.pw > 2) return false;
  // 32-bit offsets inside a sample and 32-bit tile counts over all of them, with room for a brick past the end
  const int64_t in = (int64_t)(a.td + 8) * (a.th + 8) * (a.tw + 40) * a.ct, voxels = (int64_t)a.n * (a.od + 4) * (a.oh + 4) * (a.ow + 32);
  return in < (int64_t)1 << 31 && (int64_t)a.od * a.oh < (int64_t)1 << 31 && voxels / kGVox < (int64_t)1 << 30;
}

int stem_gn_records(const StemArgs& a, int groups) {
  return gn_partials_fit(a.cw, groups, a.cw) ? fwd_plan(a).wgs : 0;
}

int stem_fwd(const StemArgs& a, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t st, const GnPartialOut& gn) {
  return dtype == SFH_BF16 ? fwd_of<bf16_t>(a, x, w, bias, y, st, gn) : fwd_of<fp16_t>(a, x, w, bias, y, st, gn);
}

int stem_wgrad_splits(const StemArgs& a) { return wgrad_plan(a).wgs; }

size_t stem_wgrad_workspace_bytes(const StemArgs& a) { return (size_t)wgrad_plan(a).wgs * 27 * a.ct * a.cw * sizeof(float); }

int stem_wgrad(const StemArgs& a, int dtype, const void* x, const void* gy, void* gw, int gw_dtype, void* ws, hipStream_t st) {
  return dtype == SFH_BF16 ? wgrad_of<bf16_t>(a, x, gy, gw, gw_dtype, ws, st) : wgrad_of<fp16_t>(a, x, gy, gw, gw_dtype, ws, st);
}

}  // namespace sfh
