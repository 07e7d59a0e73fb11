// Tiled fp32 convolution on the fp32 matrix pipe of gfx950 (3x3x3, stride 1, dilation 1): forward and data gradient.
//
// The reference runs its fp32 convolutions through the same tiled kernel as the 16-bit ones with the dot product at
// full IEEE fp32 precision (triton_conv3d/gather_gemm.py:1334, input_precision="ieee"). Here that is
// v_mfma_f32_32x32x2_f32: fp32 operands, fp32 products, fp32 accumulation -- no down-conversion anywhere, so the
// 1e-5 bar of the fp32 configuration holds; dense fp32 MFMA peak is 157.3 TFLOP/s.
//
// GEMM view (gather_gemm.py:112-341): M = output voxels, N = produced channels, K = taps x reduction channels.
//   * A workgroup owns a TD x TH x TW brick of output voxels and one block of 32 produced channels; the input brick
//     with its halo is staged in LDS per chunk of 16 reduction channels as four 16-byte channel planes (plane p =
//     channels 4p .. 4p+3 of every brick voxel; planes 64 bytes apart modulo 256, so a wavefront's ds_read_b128 of rows
//     of 8 or more voxels is conflict free and every tap is an immediate offset).
//   * One MFMA contracts 2 reduction channels: k-slot kg (= lane / 32) at step kk of a chunk is channel 8 kg + kk, so a
//     lane's operands of the 8 steps of a tap are 8 consecutive channels: two 16-byte LDS reads of activations and 32 bytes
//     of the weight. A channels-last weight is read where it lies: forward two 16-byte loads of a row, data gradient eight of one
//     element, 32 produced channels side by side. An fp32 MFMA takes 64 cycles, so a tap's 8 per sub-tile hide either (a packing
//     launch in front, which other layouts still take, was 3 to 4 us of the call):
//       packed[cout/32][cred/16][tap][q(2)][lane(64)][4],  lane = cout % 32 + 32 kg,  channel = 16 cc + 8 kg + 4 q + e.
//   * The weight is the ROW operand, so a lane ends up with four runs of four consecutive output channels of one voxel
//     and stores 16-byte pieces.
// The data gradient runs this kernel with the weight transposed and tap-flipped and padding k-1-p
// (triton_conv3d/bwd_data.py:344-363).
#include "conv_f32.hpp"
#include "reduce.hpp"

namespace sfh {
namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kChunk = 16;  // reduction channels staged per pass (4 planes of 4)
constexpr int kTaps = 27;

constexpr int plane_bytes(int voxels) {  // smallest size >= voxels*16 that is 64 modulo 256
  return ((voxels * 16 - 64 + 255) / 256) * 256 + 64;
}

// KS: wavefronts that share a sub-tile's reduction, each a chunk of channels of its own; they meet in LDS in that order. WM: groups of
// such wavefronts, each with its sub-tiles.
template <int TD_, int TH_, int TW_, int WM_ = 4, int KS_ = 1>
struct FTile {
  static constexpr int TD = TD_, TH = TH_, TW = TW_, WM = WM_, KS = KS_;
  static constexpr int BD = TD + 2, BH = TH + 2, BW = TW + 2;
  static constexpr int BV = BD * BH * BW;
  static constexpr int PLANE = plane_bytes(BV);
  static constexpr int CHUNK = 4 * PLANE;
  static constexpr int MEET = (KS - 1) * WM * 16 * 64 * 4;
  static constexpr int LDS = KS * CHUNK > MEET ? KS * CHUNK : MEET;
  static constexpr int THREADS = 64 * WM * KS;
  static constexpr int MS = TD * TH * TW / (32 * WM);  // 32-voxel sub-tiles per wavefront
  // One sub-tile to a wavefront is what a volume gets that does not fill the chip: nothing else on the SIMD hides a trip to
  // memory or LDS, and there are registers for requesting the next chunk's brick and the next tap's activations ahead.
  // 32 -> 32 channels on 32^3: 27.4 -> 20.5 us a launch (its MFMAs alone 11.5; in bricks of
  // 8-voxel rows 21.3 in a trace with idle time between passes).
  static constexpr bool AHEAD = MS == 1;
  static_assert(TD * TH * TW % (32 * WM) == 0, "tile must split into WM wavefronts of 32-voxel sub-tiles");
  static_assert(KS == 1 || MS == 1, "the parts of a reduction meet in one sub-tile a wavefront");
  static_assert((THREADS > 256 ? 1 : 2) * LDS <= 160 * 1024, "eight wavefronts in the 160 KB LDS of a CU");
  static_assert(PLANE + (2 * BH * BW + 2 * BW + 2) * 16 < 65536, "ds_read immediate range");
};

// The bricks. Rows of 8 or 16 voxels: 32-voxel rows spend three quarters of the matrix pipe on nothing where a volume is 8 wide.
using WholeTile = FTile<8, 8, 8>;                                                       // 512 voxels, four sub-tiles a wavefront
template <int TW> using FlatTile = FTile<TW == 8 ? 4 : 2, 4, TW>;                       // 128 voxels
template <int TW> using HalvedTile = FTile<2, TW == 8 ? 4 : 2, TW, 2, 2>;               // 64 voxels, the reduction in two parts
using QuarteredTile = FTile<2, 2, 8, 1, 4>;                                             // 32 voxels, in four

template <typename C>
__device__ __forceinline__ constexpr int tap_off(int tap) {
  const int kd = tap / 9, kh = (tap / 3) % 3, kw = tap % 3;
  return ((kd * C::BH + kh) * C::BW + kw) * 16;
}

// wt: the weight in the form W (conv_f32.hpp)
template <typename C, F32Weight W>
__global__ void __launch_bounds__(C::THREADS, 2)
conv_f32_kernel(MfmaConvArgs a, const float* __restrict__ x, const float* __restrict__ wt, const float* __restrict__ bias,
                float* __restrict__ y, int tiles_d, int tiles_h, int tiles_w, int nblocks, uint32_t total) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) char lds[C::LDS];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = (tid >> 6) % C::WM;
  const int part = C::KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((tid >> 6) / C::WM);
  const int j = lane & 31, kg = lane >> 5;

  uint32_t t = xcd_remap(blockIdx.x, total);
  const int nb = t % nblocks; t /= nblocks;
  const int tw_i = t % tiles_w; t /= tiles_w;
  const int th_i = t % tiles_h; t /= tiles_h;
  const int td_i = t % tiles_d;
  const int n = t / tiles_d;
  const int od0 = td_i * C::TD, oh0 = th_i * C::TH, ow0 = tw_i * C::TW;
  const int id0 = od0 - a.pd, ih0 = oh0 - a.ph, iw0 = ow0 - a.pw;

  // LDS byte offset of the sub-tile voxel at tap (0,0,0) in the lane's first plane (planes 2 kg and 2 kg + 1 are its)
  int lbase[C::MS];
#pragma unroll
  for (int ms = 0; ms < C::MS; ++ms) {
    const int v = (wave * C::MS + ms) * 32 + j;
    const int tw = v % C::TW, th = (v / C::TW) % C::TH, td = v / (C::TW * C::TH);
    lbase[ms] = part * C::CHUNK + 2 * kg * C::PLANE + ((td * C::BH + th) * C::BW + tw) * 16;
  }
  f32x16_t acc[C::MS];
#pragma unroll
  for (int ms = 0; ms < C::MS; ++ms)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[ms][r] = 0.f;

  const int ncc = a.cred / kChunk;
  constexpr int PIECES = C::KS * C::BV * 4;  // voxel by voxel the pieces of KS chunks, which lie side by side
  constexpr int ITERS = (PIECES + C::THREADS - 1) / C::THREADS;
  constexpr int BATCH = C::AHEAD ? ITERS : 8;  // staging loads in flight before the first LDS write
  const float* xn = x + (int64_t)n * a.id * a.ih * a.iw * a.cred;
  auto request = [&](int cc, int it0, float4 (&v)[BATCH]) {
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      if (it0 + u < ITERS) {
        // unconditional load from a clamped address, masked afterwards (a load under a branch waits for the one before)
        const int p = (it0 + u) * C::THREADS + tid;
        const int vox = p / (4 * C::KS), piece = p % (4 * C::KS);
        const int bw = vox % C::BW, bh = (vox / C::BW) % C::BH, bd = vox / (C::BW * C::BH);
        const int id = id0 + bd, ih = ih0 + bh, iw = iw0 + bw;
        const bool in = p < PIECES && (C::KS == 1 || cc * kChunk + piece * 4 < a.cred) && (unsigned)id < (unsigned)a.id && (unsigned)ih < (unsigned)a.ih && (unsigned)iw < (unsigned)a.iw;
        const int64_t at = in ? (((int64_t)id * a.ih + ih) * a.iw + iw) * a.cred + cc * kChunk + piece * 4 : 0;
        const float4 got = *reinterpret_cast<const float4*>(xn + at);
        v[u] = in ? got : make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
  };
  auto stage = [&](int it0, const float4 (&v)[BATCH]) {
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      if (it0 + u < ITERS) {
        const int p = (it0 + u) * C::THREADS + tid;
        if (p < PIECES) *reinterpret_cast<float4*>(lds + p % (4 * C::KS) / 4 * C::CHUNK + (p & 3) * C::PLANE + p / (4 * C::KS) * 16) = v[u];
      }
    }
  };
  // A fragment's place is a chunk's, which the wavefront shares, a tap's and the lane's. The taps of a chunk are followed by the next
  // chunk's, so the requests ahead run on over the end of a chunk. A weight where it lies is read through a buffer: one scalar addition
  // a tap (64-bit addresses of eight rows were half of the instructions of a tap, and 27 taps of them spilled scalar registers).
  const int last = part < ncc ? part + (ncc - 1 - part) / C::KS * C::KS : -1;  // the wavefront's last chunk
  const int first_chunk = part < ncc ? part : 0;
  const float* wcc = wt + ((int64_t)nb * ncc + first_chunk) * (kTaps * 2 * 256) + lane * 4;  // kPacked
  __amdgpu_buffer_rsrc_t wbuf;
  int wbase = 0, wchunk = 0, wtap = 0, wlane[8];  // bytes
  if constexpr (W == F32Weight::kRows) {
    wbase = (nb * 32 * kTaps * a.cred + first_chunk * kChunk) * 4;
    wchunk = C::KS * kChunk * 4;
    wtap = a.cred * 4;
    wlane[0] = (j * (kTaps * a.cred) + 8 * kg) * 4;
  } else if constexpr (W == F32Weight::kColumns) {
    wbase = ((first_chunk * kChunk * kTaps + kTaps - 1) * a.cout + nb * 32) * 4;
    wchunk = C::KS * kChunk * kTaps * a.cout * 4;
    wtap = -a.cout * 4;
#pragma unroll
    for (int e = 0; e < 8; ++e) wlane[e] = ((8 * kg + e) * (kTaps * a.cout) + j) * 4;
  }
  if constexpr (W != F32Weight::kPacked)
    wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(wt), 0, kTaps * a.cred * a.cout * 4, 0x00020000);
  auto weights = [&](bool next, int tap, float4 (&out)[2]) {
    if constexpr (W == F32Weight::kPacked) {
#pragma unroll
      for (int q = 0; q < 2; ++q) out[q] = *reinterpret_cast<const float4*>(wcc + ((tap + (next ? C::KS * kTaps : 0)) * 2 + q) * 256);
    } else {
      const int at = wbase + (next ? wchunk : 0) + tap * wtap;
      if constexpr (W == F32Weight::kRows) {
#pragma unroll
        for (int q = 0; q < 2; ++q) out[q] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(wbuf, wlane[0] + 16 * q, at, 0));
      } else {
        float got[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) got[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wbuf, wlane[e], at, 0));
        out[0] = make_float4(got[0], got[1], got[2], got[3]);
        out[1] = make_float4(got[4], got[5], got[6], got[7]);
      }
    }
  };
  constexpr int WDEPTH = 3;  // taps requested ahead
  static_assert(kTaps % WDEPTH == 0, "a chunk ends where the ring of requests began");
  float4 wq[WDEPTH][2];
#pragma unroll
  for (int d = 0; d < WDEPTH; ++d) weights(false, d, wq[d]);
  float4 v[BATCH];
  if (C::AHEAD) request(0, 0, v);
  for (int cc = 0; cc < ncc; cc += C::KS) {
    const bool more = cc + C::KS < ncc;  // of the workgroup; `ahead`: of this wavefront
    const bool ahead = cc + part < last;
    __syncthreads();  // every wave is done reading the previous chunk
    if constexpr (C::AHEAD) {
      stage(0, v);
    } else {
#pragma unroll
      for (int it0 = 0; it0 < ITERS; it0 += BATCH) {
        request(cc, it0, v);
        stage(it0, v);
      }
    }
    __syncthreads();
    if (C::AHEAD && more) request(cc + C::KS, 0, v);
    if (cc + part > last) continue;

    constexpr int ADEPTH = C::AHEAD ? 2 : 1;  // taps whose activations are held
    float4 af[ADEPTH][C::MS][2];
    auto activations = [&](int tap) {
#pragma unroll
      for (int ms = 0; ms < C::MS; ++ms) {
        af[tap % ADEPTH][ms][0] = *reinterpret_cast<const float4*>(lds + lbase[ms] + tap_off<C>(tap));
        af[tap % ADEPTH][ms][1] = *reinterpret_cast<const float4*>(lds + lbase[ms] + C::PLANE + tap_off<C>(tap));
      }
    };
    if (C::AHEAD) activations(0);
#pragma unroll
    for (int tap = 0; tap < kTaps; ++tap) {
      float4 wf[2] = {wq[tap % WDEPTH][0], wq[tap % WDEPTH][1]};
      if (tap + WDEPTH < kTaps || ahead) {
        const bool next = tap + WDEPTH >= kTaps;
        weights(next, next ? tap + WDEPTH - kTaps : tap + WDEPTH, wq[tap % WDEPTH]);
      }
      if constexpr (C::AHEAD) {
        if (tap + 1 < kTaps) activations(tap + 1);
        __builtin_amdgcn_sched_barrier(0);
      } else {
        activations(tap);
      }
      // the sub-tiles take turns, so consecutive MFMAs do not wait for one another's result
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float wv[4] = {wf[q].x, wf[q].y, wf[q].z, wf[q].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int ms = 0; ms < C::MS; ++ms) {
            const float4 act = af[tap % ADEPTH][ms][q];
            const float av[4] = {act.x, act.y, act.z, act.w};
            acc[ms] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[e], av[e], acc[ms], 0, 0, 0);
          }
        }
      }
      if constexpr (C::AHEAD) __builtin_amdgcn_sched_barrier(0);
    }
    wcc += C::KS * kTaps * 2 * 256;
    wbase += wchunk;
  }

  if constexpr (C::KS > 1) {
    float4* meet = reinterpret_cast<float4*>(lds);
    __syncthreads();  // the last chunks have been read
    if (part > 0) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        meet[(((part - 1) * C::WM + wave) * 4 + g) * 64 + lane] =
            make_float4(acc[0][4 * g], acc[0][4 * g + 1], acc[0][4 * g + 2], acc[0][4 * g + 3]);
    }
    __syncthreads();
    if (part > 0) return;
#pragma unroll
    for (int p = 1; p < C::KS; ++p)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 o = meet[(((p - 1) * C::WM + wave) * 4 + g) * 64 + lane];
        acc[0][4 * g] += o.x; acc[0][4 * g + 1] += o.y; acc[0][4 * g + 2] += o.z; acc[0][4 * g + 3] += o.w;
      }
  }
  // Accumulator register r of a lane is output channel 8 * (r / 4) + 4 * kg + r % 4 of the sub-tile's voxel j.
#pragma unroll
  for (int ms = 0; ms < C::MS; ++ms) {
    const int v = (wave * C::MS + ms) * 32 + j;
    const int tw = v % C::TW, th = (v / C::TW) % C::TH, td = v / (C::TW * C::TH);
    const int od = od0 + td, oh = oh0 + th, ow = ow0 + tw;
    if (od >= a.od || oh >= a.oh || ow >= a.ow) continue;
    float* yp = y + ((((int64_t)n * a.od + od) * a.oh + oh) * a.ow + ow) * a.cout + nb * 32;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int co = 8 * g + 4 * kg;
      float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
      if (bias != nullptr) b = *reinterpret_cast<const float4*>(bias + nb * 32 + co);
      *reinterpret_cast<float4*>(yp + co) =
          make_float4(acc[ms][4 * g] + b.x, acc[ms][4 * g + 1] + b.y, acc[ms][4 * g + 2] + b.z, acc[ms][4 * g + 3] + b.w);
    }
  }
#endif
}

// One thread per packed 16-byte piece: the 4 consecutive reduction channels of one (output channel, tap, k-slot, q).
__global__ void __launch_bounds__(256)
pack_f32_kernel(const float* __restrict__ w, float* __restrict__ packed, int cred, int taps_kh_kw, int kw, int flip, int64_t s_out,
                int64_t s_red, int64_t s_kd, int64_t s_kh, int64_t s_kw, int64_t pieces) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= pieces) return;
  const int lane = (int)(idx % 64), q = (int)(idx / 64 % 2);
  const int ncc = cred / kChunk;
  int tap, cc, nblk;
  if (pieces <= 0x7fffffff) {  // (64-bit divisions by numbers that are not constants would be most of the kernel)
    uint32_t r = (uint32_t)idx / 128u;
    tap = (int)(r % kTaps); r /= kTaps;
    cc = (int)(r % (uint32_t)ncc);
    nblk = (int)(r / (uint32_t)ncc);
  } else {
    int64_t r = idx / 128;
    tap = (int)(r % kTaps); r /= kTaps;
    cc = (int)(r % ncc);
    nblk = (int)(r / ncc);
  }
  const int co = nblk * 32 + (lane & 31);
  const int ci = cc * kChunk + (lane >> 5) * 8 + q * 4;
  if (flip) tap = kTaps - 1 - tap;
  const int tkw = tap % kw, tkh = (tap / kw) % (taps_kh_kw / kw), tkd = tap / taps_kh_kw;
  const float* src = w + co * s_out + ci * s_red + tkd * s_kd + tkh * s_kh + tkw * s_kw;
  *reinterpret_cast<float4*>(packed + idx * 4) = make_float4(src[0], src[s_red], src[2 * s_red], src[3 * s_red]);
}

template <typename C>
int launch(const MfmaConvArgs& a, const void* x, const void* w, F32Weight form, const void* bias, void* y, hipStream_t st) {
  const int tiles_d = (int)cdiv(a.od, C::TD), tiles_h = (int)cdiv(a.oh, C::TH), tiles_w = (int)cdiv(a.ow, C::TW);
  const int nblocks = a.cout / 32;
  const int64_t total = (int64_t)a.n * tiles_d * tiles_h * tiles_w * nblocks;
  if (total == 0) return SFH_OK;
  if (total > 0x7fffffffLL) return fail(SFH_ERR_UNSUPPORTED, "conv fp32: %lld workgroups exceed the grid limit", (long long)total);
#define SFH_LAUNCH_F32(W)                                                                                                         \
  hipLaunchKernelGGL((conv_f32_kernel<C, W>), dim3((unsigned)total), dim3(C::THREADS), 0, st, a, (const float*)x, (const float*)w, \
                     (const float*)bias, (float*)y, tiles_d, tiles_h, tiles_w, nblocks, (uint32_t)total)
  if (form == F32Weight::kRows) SFH_LAUNCH_F32(F32Weight::kRows);
  else if (form == F32Weight::kColumns) SFH_LAUNCH_F32(F32Weight::kColumns);
  else SFH_LAUNCH_F32(F32Weight::kPacked);
#undef SFH_LAUNCH_F32
  return check_launch("conv_f32_kernel");
}

// What a brick costs, us: the matrix pipe's time on the CU with the most workgroups (a wavefront's 216 MFMAs of a chunk take 5.76 us;
// workgroups that share a CU share its pipes), stretched by what a wavefront waits for, and the launches around it. The slopes and
// constants are fitted to sweeps of every brick over 16 problems of 32 to 512 channels on 4x8x8 to 64^3, within 15 % on each; the
// choice is the fastest brick or within 4 % of it. One brick of 32-voxel rows (512 voxels, or 128 below a workgroup per CU) -> this, us
// with the packing: 256 -> 256 channels at 8^3 124 -> 43, 512 -> 512 at 4x8x8 244 -> 82, 512 -> 256 at 8x16x16 240 -> 133, 128 -> 128 at 16^3 65 -> 38,
// 64 -> 32 at 16x32x32 35 -> 22 (parts of the reduction on CUs that had no workgroup), two samples of 64 -> 32 at 20x33x41 93 -> 66,
// 128 -> 64 at 30x17x40 180 -> 95, 256 -> 128 at 20x32x9 355 -> 159 (rows that were padding), 32 -> 32 at 8^3 20 -> 14, at 32^3 22.5 -> 21, 64 -> 64
// at 64^3 466 -> 454 (no register spilled). A reduction in eight parts was nowhere faster than in four. Relative error against 64 bits, e-7:
// 256 -> 256 at 8^3 13.6 -> 6.8, 128 -> 128 at 8x10x12 9.8 -> 4.9, 32 -> 32 at 16x16x24 5.1 -> 3.6. A pure function of the shape.
template <typename C>
double tile_us(const MfmaConvArgs& a, double slope, double fixed) {
  const int64_t wgs = (int64_t)a.n * cdiv(a.od, C::TD) * cdiv(a.oh, C::TH) * cdiv(a.ow, C::TW) * (a.cout / 32);
  const double waves = C::WM * C::KS / 4.0;
  return slope * 5.76 * (double)cdiv(wgs, kComputeUnits) * waves * C::MS * (double)cdiv(a.cred / kChunk, C::KS) + fixed;
}
double tile_us(const MfmaConvArgs& a, int c) {
  switch (c) {
    case 0: return tile_us<WholeTile>(a, 1.16, 20.);
    case 1: return tile_us<FlatTile<8>>(a, 1.245, 10.);
    case 2: return tile_us<FlatTile<16>>(a, 1.255, 10.);
    case 3: return tile_us<HalvedTile<8>>(a, 1.25, 10.);
    case 4: return tile_us<HalvedTile<16>>(a, 1.27, 10.);
    default: return tile_us<QuarteredTile>(a, 1.3, 9.5);
  }
}

// ---- weight gradient ---------------------------------------------------------------------------------------------
//   gw[co][tap][ci] = sum over output voxels v of gy[v][co] * x[v + tap - pad][ci]
// GEMM view (triton_conv3d/reduce_gemm.py:137-393): M = Cout, N = 27 x Cin, K = output voxels. One fp32 MFMA contracts
// TWO voxels and a lane supplies ONE value per operand: row operand gy[voxel 2s + kg][co = lane % 32], column operand
// x[that voxel + tap][ci = lane % 32] -- both are 32 consecutive floats of a channels-last row, so unlike the 16-bit
// kernel nothing has to be transposed. A workgroup owns the nine taps of one kd of a (32 co, 32 ci) block and a range of steps; a
// step is 64 voxels of the output, four rows of 16, whose gy and whose x rows with their halo lie in LDS as they lie in memory. Its twelve
// wavefronts are three kh x the rows; along W the taps share operands (a pair of kw = 2 is the next pair of kw = 0), so three
// MFMAs take three LDS reads. The rows meet in LDS before the slice is written. Split-K over the steps: fp32 partial slices
// [Cout][27][Cin] at fixed workspace slots, summed in fixed order afterwards (reduce_gemm.py:396-435) -- no float atomics,
// split count a pure function of shape.
//
// What bounds it is the matrix pipe, below 64^3 with the launch, the first step's trip to memory and the slices (36 KB a
// workgroup). Before, a lane's value per operand was a load of its own, 1.14 per MFMA: the CU's address path needs as long for one as
// its matrix pipes for an MFMA, and a workgroup owned all taps, three times the slices. us with the slice sum, before -> now:
// 32 -> 32 channels at 32^3 45.6 -> 34.0, at 16x24x20 29.4 -> 17.7, at 64^3 (two samples) 384 -> 293 (its MFMAs alone 188); 64 -> 64 at 64^3
// 752 -> 578; 128 -> 128 at 16^3 67 -> 49; 256 -> 256 at 8x16x16 114 -> 97; 512 -> 512 at 4x8x8 56.6 -> 52.
constexpr int kRowWaves = 4;                  // wavefronts that share the rows of a step
constexpr int kWgradThreads = 64 * 3 * kRowWaves;
typedef float Quad __attribute__((ext_vector_type(4), aligned(4)));  // the operands may be views 4 bytes off the 16-byte grid

// SEG: voxels of a step's rows, 16, or 8 with twice the rows where a row has no more.
template <int SEG>
__global__ void __launch_bounds__(kWgradThreads, 3)
wgrad_f32_kernel(WgradArgs a, const float* __restrict__ x, const float* __restrict__ gy, float* __restrict__ partial, int nsplit, int per,
                 int steps, int cibs) {
  constexpr int kRows = kRowWaves * (16 / SEG), kSeg = SEG;
  constexpr int kXSeg = kSeg + 2, kXPieces = (kRows + 2) * kXSeg * 8, kGyPieces = kRows * kSeg * 8;  // 16-byte pieces of 32 channels
  constexpr int kPiecesPer = (kXPieces + kGyPieces + kWgradThreads - 1) / kWgradThreads;
  constexpr int kStep = (kXPieces + kGyPieces) * 16, kMeet = (kRowWaves - 1) * 3 * 3 * 16 * 64 * 4;
  __shared__ __attribute__((aligned(16))) char lds[2 * kStep > kMeet ? 2 * kStep : kMeet];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = wave % 3, row = wave / 3;
  const int i = lane & 31, kg = lane >> 5;
  int b = blockIdx.x;
  const int split = b % nsplit; b /= nsplit;
  const int kd = b % 3; b /= 3;
  const int cib = b % cibs, cob = b / cibs;
  const int segs = (a.ow + kSeg - 1) / kSeg, row_tiles = (a.oh + kRows - 1) / kRows;
  const int begin = split * per, end = steps - begin < per ? steps : begin + per;
  // The range's steps in turn, segments first: positions are kept and moved on (all of it scalar), a thread's places in a step and
  // its offsets from the step's first voxel are constants.
  const int next_plane = begin / segs / row_tiles;
  int next_seg = begin % segs, next_tile = begin / segs % row_tiles;
  int next_od = next_plane % a.od, next_n = next_plane / a.od;
  int rr[kPiecesPer], vv[kPiecesPer];
  int64_t off[kPiecesPer];
  bool of_x[kPiecesPer], used[kPiecesPer];
#pragma unroll
  for (int k = 0; k < kPiecesPer; ++k) {
    const int p = k * kWgradThreads + tid, q = p - kXPieces;
    of_x[k] = p < kXPieces;
    used[k] = q < kGyPieces;
    rr[k] = of_x[k] ? p / (kXSeg * 8) - a.ph : q / (kSeg * 8);
    vv[k] = of_x[k] ? p / 8 % kXSeg - a.pw : q / 8 % kSeg;
    off[k] = of_x[k] ? ((int64_t)rr[k] * a.iw + vv[k]) * a.cin + cib * 32 + (p & 7) * 4
                     : ((int64_t)rr[k] * a.ow + vv[k]) * a.cout + cob * 32 + (p & 7) * 4;
  }
  struct Ahead { float4 piece[kPiecesPer]; int oh, ow; } ahead[2];
  auto request = [&](Ahead& o) {
    const int oh = next_tile * kRows, ow = next_seg * kSeg, id = next_od + kd - a.pd;
    const bool plane_in = (unsigned)id < (unsigned)a.id;
    const float* xs = x + ((((int64_t)next_n * a.id + id) * a.ih + oh) * a.iw + ow) * a.cin;
    const float* gs = gy + ((((int64_t)next_n * a.od + next_od) * a.oh + oh) * a.ow + ow) * a.cout;
#pragma unroll
    for (int k = 0; k < kPiecesPer; ++k) {
      const unsigned h = (unsigned)(rr[k] + oh), w = (unsigned)(vv[k] + ow);
      const bool in = used[k] && (of_x[k] ? plane_in && h < (unsigned)a.ih && w < (unsigned)a.iw : h < (unsigned)a.oh && w < (unsigned)a.ow);
      const float* src = (of_x[k] ? xs : gs) + off[k];
      const Quad got = *reinterpret_cast<const Quad*>(in ? src : x);  // (unconditional, masked afterwards: nothing waits for it here)
      o.piece[k] = in ? make_float4(got.x, got.y, got.z, got.w) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    o.oh = oh; o.ow = ow;
    if (++next_seg == segs) {
      next_seg = 0;
      if (++next_tile == row_tiles) {
        next_tile = 0;
        if (++next_od == a.od) { next_od = 0; ++next_n; }
      }
    }
  };

  f32x16_t sums[2][3];  // of the even and the odd steps: against 64 bits 1.7e-7 at 32^3 instead of 2.1e-7 in one chain
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) sums[h][t][r] = 0.f;
  // Two steps ahead: a wavefront requests behind its MFMAs, where the addresses cost the matrix pipe nothing.
  auto run = [&](Ahead& o, f32x16_t (&acc)[3], char* tile, bool more) {
#pragma unroll
    for (int k = 0; k < kPiecesPer; ++k) {
      const int p = k * kWgradThreads + tid;
      if (p < kXPieces + kGyPieces) *reinterpret_cast<float4*>(tile + p * 16) = o.piece[k];
    }
    __syncthreads();  // the other phase was read before the barrier of the step behind it
#pragma unroll
    for (int rw = row; rw < row + kRows; rw += kRowWaves) {
      if (o.oh + rw >= a.oh) break;
      const int left = a.ow - o.ow;  // voxels of the row from the step's first on
      const float* xr = reinterpret_cast<const float*>(tile) + ((rw + kh) * kXSeg + kg) * 32 + i;
      const float* gr = reinterpret_cast<const float*>(tile + kXPieces * 16) + (rw * kSeg + kg) * 32 + i;
      float even = xr[0];
#pragma unroll
      for (int u = 0; u < kSeg / 2; ++u) {
        if (2 * u >= left) break;
        const float g = gr[u * 64], odd = xr[u * 64 + 32], after = xr[u * 64 + 64];
        // a voxel that belongs to no output of the row meets a zero of gy: it must be zero itself, 0 x infinity is not
        const bool in = 2 * u + kg < left;
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(g, in ? even : 0.f, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(g, in ? odd : 0.f, acc[1], 0, 0, 0);
        acc[2] = __builtin_amdgcn_mfma_f32_32x32x2f32(g, in ? after : 0.f, acc[2], 0, 0, 0);
        even = after;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) request(o);
  };
  if (begin < end) request(ahead[0]);
  if (begin + 1 < end) request(ahead[1]);
  for (int step = begin; step < end; step += 2) {
    run(ahead[0], sums[0], lds, step + 2 < end);
    if (step + 1 < end) run(ahead[1], sums[1], lds + kStep, step + 3 < end);
  }

  f32x16_t(&acc)[3] = sums[0];
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] += sums[1][t][r];
  __syncthreads();  // the tiles are not read any more
  float* meet = reinterpret_cast<float*>(lds);
  if (row > 0) {
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) meet[((((row - 1) * 3 + kh) * 3 + t) * 16 + r) * 64 + lane] = acc[t][r];
  }
  __syncthreads();
  if (row > 0) return;
  // result register r of a lane: column ci = lane % 32, row co = 8 * (r / 4) + 4 * kg + r % 4
  float* dst = partial + (int64_t)split * a.cout * kTaps * a.cin + ((int64_t)cob * 32 * kTaps + kd * 9 + kh * 3) * a.cin + cib * 32 + i;
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int co = 8 * (r / 4) + 4 * kg + (r % 4);
      float sum = acc[t][r];
#pragma unroll
      for (int q = 0; q < kRowWaves - 1; ++q) sum += meet[(((q * 3 + kh) * 3 + t) * 16 + r) * 64 + lane];
      dst[((int64_t)co * kTaps + t) * a.cin] = sum;
    }
}

}  // namespace

bool f32_conv_supported(const MfmaConvArgs& a) {
  if (a.kd != 3 || a.kh != 3 || a.kw != 3) return false;
  if (a.cred % kChunk != 0 || a.cout % 32 != 0) return false;
  if (a.pd < 0 || a.ph < 0 || a.pw < 0 || a.pd > 2 || a.ph > 2 || a.pw > 2) return false;
  if (a.n < 1 || a.od < 1 || a.oh < 1 || a.ow < 1) return false;
  return true;
}

size_t f32_conv_packed_weight_bytes(const MfmaConvArgs& a) { return align_up((size_t)a.cout * a.cred * kTaps * 4, 256); }

int f32_pack_weight(const MfmaConvArgs& a, const void* w, int64_t s_out, int64_t s_red, int64_t s_kd, int64_t s_kh, int64_t s_kw, int flip,
                    void* packed, hipStream_t st) {
  const int64_t pieces = (int64_t)a.cout * a.cred * kTaps / 4;
  if (pieces <= 0) return SFH_OK;
  hipLaunchKernelGGL(pack_f32_kernel, dim3((unsigned)cdiv(pieces, 256)), dim3(256), 0, st, (const float*)w, (float*)packed, a.cred,
                     a.kh * a.kw, a.kw, flip, s_out, s_red, s_kd, s_kh, s_kw, pieces);
  return check_launch("pack_f32_kernel");
}

// The brick of the least time.
static int choose_brick(const MfmaConvArgs& a) {
  int best = 0;
  for (int c = 1; c < 6; ++c)
    if (tile_us(a, c) < tile_us(a, best)) best = c;
  return best;
}

// A channels-last weight is read where it lies: no packing launch, and where the weights are much of what a launch reads the packed
// ones were written and read once more. Of 70 drawn problems of 32 to 512 channels, us, packed -> as it lies: 32 -> 32 at 32^3 22.7 -> 18.5 and
// 21.6 -> 18.7 (data gradient), at 8^3 13.9 -> 10.8 and 14.1 -> 11.5, 128 -> 128 at 16^3 39.9 -> 32.5 and 38.3 -> 33.2, 512 -> 512 at
// 4x8x8 100.7 -> 62.6 and 100.2 -> 63.4, at 16^3 486 -> 415 and 484 -> 429, 64 -> 64 at 64^3 451 -> 417 and 451 -> 425. The line: where many
// workgroups of few wavefronts a sub-tile share a CU, the data gradient's eight loads a tap are what it waits for (packed / as it lies: 64
// channels at 63x9x30 45.4 / 52.2, at 33x25x16 61.8 / 68.7, of 128 channels level, of 256 276 / 263), and a forward with fewer
// produced channels than it reads shares its lines with few (two samples of 64 -> 32 at 20x33x41 65.8 / 71.7, 256 -> 128 at 20x32x9 158.5 / 163.2).
F32Weight f32_weight_form(const MfmaConvArgs& a, const void* w, const int64_t w_stride[5], bool dgrad) {
  const int64_t inner = dgrad ? a.cout : a.cred;  // Cin
  const bool dense = w_stride[1] == 1 && w_stride[4] == inner && w_stride[3] == 3 * inner && w_stride[2] == 9 * inner && w_stride[0] == 27 * inner;
  if (!dense || (int64_t)a.cout * a.cred * kTaps > 0x1fffffffLL) return F32Weight::kPacked;
  const int brick = choose_brick(a);
  const int64_t bricks = (int64_t)a.n * cdiv(a.od, 2) * cdiv(a.oh, 2) * cdiv(a.ow, brick == 4 ? 16 : 8);
  const bool crowded = brick >= 4 && bricks * (a.cout / 32) > 3 * kComputeUnits;
  if (dgrad) return crowded && a.cred <= 128 ? F32Weight::kPacked : F32Weight::kColumns;
  return (crowded && a.cout < a.cred) || (reinterpret_cast<uintptr_t>(w) & 15u) != 0 ? F32Weight::kPacked : F32Weight::kRows;
}

int f32_conv(const MfmaConvArgs& a, const void* x, const void* w, F32Weight form, const void* bias, void* y, hipStream_t st) {
  switch (choose_brick(a)) {
    case 0: return launch<WholeTile>(a, x, w, form, bias, y, st);
    case 1: return launch<FlatTile<8>>(a, x, w, form, bias, y, st);
    case 2: return launch<FlatTile<16>>(a, x, w, form, bias, y, st);
    case 3: return launch<HalvedTile<8>>(a, x, w, form, bias, y, st);
    case 4: return launch<HalvedTile<16>>(a, x, w, form, bias, y, st);
    default: return launch<QuarteredTile>(a, x, w, form, bias, y, st);
  }
}

}  // namespace sfh

namespace sfh {

// Steps of a weight gradient, and how many a workgroup takes: about one workgroup per CU over the blocks and kd, and no more slices
// than the longest range asks for.
static int wgrad_segment(const WgradArgs& a) { return a.ow <= 8 ? 8 : 16; }
static int64_t wgrad_steps(const WgradArgs& a) {
  const int seg = wgrad_segment(a);
  return (int64_t)a.n * a.od * cdiv(a.oh, kRowWaves * (16 / seg)) * cdiv(a.ow, seg);
}

static int64_t wgrad_per(const WgradArgs& a) {
  const int64_t units = 3 * (int64_t)(a.cout / 32) * (a.cin / 32), steps = wgrad_steps(a);
  const int64_t s = kComputeUnits / units;
  return s > 1 ? cdiv(steps, s) : steps;
}

bool f32_wgrad_supported(const WgradArgs& a) {
  // places along a row and a column and the count of steps are 32-bit, the offsets they make 64-bit
  constexpr int64_t kLast = 0x7fffffffLL - 64;
  if (a.n < 1 || a.od < 1 || a.oh > kLast || a.ow > kLast || a.ih > kLast || a.iw > kLast || wgrad_steps(a) > 0x7fffffffLL) return false;
  return a.cin % 32 == 0 && a.cout % 32 == 0 && a.n >= 1 && a.od >= 1 && a.oh >= 1 && a.ow >= 1 && a.pd >= 0 && a.ph >= 0 && a.pw >= 0;
}

int f32_wgrad_splits(const WgradArgs& a) { return (int)cdiv(wgrad_steps(a), wgrad_per(a)); }

size_t f32_wgrad_workspace_bytes(const WgradArgs& a) {
  return align_up((size_t)f32_wgrad_splits(a) * a.cout * kTaps * a.cin * sizeof(float), 256);
}

int f32_wgrad(const WgradArgs& a, const void* x, const void* gy, void* gw, void* workspace, hipStream_t st) {
  const int nsplit = f32_wgrad_splits(a);
  const int cibs = a.cin / 32, cobs = a.cout / 32;
  const int64_t total = (int64_t)nsplit * 3 * cibs * cobs;
  if (total > 0x7fffffffLL) return fail(SFH_ERR_UNSUPPORTED, "conv fp32 wgrad: too many workgroups");
  float* slices = (float*)(nsplit == 1 ? gw : workspace);  // one slice is the gradient itself
  const int per = (int)wgrad_per(a), steps = (int)wgrad_steps(a);
  if (wgrad_segment(a) == 8)
    hipLaunchKernelGGL(wgrad_f32_kernel<8>, dim3((unsigned)total), dim3(kWgradThreads), 0, st, a, (const float*)x, (const float*)gy, slices,
                       nsplit, per, steps, cibs);
  else
    hipLaunchKernelGGL(wgrad_f32_kernel<16>, dim3((unsigned)total), dim3(kWgradThreads), 0, st, a, (const float*)x, (const float*)gy, slices,
                       nsplit, per, steps, cibs);
  if (int rc = check_launch("wgrad_f32_kernel")) return rc;
  if (nsplit == 1) return SFH_OK;
  return sum_slices(SFH_FP32, (const float*)workspace, gw, (int64_t)a.cout * kTaps * a.cin, nsplit, st);
}

}  // namespace sfh
