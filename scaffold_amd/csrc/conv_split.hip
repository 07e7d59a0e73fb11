// MFMA implicit-GEMM convolution for the small volumes of a deep network level (3x3x3, stride 1, bf16 / fp16, 64 or
// more reduction channels): forward and data gradient (GEMM view as triton_conv3d/gather_gemm.py:112-341: M = output
// voxels, N = produced channels, K = taps x reduction channels).
//
// A level of 16 x 32 x 32 voxels or fewer has too few 256-voxel bricks to give every CU a workgroup unless the
// reduction is cut into slices, and slices that meet in memory cost fp32 partial tiles written and read plus a launch
// of their own. Here the reduction is cut INSIDE the workgroup:
//
//   * A workgroup owns a brick of only 64 output voxels (2 x 4 x 8, 4 x 4 x 4 or 2 x 2 x 16) and 64 produced channels -- four 32-voxel x
//     32-channel accumulator blocks -- so even a level of 2048 voxels has 32 x Cout/64 of them; where those would leave
//     half of the CUs idle, 32 produced channels.
//   * Its four wavefronts split the REDUCTION, not the voxels: a round stages the halo bricks of R 32-channel chunks
//     (R = 4, or 2 when there are only two) side by side in LDS, and every wavefront runs all four accumulator blocks
//     over its own share -- one chunk each, or half a chunk's k-steps each when R = 2. A weight fragment then feeds
//     four MFMAs (two in the brick kernel at this size), every fragment of the workgroup is fetched by exactly one
//     wavefront (the brick kernel's four wavefronts fetch the same ones), and the chunks of a round are staged with
//     one trip to memory instead of one per chunk.
//     (In the place of the bricks' slices the shares are those of the slices, so that the sums are too: SplitForm.)
//   * At the end the wavefronts' partial accumulators meet in LDS: wavefront u collects block u from the other three
//     in wavefront order (a fixed order: the same bits on every run), adds the bias, rounds once, leaves the GroupNorm
//     records of what it stores (gn_stats.hpp) and writes 16-byte pieces.
//
// LDS layout per chunk as in conv_mfma.hip (four 16-byte channel planes, 64 bytes mod 256 apart); chunk slots are a
// further 16 bytes apart so that the staging writes of one voxel's pieces fall into different banks.
// The data gradient runs this kernel with the weight packed transposed and tap-flipped and padding k-1-p
// (triton_conv3d/bwd_data.py:344-363). Launch geometry is a pure function of the shape.
#include "conv_mfma.hpp"
#include "mma.hpp"
#include "gn_stats.hpp"

namespace sfh {
namespace {

constexpr int kChunk = 32;
constexpr int kBrickVoxels = 64;
constexpr int MS = 2, kBlocks = 2;                              // accumulator blocks: voxel halves x at most two channel blocks
constexpr int TAPS = 27, NIT = TAPS * 2, FRAG = 512;
// An output brick of 64 voxels: half ms is its voxels 32 ms .. 32 ms + 31 in memory order. PITCH: of its rows in LDS where a workgroup has one
// channel block. LDS of a chunk's brick, NSUB channel blocks to a workgroup: row pitch, channel plane (64 modulo 256), chunk slot. A fragment
// read covers sixteen voxels at a time: two rows of 8, 128 modulo 256 apart, four of 4, 64 apart, or one of 16 share no bank. Two workgroups to a
// CU (NSUB = 2) have no room for that pitch, and do not miss it; alone on its CU one reads 5 % faster (13.8 -> 13.1 us at 256 -> 256, 8x16x16).
template <int TD_, int TH_, int TW_, int PITCH_>
struct Shape {
  static constexpr int TD = TD_, TH = TH_, TW = TW_, PITCH = PITCH_;
  static constexpr int BD = TD + 2, BH = TH + 2, BW = TW + 2, BV = BD * BH * BW;  // with the halo
  static_assert(TD * TH * TW == kBrickVoxels && PITCH >= BW * 16, "two blocks of 32 voxels");
};
template <typename S, int NSUB>
struct Brick {
  static constexpr int ROW = NSUB == 1 ? S::PITCH : S::BW * 16;
  static constexpr int PLANE = ((S::BD * S::BH * ROW - 64 + 255) / 256) * 256 + 64;
  static constexpr int SLOT = 4 * PLANE + 16;
  // byte offset of a brick voxel in its plane (dense rows: not by row and column, which is 130 instructions a round of four chunks and 1 % of the time)
  static __device__ __forceinline__ int at(int vox) { return ROW == S::BW * 16 ? vox * 16 : vox / S::BW * ROW + vox % S::BW * 16; }
  // byte offset of (tap, k-step) relative to a lane's voxel at tap (0, 0, 0)
  static constexpr int tap_off(int tap) { return ((tap / 9) * S::BH + (tap / 3) % 3) * ROW + tap % 3 * 16; }
};

// R: chunks per round. PAIR: the input is two tensors whose channels follow each other (the first `c_first` in x, the
// rest in x1). Independently, a non-null y1 splits the OUTPUT the same way. chunk_stride: 1, a round's slots are R chunks that follow each other;
// more, a slot's rounds are that many that do. FORM, of launches that add as the bricks' slices do (split_rule):
//   kApart   the reduction is two rounds, and the first one's sums are set aside. They want 32 registers more: one workgroup to a CU, which the
//            brick's LDS leaves room for anyway (with two 11 to 17 registers were spilled and every other launch of one block took 0.5 us longer).
//   kHalves  (R = 2, one block) a wavefront has one of the two voxel halves and all 32 channels of its chunks, in place of both halves and 16.
//   kPairs   (R = 4, two blocks) a wavefront has one of the two blocks and two chunks a round: every weight still goes to one wavefront
//            only, which the halves' do not.
enum SplitForm { kOrdinary, kApart, kHalves, kPairs };
template <typename T, typename S, int R, int NSUB, bool PAIR, SplitForm FORM = kOrdinary>
__global__ void __launch_bounds__(256, FORM == kApart ? 1 : 2)
conv_split_kernel(MfmaConvArgs a, const T* __restrict__ x, const T* __restrict__ wp, const T* __restrict__ bias, T* __restrict__ y,
                  int tiles_d, int tiles_h, int tiles_w, int nblocks, uint32_t total, GnPartialOut gn, const T* __restrict__ x1,
                  T* __restrict__ y1, int c_first, int chunk_stride) {
  using B = Brick<S, NSUB>;
  constexpr int TD = S::TD, TH = S::TH, TW = S::TW, BH = S::BH, BW = S::BW;
  constexpr int PLANE = B::PLANE, SLOT = B::SLOT;
  constexpr bool APART = FORM == kApart, HALVES = FORM == kHalves, PAIRS = FORM == kPairs, WHOLE = R == 4 || HALVES;  // WHOLE: both k-steps of a tap
  static_assert(FORM == kOrdinary || (NSUB == (PAIRS ? 2 : 1) && R == (HALVES ? 2 : 4)), "forms");
  constexpr int MSW = HALVES ? 1 : MS, NSW = PAIRS ? 1 : NSUB, CHW = PAIRS ? 2 : 1;  // voxel halves, blocks and chunks of a wavefront
  constexpr int ROUNDS = APART ? 2 : 1;
  constexpr int RED_BYTES = ROUNDS * MS * NSUB * 3 * 4096;  // every block from the three wavefronts that do not own it
  constexpr int LDS = R * SLOT > RED_BYTES ? R * SLOT : RED_BYTES;
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int j = lane & 31, kg = lane >> 5;

  uint32_t t = xcd_remap(blockIdx.x, total);
  const int nb = t % nblocks; t /= nblocks;
  const int tw_i = t % tiles_w; t /= tiles_w;
  const int th_i = t % tiles_h; t /= tiles_h;
  const int td_i = t % tiles_d;
  const int n = t / tiles_d;
  const int od0 = td_i * TD, oh0 = th_i * TH, ow0 = tw_i * TW;

  // This wavefront's share of a round: chunk slot `slot`; with R = 2 also one of the two k-steps of every tap, or one of the voxel halves.
  const int slot = PAIRS ? wave & ~1 : R == 4 ? wave : wave >> 1;
  const int khalf = WHOLE ? 0 : wave & 1, half = HALVES ? wave & 1 : 0, block = PAIRS ? wave & 1 : 0;
  constexpr int NITC = WHOLE ? NIT : TAPS, NITS = CHW * NITC;  // iterations of a wavefront per chunk, per round
  constexpr int WSTEP = WHOLE ? FRAG : 2 * FRAG;
  int abase[MSW];  // LDS byte address of the lane's voxel of block row ms at tap (0, 0, 0), in its k-half plane
#pragma unroll
  for (int ms = 0; ms < MSW; ++ms) {
    const int v = (half + ms) * 32 + j, tw = v % TW, th = v / TW % TH, td = v / (TW * TH);
    abase[ms] = slot * SLOT + (kg + 2 * khalf) * PLANE + (td * BH + th) * B::ROW + tw * 16;
  }
  auto a_off = [](int k) constexpr { return k / NITC * SLOT + (WHOLE ? B::tap_off(k % NITC / 2) + (k % 2) * 2 * PLANE : B::tap_off(k)); };

  f32x16_t acc[MSW][NSW], first[MSW];  // first: the first round's sums, where they are chains apart
#pragma unroll
  for (int ms = 0; ms < MSW; ++ms)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
#pragma unroll
      for (int ns = 0; ns < NSW; ++ns) acc[ms][ns][r] = 0.f;
      first[ms][r] = 0.f;
    }

  const int ncc = a.cred / kChunk;
  const int id0 = od0 - a.pd, ih0 = oh0 - a.ph, iw0 = ow0 - a.pw;
  constexpr int PIECES = S::BV * 4 * R;
  constexpr int ITERS = (PIECES + 255) / 256;
  constexpr int WDEPTH = 16 / NSW;  // weight fragments (per output block) in flight per wavefront
  const int64_t wns = (int64_t)ncc * (NIT * FRAG);  // next 32-channel output block

  for (int c0 = 0; c0 < ncc; c0 += R) {
    // The wavefront's first weight fragments are requested before the bricks are staged: they depend on nothing in LDS.
    const int stride = NSUB == 1 ? chunk_stride : 1;  // (two blocks have no registers for it)
    const int first_chunk = PAIRS ? c0 / 2 : stride == 1 ? c0 : c0 / R;  // slot 0's
    auto chunk_of = [&](int q) { return PAIRS ? first_chunk + (q >> 1) * (ncc >> 1) + (q & 1) : first_chunk + q * stride; };
    const T* wcc = wp + ((int64_t)(nb * NSUB + block) * ncc + chunk_of(slot)) * (NIT * FRAG) + khalf * FRAG + lane * 8;
    uint4 wq[NITS][NSW];  // fully unrolled: every slot is its own register set, live for WDEPTH iterations
#pragma unroll
    for (int k = 0; k < WDEPTH; ++k)
#pragma unroll
      for (int ns = 0; ns < NSW; ++ns) wq[k][ns] = *reinterpret_cast<const uint4*>(wcc + ns * wns + k * WSTEP);
    __syncthreads();  // every wavefront is done reading the previous round
    {
      // A voxel's 4 R pieces (R chunks of 4) are consecutive threads: 64 R contiguous bytes when the chunks lie in one tensor.
      uint4 v[ITERS];
#pragma unroll
      for (int u = 0; u < ITERS; ++u) {
        const int p = u * 256 + tid;
        const int q = p % (4 * R), vox = p / (4 * R);
        const int cc = chunk_of(q >> 2), piece = q & 3;
        const int bw = vox % BW, bh = (vox / BW) % BH, bd = vox / (BW * BH);
        const int id = id0 + bd, ih = ih0 + bh, iw = iw0 + bw;
        const bool in = p < PIECES && (unsigned)id < (unsigned)a.id && (unsigned)ih < (unsigned)a.ih && (unsigned)iw < (unsigned)a.iw;
        int row = a.cred, ch = cc * kChunk;
        const T* xb = x;
        if constexpr (PAIR) {
          const bool second = ch >= c_first;
          row = second ? a.cred - c_first : c_first;
          xb = second ? x1 : x;
          ch = second ? ch - c_first : ch;
        }
        v[u] = make_uint4(0, 0, 0, 0);
        if (in) v[u] = *reinterpret_cast<const uint4*>(xb + ((((int64_t)n * a.id + id) * a.ih + ih) * a.iw + iw) * row + ch + piece * 8);
      }
#pragma unroll
      for (int u = 0; u < ITERS; ++u) {
        const int p = u * 256 + tid;
        const int q = p % (4 * R), vox = p / (4 * R);
        if (p < PIECES) *reinterpret_cast<uint4*>(lds + (q >> 2) * SLOT + (q & 3) * PLANE + B::at(vox)) = v[u];
      }
    }
    __syncthreads();

    // Software pipeline over the wavefront's iterations: the weight fragments of iteration k + WDEPTH and the
    // activation fragments of iteration k + 1 are requested between the MFMAs of iteration k, one behind each.
    uint4 aq[2][MSW];
#pragma unroll
    for (int ms = 0; ms < MSW; ++ms) aq[0][ms] = *reinterpret_cast<const uint4*>(lds + abase[ms] + a_off(0));
#pragma unroll
    for (int k = 0; k < NITS; ++k) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < MSW * NSW; ++m) {
        const int ms = m / NSW, ns = m % NSW;
        acc[ms][ns] = Mma32<T>::run(wq[k][ns], aq[k & 1][ms], acc[ms][ns]);
        __builtin_amdgcn_sched_barrier(0);
        if (m < NSW && k + WDEPTH < NITS) wq[k + WDEPTH][m] = *reinterpret_cast<const uint4*>(wcc + m * wns + (k + WDEPTH) * WSTEP);
        if (NSW == 1 ? true : m >= NSW) {
          constexpr int first = NSW == 1 ? 0 : NSW;
          if (k + 1 < NITS) aq[(k + 1) & 1][m - first] = *reinterpret_cast<const uint4*>(lds + abase[m - first] + a_off(k + 1));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (APART) {
      if (c0 == 0) {
#pragma unroll
        for (int ms = 0; ms < MSW; ++ms)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            first[ms][r] = acc[ms][0][r];
            acc[ms][0][r] = 0.f;
          }
      }
    }
  }

  // The four partial results of every block meet in LDS, those of the first round before those of the second where they are apart: wavefront
  // u collects block u = ms * NSUB + ns.
  __syncthreads();  // the bricks are not read any more
  float4* red = reinterpret_cast<float4*>(lds);
  auto mine_of = [&](int round, int u) -> const f32x16_t& { return APART && round == 0 ? first[u / NSUB] : acc[u / NSUB % MSW][u % NSUB % NSW]; };
  auto send = [&](int place, const f32x16_t& v) {
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) red[(place * 4 + r4) * 64 + lane] = make_float4(v[4 * r4], v[4 * r4 + 1], v[4 * r4 + 2], v[4 * r4 + 3]);
  };
  auto receive = [&](int place) {
    f32x16_t v;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const float4 e = red[(place * 4 + r4) * 64 + lane];
      v[4 * r4] = e.x; v[4 * r4 + 1] = e.y; v[4 * r4 + 2] = e.z; v[4 * r4 + 3] = e.w;
    }
    return v;
  };
  if constexpr (HALVES) {
    send(half * 2 + slot, acc[0][0]);
  } else if constexpr (PAIRS) {
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) send((ms * NSUB + block) * 2 + (slot >> 1), acc[ms][0]);
  } else {
#pragma unroll
  for (int round = 0; round < ROUNDS; ++round)
#pragma unroll
    for (int u = 0; u < MS * NSUB; ++u) {
      if (u != wave) {
        const int from = wave < u ? wave : wave - 1;  // this wavefront's place among block u's three senders
        send((round * MS * NSUB + u) * 3 + from, mine_of(round, u));
      }
    }
  }
  __syncthreads();
  f32x16_t tot;
#pragma unroll
  for (int r = 0; r < 16; ++r) tot[r] = 0.f;
  if constexpr (HALVES || PAIRS) {
    if (wave < MS * NSUB) {
      tot = receive(wave * 2);
      const f32x16_t second = receive(wave * 2 + 1);
#pragma unroll
      for (int r = 0; r < 16; ++r) tot[r] += second[r];
    }
  } else
#pragma unroll
  for (int u = 0; u < MS * NSUB; ++u) {
    if (u == wave) {
      // wavefronts 0, 1, 2, 3 in that order, this one's own share from its registers
#pragma unroll
      for (int round = 0; round < ROUNDS; ++round)
#pragma unroll
        for (int src = 0; src < 4; ++src) {
          f32x16_t part;
          if (src == u) {
            part = mine_of(round, u);
          } else {
            part = receive((round * MS * NSUB + u) * 3 + (src < u ? src : src - 1));
          }
          if (round == 0 && src == 0) tot = part;
          else
#pragma unroll
            for (int r = 0; r < 16; ++r) tot[r] += part[r];
        }
    }
  }

  // Epilogue of block (ms, ns) = (wave / NSUB, wave % NSUB). Accumulator register r of a lane is output channel
  // 8 * (r / 4) + 4 * kg + r % 4 of voxel j of the block row; the two lanes of a voxel trade runs so that each stores
  // two 16-byte pieces.
  const int ms_o = wave / NSUB, ns_o = wave % NSUB;
  const bool owns = MS * NSUB == 4 || wave < MS * NSUB;
  const int own_v = ms_o * 32 + j;
  const int od = od0 + own_v / (TW * TH), oh = oh0 + own_v / TW % TH, ow = ow0 + own_v % TW;
  const bool inside = owns && od < a.od && oh < a.oh && ow < a.ow;
  const int64_t vox = (((int64_t)n * a.od + od) * a.oh + oh) * a.ow + ow;
  const int ch = (nb * NSUB + ns_o) * 32;
  T* yp = y + vox * a.cout + ch;
  if (y1 != nullptr) yp = ch >= c_first ? y1 + vox * (a.cout - c_first) + (ch - c_first) : y + vox * c_first + ch;
  uint32_t run[4][2];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    float b0 = 0.f, b1 = 0.f, b2 = 0.f, b3 = 0.f;
    if (bias != nullptr) {
      const T* bp = bias + ch + 8 * g + 4 * kg;
      b0 = to_float(bp[0]); b1 = to_float(bp[1]); b2 = to_float(bp[2]); b3 = to_float(bp[3]);
    }
    run[g][0] = Mma32<T>::pack2(tot[4 * g] + b0, tot[4 * g + 1] + b1);
    run[g][1] = Mma32<T>::pack2(tot[4 * g + 2] + b2, tot[4 * g + 3] + b3);
  }
  RunSums mine;
  mine.clear();
  if (gn.part != nullptr) mine.template add<T>(run, inside, true);
  uint4 piece[2];
  trade_channel_runs(run, piece);  // all lanes take part, also those of voxels past the edge
  if (inside) {
    *reinterpret_cast<uint4*>(yp + 8 * kg) = piece[0];
    *reinterpret_cast<uint4*>(yp + 16 + 8 * kg) = piece[1];
  }
  if (gn.part != nullptr) {
    // this wavefront's sums belong to channel block ns_o; for the other block it counts nothing
    RunSums rs[NSUB];
#pragma unroll
    for (int ns = 0; ns < NSUB; ++ns) {
      const bool own = owns && ns == ns_o;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        rs[ns].s1[g] = own ? mine.s1[g] : 0.f;
        rs[ns].s2[g] = own ? mine.s2[g] : 0.f;
        rs[ns].k[g] = mine.k[g];
      }
      rs[ns].cnt = own ? mine.cnt : 0.f;
    }
    __syncthreads();  // every wavefront has collected its block: the LDS is free
    constexpr int SPAN = 32 * NSUB;
    const int per_tile = gn.cg > SPAN ? gn.cg / SPAN : 1;  // workgroups that share a group of this tile
    const int tile = (td_i * tiles_h + th_i) * tiles_w + tw_i;
    write_group_partials<4, NSUB>(rs, reinterpret_cast<float*>(lds), gn, n, tile * per_tile + nb % per_tile, nb * SPAN, tid);
  }
}

typedef Shape<2, 4, 8, 384> Flat;    // 240 voxels with the halo
typedef Shape<4, 4, 4, 192> Cube;    // 216
typedef Shape<2, 2, 16, 288> Rows;   // 288

int64_t tiles_of(const MfmaConvArgs& a, int shape) {
  static const int log2[3][3] = {{1, 2, 3}, {2, 2, 2}, {1, 1, 4}};
  auto parts = [](int64_t extent, int log2) { return (extent + (1 << log2) - 1) >> log2; };
  return a.n * parts(a.od, log2[shape][0]) * parts(a.oh, log2[shape][1]) * parts(a.ow, log2[shape][2]);
}

// What a launch of `pairs` pairs of channel blocks takes, in hundredths of a us, fitted as the brick kernel's (conv_mfma.hip, brick_time) to 453
// problems on odd levels: 7 % (rms). Up to half a round is dealt as single blocks.
int64_t split_time(int64_t pairs, int chunks) {
  const int64_t rounds = cdiv(pairs, kComputeUnits);
  return pairs <= kComputeUnits / 2 ? 420 + 100 * chunks
                                    : 400 + 60 * rounds + chunks * (99 * rounds * kComputeUnits + 54 * pairs) / kComputeUnits;
}

// The brick that is done soonest: a volume of odd extents takes fewer of one shape than of another, and a round of workgroups less is what
// that mostly saves. At equal counts 4x4x4 takes 0.99 of the time of 2x4x8 (its halo is smaller) and 2x2x16 1.06. A voxel's sums do not depend on
// the brick. us, 2x4x8 / 4x4x4 / 2x2x16: 512 -> 512 at 12x10x14 50.0 / 49.0 / 38.9 (288, 288 and 240 pairs), 256 -> 512 28.0 / 27.2 / 22.9, 128 -> 128 at 19x17x58
// 29.6 / 24.4 / 26.8, 512 -> 512 at 7x9x4 22.1 / 19.5 / 32.2, 256 -> 256 at 8x16x16 13.4 / 12.8 / 13.5; over 136 odd levels the choice is 4.4 % ahead of 2x4x8.
int split_shape(const MfmaConvArgs& a) {
  static const int weight[3] = {100, 99, 106};
  const int pair = a.cout / (32 * kBlocks), chunks = a.cred / kChunk;
  int best = 0;
  int64_t least = 0;
  for (int s = 0; s < 3; ++s) {
    const int64_t time = split_time(tiles_of(a, s) * pair, chunks) * weight[s];
    if (s > 0 && time >= least) continue;
    least = time;
    best = s;
  }
  return best;
}

int64_t split_tiles(const MfmaConvArgs& a) { return tiles_of(a, split_shape(a)); }

// One channel block per workgroup where pairs would leave half of the CUs idle: each workgroup then has half the weights to fetch and
// half the MFMAs (the bits of the output do not depend on it). us, caches warm / cold: 256 -> 256 at 8x16x16 16.0 / 18.9 -> 13.1 / 16.2,
// 128 -> 256 10.2 / 13.8 -> 8.7 / 11.4, 256 -> 256 at 5x7x9 (two samples) 15.0 / 20.5 -> 11.8 / 15.1. With 129 to 256 pairs it loses:
// 256 -> 256 at 10x16x16 16.5 / 22.0 -> 19.2 / 22.2, at 16^3 17.6 -> 19.6 (each CU fetches the same weights and stages twice the bricks).
int split_blocks(int64_t tiles, int cout) { return tiles * (cout / (32 * kBlocks)) <= kComputeUnits / 2 ? 1 : kBlocks; }

// Whether a problem is this kernel's, and how many of the bricks' slices it adds like (0: in its own order): see mfma_conv_split_applies.
struct SplitRule { bool use; int slices; };
SplitRule split_rule(const MfmaConvArgs& a, bool records);

// A launch: its brick (0: 2x4x8, 1: 4x4x4, 2: 2x2x16), their number and the channel blocks of a workgroup. GroupNorm records are sums of bricks: a
// launch that leaves them keeps 2x4x8, so that the statistics behind it, and with them all that a network computes from there on, do not hang on
// an estimate of times (us it costs: where a brick less saves a round, 512 -> 512 at 12x10x14, 39 -> 50; elsewhere 1 to 5 %). Launches that add
// as slices do are few pairs: one block, and where two or eight are followed the smallest halo.
struct SplitPlan { SplitForm form; int chunk_stride, shape, blocks; int64_t tiles; };
SplitPlan split_plan(const MfmaConvArgs& a, bool records) {
  const int slices = split_rule(a, records).slices;
  const SplitForm form = slices == 8 ? kApart : slices != 2 ? kOrdinary : a.cred <= 4 * kChunk ? kHalves : kPairs;
  const int shape = records ? 0 : form != kOrdinary ? 1 : split_shape(a);
  const int64_t tiles = tiles_of(a, shape);
  return SplitPlan{form, slices == 2 || slices == 4 ? a.cred / kChunk / slices : 1, shape,
                   form == kPairs ? 2 : slices > 0 ? 1 : split_blocks(tiles, a.cout), tiles};
}

template <typename T, typename S, int R, int NSUB, bool PAIR, SplitForm FORM = kOrdinary>
int launch_brick(int chunk_stride, const MfmaConvArgs& a, const void* x, const void* packed, const void* bias, void* y, hipStream_t st,
                 const GnPartialOut& gn, const void* x1, void* y1, int first) {
  const int tiles_d = (int)cdiv(a.od, S::TD), tiles_h = (int)cdiv(a.oh, S::TH), tiles_w = (int)cdiv(a.ow, S::TW);
  const int nblocks = a.cout / (32 * NSUB);
  const int64_t total = (int64_t)a.n * tiles_d * tiles_h * tiles_w * nblocks;
  if (total == 0) return SFH_OK;
  if (total > 0x7fffffffLL) return fail(SFH_ERR_UNSUPPORTED, "conv split: %lld workgroups exceed the grid limit", (long long)total);
  hipLaunchKernelGGL((conv_split_kernel<T, S, R, NSUB, PAIR, FORM>), dim3((unsigned)total), dim3(256), 0, st, a, (const T*)x, (const T*)packed,
                     (const T*)bias, (T*)y, tiles_d, tiles_h, tiles_w, nblocks, (uint32_t)total, gn, (const T*)x1, (T*)y1, first, chunk_stride);
  return check_launch("conv_split_kernel");
}

template <typename T, int R, int NSUB, bool PAIR>
int launch_split(const SplitPlan& p, const MfmaConvArgs& a, const void* x, const void* packed, const void* bias, void* y, hipStream_t st,
                 const GnPartialOut& gn, const void* x1, void* y1, int first) {
  switch (p.shape) {
    case 1: return launch_brick<T, Cube, R, NSUB, PAIR>(p.chunk_stride, a, x, packed, bias, y, st, gn, x1, y1, first);
    case 2: return launch_brick<T, Rows, R, NSUB, PAIR>(p.chunk_stride, a, x, packed, bias, y, st, gn, x1, y1, first);
    default: return launch_brick<T, Flat, R, NSUB, PAIR>(p.chunk_stride, a, x, packed, bias, y, st, gn, x1, y1, first);
  }
}

template <typename T>
int launch_split_typed(const MfmaConvArgs& a, const void* x, const void* packed, const void* bias, void* y, hipStream_t st,
                       const GnPartialOut& gn, const void* x1, void* y1, int first) {
  const SplitPlan p = split_plan(a, gn.part != nullptr);
  const bool four = (a.cred / kChunk) % 4 == 0;
  if (p.form == kApart)
    return x1 != nullptr ? launch_brick<T, Cube, 4, 1, true, kApart>(1, a, x, packed, bias, y, st, gn, x1, y1, first)
                         : launch_brick<T, Cube, 4, 1, false, kApart>(1, a, x, packed, bias, y, st, gn, x1, y1, first);
  if (p.form == kHalves)
    return x1 != nullptr ? launch_brick<T, Cube, 2, 1, true, kHalves>(p.chunk_stride, a, x, packed, bias, y, st, gn, x1, y1, first)
                         : launch_brick<T, Cube, 2, 1, false, kHalves>(p.chunk_stride, a, x, packed, bias, y, st, gn, x1, y1, first);
  if (p.form == kPairs)
    return x1 != nullptr ? launch_brick<T, Cube, 4, 2, true, kPairs>(1, a, x, packed, bias, y, st, gn, x1, y1, first)
                         : launch_brick<T, Cube, 4, 2, false, kPairs>(1, a, x, packed, bias, y, st, gn, x1, y1, first);
#define SFH_SPLIT(NSUB)                                                                                         \
  x1 != nullptr ? (four ? launch_split<T, 4, NSUB, true>(p, a, x, packed, bias, y, st, gn, x1, y1, first)   \
                        : launch_split<T, 2, NSUB, true>(p, a, x, packed, bias, y, st, gn, x1, y1, first))  \
                : (four ? launch_split<T, 4, NSUB, false>(p, a, x, packed, bias, y, st, gn, x1, y1, first)  \
                        : launch_split<T, 2, NSUB, false>(p, a, x, packed, bias, y, st, gn, x1, y1, first))
  return p.blocks == 1 ? SFH_SPLIT(1) : SFH_SPLIT(2);
#undef SFH_SPLIT
}

}  // namespace

// Serves 64 or more reduction channels in an even number of 32-channel chunks and produced channels in blocks of 64, on
// planes of at most 32 x 32 voxels whose bricks times block pairs number 24 or more per two planes. Measured against the
// brick kernel on every convolution of a five-level U-Net step: 10-25 % faster at 16 x 32 x 32 and 8 x 16 x 16, where the
// brick kernel runs as one round of workgroups or needs slices; slower on 32 x 64 x 64 (several rounds of bricks overlap
// staging and MFMAs by themselves, and 64-voxel bricks stage 3.75 voxels per output voxel) and at 4 x 8 x 8 (a handful
// of workgroups cannot pull 7-14 MiB of weights fast enough: that level needs the slices over many CUs). For the same
// reason it leaves reductions of 512 channels or more to the slices where its workgroups would number 32 or fewer per
// two planes (8 x 16 x 16 with 256 produced channels: 128 workgroups of 1.7 MiB of weights each, 41 us against 30 with
// the weights cold; eight wavefronts per workgroup instead of four changed nothing, which is how the bound was found).
// That line looks at a plane only; volumes below it come here too once pairs of blocks number a quarter of the CUs (a
// workgroup of one block needs no slices and no launch that sums them). us, slices and their sum -> here: 64 -> 64 at 16^3 10.4 -> 5.6,
// 64 -> 128 at 16^3 11.9 -> 6.0, 128 -> 128 at 16^3 14.9 -> 8.6, 256 -> 128 at 20x12x14 22 -> 12.5, 512 -> 256 at 16^3 44 -> 32. Few pairs of a
// long reduction lose (512 -> 512 at 8^3, 64 pairs: 17.4 -> 23.2; 256 -> 256 at 4x8x8, 16 pairs: 10.1 -> 10.6), so the line is higher for
// those. Some below it would gain as well (128 -> 128 at 8^3, 16 pairs: 9.7 -> 7.7; 256 -> 128 at 8x16x16, 64: 14.9 -> 11.4; 512 -> 256 at
// 8x16x16, 128: 27.8 -> 22.9): their sliced geometry is what the tests of the launch query hold the last two to.
// Past three rounds of pairs the brick kernel's launches have no slices either and stage less: a volume below the plane's line comes here only
// where the bricks leave more over, by the busiest CU's share, than the 10 % that 64-voxel bricks lose at equal shares, or where
// the times say that a third is gained. us, bricks -> here: 64 -> 64 at 256x16x16 (1024 pairs, equal shares) 19.2 -> 21.2, 128 -> 128 at 128x16x16 31.0 -> 33.9; 128 -> 64
// at 200x20x20 (1500 pairs, 768 against 993 voxel blocks) 56 -> 46, 64 -> 64 at 64x24x24 (576 pairs) 17.9 -> 16.0. Planes past 32 x 32 come here by the times,
// from about a round of pairs on and where a third is gained (another order of sums is worth no less): 64 -> 64 at 17x36x35
// 15.9 -> 9.7, at 9x27x50 12.1 -> 7.9, 128 -> 128 at 10x28x56 25.8 -> 17.0.
// All that is for the forward, with GroupNorm records or without (the result is the same bits either way). A data gradient comes here by the rules
// before the times: nothing is gained by another order of its sums that is worth a step's gradients in other bits. Where the slices' bits
// are kept (below), it comes here by the fewer pairs too.
// The times take nothing away from this kernel: its four partial sums to a voxel are nearer the 64-bit result than the bricks' one chain (fp16
// results of 64 to 512 channels that are not the rounded 64-bit ones: 1.5e-3 here, 1.9e-3 in bricks, 28 problems of both directions), so 256 -> 256 at 32^3 stays at
// 109 us though bricks take 102. Eight slices are nearer still (1.35e-3, 1.75e-3 here with four sums; four: level).
// What the bricks would sum in slices comes here with the slices' bits, so that it may in both directions: of four a wavefront takes one's chunks in
// their order; of two, up to 128 channels, a voxel half of one's, past that one of two blocks of one's; eight of one chunk (256 channels) are two
// rounds whose sums meet at the end. Where none of these is, eight slices stay (nearer the exact value still, 1.35e-3, 1.75e-3 here with four sums), and four become this
// kernel's sums where a third of the time is gained. A launch that leaves GroupNorm records stays with the slices, whose records are sums of other voxels.
// us, slices and their sum -> here, with their bits: 64 -> 128 at 14x13x6 9.3 -> 6.0, 64 -> 512 at 7x3x6 8.8 -> 6.0, 128 -> 64 (data gradient) at 14x13x6 9.4 -> 6.0,
// three samples of 128 -> 256 at 10x3x6 12.8 -> 8.9, 128 -> 512 at 3x4x9 9.0 -> 7.0, 256 -> 256 at 11x4x9 12.6 -> 10.3, at 8x4x20 (eight) 12.0 -> 11.4, at 5x8x14 11.2 -> 11.7,
// 512 -> 512 at 9x9x6 38.4 -> 31.2 (four sums 24.2; by voxel halves, whose every weight goes to two wavefronts, 39.8), 512 -> 256 at 10x8x22 39.1 -> 31.3. Eight would
// lose where rows are short or 512 channels are produced (256 -> 256 at 14x6x4 10.2 -> 11.5, 256 -> 512 at 6x7x5 10.2 -> 14.6).
// The data gradient of a depth shard's slab (D + 2 planes from D) and of the padded volume (D from D) must come from the same
// kernel, or a shard and the whole volume would disagree in the last bit: the depth counted is the smaller of the two.
constexpr int kSplitMaxPlane = 32 * 32, kSplitMinPerDepth = 24, kSplitFewPerDepth = 32, kSplitFewMaxChunks = 16;
constexpr int kSplitBigPlanePairs = 240;
// Pairs from which a volume below the plane's line comes here, and the fewer from which it does in the place of slices (figures above; longer reductions where
// the times say that three tenths are gained).
int64_t split_line(int chunks) { return chunks <= 4 ? kComputeUnits / 4 : chunks <= 8 ? kComputeUnits / 4 + 1 : kComputeUnits / 2 + 1; }
int64_t split_line_few(int chunks, int cout) { return chunks <= 4 && cout >= 128 ? 24 : chunks <= 8 && cout >= 256 ? 48 : split_line(chunks); }

namespace {
SplitRule split_rule(const MfmaConvArgs& a, bool records) {
  if (a.kd != 3 || a.kh != 3 || a.kw != 3) return {};
  if (a.cred < 2 * kChunk || a.cred % (2 * kChunk) != 0 || a.cout % (32 * kBlocks) != 0) return {};
  const int chunks = a.cred / kChunk, pair = a.cout / (32 * kBlocks);
  MfmaConvArgs core = a;
  core.od = a.id < a.od ? a.id : a.od;
  const int64_t per_depth = (int64_t)a.n * cdiv(a.oh, Flat::TH) * cdiv(a.ow, Flat::TW) * pair;
  const int64_t pairs = per_depth * cdiv(core.od, Flat::TD), rounds = cdiv(pairs, kComputeUnits);
  const bool kept = a.gradient != 0;  // the order of sums does not go by the times
  auto sooner = [&](int percent) { return 100 * split_time(split_tiles(core) * pair, chunks) < percent * mfma_conv_brick_time(core); };
  if ((int64_t)a.oh * a.ow > kSplitMaxPlane) return {!kept && pairs > kSplitBigPlanePairs && sooner(68), 0};
  const bool few = per_depth <= kSplitFewPerDepth && chunks >= kSplitFewMaxChunks;
  if (!few && per_depth >= kSplitMinPerDepth) return {true, 0};
  if (pairs >= split_line(chunks))
    return {rounds <= 3 || rounds * (kBrickVoxels * kBlocks) * 110 < mfma_conv_brick_cost(core) || (!kept && sooner(68)), 0};
  const int slices = mfma_conv_brick_slices(core);
  const bool like_slices = slices == 8 ? chunks == 8 && a.cout <= 256 && a.ow > 8 : slices == 4 || (slices == 2 && chunks > 4) ? chunks % 4 == 0 : slices == 2;
  const bool same_bits = like_slices && (a.gradient || core.od == a.od || mfma_conv_brick_slices(a) == slices);
  if (same_bits ? records : slices > 4 || kept) return {};
  const bool enough = pairs >= split_line_few(chunks, a.cout) && (same_bits || sooner(68));
  return {enough || (chunks >= kSplitFewMaxChunks && sooner(70)), same_bits ? slices : 0};
}
}  // namespace

bool mfma_conv_split_applies(const MfmaConvArgs& a, bool records) { return split_rule(a, records).use; }

MfmaConvGeometry mfma_conv_split_geometry(const MfmaConvArgs&) { return MfmaConvGeometry{kKernelSplit, kBrickVoxels, kBlocks, 1}; }

int mfma_conv_split_gn_records(const MfmaConvArgs& a, int groups) {
  const SplitPlan p = split_plan(a, true);
  const int span = 32 * p.blocks;
  if (!gn_partials_fit(a.cout, groups, span)) return 0;
  const int cg = a.cout / groups;
  const int64_t records = p.tiles / a.n * (cg > span ? cg / span : 1);
  return records <= 0x7fffffff ? (int)records : 0;
}

bool mfma_conv_split_pair_ok(const MfmaConvArgs& a, int first, bool as_output) {
  const int channels = as_output ? a.cout : a.cred;
  return first > 0 && first < channels && first % 32 == 0;
}

int mfma_conv_split(const MfmaConvArgs& a, int dtype, const void* x, const void* packed, const void* bias, void* y, hipStream_t st,
                    const GnPartialOut* gn, const ChannelPair* in2, const ChannelPair* out2) {
  if (in2 != nullptr && out2 != nullptr) return fail(SFH_ERR_UNSUPPORTED, "conv split: input and output cannot both be pairs");
  if (out2 != nullptr && gn != nullptr && gn->part != nullptr)
    return fail(SFH_ERR_UNSUPPORTED, "conv split: no GroupNorm partials of an output written as two tensors");
  if (in2 != nullptr && (in2->second == nullptr || !mfma_conv_split_pair_ok(a, in2->first, false)))
    return fail(SFH_ERR_UNSUPPORTED, "conv split: the input cannot be cut at channel %d of %d", in2->first, a.cred);
  if (out2 != nullptr && (out2->second == nullptr || !mfma_conv_split_pair_ok(a, out2->first, true)))
    return fail(SFH_ERR_UNSUPPORTED, "conv split: the output cannot be cut at channel %d of %d", out2->first, a.cout);
  GnPartialOut out{nullptr, 0, 0, 0};
  if (gn != nullptr && gn->part != nullptr) {
    if (gn->records != mfma_conv_split_gn_records(a, gn->groups) || gn->records == 0)
      return fail(SFH_ERR_INVALID, "conv split: GroupNorm partials asked for %d records, this launch leaves %d", gn->records,
                  mfma_conv_split_gn_records(a, gn->groups));
    out = *gn;
    out.cg = a.cout / gn->groups;
  }
  const void* x1 = in2 != nullptr ? in2->second : nullptr;
  void* y1 = out2 != nullptr ? out2->second : nullptr;
  const int first = in2 != nullptr ? in2->first : (out2 != nullptr ? out2->first : 0);
  if (dtype == SFH_BF16) return launch_split_typed<bf16_t>(a, x, packed, bias, y, st, out, x1, y1, first);
  return launch_split_typed<fp16_t>(a, x, packed, bias, y, st, out, x1, y1, first);
}

}  // namespace sfh
