// Learned initial guess for the Poisson solve: a 3-D convolutional
// encoder-decoder that maps (charge density, conductor mask) to the potential,
// trained on (rho, phi) pairs that the multigrid solver itself produces. The
// multigrid solve always iterates from the guess to the same residual, so the
// network only changes where the iteration starts. The reference has no
// counterpart (its solver is SOR from the previous potential,
// RootGridField.cpp:41-103).
//
// Network (levels 0..3 at n, n/2, n/4, n/8 voxels per axis; 3x3x3 kernels,
// zero padding, BF16 weights and activations, FP32 accumulation):
//   e0a 8->16, e0b 16->16 = S0 | pool | e1a 16->32, e1b 32->32 = S1 | pool |
//   e2a 32->48, e2b 48->48 = S2 | pool | e3a 48->64, e3b 64->64 = B3 |
//   d2a up(B3) 64->48 (+S2), d2b 48->48 | d1a up 48->32 (+S1), d1b 32->32 |
//   d0a up 32->16 (+S0), d0b 16->16 | out 16->1 (linear).
// Every layer but `out` is relu(conv(x) + b [+ skip]); pool is a 2x2x2 mean,
// up is nearest-neighbour (read through the index map, never materialised).
//
// Convolutions are implicit GEMMs on v_mfma_f32_16x16x32_bf16: activations
// are channels-last [voxel][channel], a K step of 32 is four 8-channel chunks
// of (tap, channel) pairs, one chunk per 16-lane group, loaded as 16 bytes.
// The data-gradient is the same kernel with the taps mirrored and the channel
// roles swapped; the weight-gradient reduces over voxels with the voxels as
// the MFMA K dimension.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <type_traits>

#include "fopis_internal.hpp"

namespace fopis {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __host__ inline float bf2f(uint16_t h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }

// FP32 -> BF16, round to nearest even (NaN kept quiet).
__device__ __host__ inline uint16_t f2bf(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ inline bf16x8 load8(const uint16_t* p) {
  const u32x4 raw = *reinterpret_cast<const u32x4*>(p);
  return __builtin_bit_cast(bf16x8, raw);
}

__device__ inline bf16x8 zero8() {
  const u32x4 z = {0u, 0u, 0u, 0u};
  return __builtin_bit_cast(bf16x8, z);
}

// See poisson.hip: XCD x runs a contiguous run of the logical workgroup ids.
__device__ inline int xcd_block(int p, int n) {
  const int per = n >> 3, rem = n & 7, x = p & 7, slot = p >> 3;
  return x * per + min(x, rem) + slot;
}

// ---------------------------------------------------------------- conv forward

enum { EPI_BF16 = 0, EPI_F32 = 1, EPI_PHI = 2 };

struct ConvArgs {
  const uint16_t* x;     // input [voxel][cin] (at half resolution when up)
  const uint16_t* w;     // packed weights [nqp][cout][8]
  const float* bias;     // [cout]
  const uint16_t* add;   // [voxel][cout] added before the activation, or null
  const uint16_t* gate;  // [voxel][cout]: the result is kept where this is > 0 (a ReLU's backward), or null
  uint16_t* y;           // EPI_BF16: [voxel][cout]
  float* y32;            // EPI_F32: channel 0, [voxel]
  double* phi;           // EPI_PHI: glue-layout potential
  const double* scal;    // EPI_PHI: scal[0] = input scale sigma
  double phi_k;          // EPI_PHI: phi = out * sigma * phi_k
  int phi_add;           // EPI_PHI: add to phi instead of replacing it
  int64_t gsx, gsy, goff;
  int vn0, vn1, vn2;     // EPI_PHI: voxels that map to interior nodes
  int n0, n1, n2;        // output grid
  int cin, cout;
  int up;                // 1: x is at half resolution (nearest-neighbour upsampling on read)
  int nbrick;            // output bricks
  int relu;
};

// Output bricks of kBI x kBJ x 16 voxels: the brick's input with a one-voxel
// halo (kBI+2, kBJ+2, 18) is staged once in LDS, channel rows padded by 8
// elements to spread the 16 lanes of a fragment read over the banks; each
// of the 4 waves then owns kBI*kBJ/4 rows of 16 voxels (its M tiles) and reads
// its A fragments from LDS, B fragments (weights) from global memory through
// the caches.
constexpr int kBI = 4, kBJ = 4, kBK = 16;
constexpr int kHI = kBI + 2, kHJ = kBJ + 2, kHK = kBK + 2;
constexpr int kHalo = kHI * kHJ * kHK;
constexpr int kRowsPerWave = kBI * kBJ / 4;
static_assert(kRowsPerWave == kBJ, "wave w owns the brick's plane w");
static_assert(kHI + kHJ + kHK <= 32, "one bit per halo plane");

constexpr size_t conv_lds_bytes(int cin) { return (size_t)kHalo * (cin + 8) * sizeof(uint16_t); }

// LDS element offset, from a row's own voxel, of the 8-channel chunk q of the
// K axis (q = tap * cin / 8 + channel / 8); chunks past the last tap sit at 0.
template <int CIN>
constexpr int chunk_off(int q) {
  constexpr int cpt = CIN / 8;
  if (q >= 27 * cpt) return 0;
  const int tap = q / cpt;
  return ((tap / 9 * kHJ + (tap / 3) % 3) * kHK + tap % 3) * (CIN + 8) + (q % cpt) * 8;
}

template <int MASK>
__device__ inline float quad_swap(float v) {  // the value of lane ^ MASK, MASK 1 or 2
  constexpr int ctrl = MASK == 1 ? 0xB1 : 0x4E;
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, true));
}

// Two floats rounded to BF16 (nearest even), the first in the low half.
__device__ inline uint32_t pack_bf16(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// Waves per SIMD that k_conv's registers leave room for: as many as hold what a
// thread keeps without scratch memory: the next brick's units (1.9 registers
// per input channel) and, with one tile, all weights (3.4 per channel). One more than that spills: 64 -> 64 at 16^3 14.9 -> 26.8 us with two,
// 48 -> 48 at 32^3 23.3 -> 25.9, 32 -> 16 upsampled to 128^3 115 -> 222 with three,
// 48 -> 32 to 64^3 34 -> 39. One fewer leaves the chip waiting: 32 -> 32 at 64^3
// takes 37 us with one, 30 with two or three.
constexpr int conv_waves(int cin, int nt) {
  if (cin >= 56 || (nt == 1 && cin >= 40)) return 1;
  return cin >= 48 || nt > 2 || (nt == 1 && cin >= 24) ? 2 : 3;
}

// NT tiles of 16 output channels per workgroup, tiles blockIdx.y * NT on.
// The input channel count is a template argument, so that the K loop unrolls
// and every fragment's LDS address is a lane base plus an immediate: with the
// count at run time a K step spent ~80 vector instructions (a division by
// cin/8 among them) on the addresses of four 16-cycle MFMAs, and those
// bounded the kernel. A workgroup walks a run of neighbouring bricks: each
// thread's voxels sit at the same offsets from every brick's corner, computed
// once, and one bit per halo plane tells which of them lie outside the grid;
// the next brick's voxels are loaded while the current brick is multiplied;
// with one tile the weights stay in registers (all of their loads are then in
// flight before the first brick arrives, which is what a small grid waits
// for). The result leaves through a 4x4 exchange between the four lanes that hold
// neighbouring channels, so that a lane stores (and loads the addend and the
// gate as) four channels of one voxel, 8 bytes, instead of four times 2 bytes.
// Bound by LDS reads (one per product with 16 output channels) and the
// latency of a brick's stage-multiply-store chain: at 128^3, 16 -> 16, a compute
// unit's LDS is busy 60 % of the time (half of it bank conflicts), the vector
// units 45 %, the matrix cores 25 %, and waves wait 41 % of theirs; at 16^3, 64 ->
// 64, LDS 21 %, matrix cores 10 %, waves wait 54 %. 16 -> 16 channels at 128^3:
// 115 -> 58 us (2.3 TB/s, 0.5 PFLOP/s), 32 -> 16 upsampled: 222 -> 113 us,
// 64 -> 64 at 16^3: 38 -> 15 us.
template <int CIN, int NT, int EPI>
__global__ __launch_bounds__(256, conv_waves(CIN, NT)) void k_conv(ConvArgs A) {
  extern __shared__ __attribute__((aligned(16))) uint16_t xs[];
  constexpr int MT = kRowsPerWave;
  constexpr int CPT = CIN / 8, NQ = 27 * CPT, NS = (NQ + 3) / 4, LS = CIN + 8;
  constexpr bool kWReg = NT == 1;
  const int cout = A.cout, ct0 = blockIdx.y * NT * 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = lane & 15, grp = lane >> 4;
  const int nb1 = (A.n1 + kBJ - 1) / kBJ, nb2 = (A.n2 + kBK - 1) / kBK;
  const int in1 = A.n1 >> A.up, in2 = A.n2 >> A.up;
  const int per = (A.nbrick + (int)gridDim.x - 1) / (int)gridDim.x;
  const int first = xcd_block(blockIdx.x, gridDim.x) * per, last = min(first + per, A.nbrick);
  if (first >= last) return;

  // the thread's units (16 bytes of one halo voxel): offset from the brick's
  // corner in x, and one bit per halo plane along each axis
  constexpr int kUnits = kHalo * CPT, IT = (kUnits + 255) / 256;
  int rel[IT];
  uint32_t planes[IT];
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    const int e = threadIdx.x + u * 256;
    const int ch = e % CPT, hv = e / CPT;
    const int hk = hv % kHK, hj = (hv / kHK) % kHJ, hi = hv / (kHK * kHJ);
    // (bricks start at even voxels, so the halving of a coordinate splits)
    rel[u] = ((((hi - 1) >> A.up) * in1 + ((hj - 1) >> A.up)) * in2 + ((hk - 1) >> A.up)) * CIN + ch * 8;
    planes[u] = e < kUnits ? (1u << hi) | (1u << (kHI + hj)) | (1u << (kHI + kHJ + hk)) : 0xffffffffu;
  }
  u32x4 v[IT];
  auto fetch = [&](int blk) {
    const int b2 = blk % nb2, b1 = (blk / nb2) % nb1, b0 = blk / (nb2 * nb1);
    const int i0 = b0 * kBI, j0 = b1 * kBJ, k0 = b2 * kBK;
    // halo planes outside the grid: below the first voxel, from the last one on
    auto off = [](int o, int n, int h) -> uint32_t {
      const int live = min(h, n - o + 1);  // planes 1 .. live - 1 (and 0 when o > 0) are inside
      return (o > 0 ? 0u : 1u) | (((1u << h) - 1u) & ~((1u << live) - 1u));
    };
    const uint32_t out = off(i0, A.n0, kHI) | (off(j0, A.n1, kHJ) << kHI) | (off(k0, A.n2, kHK) << (kHI + kHJ));
    const uint16_t* base = A.x + (((int64_t)(i0 >> A.up) * in1 + (j0 >> A.up)) * in2 + (k0 >> A.up)) * CIN;
#pragma unroll
    for (int u = 0; u < IT; ++u) {
      v[u] = (u32x4){0u, 0u, 0u, 0u};
      if (!(planes[u] & (out | (1u << 31)))) v[u] = *reinterpret_cast<const u32x4*>(base + rel[u]);
    }
  };
  fetch(first);

  bf16x8 wreg[kWReg ? NS : 1][NT];
  if constexpr (kWReg) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)  // chunk 4s + grp, output channel ct0 + nt * 16 + row
        wreg[s][nt] = load8(A.w + (int64_t)(s * 4 + grp) * cout * 8 + (ct0 + nt * 16 + row) * 8);
  }
  float bias[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) bias[nt] = A.bias[ct0 + nt * 16 + row];

  for (int blk = first; blk < last; ++blk) {
    const int b2 = blk % nb2, b1 = (blk / nb2) % nb1, b0 = blk / (nb2 * nb1);
    const int i0 = b0 * kBI, j0 = b1 * kBJ, k0 = b2 * kBK;
    if (blk != first) __syncthreads();  // the last brick's fragments have been read
#pragma unroll
    for (int u = 0; u < IT; ++u) {
      const int e = threadIdx.x + u * 256;
      if ((u + 1) * 256 <= kUnits || e < kUnits)
        *reinterpret_cast<u32x4*>(xs + (e / CPT) * LS + (e % CPT) * 8) = v[u];
    }
    __syncthreads();
    if (blk + 1 < last) fetch(blk + 1);

    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // (the weights are read again for each brick: without this the compiler
    // moves all of their loads out of the brick loop, into scratch memory)
    int wo = (grp * cout + ct0 + row) * 8;
    asm volatile("" : "+v"(wo));
    const uint16_t* xb = xs + (wave * kHJ * kHK + row) * LS;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      bf16x8 bfr[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) bfr[nt] = kWReg ? wreg[kWReg ? s : 0][nt] : load8(A.w + s * 32 * cout + nt * 128 + wo);
      // the four lane groups' chunks: one lane offset per pattern of
      // differences (few of them), the rest an immediate
      const int o0 = chunk_off<CIN>(4 * s);
      const int d1 = chunk_off<CIN>(4 * s + 1) - o0, d2 = chunk_off<CIN>(4 * s + 2) - o0,
                d3 = chunk_off<CIN>(4 * s + 3) - o0;
      const int ld = grp == 0 ? 0 : (grp == 1 ? d1 : (grp == 2 ? d2 : d3));
      const bool qok = 4 * s + 3 < NQ || 4 * s + grp < NQ;  // chunks past the last tap (K padding) are zeroed
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const u32x4 raw = *reinterpret_cast<const u32x4*>(xb + ld + (o0 + mt * kHK * LS));
        const bf16x8 af = qok ? __builtin_bit_cast(bf16x8, raw) : zero8();
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr[nt], acc[mt][nt], 0, 0, 0);
      }
    }

    // D layout: lane holds output channel ct0 + nt*16 + row for voxels k0 + 4*grp + r of the row
    const int i = i0 + wave;
    if (i < A.n0) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int j = j0 + mt;
        if (j >= A.n1) continue;
        const int64_t vrow = ((int64_t)i * A.n1 + j) * A.n2;
        if constexpr (EPI == EPI_BF16) {
          const int q = row & 3, k = k0 + 4 * grp + q;
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            float f[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) f[r] = acc[mt][nt][r] + bias[nt];
            // lane q of a quad ends with voxel 4*grp + q, channels 4*(row/4) .. + 3
            float t;
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
              t = quad_swap<1>((q & 1) ? f[r] : f[r + 1]);
              f[r] = (q & 1) ? t : f[r];
              f[r + 1] = (q & 1) ? f[r + 1] : t;
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
              t = quad_swap<2>((q & 2) ? f[r] : f[r + 2]);
              f[r] = (q & 2) ? t : f[r];
              f[r + 2] = (q & 2) ? f[r + 2] : t;
            }
            if (k < A.n2) {
              const int64_t at = (vrow + k) * cout + ct0 + nt * 16 + (row & 12);
              if (A.add) {
                const uint2 ad = *reinterpret_cast<const uint2*>(A.add + at);
                f[0] += bf2f((uint16_t)ad.x);
                f[1] += bf2f((uint16_t)(ad.x >> 16));
                f[2] += bf2f((uint16_t)ad.y);
                f[3] += bf2f((uint16_t)(ad.y >> 16));
              }
              if (A.relu)
#pragma unroll
                for (int r = 0; r < 4; ++r) f[r] = fmaxf(f[r], 0.f);
              uint2 o = make_uint2(pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]));
              if (A.gate) {
                const uint2 gt = *reinterpret_cast<const uint2*>(A.gate + at);
                if (!(bf2f((uint16_t)gt.x) > 0.f)) o.x &= 0xffff0000u;
                if (!(bf2f((uint16_t)(gt.x >> 16)) > 0.f)) o.x &= 0xffffu;
                if (!(bf2f((uint16_t)gt.y) > 0.f)) o.y &= 0xffff0000u;
                if (!(bf2f((uint16_t)(gt.y >> 16)) > 0.f)) o.y &= 0xffffu;
              }
              *reinterpret_cast<uint2*>(A.y + at) = o;
            }
          }
        } else if (row == 0) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int k = k0 + 4 * grp + r;
            if (k >= A.n2) continue;
            const float val = acc[mt][0][r] + bias[0];
            if constexpr (EPI == EPI_F32) {
              A.y32[vrow + k] = val;
            } else if (i < A.vn0 && j < A.vn1 && k < A.vn2) {
              double* p = A.phi + A.goff + i * A.gsx + j * A.gsy + k;
              *p = (A.phi_add ? *p : 0.0) + (double)val * A.scal[0] * A.phi_k;
            }
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------- weight gradient

// dW[tap][ci][co] = sum over voxels v of x[v + tap][ci] g[v][co], and the bias
// gradient sum g[v][co]: products whose contraction runs over the voxels, so
// an MFMA operand wants eight neighbouring voxels of one channel where the
// arrays hold neighbouring channels of one voxel. A workgroup stages a brick
// of BI x BJ x 32 voxels of g, and of x with its halo, into LDS with each
// 8-voxel x 8-channel block transposed in registers (32 byte permutes), as
// rows [channel][voxel]. A lane then reads its fragment for the left tap of a
// row as 16 bytes plus the next dword, and the centre and right taps are the
// same registers shifted by one and two voxels. Each x row meets up to nine g
// rows (held in registers), 27 products per row pair of tiles: 27 products
// cost 3 to 7 LDS reads. The four waves take PI x PO tiles of 16 x 16
// channels; where the layer has fewer tiles they split the brick's rows
// (kSub) and add their sums in LDS. The bias gradient is one more product,
// with ones. Partials of a launch's workgroups go to `part`, and
// k_wgrad_reduce adds them in workgroup order.
// Bound by the latency of staging: at 64^3 a workgroup has two bricks of 216 to
// 432 products per wave, waves wait 42 to 63 % of their time, the LDS is busy
// 29 to 41 % (most of it bank conflicts), the matrix cores 7 to 14 %. The 15
// layers of a 64^3 training pair: 2.29 -> 0.22 ms (with 2-byte gathers, one per
// voxel, tap and channel), their bias sums 1.00 ms -> none.
constexpr int kWTile = 27 * 256 + 16;  // floats of one channel tile's partial: the taps, then the bias gradient
constexpr int kWRow = 40;              // LDS elements of one channel's row: 34 voxels, padded to spread the banks

struct WgradArgs {
  const uint16_t* x;  // layer input [voxel][cin] (half resolution when UP)
  const uint16_t* g;  // output gradient after the activation [voxel][cout]
  float* part;        // [pair][chunk][kWTile]
  int n0, n1, n2;     // output grid
  int cin, cout, nci, nco;  // nci, nco: tiles of 16 channels
  int nbrick;
};

template <int PI, int PO>
struct WgradShape {
  static constexpr int kSub = 4 / (PI * PO);       // waves sharing a tile pair
  static constexpr int RI = 2, RJ = kSub == 1 ? 4 : 2;  // rows of one wave
  static constexpr int SI = kSub == 4 ? 2 : 1, SJ = kSub / SI;
  static constexpr int BI = RI * SI, BJ = RJ * SJ;  // rows of the brick
  static constexpr int kXRows = (BI + 2) * (BJ + 2), kGRows = BI * BJ;
  static constexpr int kXElems = kXRows * PI * 16 * kWRow, kGElems = kGRows * PO * 16 * kWRow;
  static constexpr size_t kStage = (size_t)(kXElems + kGElems) * sizeof(uint16_t);
  static constexpr size_t kSum = kSub > 1 ? (size_t)PI * PO * kWTile * sizeof(float) : 0;
  static constexpr size_t kLds = kStage > kSum ? kStage : kSum;
  static_assert(kLds <= 81920, "two workgroups per compute unit");
};

// Eight voxels of eight channels each into eight channels of eight voxels.
__device__ inline void transpose8(const u32x4 (&v)[8], u32x4 (&t)[8]) {
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int h = 0; h < 4; ++h)
      t[c][h] = __builtin_amdgcn_perm(v[2 * h + 1][c >> 1], v[2 * h][c >> 1], (c & 1) ? 0x07060302u : 0x05040100u);
}

template <int PI, int PO, bool UP>
__global__ __launch_bounds__(256, 2) void k_wgrad(WgradArgs A) {
  using W = WgradShape<PI, PO>;
  extern __shared__ __attribute__((aligned(16))) uint16_t ws[];
  uint16_t* xs = ws;
  uint16_t* gs = ws + W::kXElems;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 15, grp = lane >> 4;
  const int ngo = (A.nco + PO - 1) / PO;
  const int ci0 = (blockIdx.y / ngo) * PI, co0 = (blockIdx.y % ngo) * PO;  // the group's first tiles
  const int sub = wave / (PI * PO), pi = (wave % (PI * PO)) / PO, po = wave % PO;
  const int si = sub / W::SJ, sj = sub % W::SJ;
  const bool live = ci0 + pi < A.nci && co0 + po < A.nco;
  const int nb1 = (A.n1 + W::BJ - 1) / W::BJ, nb2 = (A.n2 + 31) / 32;
  const int in1 = UP ? (A.n1 >> 1) : A.n1, in2 = UP ? (A.n2 >> 1) : A.n2;
  f32x4 acc[27], accb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < 27; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};

  for (int brick = blockIdx.x; brick < A.nbrick; brick += gridDim.x) {
    const int b2 = brick % nb2, b1 = (brick / nb2) % nb1, b0 = brick / (nb2 * nb1);
    const int i0 = b0 * W::BI, j0 = b1 * W::BJ, k0 = b2 * 32;
    __syncthreads();  // the last brick's fragments have been read
    // x rows: voxels k0 - 1 .. k0 + 32 in five blocks of eight (the last holds two)
    for (int u = threadIdx.x; u < W::kXRows * 5 * PI * 2; u += 256) {
      const int c8 = u % (PI * 2), o = (u / (PI * 2)) % 5, r = u / (PI * 2 * 5);
      int gi = i0 - 1 + r / (W::BJ + 2), gj = j0 - 1 + r % (W::BJ + 2);
      const int c = ci0 * 16 + c8 * 8;
      const bool ok = c < A.cin && gi >= 0 && gi < A.n0 && gj >= 0 && gj < A.n1;
      if (UP) {
        gi >>= 1;
        gj >>= 1;
      }
      const uint16_t* p = A.x + ((int64_t)gi * in1 + gj) * in2 * A.cin + c;
      u32x4 v[8], t[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int e = o * 8 + q;
        int gk = k0 - 1 + e;
        v[q] = (u32x4){0u, 0u, 0u, 0u};
        if (ok && e < 34 && gk >= 0 && gk < A.n2) {
          if (UP) gk >>= 1;
          v[q] = *reinterpret_cast<const u32x4*>(p + (int64_t)gk * A.cin);
        }
      }
      transpose8(v, t);
#pragma unroll
      for (int q = 0; q < 8; ++q)
        *reinterpret_cast<u32x4*>(xs + (r * PI * 16 + c8 * 8 + q) * kWRow + o * 8) = t[q];
    }
    for (int u = threadIdx.x; u < W::kGRows * 4 * PO * 2; u += 256) {
      const int c8 = u % (PO * 2), o = (u / (PO * 2)) % 4, r = u / (PO * 2 * 4);
      const int gi = i0 + r / W::BJ, gj = j0 + r % W::BJ;
      const int c = co0 * 16 + c8 * 8;
      const bool ok = c < A.cout && gi < A.n0 && gj < A.n1;
      const uint16_t* p = A.g + ((int64_t)gi * A.n1 + gj) * A.n2 * A.cout + c;
      u32x4 v[8], t[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int gk = k0 + o * 8 + q;
        v[q] = (u32x4){0u, 0u, 0u, 0u};
        if (ok && gk < A.n2) v[q] = *reinterpret_cast<const u32x4*>(p + (int64_t)gk * A.cout);
      }
      transpose8(v, t);
#pragma unroll
      for (int q = 0; q < 8; ++q)
        *reinterpret_cast<u32x4*>(gs + (r * PO * 16 + c8 * 8 + q) * kWRow + o * 8) = t[q];
    }
    __syncthreads();
    if (!live) continue;

    bf16x8 bfr[W::RI][W::RJ];
#pragma unroll
    for (int ri = 0; ri < W::RI; ++ri)
#pragma unroll
      for (int rj = 0; rj < W::RJ; ++rj) {
        const int r = (si * W::RI + ri) * W::BJ + sj * W::RJ + rj;
        bfr[ri][rj] = load8(gs + (r * PO * 16 + po * 16 + row) * kWRow + grp * 8);
        accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones), bfr[ri][rj], accb, 0, 0, 0);
      }
    // g is 0 past the grid, but the first voxel and row there meet x inside it
    // through the lower tap, and 0 times an infinite or NaN x is not 0: those
    // products are left out (x past the grid is 0 itself)
    const int li = A.n0 - i0 - si * W::RI, lj = A.n1 - j0 - sj * W::RJ, lk = A.n2 - k0 - grp * 8;
    u32x4 in;
#pragma unroll
    for (int h = 0; h < 4; ++h) in[h] = (2 * h < lk ? 0xffffu : 0u) | (2 * h + 1 < lk ? 0xffff0000u : 0u);
#pragma unroll
    for (int xi = 0; xi < W::RI + 2; ++xi)
#pragma unroll
      for (int xj = 0; xj < W::RJ + 2; ++xj) {
        const int r = (si * W::RI + xi) * (W::BJ + 2) + sj * W::RJ + xj;
        const uint16_t* p = xs + (r * PI * 16 + pi * 16 + row) * kWRow + grp * 8;
        const u32x4 d = *reinterpret_cast<const u32x4*>(p);
        const uint32_t d4 = *reinterpret_cast<const uint32_t*>(p + 8);
        const u32x4 f1 = {__builtin_amdgcn_alignbit(d[1], d[0], 16), __builtin_amdgcn_alignbit(d[2], d[1], 16),
                          __builtin_amdgcn_alignbit(d[3], d[2], 16), __builtin_amdgcn_alignbit(d4, d[3], 16)};
        const u32x4 f2 = {d[1], d[2], d[3], d4};
        const bf16x8 af[3] = {__builtin_bit_cast(bf16x8, d & in), __builtin_bit_cast(bf16x8, f1),
                              __builtin_bit_cast(bf16x8, f2)};
#pragma unroll
        for (int di = 0; di < 3; ++di)
#pragma unroll
          for (int dj = 0; dj < 3; ++dj) {
            const int ri = xi - di, rj = xj - dj;
            if (ri < 0 || ri >= W::RI || rj < 0 || rj >= W::RJ) continue;
            if ((di == 0 && ri >= li) || (dj == 0 && rj >= lj)) continue;
#pragma unroll
            for (int dk = 0; dk < 3; ++dk) {
              const int t = (di * 3 + dj) * 3 + dk;
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[dk], bfr[ri][rj], acc[t], 0, 0, 0);
            }
          }
      }
  }
  // D[m = ci local][n = co local]: lane holds n = row, m = 4*grp + r; the bias
  // gradient is in every m
  float* out = A.part + ((int64_t)((ci0 + pi) * A.nco + co0 + po) * gridDim.x + blockIdx.x) * kWTile;
  if constexpr (W::kSub == 1) {
    if (!live) return;
#pragma unroll
    for (int t = 0; t < 27; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) out[t * 256 + (4 * grp + r) * 16 + row] = acc[t][r];
    if (grp == 0) out[27 * 256 + row] = accb[0];
  } else {
    // the kSub waves of a tile pair add theirs in wave order
    float* red = reinterpret_cast<float*>(ws) + (pi * PO + po) * kWTile;
    for (int w = 0; w < W::kSub; ++w) {
      __syncthreads();
      if (sub != w) continue;
#pragma unroll
      for (int t = 0; t < 27; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int idx = t * 256 + (4 * grp + r) * 16 + row;
          red[idx] = (w == 0 ? 0.f : red[idx]) + acc[t][r];
        }
      if (grp == 0) red[27 * 256 + row] = (w == 0 ? 0.f : red[27 * 256 + row]) + accb[0];
    }
    __syncthreads();
    if (live)
      for (int i = lane + 64 * sub; i < kWTile; i += 64 * W::kSub) out[i] = red[i];
  }
}

// Partials into dW[tap][ci][co] and db[co], one block of 256 threads per 64
// elements of a tile: each wavefront adds a quarter of the chunks (64
// neighbouring floats per chunk), the quarters are added in order. All of a
// backward pass's layers go through one launch (15 launches of a few blocks
// each took 1.38 ms at 64^3, one takes 0.035 ms).
constexpr int kWMaxLayers = 16;
struct WreduceLayer {
  const float* part;
  float *dw, *db;
  int nchunk, cin, cout, nco;
  int block0;  // first block of the layer
};
struct WreduceArgs {
  WreduceLayer l[kWMaxLayers];
  int n;
};
// The layers of one backward pass whose partials wait for k_wgrad_reduce; it
// lives and dies with the pass, so a pass that fails leaves none behind.
struct WgradQueue {
  WreduceArgs a{};
  int blocks = 0;
};
constexpr int kWredBlocks = (kWTile + 63) / 64;  // per tile

__global__ __launch_bounds__(256) void k_wgrad_reduce(WreduceArgs A) {
  __shared__ float s[4][64];
  int li = 0;
  while (li + 1 < A.n && (int)blockIdx.x >= A.l[li + 1].block0) ++li;
  const WreduceLayer& L = A.l[li];
  const int b = blockIdx.x - L.block0;
  const int pair = b / kWredBlocks, e = (b % kWredBlocks) * 64 + (threadIdx.x & 63);
  const int w = threadIdx.x >> 6, k0 = L.nchunk * w / 4, k1 = L.nchunk * (w + 1) / 4;
  float acc = 0.f;
  if (e < kWTile) {
    const float* p = L.part + (int64_t)pair * L.nchunk * kWTile + e;
#pragma unroll 8
    for (int k = k0; k < k1; ++k) acc += p[(int64_t)k * kWTile];
  }
  s[w][threadIdx.x & 63] = acc;
  __syncthreads();
  if (w != 0 || e >= kWTile) return;
  const int l = threadIdx.x;
  const float v = ((s[0][l] + s[1][l]) + s[2][l]) + s[3][l];
  const int cit = pair / L.nco, cot = pair % L.nco;
  if (e < 27 * 256) {
    const int t = e / 256, ci = cit * 16 + (e / 16) % 16, co = cot * 16 + e % 16;
    if (ci < L.cin) L.dw[((int64_t)t * L.cin + ci) * L.cout + co] = v;
  } else if (cit == 0) {
    L.db[cot * 16 + (e - 27 * 256)] = v;
  }
}

// ---------------------------------------------------------------- elementwise

// 2x2x2 mean: coarse [nc][C] from fine [2nc][C]; one thread per 8 channels.
__global__ void k_pool(const uint16_t* xf, uint16_t* xc, int c0, int c1, int c2, int C) {
  const int cc = C >> 3;
  const int64_t n = (int64_t)c0 * c1 * c2 * cc;
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int h = (int)(e % cc);
  const int64_t v = e / cc;
  const int k = (int)(v % c2), j = (int)((v / c2) % c1), i = (int)(v / ((int64_t)c1 * c2));
  float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int c = 0; c < 2; ++c) {
        const size_t f = ((size_t)(2 * i + a) * (2 * c1) + (2 * j + b)) * (2 * c2) + (2 * k + c);
        const uint16_t* p = xf + f * C + h * 8;
        for (int q = 0; q < 8; ++q) s[q] += bf2f(p[q]);
      }
  uint16_t* o = xc + v * C + h * 8;
  for (int q = 0; q < 8; ++q) o[q] = f2bf(s[q] * 0.125f);
}

// Eight BF16 values as floats and back.
__device__ inline void widen8(const uint16_t* p, float (&f)[8]) {
  const u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
  for (int q = 0; q < 8; ++q) f[q] = bf2f((uint16_t)(v[q >> 1] >> (16 * (q & 1))));
}

__device__ inline void narrow8(const float (&f)[8], uint16_t* p) {
  u32x4 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = (uint32_t)f2bf(f[2 * q]) | ((uint32_t)f2bf(f[2 * q + 1]) << 16);
  *reinterpret_cast<u32x4*>(p) = v;
}

// Gradient through the mean pool, plus the skip-connection gradient, through
// the ReLU of the pooled layer's output y: gf[fine] = 0.125 * gc[fine / 2] +
// skip[fine] where y > 0, else 0. One thread per 8 channels.
__global__ void k_pool_bwd(const uint16_t* gc, const uint16_t* skip, const uint16_t* y, uint16_t* gf, int f0, int f1,
                           int f2, int C) {
  const int cc = C >> 3;
  const int64_t n = (int64_t)f0 * f1 * f2 * cc;
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int h = (int)(e % cc) * 8;
  const int64_t v = e / cc;
  const int k = (int)(v % f2), j = (int)((v / f2) % f1), i = (int)(v / ((int64_t)f1 * f2));
  const size_t vc = ((size_t)(i >> 1) * (f1 >> 1) + (j >> 1)) * (f2 >> 1) + (k >> 1);
  float a[8], b[8], g[8], o[8];
  widen8(gc + vc * C + h, a);
  widen8(skip + v * C + h, b);
  widen8(y + v * C + h, g);
#pragma unroll
  for (int q = 0; q < 8; ++q) o[q] = g[q] > 0.f ? 0.125f * a[q] + b[q] : 0.f;
  narrow8(o, gf + v * C + h);
}

// Gradient through nearest upsampling (coarse = sum of its 8 fine children)
// and the ReLU of the coarse layer's output y. One thread per 8 channels.
__global__ void k_upsum(const uint16_t* gf, const uint16_t* y, uint16_t* gc, int c0, int c1, int c2, int C) {
  const int cc = C >> 3;
  const int64_t n = (int64_t)c0 * c1 * c2 * cc;
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int h = (int)(e % cc) * 8;
  const int64_t v = e / cc;
  const int k = (int)(v % c2), j = (int)((v / c2) % c1), i = (int)(v / ((int64_t)c1 * c2));
  float s[8] = {0, 0, 0, 0, 0, 0, 0, 0}, g[8];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const size_t f = ((size_t)(2 * i + a) * (2 * c1) + (2 * j + b)) * (2 * c2) + (2 * k + c);
        float t[8];
        widen8(gf + f * C + h, t);
#pragma unroll
        for (int q = 0; q < 8; ++q) s[q] += t[q];
      }
  widen8(y + v * C + h, g);
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (!(g[q] > 0.f)) s[q] = 0.f;
  narrow8(s, gc + v * C + h);
}

// Weight packing. Forward: wp[q][co][j] = W[tap][c0 + j][co] with q = (tap, c0/8)
// (zero for q >= nq). Data-gradient (taps mirrored, channel roles swapped):
// wd[q'][ci][j] = W[26 - tap'][ci][o0 + j] with q' = (tap', o0/8).
__global__ void k_pack(const float* W, uint16_t* wp, int cin, int cout, int nqp, int mirror) {
  const int ci_in = mirror ? cout : cin;   // channels of the GEMM's K side
  const int co_out = mirror ? cin : cout;  // output channels
  const int cpt = ci_in >> 3;
  const int64_t n = (int64_t)nqp * co_out * 8;
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int j = (int)(e % 8), o = (int)((e / 8) % co_out), q = (int)(e / (8 * (int64_t)co_out));
  float v = 0.f;
  if (q < 27 * cpt) {
    const int tap = q / cpt, c = (q % cpt) * 8 + j;
    if (!mirror)
      v = W[((size_t)tap * cin + c) * cout + o];
    else
      v = W[((size_t)(26 - tap) * cin + o) * cout + c];
  }
  wp[e] = f2bf(v);
}

__global__ void k_adam(float* p, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ---------------------------------------------------------------- inputs, targets, loss

struct Geo {
  int n0, n1, n2;       // network grid
  int vn0, vn1, vn2;    // voxels mapped to interior nodes
  int64_t gsx, gsy;     // glue strides
  int64_t goff;         // glue index of voxel (0,0,0): node (2,2,2)
  int mcy, mcz;         // cell-mask strides: (ny+1), (nz+1)
};

// Sum of rho^2 over interior nodes (per-block partials).
__global__ __launch_bounds__(256) void k_rho2(const double* rho, Geo G, double* part) {
  __shared__ double s[256];
  const int64_t n = (int64_t)G.vn0 * G.vn1 * G.vn2;
  double acc = 0.0;
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < n; q += (int64_t)gridDim.x * 256) {
    const int k = (int)(q % G.vn2), j = (int)((q / G.vn2) % G.vn1), i = (int)(q / ((int64_t)G.vn1 * G.vn2));
    const double r = rho[G.goff + i * G.gsx + j * G.gsy + k];
    acc += r * r;
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// scal[0] = rms of rho over interior nodes (1 when rho vanishes), scal[1] = 1/scal[0].
// One block of 256 threads, fixed-order tree.
__global__ __launch_bounds__(256) void k_rho_scale(const double* part, int nb, int64_t n, double* scal) {
  __shared__ double sh[256];
  double t = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256) t += part[b];
  sh[threadIdx.x] = t;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double s = sqrt(sh[0] / (double)n);
    if (!(s > 0.0)) s = 1.0;
    scal[0] = s;
    scal[1] = 1.0 / s;
  }
}

// Node mask: 1 if any of the 8 cells around the node belongs to a conductor.
__device__ inline uint8_t node_mask(const uint8_t* cm, const Geo& G, int i, int j, int k) {
  if (!cm) return 0;
  // voxel (i,j,k) is glue node (i+2, j+2, k+2); its cells are glue cells i+1..i+2
  uint8_t m = 0;
  for (int a = 1; a <= 2; ++a)
    for (int b = 1; b <= 2; ++b)
      for (int c = 1; c <= 2; ++c) m |= cm[((size_t)(i + a) * G.mcy + (j + b)) * G.mcz + (k + c)];
  return m ? 1 : 0;
}

// Training pair from the context fields: rho_hat = rho/sigma (BF16), node
// mask, phi_hat = phi * eps0 / sigma (FP32 in, BF16 stored).
__global__ void k_store_pair(const double* rho, const double* phi, const uint8_t* cm, Geo G, const double* scal,
                             double eps0, uint16_t* drho, uint8_t* dmask, uint16_t* dphi) {
  const int64_t n = (int64_t)G.n0 * G.n1 * G.n2;
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const int k = (int)(v % G.n2), j = (int)((v / G.n2) % G.n1), i = (int)(v / ((int64_t)G.n1 * G.n2));
  float r = 0.f, p = 0.f;
  uint8_t m = 0;
  if (i < G.vn0 && j < G.vn1 && k < G.vn2) {
    const int64_t g = G.goff + i * G.gsx + j * G.gsy + k;
    r = (float)(rho[g] * scal[1]);
    p = (float)(phi[g] * eps0 * scal[1]);
    m = node_mask(cm, G, i, j, k);
  }
  drho[v] = f2bf(r);
  dmask[v] = m;
  dphi[v] = f2bf(p);
}

// Network input [voxel][8]: channel 0 rho_hat, channel 1 mask, 2..7 zero.
__global__ void k_features_pair(const uint16_t* drho, const uint8_t* dmask, uint16_t* x0, int64_t n) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  u32x4 o = {(uint32_t)drho[v] | ((uint32_t)(dmask[v] ? 0x3f80u : 0u) << 16), 0u, 0u, 0u};
  *reinterpret_cast<u32x4*>(x0 + v * 8) = o;
}

__global__ void k_features_field(const double* rho, const uint8_t* cm, Geo G, const double* scal, uint16_t* x0) {
  const int64_t n = (int64_t)G.n0 * G.n1 * G.n2;
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const int k = (int)(v % G.n2), j = (int)((v / G.n2) % G.n1), i = (int)(v / ((int64_t)G.n1 * G.n2));
  uint16_t r = 0;
  uint8_t m = 0;
  if (i < G.vn0 && j < G.vn1 && k < G.vn2) {
    r = f2bf((float)(rho[G.goff + i * G.gsx + j * G.gsy + k] * scal[1]));
    m = node_mask(cm, G, i, j, k);
  }
  u32x4 o = {(uint32_t)r | ((uint32_t)(m ? 0x3f80u : 0u) << 16), 0u, 0u, 0u};
  *reinterpret_cast<u32x4*>(x0 + v * 8) = o;
}

// eps0 (b - A phi) at the network's interior nodes, b = rho / eps0 and A the
// 7-point operator (6 phi minus the neighbours, dx = 1): the charge whose
// potential the warm start phi is still missing.
__global__ void k_warm_resid(const double* phi, const double* rho, double eps0, Geo G, double* out) {
  const int64_t n = (int64_t)G.vn0 * G.vn1 * G.vn2;
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int k = (int)(q % G.vn2), j = (int)((q / G.vn2) % G.vn1), i = (int)(q / ((int64_t)G.vn1 * G.vn2));
  const int64_t g = G.goff + i * G.gsx + j * G.gsy + k;
  const double ap = 6.0 * phi[g] - (phi[g - G.gsx] + phi[g + G.gsx] + phi[g - G.gsy] + phi[g + G.gsy] + phi[g - 1] +
                                    phi[g + 1]);
  out[g] = rho[g] - eps0 * ap;
}

// d = phi - phi_start at the interior nodes (in place into phi_start).
__global__ void k_phi_delta(const double* phi, double* d, Geo G) {
  const int64_t n = (int64_t)G.vn0 * G.vn1 * G.vn2;
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int k = (int)(q % G.vn2), j = (int)((q / G.vn2) % G.vn1), i = (int)(q / ((int64_t)G.vn1 * G.vn2));
  const int64_t g = G.goff + i * G.gsx + j * G.gsy + k;
  d[g] = phi[g] - d[g];
}

// Loss 0.5/N * sum (out - target/k)^2 over voxels of interior nodes, N their count;
// gradient into channel 0 of g [voxel][16].
__global__ __launch_bounds__(256) void k_loss(const float* out, const uint16_t* target, float inv_k, Geo G,
                                              float inv_n, uint16_t* g, double* part) {
  __shared__ double s[256];
  const int64_t n = (int64_t)G.n0 * G.n1 * G.n2;
  double acc = 0.0;
  for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < n; v += (int64_t)gridDim.x * 256) {
    const int k = (int)(v % G.n2), j = (int)((v / G.n2) % G.n1), i = (int)(v / ((int64_t)G.n1 * G.n2));
    float d = 0.f;
    if (i < G.vn0 && j < G.vn1 && k < G.vn2) d = out[v] - bf2f(target[v]) * inv_k;
    acc += 0.5 * (double)d * d;
    u32x4 z = {(uint32_t)f2bf(d * inv_n), 0u, 0u, 0u};
    *reinterpret_cast<u32x4*>(g + v * 16) = z;
    *reinterpret_cast<u32x4*>(g + v * 16 + 8) = (u32x4){0u, 0u, 0u, 0u};
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// Residual loss 0.5/N * sum q^2 with q = A (k out) - rho_hat over voxels of
// interior nodes (A the 7-point operator 6 u - sum of neighbours, the output
// taken as 0 outside those voxels): the initial relative residual the
// multigrid starts from. First pass: q and the loss partials.
__global__ __launch_bounds__(256) void k_res_loss(const float* out, const uint16_t* rho_hat, float k, Geo G,
                                                  float* q, double* part) {
  __shared__ double s[256];
  const int64_t n = (int64_t)G.n0 * G.n1 * G.n2;
  double acc = 0.0;
  for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < n; v += (int64_t)gridDim.x * 256) {
    const int kk = (int)(v % G.n2), j = (int)((v / G.n2) % G.n1), i = (int)(v / ((int64_t)G.n1 * G.n2));
    float qv = 0.f;
    if (i < G.vn0 && j < G.vn1 && kk < G.vn2) {
      auto o = [&](int a, int b, int c) -> float {
        if (a < 0 || b < 0 || c < 0 || a >= G.vn0 || b >= G.vn1 || c >= G.vn2) return 0.f;
        return out[((int64_t)a * G.n1 + b) * G.n2 + c];
      };
      const float au = 6.f * out[v] - (o(i - 1, j, kk) + o(i + 1, j, kk) + o(i, j - 1, kk) + o(i, j + 1, kk) +
                                       o(i, j, kk - 1) + o(i, j, kk + 1));
      qv = k * au - bf2f(rho_hat[v]);
    }
    q[v] = qv;
    acc += 0.5 * (double)qv * qv;
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int o2 = 128; o2 > 0; o2 >>= 1) {
    if (threadIdx.x < o2) s[threadIdx.x] += s[threadIdx.x + o2];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// Second pass: d loss / d out = (k/N) A q (A is symmetric), into channel 0 of g [voxel][16].
__global__ void k_res_grad(const float* q, float k_over_n, Geo G, uint16_t* g) {
  const int64_t n = (int64_t)G.n0 * G.n1 * G.n2;
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const int kk = (int)(v % G.n2), j = (int)((v / G.n2) % G.n1), i = (int)(v / ((int64_t)G.n1 * G.n2));
  float gv = 0.f;
  if (i < G.vn0 && j < G.vn1 && kk < G.vn2) {
    auto Q = [&](int a, int b, int c) -> float {
      if (a < 0 || b < 0 || c < 0 || a >= G.vn0 || b >= G.vn1 || c >= G.vn2) return 0.f;
      return q[((int64_t)a * G.n1 + b) * G.n2 + c];
    };
    gv = k_over_n * (6.f * q[v] - (Q(i - 1, j, kk) + Q(i + 1, j, kk) + Q(i, j - 1, kk) + Q(i, j + 1, kk) +
                                   Q(i, j, kk - 1) + Q(i, j, kk + 1)));
  }
  u32x4 z = {(uint32_t)f2bf(gv), 0u, 0u, 0u};
  *reinterpret_cast<u32x4*>(g + v * 16) = z;
  *reinterpret_cast<u32x4*>(g + v * 16 + 8) = (u32x4){0u, 0u, 0u, 0u};
}

// *out = scale * sum of the partials (one block of 256 threads, fixed tree).
__global__ __launch_bounds__(256) void k_sum_into(const double* part, int nb, double scale, double* out) {
  __shared__ double s[256];
  double t = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256) t += part[b];
  s[threadIdx.x] = t;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = s[0] * scale;
}

// Training-data objects: axis-aligned boxes of cells. Cells inside get the
// box id in the cell mask; rho at nodes with all 8 cells inside is cleared,
// rho at surface nodes (some but not all cells inside) gets the box's surface
// charge times a smooth modulation 1 + 0.5 sin(...) with per-box phases.
struct Box {
  int lo[3], hi[3];  // glue cell ranges [lo, hi)
  double q;          // surface charge per node
  double ph[3];      // modulation phases
};

__global__ void k_box_mask(uint8_t* cm, int c0, int c1, int c2, const Box* boxes, int nbox) {
  const int64_t n = (int64_t)c0 * c1 * c2;
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int k = (int)(e % c2), j = (int)((e / c2) % c1), i = (int)(e / ((int64_t)c1 * c2));
  uint8_t m = 0;
  for (int b = 0; b < nbox; ++b) {
    const Box& B = boxes[b];
    if (i >= B.lo[0] && i < B.hi[0] && j >= B.lo[1] && j < B.hi[1] && k >= B.lo[2] && k < B.hi[2]) m = (uint8_t)(b + 1);
  }
  cm[e] = m;
}

__global__ void k_box_charge(double* rho, int cx, int cy, int cz, const uint8_t* cm, const Box* boxes, int nbox) {
  const int64_t n = (int64_t)cx * cy * cz;
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int k = (int)(e % cz), j = (int)((e / cz) % cy), i = (int)(e / ((int64_t)cy * cz));
  if (i < 2 || j < 2 || k < 2 || i > cx - 3 || j > cy - 3 || k > cz - 3) return;  // interior nodes only
  int inside = 0, owner = 0;
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int c = 0; c < 2; ++c) {
        // the cell map is (cx-1) x (cy-1) x (cz-1): cell (p, q, r) spans nodes p..p+1
        const uint8_t m = cm[((size_t)(i - 1 + a) * (cy - 1) + (j - 1 + b)) * (cz - 1) + (k - 1 + c)];
        if (m) {
          ++inside;
          owner = m;
        }
      }
  if (inside == 0) return;
  if (inside == 8) {
    rho[e] = 0.0;
    return;
  }
  const Box& B = boxes[owner - 1];
  const double mod = 1.0 + 0.5 * sin(0.37 * i + B.ph[0]) * sin(0.41 * j + B.ph[1]) * sin(0.43 * k + B.ph[2]);
  rho[e] += B.q * mod;
}

}  // namespace

// ---------------------------------------------------------------- host side

struct GuessLayer {
  int cin, cout, lvl, up, relu;
  int64_t woff, boff;  // offsets in the flat parameter vector
  int nq, nqp, nqd, nqpd;
  DBuf<uint16_t> wp, wd;
};

struct GuessNet {
  Geo G{};
  int lv[4][3];
  std::vector<GuessLayer> L;
  int64_t nparams = 0;
  DBuf<float> master, grad, m1, m2;
  double k_out = 1.0;
  int64_t adam_t = 0;
  // activations (BF16 channels-last) and gradients
  DBuf<uint16_t> X0, A0, S0, P0, A1, S1, P1, A2, S2, P2, A3, B3, D2, E2, D1, E1, D0, E0;
  DBuf<float> OUT;
  DBuf<uint16_t> gOUT, gE0, gD0, gE1, gD1, gE2, gD2, gB3, gA3, gP2, gS2, gA2, gP1, gS1, gA1, gP0, gS0, gA0;
  DBuf<uint16_t> T0, T1, T2;
  bool train_alloc = false;
  std::vector<DBuf<float>> wpart;  // weight- and bias-gradient partial sums, one buffer per layer
  DBuf<double> dpart, scal, loss_acc;
  DBuf<uint8_t> cellmask;  // training-data objects
  DBuf<double> rwarm;      // eps0 (b - A phi) of the warm start at the interior nodes (modes 2 and 3)
  DBuf<double> phi_start;  // mode 3: the warm start, to form phi_solution - phi_start after the solve
  int record_slot = 0;     // mode 3: the dataset slot the next pair goes to
  bool use_cellmask = false;
  DBuf<Box> boxes;
  // dataset of training pairs
  int capacity = 0;
  DBuf<uint16_t> ds_rho, ds_phi;
  DBuf<uint8_t> ds_mask;
  std::vector<double> ds_phi_rms;
  int mode = 0;
  int loss_kind = 0;  // 0: potential MSE, 1: initial multigrid residual
  DBuf<float> q;      // residual of the guess (loss_kind 1)
  uint64_t seed = 1;
};

namespace {

int64_t nvox_of(const int* d) { return (int64_t)d[0] * d[1] * d[2]; }

void add_layer(GuessNet& g, int cin, int cout, int lvl, int up, int relu) {
  GuessLayer l;
  l.cin = cin;
  l.cout = cout;
  l.lvl = lvl;
  l.up = up;
  l.relu = relu;
  l.woff = g.nparams;
  g.nparams += 27LL * cin * cout;
  l.boff = g.nparams;
  g.nparams += cout;
  l.nq = 27 * cin / 8;
  l.nqp = (l.nq + 3) / 4 * 4;
  l.nqd = 27 * cout / 8;
  l.nqpd = (l.nqd + 3) / 4 * 4;
  g.L.push_back(std::move(l));
}

enum { E0A, E0B, E1A, E1B, E2A, E2B, E3A, E3B, D2A, D2B, D1A, D1B, D0A, D0B, OUTL, NLAYER };

void pack_all(Ctx& c, GuessNet& g) {
  for (auto& l : g.L) {
    const int64_t nf = (int64_t)l.nqp * l.cout * 8;
    k_pack<<<div_up(nf, 256), 256, 0, c.stream>>>(g.master.p + l.woff, l.wp.p, l.cin, l.cout, l.nqp, 0);
    if (l.cin % 16 == 0) {
      const int64_t nd = (int64_t)l.nqpd * l.cin * 8;
      k_pack<<<div_up(nd, 256), 256, 0, c.stream>>>(g.master.p + l.woff, l.wd.p, l.cin, l.cout, l.nqpd, 1);
    }
  }
}

template <int CIN, int NT, int EPI>
void launch_conv_t(hipStream_t st, ConvArgs& a) {
  constexpr size_t lds = conv_lds_bytes(CIN);
  grant_lds(reinterpret_cast<const void*>(&k_conv<CIN, NT, EPI>), lds);
  a.nbrick = div_up(a.n0, kBI) * div_up(a.n1, kBJ) * div_up(a.n2, kBK);
  // a few workgroups per compute unit, as many as its LDS holds, so that one
  // brick's loads and stores overlap another's products
  const int most = 256 * (int)std::max<size_t>(1, std::min<size_t>(NT <= 2 ? 3 : 2, 163840 / lds));
  k_conv<CIN, NT, EPI><<<dim3(std::min(a.nbrick, most), a.cout / (16 * NT)), 256, lds, st>>>(a);
}

template <int CIN>
void launch_conv_nt(hipStream_t st, ConvArgs& a) {
  // One tile per workgroup below 512 bricks: two workgroups per compute unit
  // want more of them than there are bricks, and the weights then fit the
  // registers (64 -> 64 at 16^3: 22.7 us with all four tiles, 15.2 us; 48 ->
  // 48 at 32^3 inside the network 30.8 and 20.3 us). From 512 bricks on every
  // fragment read serves all tiles (32 -> 32 at 64^3: 30 us).
  const int nbrick = div_up(a.n0, kBI) * div_up(a.n1, kBJ) * div_up(a.n2, kBK);
  switch (nbrick < 512 ? 1 : a.cout / 16) {
    case 1: launch_conv_t<CIN, 1, EPI_BF16>(st, a); break;
    case 2: launch_conv_t<CIN, 2, EPI_BF16>(st, a); break;
    case 3: launch_conv_t<CIN, 3, EPI_BF16>(st, a); break;
    case 4: launch_conv_t<CIN, 4, EPI_BF16>(st, a); break;
  }
}

void launch_conv(hipStream_t st, ConvArgs a, int epi, bool up) {
  if (up && (a.n0 % 2 || a.n1 % 2 || a.n2 % 2)) throw Error(FOPIS_E_ARG, "conv: upsampled grid must be even");
  if (a.cout < 16 || a.cout > 64 || a.cout % 16)
    throw Error(FOPIS_E_ARG, "conv: output channels must be 16, 32, 48 or 64");
  a.up = up ? 1 : 0;
  if (epi != EPI_BF16) {  // the output layer
    if (a.cin != 16 || a.cout != 16 || up) throw Error(FOPIS_E_ARG, "conv: the output layer is 16 -> 16 channels");
    if (epi == EPI_F32)
      launch_conv_t<16, 1, EPI_F32>(st, a);
    else
      launch_conv_t<16, 1, EPI_PHI>(st, a);
    return;
  }
  switch (a.cin) {
    case 8: launch_conv_nt<8>(st, a); break;
    case 16: launch_conv_nt<16>(st, a); break;
    case 24: launch_conv_nt<24>(st, a); break;
    case 32: launch_conv_nt<32>(st, a); break;
    case 40: launch_conv_nt<40>(st, a); break;
    case 48: launch_conv_nt<48>(st, a); break;
    case 56: launch_conv_nt<56>(st, a); break;
    case 64: launch_conv_nt<64>(st, a); break;
    default: throw Error(FOPIS_E_ARG, "conv: input channels must be 8..64, multiple of 8");
  }
}

ConvArgs conv_args(const int* d, int cin, int cout, const uint16_t* x, const uint16_t* w, const float* b, int relu) {
  ConvArgs a{};
  a.x = x;
  a.w = w;
  a.bias = b;
  a.n0 = d[0];
  a.n1 = d[1];
  a.n2 = d[2];
  a.cin = cin;
  a.cout = cout;
  a.relu = relu;
  return a;
}

template <int PI, int PO>
int wgrad_chunks(const WgradArgs& a) {
  using W = WgradShape<PI, PO>;
  const int groups = div_up(a.nci, PI) * div_up(a.nco, PO);
  const int nbrick = div_up(a.n0, W::BI) * div_up(a.n1, W::BJ) * div_up(a.n2, 32);
  // one workgroup per compute unit: more of them add partials (two per unit:
  // the sum of the partials of a 64^3 pair took 54 us instead of 35, the
  // gradients the same)
  return std::min(nbrick, std::max(1, 256 / groups));
}

template <int PI, int PO, bool UP>
void launch_wgrad_t(hipStream_t st, WgradArgs& a, int nchunk) {
  using W = WgradShape<PI, PO>;
  grant_lds(reinterpret_cast<const void*>(&k_wgrad<PI, PO, UP>), W::kLds);
  a.nbrick = div_up(a.n0, W::BI) * div_up(a.n1, W::BJ) * div_up(a.n2, 32);
  k_wgrad<PI, PO, UP><<<dim3(nchunk, div_up(a.nci, PI) * div_up(a.nco, PO)), 256, W::kLds, st>>>(a);
}

// Weight and bias gradient of one layer: the partials now, dw and db when
// wgrad_flush runs. `slot` names the layer's partial buffer.
void wgrad(Ctx& c, GuessNet& g, WgradQueue& wq, int slot, const int* d, int cin, int cout, bool up, const uint16_t* x,
           const uint16_t* gy, float* dw, float* db) {
  if (wq.a.n >= kWMaxLayers) throw Error(FOPIS_E_STATE, "more layers than a weight-gradient reduction takes");
  WgradArgs a{};
  a.x = x;
  a.g = gy;
  a.n0 = d[0];
  a.n1 = d[1];
  a.n2 = d[2];
  a.cin = cin;
  a.cout = cout;
  a.nci = (cin + 15) / 16;
  a.nco = cout / 16;
  const int kind = (a.nci > 1 ? 2 : 0) + (a.nco > 1 ? 1 : 0);
  const int nchunk = kind == 0 ? wgrad_chunks<1, 1>(a) : kind == 1 ? wgrad_chunks<1, 2>(a)
                     : kind == 2 ? wgrad_chunks<2, 1>(a) : wgrad_chunks<2, 2>(a);
  const int npairs = a.nci * a.nco;
  const size_t need = (size_t)npairs * nchunk * kWTile;
  if ((int)g.wpart.size() <= slot) g.wpart.resize(slot + 1);
  if (g.wpart[slot].n < need) {
    FOPIS_HIP(hipStreamSynchronize(c.stream));
    g.wpart[slot].alloc(need);
  }
  a.part = g.wpart[slot].p;
  auto go = [&](auto up_c) {
    constexpr bool U = decltype(up_c)::value;
    if (kind == 0)
      launch_wgrad_t<1, 1, U>(c.stream, a, nchunk);
    else if (kind == 1)
      launch_wgrad_t<1, 2, U>(c.stream, a, nchunk);
    else if (kind == 2)
      launch_wgrad_t<2, 1, U>(c.stream, a, nchunk);
    else
      launch_wgrad_t<2, 2, U>(c.stream, a, nchunk);
  };
  if (up)
    go(std::true_type{});
  else
    go(std::false_type{});
  wq.a.l[wq.a.n++] = WreduceLayer{a.part, dw, db, nchunk, cin, cout, a.nco, wq.blocks};
  wq.blocks += npairs * kWredBlocks;
}

void wgrad_flush(Ctx& c, const WgradQueue& wq) {
  if (wq.a.n > 0) k_wgrad_reduce<<<wq.blocks, 256, 0, c.stream>>>(wq.a);
}

void alloc_train(GuessNet& g) {
  if (g.train_alloc) return;
  const int64_t n0 = nvox_of(g.lv[0]), n1 = nvox_of(g.lv[1]), n2 = nvox_of(g.lv[2]), n3 = nvox_of(g.lv[3]);
  g.gOUT.alloc(n0 * 16);
  g.gE0.alloc(n0 * 16);
  g.gD0.alloc(n0 * 16);
  g.gS0.alloc(n0 * 16);
  g.gA0.alloc(n0 * 16);
  g.T0.alloc(n0 * 32);
  g.gE1.alloc(n1 * 32);
  g.gD1.alloc(n1 * 32);
  g.gS1.alloc(n1 * 32);
  g.gA1.alloc(n1 * 32);
  g.gP0.alloc(n1 * 16);
  g.T1.alloc(n1 * 48);
  g.gE2.alloc(n2 * 48);
  g.gD2.alloc(n2 * 48);
  g.gS2.alloc(n2 * 48);
  g.gA2.alloc(n2 * 48);
  g.gP1.alloc(n2 * 32);
  g.T2.alloc(n2 * 64);
  g.gB3.alloc(n3 * 64);
  g.gA3.alloc(n3 * 64);
  g.gP2.alloc(n3 * 48);
  g.m1.alloc(g.nparams);
  g.m2.alloc(g.nparams);
  FOPIS_HIP(hipMemset(g.m1.p, 0, g.nparams * sizeof(float)));
  FOPIS_HIP(hipMemset(g.m2.p, 0, g.nparams * sizeof(float)));
  g.train_alloc = true;
}

// Forward pass from g.X0. epi = EPI_F32 writes g.OUT, EPI_PHI writes phi.
void forward(Ctx& c, GuessNet& g, int epi, bool phi_add = false) {
  hipStream_t st = c.stream;
  auto conv = [&](int li, const uint16_t* x, const uint16_t* add, uint16_t* y) {
    GuessLayer& l = g.L[li];
    ConvArgs a = conv_args(g.lv[l.lvl], l.cin, l.cout, x, l.wp.p, g.master.p + l.boff, l.relu);
    a.add = add;
    a.y = y;
    launch_conv(st, a, EPI_BF16, l.up != 0);
  };
  auto pool = [&](const uint16_t* xf, uint16_t* xc, int lc, int C) {
    const int* d = g.lv[lc];
    k_pool<<<div_up(nvox_of(d) * (C / 8), 256), 256, 0, st>>>(xf, xc, d[0], d[1], d[2], C);
  };
  conv(E0A, g.X0.p, nullptr, g.A0.p);
  conv(E0B, g.A0.p, nullptr, g.S0.p);
  pool(g.S0.p, g.P0.p, 1, 16);
  conv(E1A, g.P0.p, nullptr, g.A1.p);
  conv(E1B, g.A1.p, nullptr, g.S1.p);
  pool(g.S1.p, g.P1.p, 2, 32);
  conv(E2A, g.P1.p, nullptr, g.A2.p);
  conv(E2B, g.A2.p, nullptr, g.S2.p);
  pool(g.S2.p, g.P2.p, 3, 48);
  conv(E3A, g.P2.p, nullptr, g.A3.p);
  conv(E3B, g.A3.p, nullptr, g.B3.p);
  conv(D2A, g.B3.p, g.S2.p, g.D2.p);
  conv(D2B, g.D2.p, nullptr, g.E2.p);
  conv(D1A, g.E2.p, g.S1.p, g.D1.p);
  conv(D1B, g.D1.p, nullptr, g.E1.p);
  conv(D0A, g.E1.p, g.S0.p, g.D0.p);
  conv(D0B, g.D0.p, nullptr, g.E0.p);
  GuessLayer& lo = g.L[OUTL];
  ConvArgs a = conv_args(g.lv[0], lo.cin, lo.cout, g.E0.p, lo.wp.p, g.master.p + lo.boff, 0);
  if (epi == EPI_F32) {
    a.y32 = g.OUT.p;
  } else {
    a.phi = c.phi.p;
    a.scal = g.scal.p;
    a.phi_k = g.k_out / c.d.eps0;
    a.phi_add = phi_add ? 1 : 0;
    a.gsx = g.G.gsx;
    a.gsy = g.G.gsy;
    a.goff = g.G.goff;
    a.vn0 = g.G.vn0;
    a.vn1 = g.G.vn1;
    a.vn2 = g.G.vn2;
  }
  launch_conv(st, a, epi, false);
}

// Backward pass from g.gOUT; fills g.grad.
void backward(Ctx& c, GuessNet& g) {
  hipStream_t st = c.stream;
  WgradQueue wq;
  auto wg = [&](int li, const uint16_t* x, const uint16_t* gy) {
    GuessLayer& l = g.L[li];
    wgrad(c, g, wq, li, g.lv[l.lvl], l.cin, l.cout, l.up != 0, x, gy, g.grad.p + l.woff, g.grad.p + l.boff);
  };
  // data gradient of layer li at its output grid into dx ([out voxels][cin]),
  // through the ReLU of the layer's input y where that is a layer's output
  auto dg = [&](int li, const uint16_t* gy, uint16_t* dx, const uint16_t* y = nullptr) {
    GuessLayer& l = g.L[li];
    const float* zero_bias = g.master.p + g.nparams;  // cin zeros kept after the parameters
    ConvArgs a = conv_args(g.lv[l.lvl], l.cout, l.cin, gy, l.wd.p, zero_bias, 0);
    a.y = dx;
    a.gate = y;
    launch_conv(st, a, EPI_BF16, false);
  };
  auto upsum = [&](const uint16_t* gf, const uint16_t* y, uint16_t* gcoarse, int lc, int C) {
    const int* d = g.lv[lc];
    k_upsum<<<div_up(nvox_of(d) * (C / 8), 256), 256, 0, st>>>(gf, y, gcoarse, d[0], d[1], d[2], C);
  };
  auto poolb = [&](const uint16_t* gcoarse, const uint16_t* skip, const uint16_t* y, uint16_t* gf, int lf, int C) {
    const int* d = g.lv[lf];
    k_pool_bwd<<<div_up(nvox_of(d) * (C / 8), 256), 256, 0, st>>>(gcoarse, skip, y, gf, d[0], d[1], d[2], C);
  };
  wg(OUTL, g.E0.p, g.gOUT.p);
  dg(OUTL, g.gOUT.p, g.gE0.p, g.E0.p);
  wg(D0B, g.D0.p, g.gE0.p);
  dg(D0B, g.gE0.p, g.gD0.p, g.D0.p);
  wg(D0A, g.E1.p, g.gD0.p);
  dg(D0A, g.gD0.p, g.T0.p);
  upsum(g.T0.p, g.E1.p, g.gE1.p, 1, 32);
  wg(D1B, g.D1.p, g.gE1.p);
  dg(D1B, g.gE1.p, g.gD1.p, g.D1.p);
  wg(D1A, g.E2.p, g.gD1.p);
  dg(D1A, g.gD1.p, g.T1.p);
  upsum(g.T1.p, g.E2.p, g.gE2.p, 2, 48);
  wg(D2B, g.D2.p, g.gE2.p);
  dg(D2B, g.gE2.p, g.gD2.p, g.D2.p);
  wg(D2A, g.B3.p, g.gD2.p);
  dg(D2A, g.gD2.p, g.T2.p);
  upsum(g.T2.p, g.B3.p, g.gB3.p, 3, 64);
  wg(E3B, g.A3.p, g.gB3.p);
  dg(E3B, g.gB3.p, g.gA3.p, g.A3.p);
  wg(E3A, g.P2.p, g.gA3.p);
  dg(E3A, g.gA3.p, g.gP2.p);
  poolb(g.gP2.p, g.gD2.p, g.S2.p, g.gS2.p, 2, 48);
  wg(E2B, g.A2.p, g.gS2.p);
  dg(E2B, g.gS2.p, g.gA2.p, g.A2.p);
  wg(E2A, g.P1.p, g.gA2.p);
  dg(E2A, g.gA2.p, g.gP1.p);
  poolb(g.gP1.p, g.gD1.p, g.S1.p, g.gS1.p, 1, 32);
  wg(E1B, g.A1.p, g.gS1.p);
  dg(E1B, g.gS1.p, g.gA1.p, g.A1.p);
  wg(E1A, g.P0.p, g.gA1.p);
  dg(E1A, g.gA1.p, g.gP0.p);
  poolb(g.gP0.p, g.gD0.p, g.S0.p, g.gS0.p, 0, 16);
  wg(E0B, g.A0.p, g.gS0.p);
  dg(E0B, g.gS0.p, g.gA0.p, g.A0.p);
  wg(E0A, g.X0.p, g.gA0.p);
  wgrad_flush(c, wq);
}

GuessNet& net(Ctx& c) {
  if (!c.guess) throw Error(FOPIS_E_STATE, "the learned guess is not initialised (fopis_guess_init)");
  return *c.guess;
}

void features_from_slot(Ctx& c, GuessNet& g, int slot) {
  const int64_t n = nvox_of(g.lv[0]);
  k_features_pair<<<div_up(n, 256), 256, 0, c.stream>>>(g.ds_rho.p + (size_t)slot * n, g.ds_mask.p + (size_t)slot * n,
                                                         g.X0.p, n);
}

// Loss of pair `slot` on g.OUT into *dst (device) and its gradient into g.gOUT.
void launch_loss(Ctx& c, GuessNet& g, int slot, double* dst) {
  const int64_t n = nvox_of(g.lv[0]);
  const int nb = 256;
  const double nvalid = (double)g.G.vn0 * g.G.vn1 * g.G.vn2;
  if (g.loss_kind == 1) {
    if (!g.q.p) g.q.alloc(n);
    k_res_loss<<<nb, 256, 0, c.stream>>>(g.OUT.p, g.ds_rho.p + (size_t)slot * n, (float)g.k_out, g.G, g.q.p,
                                         g.dpart.p);
    k_res_grad<<<div_up(n, 256), 256, 0, c.stream>>>(g.q.p, (float)(g.k_out / nvalid), g.G, g.gOUT.p);
  } else {
    k_loss<<<nb, 256, 0, c.stream>>>(g.OUT.p, g.ds_phi.p + (size_t)slot * n, (float)(1.0 / g.k_out), g.G,
                                     (float)(1.0 / nvalid), g.gOUT.p, g.dpart.p);
  }
  k_sum_into<<<1, 256, 0, c.stream>>>(g.dpart.p, nb, 1.0 / nvalid, dst);
}

double loss_and_grad(Ctx& c, GuessNet& g, int slot, bool sync) {
  launch_loss(c, g, slot, g.loss_acc.p);
  if (!sync) return 0.0;
  double l = 0.0;
  FOPIS_HIP(hipMemcpyAsync(&l, g.loss_acc.p, sizeof(double), hipMemcpyDeviceToHost, c.stream));
  FOPIS_HIP(hipStreamSynchronize(c.stream));
  return l;
}

void compute_scale(Ctx& c, GuessNet& g, const double* rho) {
  const int nb = 1024;
  k_rho2<<<nb, 256, 0, c.stream>>>(rho, g.G, g.dpart.p);
  k_rho_scale<<<1, 256, 0, c.stream>>>(g.dpart.p, nb, (int64_t)g.G.vn0 * g.G.vn1 * g.G.vn2, g.scal.p);
}

}  // namespace

namespace {
// Normal numbers of mean 0 by Marsaglia's polar method, with the values that
// std::normal_distribution gives here. That one's conversion of each draw takes
// two long-double logarithms: the 590 000 weights of a network took 23 or 41 ms,
// by where the linker put the function, and a new network takes 5.7 now.
struct PolarNormal {
  std::mt19937_64& rng;
  double sd, saved = 0.0;
  bool have = false;
  double uniform() {  // [0, 1)
    const double u = (double)rng() * 0x1p-64;
    return u < 1.0 ? u : std::nextafter(1.0, 0.0);
  }
  double operator()() {
    have = !have;
    if (!have) return saved * sd + 0.0;
    double x, y, r2;
    do {
      x = 2.0 * uniform() - 1.0;
      y = 2.0 * uniform() - 1.0;
      r2 = x * x + y * y;
    } while (r2 > 1.0 || r2 == 0.0);
    const double m = std::sqrt(-2.0 * std::log(r2) / r2);
    saved = x * m;
    return y * m * sd + 0.0;
  }
};
}  // namespace

// ---------------------------------------------------------------- entry points

void guess_free(Ctx& c) {
  delete c.guess;
  c.guess = nullptr;
}

void guess_init(Ctx& c, uint64_t seed) {
  guess_free(c);
  GuessNet* gp = new GuessNet();
  c.guess = gp;
  GuessNet& g = *gp;
  g.seed = seed;
  const int vn[3] = {c.nx - 2, c.ny - 2, c.nz - 2};
  for (int q = 0; q < 3; ++q) {
    const int n = (vn[q] + 7) / 8 * 8;
    for (int l = 0; l < 4; ++l) g.lv[l][q] = n >> l;
  }
  g.G.n0 = g.lv[0][0];
  g.G.n1 = g.lv[0][1];
  g.G.n2 = g.lv[0][2];
  g.G.vn0 = vn[0];
  g.G.vn1 = vn[1];
  g.G.vn2 = vn[2];
  g.G.gsx = (int64_t)c.cy * c.cz;
  g.G.gsy = c.cz;
  g.G.goff = (int64_t)c.id3(2, 2, 2);
  g.G.mcy = c.cy - 1;
  g.G.mcz = c.cz - 1;
  add_layer(g, 8, 16, 0, 0, 1);
  add_layer(g, 16, 16, 0, 0, 1);
  add_layer(g, 16, 32, 1, 0, 1);
  add_layer(g, 32, 32, 1, 0, 1);
  add_layer(g, 32, 48, 2, 0, 1);
  add_layer(g, 48, 48, 2, 0, 1);
  add_layer(g, 48, 64, 3, 0, 1);
  add_layer(g, 64, 64, 3, 0, 1);
  add_layer(g, 64, 48, 2, 1, 1);
  add_layer(g, 48, 48, 2, 0, 1);
  add_layer(g, 48, 32, 1, 1, 1);
  add_layer(g, 32, 32, 1, 0, 1);
  add_layer(g, 32, 16, 0, 1, 1);
  add_layer(g, 16, 16, 0, 0, 1);
  add_layer(g, 16, 16, 0, 0, 0);  // out: only channel 0 is used
  for (auto& l : g.L) {
    l.wp.alloc((size_t)l.nqp * l.cout * 8);
    if (l.cin % 16 == 0) l.wd.alloc((size_t)l.nqpd * l.cin * 8);
  }
  // He-normal initialisation (std::mt19937_64, fixed seed); biases zero; the
  // output layer starts small and only channel 0 is live.
  std::vector<float> h(g.nparams + 64, 0.f);
  std::mt19937_64 rng(seed);
  for (int li = 0; li < NLAYER; ++li) {
    GuessLayer& l = g.L[li];
    const int cin_live = li == E0A ? 2 : l.cin;
    const double sd = std::sqrt(2.0 / (27.0 * cin_live)) * (li == OUTL ? 0.1 : 1.0);
    PolarNormal nd{rng, sd};
    for (int t = 0; t < 27; ++t)
      for (int ci = 0; ci < l.cin; ++ci)
        for (int co = 0; co < l.cout; ++co) {
          float v = (float)nd();
          if (li == E0A && ci >= 2) v = 0.f;
          if (li == OUTL && co != 0) v = 0.f;
          h[l.woff + ((size_t)t * l.cin + ci) * l.cout + co] = v;
        }
  }
  // the parameter buffer carries 64 zeros after the parameters (zero bias of the data-gradient convs)
  g.master.alloc(g.nparams + 64);
  g.grad.alloc(g.nparams + 64);
  FOPIS_HIP(hipMemcpy(g.master.p, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
  FOPIS_HIP(hipMemset(g.grad.p, 0, (g.nparams + 64) * sizeof(float)));
  const int64_t n0 = nvox_of(g.lv[0]), n1 = nvox_of(g.lv[1]), n2 = nvox_of(g.lv[2]), n3 = nvox_of(g.lv[3]);
  g.X0.alloc(n0 * 8);
  g.A0.alloc(n0 * 16);
  g.S0.alloc(n0 * 16);
  g.D0.alloc(n0 * 16);
  g.E0.alloc(n0 * 16);
  g.P0.alloc(n1 * 16);
  g.A1.alloc(n1 * 32);
  g.S1.alloc(n1 * 32);
  g.D1.alloc(n1 * 32);
  g.E1.alloc(n1 * 32);
  g.P1.alloc(n2 * 32);
  g.A2.alloc(n2 * 48);
  g.S2.alloc(n2 * 48);
  g.D2.alloc(n2 * 48);
  g.E2.alloc(n2 * 48);
  g.P2.alloc(n3 * 48);
  g.A3.alloc(n3 * 64);
  g.B3.alloc(n3 * 64);
  g.OUT.alloc(n0);
  g.dpart.alloc(1024);
  g.scal.alloc(4);
  g.loss_acc.alloc(4096);
  pack_all(c, g);
  FOPIS_HIP(hipStreamSynchronize(c.stream));
}

int64_t guess_num_params(Ctx& c) { return net(c).nparams; }

void guess_get_params(Ctx& c, float* out, double* k_out) {
  GuessNet& g = net(c);
  FOPIS_HIP(hipStreamSynchronize(c.stream));
  FOPIS_HIP(hipMemcpy(out, g.master.p, g.nparams * sizeof(float), hipMemcpyDeviceToHost));
  if (k_out) *k_out = g.k_out;
}

void guess_set_params(Ctx& c, const float* in, double k_out) {
  GuessNet& g = net(c);
  if (!(k_out > 0.0)) throw Error(FOPIS_E_ARG, "output scale must be positive");
  FOPIS_HIP(hipMemcpyAsync(g.master.p, in, g.nparams * sizeof(float), hipMemcpyHostToDevice, c.stream));
  g.k_out = k_out;
  pack_all(c, g);
  FOPIS_HIP(hipStreamSynchronize(c.stream));
}

void guess_set_loss(Ctx& c, int kind) {
  if (kind != 0 && kind != 1) throw Error(FOPIS_E_ARG, "loss kind must be 0 or 1");
  net(c).loss_kind = kind;
}

void guess_set_mode(Ctx& c, int mode) {
  if (mode < 0 || mode > 3) throw Error(FOPIS_E_ARG, "guess mode must be 0, 1, 2 or 3");
  if (mode != 0) net(c);
  if (c.guess) {
    c.guess->mode = mode;
    if (mode == 3) c.guess->record_slot = 0;
  }
}

int guess_mode(const Ctx& c) { return c.guess ? c.guess->mode : 0; }

// Modes 2 and 3 before the first solve of a step: the warm start's residual
// (in charge units) into rwarm. Mode 2 then adds the network's potential for
// that charge to phi; mode 3 keeps phi for the pair recorded after the solve.
void guess_before_solve(Ctx& c) {
  GuessNet& g = net(c);
  Phase ph(c, "guess");
  g.rwarm.alloc(c.nnode);
  const int64_t n = (int64_t)g.G.vn0 * g.G.vn1 * g.G.vn2;
  k_warm_resid<<<div_up(n, 256), 256, 0, c.stream>>>(c.phi.p, c.rho.p, c.d.eps0, g.G, g.rwarm.p);
  if (g.mode == 3) {
    g.phi_start.alloc(c.nnode);
    FOPIS_HIP(hipMemcpyAsync(g.phi_start.p, c.phi.p, c.nnode * sizeof(double), hipMemcpyDeviceToDevice, c.stream));
    return;
  }
  compute_scale(c, g, g.rwarm.p);
  const uint8_t* cm = g.use_cellmask ? g.cellmask.p : (c.have_mask ? c.mask.p : nullptr);
  k_features_field<<<div_up(nvox_of(g.lv[0]), 256), 256, 0, c.stream>>>(g.rwarm.p, cm, g.G, g.scal.p, g.X0.p);
  forward(c, g, EPI_PHI, true);
  FOPIS_HIP(hipGetLastError());
}

// Mode 3 after the solve: the pair (eps0 r0 / sigma, mask, (phi - phi_start) eps0 / sigma)
// into the next dataset slot, while there is room.
void guess_after_solve(Ctx& c) {
  GuessNet& g = net(c);
  if (g.mode != 3 || g.record_slot >= g.capacity || !g.phi_start.p) return;
  const int64_t n = (int64_t)g.G.vn0 * g.G.vn1 * g.G.vn2;
  k_phi_delta<<<div_up(n, 256), 256, 0, c.stream>>>(c.phi.p, g.phi_start.p, g.G);
  compute_scale(c, g, g.rwarm.p);
  const int slot = g.record_slot++;
  const int64_t nv = nvox_of(g.lv[0]);
  const uint8_t* cm = g.use_cellmask ? g.cellmask.p : (c.have_mask ? c.mask.p : nullptr);
  k_store_pair<<<div_up(nv, 256), 256, 0, c.stream>>>(g.rwarm.p, g.phi_start.p, cm, g.G, g.scal.p, c.d.eps0,
                                                     g.ds_rho.p + (size_t)slot * nv, g.ds_mask.p + (size_t)slot * nv,
                                                     g.ds_phi.p + (size_t)slot * nv);
  std::vector<uint16_t> h(nv);
  FOPIS_HIP(hipMemcpyAsync(h.data(), g.ds_phi.p + (size_t)slot * nv, nv * sizeof(uint16_t), hipMemcpyDeviceToHost,
                           c.stream));
  FOPIS_HIP(hipStreamSynchronize(c.stream));
  double s = 0.0;
  for (int64_t v = 0; v < nv; ++v) {
    const double x = bf2f(h[v]);
    s += x * x;
  }
  g.ds_phi_rms[slot] = std::sqrt(s / ((double)g.G.vn0 * g.G.vn1 * g.G.vn2));
}

int guess_recorded(const Ctx& c) { return c.guess ? c.guess->record_slot : 0; }

// phi at interior nodes <- network(rho[0], conductor mask).
void guess_apply(Ctx& c) {
  GuessNet& g = net(c);
  Phase ph(c, "guess");
  compute_scale(c, g, c.rho.p);
  const uint8_t* cm = g.use_cellmask ? g.cellmask.p : (c.have_mask ? c.mask.p : nullptr);
  const int64_t n = nvox_of(g.lv[0]);
  k_features_field<<<div_up(n, 256), 256, 0, c.stream>>>(c.rho.p, cm, g.G, g.scal.p, g.X0.p);
  forward(c, g, EPI_PHI);
  FOPIS_HIP(hipGetLastError());
}

void guess_dataset_alloc(Ctx& c, int capacity) {
  GuessNet& g = net(c);
  if (capacity < 1) throw Error(FOPIS_E_ARG, "dataset capacity must be >= 1");
  const int64_t n = nvox_of(g.lv[0]);
  g.ds_rho.alloc((size_t)capacity * n);
  g.ds_phi.alloc((size_t)capacity * n);
  g.ds_mask.alloc((size_t)capacity * n);
  g.capacity = capacity;
  g.ds_phi_rms.assign(capacity, 0.0);
}

static void check_slot(const GuessNet& g, int slot) {
  if (slot < 0 || slot >= g.capacity) throw Error(FOPIS_E_ARG, "dataset slot out of range");
}

// Store (rho[0], node mask, phi) of the context as pair `slot`; returns the rms of phi_hat.
double guess_dataset_store(Ctx& c, int slot) {
  GuessNet& g = net(c);
  check_slot(g, slot);
  compute_scale(c, g, c.rho.p);
  const int64_t n = nvox_of(g.lv[0]);
  const uint8_t* cm = g.use_cellmask ? g.cellmask.p : (c.have_mask ? c.mask.p : nullptr);
  k_store_pair<<<div_up(n, 256), 256, 0, c.stream>>>(c.rho.p, c.phi.p, cm, g.G, g.scal.p, c.d.eps0,
                                                    g.ds_rho.p + (size_t)slot * n, g.ds_mask.p + (size_t)slot * n,
                                                    g.ds_phi.p + (size_t)slot * n);
  std::vector<uint16_t> h(n);
  FOPIS_HIP(hipMemcpyAsync(h.data(), g.ds_phi.p + (size_t)slot * n, n * sizeof(uint16_t), hipMemcpyDeviceToHost,
                           c.stream));
  FOPIS_HIP(hipStreamSynchronize(c.stream));
  double s = 0.0;
  for (int64_t v = 0; v < n; ++v) {
    const double x = bf2f(h[v]);
    s += x * x;
  }
  const double nvalid = (double)g.G.vn0 * g.G.vn1 * g.G.vn2;
  g.ds_phi_rms[slot] = std::sqrt(s / nvalid);
  return g.ds_phi_rms[slot];
}

void guess_dataset_get(Ctx& c, int slot, uint16_t* rho_hat, uint8_t* mask, uint16_t* phi_hat) {
  GuessNet& g = net(c);
  check_slot(g, slot);
  const int64_t n = nvox_of(g.lv[0]);
  FOPIS_HIP(hipStreamSynchronize(c.stream));
  if (rho_hat) copy_out(rho_hat, g.ds_rho.p + (size_t)slot * n, n * 2, c.stream);
  if (mask) copy_out(mask, g.ds_mask.p + (size_t)slot * n, n, c.stream);
  if (phi_hat) copy_out(phi_hat, g.ds_phi.p + (size_t)slot * n, n * 2, c.stream);
}

void guess_dataset_set(Ctx& c, int slot, const uint16_t* rho_hat, const uint8_t* mask, const uint16_t* phi_hat) {
  GuessNet& g = net(c);
  check_slot(g, slot);
  const int64_t n = nvox_of(g.lv[0]);
  FOPIS_HIP(hipStreamSynchronize(c.stream));
  copy_in(g.ds_rho.p + (size_t)slot * n, rho_hat, n * 2, c.stream);
  copy_in(g.ds_mask.p + (size_t)slot * n, mask, n, c.stream);
  copy_in(g.ds_phi.p + (size_t)slot * n, phi_hat, n * 2, c.stream);
  double s = 0.0;
  for (int64_t v = 0; v < n; ++v) {
    const double x = bf2f(phi_hat[v]);
    s += x * x;
  }
  g.ds_phi_rms[slot] = std::sqrt(s / ((double)g.G.vn0 * g.G.vn1 * g.G.vn2));
}

// Loss and flat parameter gradient on pair `slot` (no update).
double guess_grad(Ctx& c, int slot, float* grad_out) {
  GuessNet& g = net(c);
  check_slot(g, slot);
  alloc_train(g);
  features_from_slot(c, g, slot);
  forward(c, g, EPI_F32);
  loss_and_grad(c, g, slot, false);
  backward(c, g);
  double l = 0.0;
  FOPIS_HIP(hipMemcpyAsync(&l, g.loss_acc.p, sizeof(double), hipMemcpyDeviceToHost, c.stream));
  FOPIS_HIP(hipStreamSynchronize(c.stream));
  if (grad_out) copy_out(grad_out, g.grad.p, g.nparams * sizeof(float), c.stream);
  FOPIS_HIP(hipGetLastError());
  return l;
}

// Adam over pairs [0, nsamples) for `epochs` passes in shuffled order; the
// learning rate follows a cosine from lr to lr_end. loss_out[e] = mean loss of epoch e.
void guess_train(Ctx& c, int nsamples, int epochs, double lr, double lr_end, uint64_t seed, double* loss_out) {
  GuessNet& g = net(c);
  if (nsamples < 1 || nsamples > g.capacity) throw Error(FOPIS_E_ARG, "nsamples out of range of the dataset");
  if (epochs < 1) throw Error(FOPIS_E_ARG, "epochs must be >= 1");
  alloc_train(g);
  {
    // output scale: rms of phi_hat over the training pairs
    double s = 0.0;
    for (int i = 0; i < nsamples; ++i) s += g.ds_phi_rms[i] * g.ds_phi_rms[i];
    s = std::sqrt(s / nsamples);
    if (g.adam_t == 0 && s > 0.0) g.k_out = s;
  }
  std::mt19937_64 rng(seed);
  std::vector<int> order(nsamples);
  for (int i = 0; i < nsamples; ++i) order[i] = i;
  const int64_t total = (int64_t)epochs * nsamples;
  int64_t step = 0;
  const int nacc = 4096;
  for (int e = 0; e < epochs; ++e) {
    std::shuffle(order.begin(), order.end(), rng);
    double esum = 0.0;
    int pending = 0;
    auto flush = [&]() {
      if (!pending) return;
      std::vector<double> h(pending);
      FOPIS_HIP(hipMemcpyAsync(h.data(), g.loss_acc.p + 1, pending * sizeof(double), hipMemcpyDeviceToHost,
                               c.stream));
      FOPIS_HIP(hipStreamSynchronize(c.stream));
      for (double x : h) esum += x;
      pending = 0;
    };
    for (int i = 0; i < nsamples; ++i) {
      const int slot = order[i];
      features_from_slot(c, g, slot);
      forward(c, g, EPI_F32);
      launch_loss(c, g, slot, g.loss_acc.p + 1 + pending);
      ++pending;
      backward(c, g);
      ++g.adam_t;
      const double frac = (double)step / std::max<int64_t>(1, total - 1);
      const double lr_t = lr_end + (lr - lr_end) * 0.5 * (1.0 + std::cos(M_PI * frac));
      const float b1 = 0.9f, b2 = 0.999f;
      const float c1 = 1.f - std::pow(b1, (float)g.adam_t), c2 = 1.f - std::pow(b2, (float)g.adam_t);
      k_adam<<<div_up(g.nparams, 256), 256, 0, c.stream>>>(g.master.p, g.grad.p, g.m1.p, g.m2.p, g.nparams,
                                                           (float)lr_t, b1, b2, 1e-8f, c1, c2);
      pack_all(c, g);
      ++step;
      if (pending == nacc - 1) flush();
    }
    flush();
    if (loss_out) loss_out[e] = esum / nsamples;
  }
  FOPIS_HIP(hipStreamSynchronize(c.stream));
  FOPIS_HIP(hipGetLastError());
}

// Mean loss over pairs [begin, end) with the current parameters.
double guess_eval(Ctx& c, int begin, int end) {
  GuessNet& g = net(c);
  if (begin < 0 || end > g.capacity || begin >= end) throw Error(FOPIS_E_ARG, "bad pair range");
  alloc_train(g);
  double s = 0.0;
  for (int i = begin; i < end; ++i) {
    features_from_slot(c, g, i);
    forward(c, g, EPI_F32);
    s += loss_and_grad(c, g, i, true);
  }
  return s / (end - begin);
}

// Training-data conductor boxes: sets the guess's own cell mask and edits rho[0].
void guess_synth_boxes(Ctx& c, int nbox, const int32_t* lohi, const double* q, uint64_t seed) {
  GuessNet& g = net(c);
  if (nbox < 0 || nbox > 8) throw Error(FOPIS_E_ARG, "nbox must be 0..8");
  const int c0 = c.cx - 1, c1 = c.cy - 1, c2 = c.cz - 1;
  std::vector<Box> hb(std::max(nbox, 1));
  std::mt19937_64 rng(seed);
  std::uniform_real_distribution<double> ud(0.0, 6.283185307179586);
  for (int b = 0; b < nbox; ++b) {
    for (int a = 0; a < 3; ++a) {
      hb[b].lo[a] = lohi[6 * b + a];
      hb[b].hi[a] = lohi[6 * b + 3 + a];
      const int lim = a == 0 ? c0 : (a == 1 ? c1 : c2);
      if (hb[b].lo[a] < 1 || hb[b].hi[a] > lim - 1 || hb[b].lo[a] >= hb[b].hi[a])
        throw Error(FOPIS_E_ARG, "box outside the grid's interior cells");
    }
    hb[b].q = q[b];
    for (int a = 0; a < 3; ++a) hb[b].ph[a] = ud(rng);
  }
  g.cellmask.alloc((size_t)c0 * c1 * c2);
  g.boxes.alloc(hb.size());
  FOPIS_HIP(hipMemcpyAsync(g.boxes.p, hb.data(), hb.size() * sizeof(Box), hipMemcpyHostToDevice, c.stream));
  const int64_t nm = (int64_t)c0 * c1 * c2;
  k_box_mask<<<div_up(nm, 256), 256, 0, c.stream>>>(g.cellmask.p, c0, c1, c2, g.boxes.p, nbox);
  k_box_charge<<<div_up((int64_t)c.nnode, 256), 256, 0, c.stream>>>(c.rho.p, c.cx, c.cy, c.cz, g.cellmask.p,
                                                                     g.boxes.p, nbox);
  g.use_cellmask = nbox > 0;
  FOPIS_HIP(hipStreamSynchronize(c.stream));
  FOPIS_HIP(hipGetLastError());
}

void guess_clear_boxes(Ctx& c) { net(c).use_cellmask = false; }

// ---- single-layer entry points (host buffers) for tests and benchmarks

namespace {
struct TmpStream {
  hipStream_t s = nullptr;
  TmpStream() { FOPIS_HIP(hipStreamCreate(&s)); }
  ~TmpStream() {
    if (s) (void)hipStreamDestroy(s);
  }
};

void check_conv_shape(int n0, int n1, int n2, int cin, int cout, int up) {
  if (n0 < 1 || n1 < 1 || n2 < 1) throw Error(FOPIS_E_ARG, "grid must be positive");
  if (cin < 8 || cin > 64 || cin % 8) throw Error(FOPIS_E_ARG, "cin must be 8..64, multiple of 8");
  if (cout < 16 || cout > 64 || cout % 16) throw Error(FOPIS_E_ARG, "cout must be 16, 32, 48 or 64");
  if (up && (n0 % 2 || n1 % 2 || n2 % 2)) throw Error(FOPIS_E_ARG, "upsampled grid must be even");
}
}  // namespace

void nn_conv3d(int n0, int n1, int n2, int cin, int cout, int up, int relu, const uint16_t* x, const float* w,
               const float* b, const uint16_t* add, uint16_t* y, int reps, float* ms) {
  check_conv_shape(n0, n1, n2, cin, cout, up);
  TmpStream ts;
  const int64_t nv = (int64_t)n0 * n1 * n2, nin = up ? nv / 8 : nv;
  const int nq = 27 * cin / 8, nqp = (nq + 3) / 4 * 4;
  DBuf<uint16_t> dx, dy, dadd, dwp;
  DBuf<float> dw, db;
  dx.alloc(nin * cin);
  dy.alloc(nv * cout);
  dw.alloc(27LL * cin * cout);
  db.alloc(cout);
  dwp.alloc((size_t)nqp * cout * 8);
  if (add) dadd.alloc(nv * cout);
  const HostSeg up_seg[4] = {{const_cast<uint16_t*>(x), dx.p, (size_t)(nin * cin * 2)},
                             {const_cast<float*>(w), dw.p, (size_t)(27LL * cin * cout * 4)},
                             {const_cast<float*>(b), db.p, (size_t)cout * 4},
                             {const_cast<uint16_t*>(add), dadd.p, (size_t)(nv * cout * 2)}};
  host_copy(up_seg, add ? 4 : 3, false, ts.s);
  k_pack<<<div_up((int64_t)nqp * cout * 8, 256), 256, 0, ts.s>>>(dw.p, dwp.p, cin, cout, nqp, 0);
  const int dims[3] = {n0, n1, n2};
  ConvArgs a = conv_args(dims, cin, cout, dx.p, dwp.p, db.p, relu);
  a.add = add ? dadd.p : nullptr;
  a.y = dy.p;
  launch_conv(ts.s, a, EPI_BF16, up != 0);
  if (reps > 0 && ms) {
    hipEvent_t e0, e1;
    FOPIS_HIP(hipEventCreate(&e0));
    FOPIS_HIP(hipEventCreate(&e1));
    FOPIS_HIP(hipEventRecord(e0, ts.s));
    for (int r = 0; r < reps; ++r) launch_conv(ts.s, a, EPI_BF16, up != 0);
    FOPIS_HIP(hipEventRecord(e1, ts.s));
    FOPIS_HIP(hipEventSynchronize(e1));
    FOPIS_HIP(hipEventElapsedTime(ms, e0, e1));
    *ms /= reps;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
  }
  FOPIS_HIP(hipStreamSynchronize(ts.s));
  FOPIS_HIP(hipGetLastError());
  copy_out(y, dy.p, nv * cout * 2, ts.s);
}

void nn_conv3d_backward(int n0, int n1, int n2, int cin, int cout, int up, const uint16_t* x, const float* w,
                        const uint16_t* gy, float* dw_out, float* db_out, uint16_t* dx_out) {
  check_conv_shape(n0, n1, n2, cin, cout, up);
  if (dx_out && cin % 16) throw Error(FOPIS_E_ARG, "data gradient needs cin multiple of 16");
  TmpStream ts;
  const int64_t nv = (int64_t)n0 * n1 * n2, nin = up ? nv / 8 : nv;
  DBuf<uint16_t> dx, dg, dwd, ddx;
  DBuf<float> dw, dgw, dgb, zb;
  dx.alloc(nin * cin);
  dg.alloc(nv * cout);
  dw.alloc(27LL * cin * cout);
  dgw.alloc(27LL * cin * cout);
  dgb.alloc(cout);
  zb.alloc(64);
  const HostSeg up_seg[3] = {{const_cast<uint16_t*>(x), dx.p, (size_t)(nin * cin * 2)},
                             {const_cast<uint16_t*>(gy), dg.p, (size_t)(nv * cout * 2)},
                             {const_cast<float*>(w), dw.p, (size_t)(27LL * cin * cout * 4)}};
  host_copy(up_seg, 3, false, ts.s);
  FOPIS_HIP(hipMemsetAsync(zb.p, 0, 64 * 4, ts.s));
  // weight and bias gradients through a throwaway network object
  GuessNet tmp;
  Ctx cc;
  cc.stream = ts.s;
  const int dims[3] = {n0, n1, n2};
  WgradQueue wq;
  wgrad(cc, tmp, wq, 0, dims, cin, cout, up != 0, dx.p, dg.p, dgw.p, dgb.p);
  wgrad_flush(cc, wq);
  cc.stream = nullptr;
  if (dx_out) {
    const int nqd = 27 * cout / 8, nqpd = (nqd + 3) / 4 * 4;
    dwd.alloc((size_t)nqpd * cin * 8);
    k_pack<<<div_up((int64_t)nqpd * cin * 8, 256), 256, 0, ts.s>>>(dw.p, dwd.p, cin, cout, nqpd, 1);
    ddx.alloc(nv * cin);
    ConvArgs a = conv_args(dims, cout, cin, dg.p, dwd.p, zb.p, 0);
    a.y = ddx.p;
    launch_conv(ts.s, a, EPI_BF16, false);
    copy_out(dx_out, ddx.p, nv * cin * 2, ts.s);
  }
  FOPIS_HIP(hipStreamSynchronize(ts.s));
  FOPIS_HIP(hipGetLastError());
  copy_out(dw_out, dgw.p, 27LL * cin * cout * 4, ts.s);
  FOPIS_HIP(hipMemcpy(db_out, dgb.p, cout * 4, hipMemcpyDeviceToHost));
}

}  // namespace fopis
