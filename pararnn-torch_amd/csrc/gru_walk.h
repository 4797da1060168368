// Walks over time for 64-wide head GRUs: device code shared by the Newton
// walk and the adjoint walk (gru_walk.hip), and their launchers.
//
// A workgroup of 256 lanes owns one (sequence, head).  Its lanes play two
// roles at once:
//  * the walk, one step at a time: 16 groups of 4 channels x 16 parts of the
//    contraction index.  A lane keeps 4 entries of each of the three matrices
//    for the 4 channels of its group (a product reads one 16-byte LDS word) and
//    the 16 parts of a group, a DPP row, meet through five DPP adds; LDS and a
//    barrier only broadcast the two vectors the products read;
//  * the gates of the next block of 16 steps, which do not depend on the walk,
//    as fp32 MFMA products (16 steps x 64 channels x 64, wave w the columns
//    16 w .. + 15), a few MFMA per walk step, in the shadow of the walk's LDS
//    and barrier latencies.
// The gates become the per-step scalars that the walk multiplies by, written
// to LDS once per channel, so that the walk's chain per step is the three
// products and six fused multiply-adds.
#pragma once

#include "gru_wide.h"

namespace prnn {
namespace gruk {

using gruw::dppf;
using gruw::floatx4;
using gruw::lerp_t;
using gruw::Scalars;
using gruw::scalars;

constexpr int DH = 64;
constexpr int kBlk = 16;          // steps per block
constexpr int kThreads = 256;
constexpr int kPad = DH + 4;      // LDS row stride of the MFMA operands (bank spread)
constexpr int kEnt = 4;           // contraction entries per lane
constexpr int kParts = DH / kEnt;
constexpr int kChan = 4;          // channels per lane group

struct Lane {
  int c, part;         // walk: channel and part; `wr` lanes write the channel
  bool wr;
  int li, g, wave, col;  // MFMA: lane % 16, lane / 16, output channel
};

__device__ __forceinline__ Lane lane_roles() {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  Lane o;
  o.part = lane & (kParts - 1);
  // channel 2 b1 + b0 of the group with (b1, b0) the part's upper bits (see dot_seg)
  o.c = kChan * (4 * wave + (lane >> 4)) + (o.part >> 2);
  o.wr = (o.part & 3) == 0;
  o.li = lane & 15;
  o.g = lane >> 4;
  o.wave = wave;
  o.col = 16 * wave + o.li;
  return o;
}

// Entries k in [4 part, 4 part + 4) of columns (COL) or rows c ^ i, i = 0 .. 3, of
// a head's (in, out) matrix: a[4 kk + i].
constexpr int kKeep = kChan * kEnt;
template <typename TX, bool COL>
__device__ __forceinline__ void load_group(const TX* A, const Lane& l, float a[kKeep]) {
#pragma unroll
  for (int kk = 0; kk < kEnt; ++kk)
#pragma unroll
    for (int i = 0; i < kChan; ++i) {
      const int k = l.part * kEnt + kk, ch = l.c ^ i;
      a[kChan * kk + i] = ld(A + (COL ? k * DH + ch : ch * DH + k));
    }
}

// The lane's entries of a vector in LDS.
using Seg = float4;
__device__ __forceinline__ Seg load_seg(const float* __restrict__ v, const Lane& l) {
  return *reinterpret_cast<const float4*>(v + l.part * kEnt);
}

// sum_k a v for this lane's channel c.  s[i] is the lane's part of channel c ^ i;
// parts p and 15 - p (row_mirror) differ in both upper bits, so what this lane
// keeps, channels c and c ^ 1, are the other's s[3] and s[2]; then p and p ^ 7
// (row_half_mirror), which keep c and c ^ 1; then the four parts of a quad.  The
// halving costs no selects, as a lane's own channel is always s[0].
__device__ __forceinline__ float dot_seg(const float a[kKeep], const Seg& v) {
  const float e[kEnt] = {v.x, v.y, v.z, v.w};
  float s[kChan];
#pragma unroll
  for (int i = 0; i < kChan; ++i) s[i] = a[i] * e[0];
#pragma unroll
  for (int k = 1; k < kEnt; ++k)
#pragma unroll
    for (int i = 0; i < kChan; ++i) s[i] = fmaf(a[kChan * k + i], e[k], s[i]);
  s[1] += dppf<0x140>(s[2]);
  s[0] += dppf<0x140>(s[3]);
  s[0] += dppf<0x141>(s[1]);
  s[0] += dppf<0xB1>(s[0]);
  s[0] += dppf<0x4E>(s[0]);
  return s[0];
}

// The gate products of one block, in slices.  Row i of the block's previous
// states is hp[i] (LDS); lane (li, g) supplies row li's entries 16 g .. + 15
// and holds column `col` of each matrix at the same entries.
struct GateOps {
  float bz[16], br[16], bn[16];
  template <typename TX>
  __device__ __forceinline__ void load(const TX* az, const TX* ar, const TX* an, const Lane& l) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int at = (16 * l.g + k) * DH + l.col;
      bz[k] = ld(az + at);
      br[k] = ld(ar + at);
      bn[k] = ld(an + at);
    }
  }
};

struct GateAcc {
  float av[16];
  floatx4 z, r, n, n1;  // n in two chains
};

__device__ __forceinline__ floatx4 mma(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void load_rows(const float (*rows)[kPad], const Lane& l, float av[16]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 f = *reinterpret_cast<const float4*>(&rows[l.li][16 * l.g + 4 * q]);
    av[4 * q] = f.x;
    av[4 * q + 1] = f.y;
    av[4 * q + 2] = f.z;
    av[4 * q + 3] = f.w;
  }
}

// Slice s = 0 .. 31 of a block's gates, two beside each walk step (one in the
// shadow of each of its LDS reads): h A_z and h A_r (slices 0-15), the gates z, r
// and the rows h r (16), (h r) A_n (18-25), then `done` with z, r, n at rows 4 g
// + v (26).  A barrier separates slices 16 and 18.  x: the block's wx at the
// lane's rows and column, as loaded; free after slice 26.
constexpr int kSlices = 32;
template <typename TX, typename Done>
__device__ __forceinline__ void gate_slice(int s, const GateOps& b, GateAcc& a,
                                           const float (*hp)[kPad], float (*hr)[kPad],
                                           const TX x[3][4], const Lane& l, Done&& done) {
  if (s == 0) {
    load_rows(hp, l, a.av);
    a.z = a.r = a.n = a.n1 = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  if (s < 16) {
    a.z = mma(a.av[s], b.bz[s], a.z);
    a.r = mma(a.av[s], b.br[s], a.r);
  }
  if (s == 16) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 4 * l.g + v;
      a.z[v] = fsigmoid(a.z[v] + to_f32(x[0][v]));
      a.r[v] = fsigmoid(a.r[v] + to_f32(x[1][v]));
      hr[row][l.col] = hp[row][l.col] * a.r[v];
    }
  }
  if (s == 18) load_rows(hr, l, a.av);
  if (s >= 18 && s < 26) {
    a.n = mma(a.av[2 * (s - 18)], b.bn[2 * (s - 18)], a.n);
    a.n1 = mma(a.av[2 * (s - 18) + 1], b.bn[2 * (s - 18) + 1], a.n1);
  }
  if (s == 26) {
#pragma unroll
    for (int v = 0; v < 4; ++v) a.n[v] = ftanh((a.n[v] + a.n1[v]) + to_f32(x[2][v]));
    done();
  }
}

// The adjoint walk of every (sequence, block head); see gru_walk.hip.
template <typename TX>
void launch_walk_reverse(const TX* wx, const TX* az, const TX* ar, const TX* an, const TX* h0,
                         const TX* states, const TX* grad, TX* g_wx, float* r_out, float* g_h0,
                         int T, int H, int n_rows, int n_chunks, int chunk, const int* cu,
                         hipStream_t stream);

}  // namespace gruk
}  // namespace prnn
