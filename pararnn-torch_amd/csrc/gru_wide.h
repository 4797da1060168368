// Device code shared by the wide-head kernels (gru_wide.hip: the walks, the
// gates and the one-launch Newton solve; gru_wide_rev.hip: the adjoint walk):
// lane roles, the A entries a lane keeps, the pair products, the staging of
// a block's per-step inputs and the argument checks.
#pragma once

#include <type_traits>

#include "prnn_common.h"
#include "pararnn_amd.h"
#include "prnn_host.h"

namespace prnn {
namespace gruw {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int DW = 128;       // widest head
constexpr int kParts = 16;    // parts of the contraction index
constexpr int kKP = DW / kParts;  // contraction entries per lane (8)
constexpr int kCh = 4;        // channels per lane group
constexpr int kK = kCh * kKP;  // entries per lane and matrix (32)
constexpr int kThreads = DW / kCh * kParts;
// A broadcast vector sits in LDS in two halves of 64 entries, the second
// shifted by four words (bank spread of the segments one wave reads).
constexpr int kVec = DW + 4;
__device__ __forceinline__ int slot(int c) { return c + (c >> 6) * 4; }

// torch.lerp(start, end, weight) for fp32 (the cell's update).
__device__ __forceinline__ float lerp_t(float s, float e, float w) {
  return w < 0.5f ? s + w * (e - s) : e - (e - s) * (1.f - w);
}

// Steps [t0, t1) of batch row `row` that workgroup `seq / H` walks: a batch
// row (rectangular) or a packed sequence of one stream (cu != nullptr).
struct Span {
  int row, t0, t1, seq;
};
__device__ __forceinline__ Span span_of(int s, int T, const int* cu) {
  if (cu == nullptr) return Span{s, 0, T, s};
  return Span{0, cu[s], cu[s + 1], s};
}

// Lane roles.  The 16 lanes of a DPP row hold a group of four channels and the
// 16 parts of the contraction index, entries k in [8 j, 8 j + 8) for part j: a
// product reads 8 entries of the broadcast vector (two 16-byte LDS words) and
// feeds four channels (the walks are bound by LDS reads and VALU issue; with 8
// parts of 16 entries and two channels the one-launch solve took 0.72 us per
// step).  After the reduction the lanes 4 q .. 4 q + 3 hold channel q of the
// group; the first of them writes it.
struct Role {
  int part, c;
  bool wr;
};
__device__ __forceinline__ Role role() {
  const int lane = threadIdx.x & 63;
  Role o;
  o.part = lane & (kParts - 1);
  o.c = kCh * ((threadIdx.x >> 6) * 4 + (lane >> 4)) + (o.part >> 2);
  o.wr = (o.part & 3) == 0;
  return o;
}

// Entries k in [8 j, 8 j + 8) of columns (COL) or rows c ^ i, i = 0 .. 3, of a
// head's A ((in, out) layout, d_head x d_head), zero outside the head:
// a[4 kk + i] = A[k][c ^ i] (COL) or A[c ^ i][k].
template <typename TX, bool COL>
__device__ __forceinline__ void load_group(const TX* A, int dh, const Role& ro, float a[kK]) {
#pragma unroll
  for (int kk = 0; kk < kKP; ++kk)
#pragma unroll
    for (int i = 0; i < kCh; ++i) {
      const int k = ro.part * kKP + kk, ch = ro.c ^ i;
      const bool in = ch < dh && k < dh;
      a[kCh * kk + i] =
          in ? ld(A + (COL ? static_cast<size_t>(k) * dh + ch : static_cast<size_t>(ch) * dh + k))
             : 0.f;
    }
}

// A step's per-channel inputs (z, r, n, the previous state, and the iterate
// or dL/dH) are staged through LDS kS steps at a time: while a block of kS
// steps is walked from LDS, every lane holds its share of the next block's
// loads in registers and writes them to the other LDS buffer at the end of
// the block.  A walk step is short, so loads issued per step would expose
// the memory latency every step; here it overlaps kS steps of work.
constexpr int kS = 16;                     // steps per staged block
constexpr int kIn = 5;                     // inputs per step and channel
constexpr int kPer = kIn * kS * DW / kThreads;  // staged values per lane (20)

struct Staged {
  float v[kPer];
};

// Lane `tid` loads values j = 0 .. kPer-1 of the block whose steps are
// t_first + dir * s (s < kS): input j / 4, step s = tid / DW + 4 (j % 4),
// channel tid % DW (clamped into the head and the sequence: the values
// outside are never used).
template <typename TG>
__device__ __forceinline__ Staged load_block(const float* __restrict__ z,
                                             const float* __restrict__ r,
                                             const float* __restrict__ n,
                                             const float* __restrict__ hp,
                                             const TG* __restrict__ x, size_t row_base, int d,
                                             int head, int dh, int t_first, int dir, int t_lo,
                                             int t_hi) {
  const int cc = min(static_cast<int>(threadIdx.x) & (DW - 1), dh - 1);
  const size_t colb = row_base + static_cast<size_t>(head) * dh + cc;
  Staged st;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int s = static_cast<int>(threadIdx.x) / DW + 4 * (j % 4);
    const int t = min(max(t_first + dir * s, t_lo), t_hi);
    const size_t at = colb + static_cast<size_t>(t) * d;
    const int a = j / 4;
    st.v[j] = a == 0 ? z[at] : a == 1 ? r[at] : a == 2 ? n[at] : a == 3 ? hp[at] : ld(x + at);
  }
  return st;
}

// Calls put(step, channel, z, r, n, hp, x) for the lane's four elements; dead
// channels hold zeros.
template <typename Put>
__device__ __forceinline__ void take_block(const Staged& st, int dh, Put&& put) {
  const int cc = static_cast<int>(threadIdx.x) & (DW - 1);
  const bool in = cc < dh;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    auto at = [&](int i) { return in ? st.v[4 * i + j] : 0.f; };
    put(static_cast<int>(threadIdx.x) / DW + 4 * j, cc, at(0), at(1), at(2), at(3), at(4));
  }
}

// A lane's value from the lane the DPP control names (every lane has a
// source for the controls used here).  Written as an update with old = 0 and
// bound_ctrl so that the compiler folds the move into the add that consumes
// it (v_add_f32 with a DPP operand): one instruction per reduction step.
template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// The lane's entries of a vector in LDS.
struct Seg {
  float4 x, y;
};
__device__ __forceinline__ Seg load_seg(const float* __restrict__ v, const Role& ro) {
  const float4* p = reinterpret_cast<const float4*>(v + slot(ro.part * kKP));
  return Seg{p[0], p[1]};
}

// sum_k A v for this lane's channel c (every lane of the channel gets it).
// s[i] is the lane's part of channel c ^ i.  Parts p and 15 - p (row_mirror)
// differ in both upper bits, so what this lane keeps, channels c and c ^ 1, are
// the other's s[3] and s[2]; then p and p ^ 7 (row_half_mirror), which keep c and
// c ^ 1; then the four parts of a quad.  The halving costs no selects, as a
// lane's own channel is always s[0].
__device__ __forceinline__ float dot_seg(const float a[kK], const Seg& v) {
  const float e[kKP] = {v.x.x, v.x.y, v.x.z, v.x.w, v.y.x, v.y.y, v.y.z, v.y.w};
  float s[kCh];
#pragma unroll
  for (int i = 0; i < kCh; ++i) s[i] = a[i] * e[0];
#pragma unroll
  for (int k = 1; k < kKP; ++k)
#pragma unroll
    for (int i = 0; i < kCh; ++i) s[i] = fmaf(a[kCh * k + i], e[k], s[i]);
  s[1] += dppf<0x140>(s[2]);
  s[0] += dppf<0x140>(s[3]);
  s[0] += dppf<0x141>(s[1]);
  s[0] += dppf<0xB1>(s[0]);
  s[0] += dppf<0x4E>(s[0]);
  return s[0];
}
__device__ __forceinline__ float dot(const float a[kK], const float* __restrict__ v,
                                     const Role& ro) {
  return dot_seg(a, load_seg(v, ro));
}

// The scalars of a step and channel, formed once when a block is staged (each
// channel's lanes would repeat them): J v = d1 v + d2 (A_z^T v) + d3 A_n^T (r v +
// d5 (A_r^T v)) with d1 = 1 - z, d2 = (n - h) z (1 - z), d3 = z (1 - n^2),
// d5 = h r (1 - r) (reference cells/para_gru.py:385-412).
struct Scalars {
  float d1, d2, d3, d5;
};
__device__ __forceinline__ Scalars scalars(float z, float r, float n, float h) {
  return Scalars{1.f - z, (n - h) * z * (1.f - z), z * (1.f - n * n), h * r * (1.f - r)};
}

static int check(int B, int T, int H, int dh, int dtype, const int* cu, int n_seq) {
  if (B < 1 || T < 1 || H < 1)
    return fail(PRNN_ERR_VALUE, "B, T, n_heads must be >= 1, got B=%d T=%d n_heads=%d", B, T, H);
  if (dh < 1 || dh > DW) return fail(PRNN_ERR_TYPE, "d_head must be in [1, %d], got %d", DW, dh);
  if (check_dtype(dtype) != PRNN_OK) return PRNN_ERR_TYPE;
  // one batch row's outputs are addressed with 32-bit buffer offsets
  if (static_cast<long long>(T) * 3 * H * dh * sizeof(float) >= (1ll << 32))
    return fail(PRNN_ERR_VALUE, "a batch row of T * 3 * d fp32 values must stay below 4 GiB");
  if (cu != nullptr && (B != 1 || n_seq < 1 || n_seq > T))
    return fail(PRNN_ERR_VALUE, "a packed stream has B = 1 and n_seq in [1, T], got B=%d n_seq=%d",
                B, n_seq);
  return PRNN_OK;
}

}  // namespace gruw
}  // namespace prnn
