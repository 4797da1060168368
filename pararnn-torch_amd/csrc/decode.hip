// T = 1 decode: one recurrent step per call, for the serving loop
// (reference kernels/decode.py:119-597).  These kernels are cell.step: project
// the input, or take it projected, read the state row
// (or the pool slot block_table[b]), the recurrent parameters (clamped to
// +-cap in-kernel, as the reference does so a captured graph allocates
// nothing) and the step's wx, and write the next state row.  fp32 algebra,
// 16-bit storage (bf16, fp16) widened on load and rounded on store.
//
//  slstm_decode_kernel     ParaSLSTM mix='diag': one thread per channel.
//  gru_diag_decode_kernel  ParaGRU mix='diag': one thread per channel.
//  gru_head_decode_kernel  ParaGRU mix='head' (d_head = 64): one wave per
//                          (b, head); lane j forms column j of h A_z, h A_r,
//                          (h r) A_n from the head's A columns with h broadcast
//                          through LDS.  (The reference runs this mix through
//                          the eager cell.step.)
//  project_kernel          W_x(x) of the step, and for the diagonal mixes the
//                          step with it, further down.
#include <cstdint>

#include "prnn_common.h"
#include "pararnn_amd.h"
#include "prnn_host.h"

namespace prnn {
namespace decode {

__device__ __forceinline__ float cap_to(float v, float cap, bool has_cap) {
  return has_cap ? fminf(fmaxf(v, -cap), cap) : v;
}

__device__ __forceinline__ int slot_of(const int* bt, int b) { return bt ? bt[b] : b; }

// torch.lerp(start, end, weight) for fp32 (the head cell's update).
__device__ __forceinline__ float lerp_t(float s, float e, float w) {
  return w < 0.5f ? s + w * (e - s) : e - (e - s) * (1.f - w);
}

// One channel's sLSTM step from the gates' pre-activations z; s and o point at
// its c, the other components d apart.
template <typename TX>
__device__ __forceinline__ void slstm_step(const TX* s, TX* o, int d, const float z[4], float eps) {
  const float c = ld(s), n = ld(s + d), m = ld(s + 2 * d);
  const float left = z[1] + m;
  const float mn = fmaxf(left, z[0]);
  // one of f, i is exactly e^0 = 1 (the larger exponent is the stabiliser)
  const float e = fexp(-fabsf(left - z[0]));
  const bool lf = left >= z[0];
  const float f = lf ? 1.f : e, i = lf ? e : 1.f;
  const float nn = f * n + i;
  const float cn = f * c + i * ftanh(z[2]);
  const float hn = fsigmoid(z[3]) * (cn / (nn + eps));
  st(o, cn);
  st(o + d, nn);
  st(o + 2 * d, mn);
  st(o + 3 * d, hn);
}

template <typename TX>
__global__ __launch_bounds__(256) void slstm_decode_kernel(
    const TX* __restrict__ state, const TX* __restrict__ wx, const TX* __restrict__ r,
    TX* __restrict__ out, const int* __restrict__ bt, int d, float eps, float cap, int has_cap) {
  const int b = blockIdx.y;
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= d) return;
  const size_t row = static_cast<size_t>(slot_of(bt, b)) * 4 * d;
  const TX* x = wx + static_cast<size_t>(b) * 4 * d + j;
  float z[4];
  const float h = ld(state + row + 3 * d + j);
#pragma unroll
  for (int g = 0; g < 4; ++g) z[g] = cap_to(ld(r + g * d + j), cap, has_cap) * h + ld(x + g * d);
  slstm_step(state + row + j, out + row + j, d, z, eps);
}

// One channel's diagonal GRU step; v: the projected input's z, r, n.
__device__ __forceinline__ float gru_step(float h, float az, float ar, float an, const float* v) {
  const float z = fsigmoid(az * h + v[0]);
  const float rr = fsigmoid(ar * h + v[1]);
  const float n = ftanh(an * (h * rr) + v[2]);
  return (1.f - z) * h + z * n;
}

template <typename TX>
__global__ __launch_bounds__(256) void gru_diag_decode_kernel(
    const TX* __restrict__ hin, const TX* __restrict__ wx, const TX* __restrict__ a_z,
    const TX* __restrict__ a_r, const TX* __restrict__ a_n, TX* __restrict__ out,
    const int* __restrict__ bt, int d, float cap, int has_cap) {
  const int b = blockIdx.y;
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= d) return;
  const size_t row = static_cast<size_t>(slot_of(bt, b)) * d;
  const float h = ld(hin + row + j);
  const TX* x = wx + static_cast<size_t>(b) * 3 * d + j;
  const float v[3] = {ld(x), ld(x + d), ld(x + 2 * d)};
  st(out + row + j, gru_step(h, cap_to(ld(a_z + j), cap, has_cap), cap_to(ld(a_r + j), cap, has_cap),
                             cap_to(ld(a_n + j), cap, has_cap), v));
}

constexpr int DH = 64;

template <typename TX>
__global__ __launch_bounds__(64) void gru_head_decode_kernel(
    const TX* __restrict__ hin, const TX* __restrict__ wx, const TX* __restrict__ a_z,
    const TX* __restrict__ a_r, const TX* __restrict__ a_n, TX* __restrict__ out,
    const int* __restrict__ bt, int H, float cap, int has_cap) {
  __shared__ float s_v[DH];
  const int b = blockIdx.y, head = blockIdx.x, j = threadIdx.x;
  const int d = H * DH;
  const size_t row = static_cast<size_t>(slot_of(bt, b)) * d + head * DH;
  const float h = ld(hin + row + j);
  const TX* x = wx + static_cast<size_t>(b) * 3 * d + head * DH + j;
  const size_t hoff = static_cast<size_t>(head) * DH * DH + j;  // column j of the head's (in, out) matrices
  s_v[j] = h;
  __syncthreads();
  float gz = 0.f, gr = 0.f;
#pragma unroll 8
  for (int i = 0; i < DH; ++i) {
    const float v = s_v[i];
    gz += v * cap_to(ld(a_z + hoff + i * DH), cap, has_cap);
    gr += v * cap_to(ld(a_r + hoff + i * DH), cap, has_cap);
  }
  const float z = fsigmoid(gz + ld(x));
  const float rr = fsigmoid(gr + ld(x + d));
  __syncthreads();
  s_v[j] = h * rr;
  __syncthreads();
  float gn = 0.f;
#pragma unroll 8
  for (int i = 0; i < DH; ++i) gn += s_v[i] * cap_to(ld(a_n + hoff + i * DH), cap, has_cap);
  const float n = ftanh(gn + ld(x + 2 * d));
  st(out + row + j, lerp_t(h, n, z));
}

// ---- the step's projection --------------------------------------------------
// wx = x W^T + bias for the few rows of a step, rounded to the storage type as a
// GEMM's result is, and (MIX) the cell's step on it while it is on the chip.
//
// Bound: reading W once (8.4 MB at d = d_in = 1024 in 16 bits: 1.6 us at the rate
// of a large copy), and on the host the dispatch of a GEMM: a live bf16 step of
// 64 rows at d = 1024 took 38 us, 20 of them in the library call, and takes 19; the
// GPU's part, replayed from a graph, 8.6 -> 7.1 us (1 row: 8.3 -> 4.2).  Beyond the
// reads a workgroup's chain counts: operands, products, partial sums through LDS,
// state.
//
// A workgroup takes 4 NT channels of every gate -- NT MFMA column tiles, whose
// columns are 4 gates x 4 channels -- for 16 MT rows, so the step's inputs meet in
// one workgroup.  Its KW waves split the contraction: each holds its whole share
// of both operands in flight, and their partial sums meet in LDS in a fixed order.
// Products are exact (16-bit) or fp32, sums fp32.
enum Mix { kProject = 0, kSlstm = 1, kGruDiag = 2 };

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// 16 bytes of each operand: k entries of row (A) or column (B) lane % 16; the four
// lane groups hold different k, the same on both sides.
template <typename TX>
__device__ __forceinline__ f32x4 mma(const uint4& a, const uint4& b, f32x4 c);
template <>
__device__ __forceinline__ f32x4 mma<bf16>(const uint4& a, const uint4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mma<f16>(const uint4& a, const uint4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mma<float>(const uint4& a, const uint4& b, f32x4 c) {
  const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], c, 0, 0, 0);
  return c;
}

struct Step {
  const void *x, *w, *bias;
  const void *state, *r0, *r1, *r2;  // r0: the sLSTM's R, or the GRU's a_z, a_r, a_n
  void* out;                         // next state, or wx (kProject)
  const int* bt;
  int B, d, d_in, gates;
  float eps, cap;
  int has_cap;
};

template <typename TX, int MIX, int NT, int MT>
__global__ __launch_bounds__(512) void project_kernel(Step p) {
  constexpr int kE = 16 / sizeof(TX);  // entries per 16-byte load
  constexpr int KW = 8;                // waves
  constexpr int kLoads = 4;            // such loads per lane, row and turn
  constexpr int kTurn = 4 * kLoads * kE;
  constexpr int COLS = 16 * NT, ROWS = 16 * MT;
  __shared__ float s_acc[KW][ROWS][COLS + 4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int c0 = blockIdx.x * 4 * NT, b0 = blockIdx.y * ROWS;
  const TX* x = static_cast<const TX*>(p.x);
  const TX* w = static_cast<const TX*>(p.w);
  // rows past the batch, channels past d and absent gates read a valid row whose
  // result is not used
  const TX *ax[MT], *bw[NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
    ax[m] = x + static_cast<size_t>(min(b0 + 16 * m + col, p.B - 1)) * p.d_in;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int g = min(col >> 2, p.gates - 1), c = min(c0 + 4 * n + (col & 3), p.d - 1);
    bw[n] = w + (static_cast<size_t>(g) * p.d + c) * p.d_in;
  }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int kb = wave * kTurn; kb < p.d_in; kb += KW * kTurn) {
    uint4 a[MT][kLoads], b[NT][kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int k = kb + (j * 4 + grp) * kE;
      const bool in = k < p.d_in;  // d_in is a multiple of kE
#pragma unroll
      for (int n = 0; n < NT; ++n)
        b[n][j] = in ? *reinterpret_cast<const uint4*>(bw[n] + k) : uint4{0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < MT; ++m)
        a[m][j] = in ? *reinterpret_cast<const uint4*>(ax[m] + k) : uint4{0, 0, 0, 0};
    }
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = mma<TX>(a[m][j], b[n][j], acc[m][n]);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        s_acc[wave][16 * m + 4 * grp + i][16 * n + col] = acc[m][n][i];
  __syncthreads();
  const TX* bias = static_cast<const TX*>(p.bias);
  for (int it = threadIdx.x; it < ROWS * 4 * NT; it += 64 * KW) {
    const int row = it / (4 * NT), ch = it % (4 * NT);
    const int b = b0 + row, c = c0 + ch;
    if (b >= p.B || c >= p.d) continue;
    float v[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (g < p.gates) {
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < KW; ++k) s += s_acc[k][row][(ch >> 2) * 16 + 4 * g + (ch & 3)];
        if (bias != nullptr) s += ld(bias + static_cast<size_t>(g) * p.d + c);
        v[g] = round_to<TX>(s);
      }
    }
    if constexpr (MIX == kProject) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if (g < p.gates)
          st(static_cast<TX*>(p.out) + (static_cast<size_t>(b) * p.gates + g) * p.d + c, v[g]);
    } else {
      const size_t at =
          static_cast<size_t>(slot_of(p.bt, b)) * (MIX == kSlstm ? 4 : 1) * p.d + c;
      const TX* s = static_cast<const TX*>(p.state) + at;
      TX* o = static_cast<TX*>(p.out) + at;
      const TX *r0 = static_cast<const TX*>(p.r0) + c, *r1 = static_cast<const TX*>(p.r1) + c,
               *r2 = static_cast<const TX*>(p.r2) + c;
      if constexpr (MIX == kSlstm) {
        const float h = ld(s + 3 * p.d);
        float z[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) z[g] = cap_to(ld(r0 + g * p.d), p.cap, p.has_cap) * h + v[g];
        slstm_step(s, o, p.d, z, p.eps);
      } else {
        st(o, gru_step(ld(s), cap_to(ld(r0), p.cap, p.has_cap), cap_to(ld(r1), p.cap, p.has_cap),
                       cap_to(ld(r2), p.cap, p.has_cap), v));
      }
    }
  }
}

// Tiles: 4 channels per workgroup while that gives every CU at most one, 8 beyond
// (the rows of x, read by every workgroup, then cost half as much: bf16 B=64,
// d=1024 9.2 -> 7.1 us); 32 batch rows, 64 where that would still be more than
// one workgroup per CU (B=128: 11.0 -> 9.6 us).
template <int MIX>
int launch_project(const Step& p, int dtype, hipStream_t s) {
  return with_storage(dtype, [&](auto tag) {
    using TX = decltype(tag);
    const unsigned g4 = (p.d + 3) / 4, g8 = (p.d + 7) / 8, r32 = (p.B + 31) / 32;
    const dim3 wg(512);
    if (static_cast<long long>(g4) * r32 <= 256) {
      if (p.B <= 16)
        project_kernel<TX, MIX, 1, 1><<<dim3(g4), wg, 0, s>>>(p);
      else
        project_kernel<TX, MIX, 1, 2><<<dim3(g4, r32), wg, 0, s>>>(p);
    } else if (p.B <= 16) {
      project_kernel<TX, MIX, 2, 1><<<dim3(g8), wg, 0, s>>>(p);
    } else if (static_cast<long long>(g8) * r32 <= 256) {
      project_kernel<TX, MIX, 2, 2><<<dim3(g8, r32), wg, 0, s>>>(p);
    } else {
      project_kernel<TX, MIX, 2, 4><<<dim3(g8, (p.B + 63) / 64), wg, 0, s>>>(p);
    }
    PRNN_HIP(hipGetLastError());
    return static_cast<int>(PRNN_OK);
  });
}

static int check(int B, int d, int dtype) {
  if (B < 1 || d < 1) return fail(PRNN_ERR_VALUE, "B and d must be >= 1, got B=%d d=%d", B, d);
  if (check_dtype(dtype) != PRNN_OK) return PRNN_ERR_TYPE;
  if (B > 65535) return fail(PRNN_ERR_VALUE, "batch %d exceeds 65535", B);
  return PRNN_OK;
}

}  // namespace decode
}  // namespace prnn

using namespace prnn;

extern "C" PRNN_API int prnn_slstm_decode(const void* state, const void* wx, const void* r,
                                          void* out, const int* block_table, int B, int d,
                                          float eps, float cap, int has_cap, int dtype,
                                          void* stream) {
  int rc = decode::check(B, d, dtype);
  if (rc != PRNN_OK) return rc;
  if (!state || !wx || !r || !out)
    return fail(PRNN_ERR_VALUE, "state, wx, r and out must be non-null");
  const dim3 grid((d + 255) / 256, B);
  hipStream_t s = static_cast<hipStream_t>(stream);
  with_storage(dtype, [&](auto tag) {
    using TX = decltype(tag);
    decode::slstm_decode_kernel<TX><<<grid, dim3(256), 0, s>>>(
        static_cast<const TX*>(state), static_cast<const TX*>(wx), static_cast<const TX*>(r),
        static_cast<TX*>(out), block_table, d, eps, cap, has_cap);
    return PRNN_OK;
  });
  PRNN_HIP(hipGetLastError());
  return PRNN_OK;
}

extern "C" PRNN_API int prnn_gru_decode(const void* h, const void* wx, const void* a_z,
                                        const void* a_r, const void* a_n, void* out,
                                        const int* block_table, int B, int d, int n_heads,
                                        float cap, int has_cap, int dtype, void* stream) {
  int rc = decode::check(B, d, dtype);
  if (rc != PRNN_OK) return rc;
  if (!h || !wx || !a_z || !a_r || !a_n || !out)
    return fail(PRNN_ERR_VALUE, "h, wx, a_z, a_r, a_n and out must be non-null");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (n_heads > 0) {
    if (d != n_heads * decode::DH)
      return fail(PRNN_ERR_TYPE, "head decode needs d_head = 64, got d=%d n_heads=%d", d,
                  n_heads);
    const dim3 grid(n_heads, B);
    with_storage(dtype, [&](auto tag) {
      using TX = decltype(tag);
      decode::gru_head_decode_kernel<TX><<<grid, dim3(64), 0, s>>>(
          static_cast<const TX*>(h), static_cast<const TX*>(wx), static_cast<const TX*>(a_z),
          static_cast<const TX*>(a_r), static_cast<const TX*>(a_n), static_cast<TX*>(out),
          block_table, n_heads, cap, has_cap);
      return PRNN_OK;
    });
  } else {
    const dim3 grid((d + 255) / 256, B);
    with_storage(dtype, [&](auto tag) {
      using TX = decltype(tag);
      decode::gru_diag_decode_kernel<TX><<<grid, dim3(256), 0, s>>>(
          static_cast<const TX*>(h), static_cast<const TX*>(wx), static_cast<const TX*>(a_z),
          static_cast<const TX*>(a_r), static_cast<const TX*>(a_n), static_cast<TX*>(out),
          block_table, d, cap, has_cap);
      return PRNN_OK;
    });
  }
  PRNN_HIP(hipGetLastError());
  return PRNN_OK;
}

namespace prnn {
namespace decode {

static int check_project(const void* x, const void* w, int B, int d, int d_in, int dtype) {
  const int rc = check(B, d, dtype);
  if (rc != PRNN_OK) return rc;
  const int size = dtype == PRNN_F32 ? 4 : 2;
  if (d_in < 1 || d_in * static_cast<long long>(size) % 16 != 0)
    return fail(PRNN_ERR_VALUE, "rows of x and W must be whole 16-byte words, got d_in=%d", d_in);
  if (!x || !w || reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16)
    return fail(PRNN_ERR_VALUE, "x and W must be non-null and 16-byte aligned");
  return PRNN_OK;
}

}  // namespace decode
}  // namespace prnn

extern "C" PRNN_API int prnn_slstm_decode_x(const void* state, const void* x, const void* w,
                                            const void* bias, const void* r, void* out,
                                            const int* block_table, int B, int d, int d_in,
                                            float eps, float cap, int has_cap, int dtype,
                                            void* stream) {
  const int rc = decode::check_project(x, w, B, d, d_in, dtype);
  if (rc != PRNN_OK) return rc;
  if (!state || !r || !out) return fail(PRNN_ERR_VALUE, "state, r and out must be non-null");
  const decode::Step p{x,  w, bias, state, r, r, r, out, block_table, B, d, d_in, 4,
                       eps, cap, has_cap};
  return decode::launch_project<decode::kSlstm>(p, dtype, static_cast<hipStream_t>(stream));
}

extern "C" PRNN_API int prnn_gru_decode_x(const void* h, const void* x, const void* w,
                                          const void* bias, const void* a_z, const void* a_r,
                                          const void* a_n, void* wx, void* out,
                                          const int* block_table, int B, int d, int d_in,
                                          int n_heads, float cap, int has_cap, int dtype,
                                          void* stream) {
  const int rc = decode::check_project(x, w, B, d, d_in, dtype);
  if (rc != PRNN_OK) return rc;
  if (!h || !a_z || !a_r || !a_n || !out)
    return fail(PRNN_ERR_VALUE, "h, a_z, a_r, a_n and out must be non-null");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (n_heads == 0) {
    const decode::Step p{x, w, bias, h, a_z, a_r, a_n, out, block_table, B, d, d_in, 3,
                         0.f, cap, has_cap};
    return decode::launch_project<decode::kGruDiag>(p, dtype, s);
  }
  if (!wx) return fail(PRNN_ERR_VALUE, "wx must be non-null for a head GRU");
  if (d != n_heads * decode::DH)
    return fail(PRNN_ERR_TYPE, "head decode needs d_head = 64, got d=%d n_heads=%d", d, n_heads);
  const decode::Step p{x, w, bias, nullptr, nullptr, nullptr, nullptr, wx, nullptr, B, d, d_in, 3,
                       0.f, cap, has_cap};
  const int pr = decode::launch_project<decode::kProject>(p, dtype, s);
  if (pr != PRNN_OK) return pr;
  return prnn_gru_decode(h, wx, a_z, a_r, a_n, out, block_table, B, d, n_heads, cap, has_cap,
                         dtype, stream);
}
