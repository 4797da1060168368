// max |f(H_{t-1}, x_t) - H_t| of a ParaGRU mix='head' trajectory, any head
// width up to 128: the residual gate of the Newton solve (reference
// solvers/newton/__init__.py:582-636).
//
// The tensor-op form is three batched products over every row, ~15 elementwise
// passes and a reduction.  Here a block keeps one head's three matrices in
// registers and walks tiles of 32 rows (row = one (b, t)): the previous
// states go to LDS once, the products run as fp32 MFMA and the gates, the new
// state and the difference stay in registers.  Every intermediate is rounded
// to the storage type where the tensor ops round theirs (products and sums in
// fp32, as the batched products accumulate).
//
// Bound: the fp32 products and the accurate exp / tanh between two barriers
// per tile; 8 heads of 64, B = 4, T = 32768, fp32 (1.07 GB read once, 26 GFLOP):
// 0.48 ms = 2.2 TB/s, against 2.0 ms of tensor ops and 1.6 ms for projecting
// the input again.
#include "prnn_host.h"

#include <algorithm>

namespace prnn {
namespace gru {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kResRows = 32;

// D(16x16) += A(16x4) B(4x16): lane l holds A[l%16][l/16], B[l/16][l%16],
// D[4(l/16)+v][l%16].
__device__ __forceinline__ floatx4 mma(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The tensor ops' sigmoid and lerp (accurate exp, IEEE division).
__device__ __forceinline__ float sigmoid_op(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float lerp_op(float s, float e, float w) {
  return fabsf(w) < 0.5f ? s + w * (e - s) : e - (e - s) * (1.f - w);
}

// KP: head width padded to 64 or 128 (zero rows and columns), one wave per 16
// columns.  The contraction of lane group g = lane / 16
// runs over k = g KP/4 .. + KP/4 - 1 (any order serves, as both operands
// agree), so a lane's A operands are contiguous in LDS.
template <typename TX, int KP>
__global__ __launch_bounds__(4 * KP) void gru_residual_kernel(
    const TX* __restrict__ wx, const TX* __restrict__ a_z, const TX* __restrict__ a_r,
    const TX* __restrict__ a_n, const TX* __restrict__ h0, const TX* __restrict__ states,
    unsigned* __restrict__ out, long long rows, int T, int H, int dh, long long n_tiles,
    const int* __restrict__ cu, int n_seq) {
  constexpr int KG = KP / 4, W = KP / 16, S = KP + 4;
  __shared__ __attribute__((aligned(16))) float sh[kResRows][S], su[kResRows][S];
  __shared__ long long s_src[kResRows];
  __shared__ unsigned s_max[W];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, g = lane >> 4;
  const int head = blockIdx.x % H;
  const int col = 16 * wave + li;
  const size_t d = static_cast<size_t>(H) * dh;
  auto rt_ = [](float v) { return round_to<TX>(v); };

  float bz[KG], br[KG], bn[KG];
#pragma unroll
  for (int k = 0; k < KG; ++k) {
    const int row = g * KG + k;
    const bool in = row < dh && col < dh;
    const size_t at = (static_cast<size_t>(head) * dh + (in ? row : 0)) * dh + (in ? col : 0);
    bz[k] = in ? ld(a_z + at) : 0.f;
    br[k] = in ? ld(a_r + at) : 0.f;
    bn[k] = in ? ld(a_n + at) : 0.f;
  }

  unsigned top = 0u;  // |F| as its bit pattern: NaN above infinity
  for (long long tile = blockIdx.x / H; tile < n_tiles; tile += gridDim.x / H) {
    const long long row0 = tile * kResRows;
    __syncthreads();  // the previous tile's reads of LDS are done
    if (threadIdx.x < kResRows) {
      // element offset of the row's previous state in `states`, -1 for zeros,
      // or -2 - (offset in h0)
      const long long k = row0 + threadIdx.x;
      long long src = -1;
      if (k < rows) {
        int q = -1;
        if (cu != nullptr) {
          int lo = 0, hi = n_seq;
          while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (cu[mid] <= k)
              lo = mid;
            else
              hi = mid;
          }
          if (cu[lo] == k) q = lo;
        } else if (k % T == 0) {
          q = static_cast<int>(k / T);
        }
        if (q < 0)
          src = (k - 1) * static_cast<long long>(d) + head * dh;
        else if (h0 != nullptr)
          src = -2 - (q * static_cast<long long>(d) + head * dh);
      }
      s_src[threadIdx.x] = src;
    }
    // this lane's inputs, in flight over the staging and the products
    float zx[2][4], rx[2][4], nx[2][4], hv[2][4];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long long k = row0 + 16 * r + 4 * g + v;
        const bool in = k < rows && col < dh;
        const size_t at = (in ? k : 0) * d + head * dh + (in ? col : 0);
        const TX* x = wx + (in ? k : 0) * 3 * d + head * dh + (in ? col : 0);
        zx[r][v] = ld(x);
        rx[r][v] = ld(x + d);
        nx[r][v] = ld(x + 2 * d);
        hv[r][v] = ld(states + at);
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kResRows * KP / (64 * W); ++i) {
      const int idx = threadIdx.x + 64 * W * i, s = idx / KP, j = idx % KP;
      const long long src = s_src[s];
      float v = 0.f;
      if (j < dh) {
        if (src >= 0)
          v = ld(states + src + j);
        else if (src <= -2)
          v = ld(h0 + (-2 - src) + j);
      }
      sh[s][j] = v;
    }
    __syncthreads();
    floatx4 gz[2], gr[2], gn[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) gz[r] = gr[r] = gn[r] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const float* a = &sh[16 * r + li][g * KG];
#pragma unroll
      for (int k = 0; k < KG; k += 4) {
        const float4 a4 = *reinterpret_cast<const float4*>(a + k);
        const float av[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          gz[r] = mma(av[q], bz[k + q], gz[r]);
          gr[r] = mma(av[q], br[k + q], gr[r]);
        }
      }
    }
    float z[2][4], hp[2][4];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int s = 16 * r + 4 * g + v;
        hp[r][v] = sh[s][col];
        z[r][v] = rt_(sigmoid_op(rt_(rt_(gz[r][v]) + zx[r][v])));
        su[s][col] = rt_(hp[r][v] * rt_(sigmoid_op(rt_(rt_(gr[r][v]) + rx[r][v]))));
      }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const float* a = &su[16 * r + li][g * KG];
#pragma unroll
      for (int k = 0; k < KG; k += 4) {
        const float4 a4 = *reinterpret_cast<const float4*>(a + k);
        const float av[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) gn[r] = mma(av[q], bn[k + q], gn[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long long k = row0 + 16 * r + 4 * g + v;
        const float n = rt_(tanhf(rt_(rt_(gn[r][v]) + nx[r][v])));
        const float f = rt_(rt_(lerp_op(hp[r][v], n, z[r][v])) - hv[r][v]);
        if (k < rows && col < dh) top = max(top, __float_as_uint(f) & 0x7fffffffu);
      }
  }
#pragma unroll
  for (int k = 32; k >= 1; k >>= 1)
    top = max(top, static_cast<unsigned>(__shfl_xor(static_cast<int>(top), k)));
  if (lane == 0) s_max[wave] = top;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < W; ++w) top = max(top, s_max[w]);
    atomicMax(out, top);
  }
}

// About 8 blocks per CU over all heads, each at least one tile of rows; a
// block loads its head's matrices once, so more blocks would only reload them.
constexpr int kResBlocks = 2048;

}  // namespace gru
}  // namespace prnn

using namespace prnn;

extern "C" PRNN_API int prnn_gru_head_residual(const void* wx, const void* a_z, const void* a_r,
                                               const void* a_n, const void* h0,
                                               const void* states, float* out, int B, int T,
                                               int n_heads, int d_head, int dtype,
                                               const int* cu_seqlens, int n_seq, void* stream) {
  if (B < 1 || T < 1 || n_heads < 1 || n_heads > (1 << 20))
    return fail(PRNN_ERR_VALUE, "B, T, n_heads must be >= 1 (n_heads <= 2^20), got B=%d T=%d "
                "n_heads=%d", B, T, n_heads);
  if (d_head < 1 || d_head > 128)
    return fail(PRNN_ERR_TYPE, "d_head must be in [1, 128], got %d", d_head);
  int rc = check_dtype(dtype);
  if (rc != PRNN_OK) return rc;
  if (cu_seqlens != nullptr && (B != 1 || n_seq < 1 || n_seq > T))
    return fail(PRNN_ERR_VALUE, "a packed stream has B = 1 and n_seq in [1, T], got B=%d n_seq=%d",
                B, n_seq);
  if (!wx || !a_z || !a_r || !a_n || !states || !out)
    return fail(PRNN_ERR_VALUE, "wx, a_z, a_r, a_n, states and out must be non-null");
  hipStream_t s = static_cast<hipStream_t>(stream);
  rc = clear_words(reinterpret_cast<int*>(out), 1, s);
  if (rc != PRNN_OK) return rc;
  const long long rows = static_cast<long long>(B) * T;
  const long long n_tiles = (rows + gru::kResRows - 1) / gru::kResRows;
  const long long per_head =
      std::max<long long>(1, std::min<long long>(n_tiles, gru::kResBlocks / n_heads));
  const dim3 grid(static_cast<unsigned>(per_head * n_heads));
  return with_storage(dtype, [&](auto tag) {
    using TX = decltype(tag);
    const TX *x = static_cast<const TX*>(wx), *az = static_cast<const TX*>(a_z),
             *ar = static_cast<const TX*>(a_r), *an = static_cast<const TX*>(a_n),
             *h = static_cast<const TX*>(h0), *st = static_cast<const TX*>(states);
    unsigned* o = reinterpret_cast<unsigned*>(out);
    if (d_head <= 64)
      gru::gru_residual_kernel<TX, 64><<<grid, dim3(256), 0, s>>>(x, az, ar, an, h, st, o, rows, T,
                                                              n_heads, d_head, n_tiles,
                                                              cu_seqlens, n_seq);
    else
      gru::gru_residual_kernel<TX, 128><<<grid, dim3(512), 0, s>>>(x, az, ar, an, h, st, o, rows, T,
                                                               n_heads, d_head, n_tiles,
                                                               cu_seqlens, n_seq);
    PRNN_HIP(hipGetLastError());
    return static_cast<int>(PRNN_OK);
  });
}
