// max |f(H_{t-1}, x_t) - H_t| of a ParaSLSTM mix='diag' trajectory: the
// residual gate of the Newton solve (reference solvers/newton/__init__.py:
// 582-636) and of its host-checked loops.
//
// The reference evaluates the cell once more over the whole trajectory as a
// chain of tensor ops and reduces |pred - H|: about 30 passes over memory.
// Here a wave walks L steps of 64 channels with the previous state in
// registers, so wx and the states are read once, and the maximum leaves the
// chip as one word.  The cell is cell_jac_eager, which rounds every
// intermediate to the storage type where the tensor ops round it, so the value
// that the gate compares is the tensor ops' (the Jacobian half of that
// function is dead code here).
//
// Bound: memory.  Measured at d = 512, B = 8, T = 16384, fp32 (2.15 GB read):
// 0.43 ms = 5.0 TB/s, the rate of a large copy; the tensor ops took 6.1 ms,
// and 2.1 ms more to project the input again.
#include "slstm_scan.h"

#include <algorithm>

namespace prnn {
namespace slstm {

// Steps a wave reads ahead of its arithmetic: 8 of fp32 (64 registers of
// inputs), 16 of 16-bit storage (packed two to a register).  The row before
// the first step is read again, 1 / L more.
template <typename TX>
constexpr int kResSteps = sizeof(TX) == 4 ? 8 : 16;
constexpr int kResBlocks = 2048;  // 8 four-wave blocks per CU; each ends in one atomic

template <typename TX, bool PK>
__global__ __launch_bounds__(256) void slstm_residual_kernel(
    const TX* __restrict__ wx, const TX* __restrict__ rmix, const TX* __restrict__ h0,
    const TX* __restrict__ states, unsigned* __restrict__ out, int T, int d, int n_cb, int n_seg,
    int n_tasks, float eps, Packed pk) {
  constexpr int L = kResSteps<TX>;
  constexpr uint32_t SZ = sizeof(TX);
  using XS = RowStash<TX>;
  __shared__ unsigned s_max[4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t row4 = static_cast<size_t>(4) * d;
  // |F| as its bit pattern: ordered like the value, with NaN above infinity
  unsigned top = 0u;
  for (int task = blockIdx.x * 4 + wave; task < n_tasks; task += gridDim.x * 4) {
    const int cb = task % n_cb, rest = task / n_cb;
    const int seg = rest % n_seg, b = rest / n_seg;
    const int c0 = cb * kCB, t0 = seg * L;
    const bool live = c0 + lane < d;
    const int n = min(L, T - t0);
    const size_t first = static_cast<size_t>(b) * T + t0;
    const uint32_t voff = live ? lane * SZ : kOOB;
    const uint32_t span = ((n - 1) * row4 + 3 * d + (d - c0)) * SZ;
    Heads hd{0ull, 0};
    if constexpr (PK) hd = find_heads(pk, t0, n);
    float r[4] = {0.f, 0.f, 0.f, 0.f}, prev[4] = {0.f, 0.f, 0.f, 0.f};
    if (live) {
#pragma unroll
      for (int g = 0; g < 4; ++g) r[g] = ld(rmix + g * d + c0 + lane);
      if (t0 > 0) {
        const TX* p = states + (first - 1) * row4 + c0 + lane;
#pragma unroll
        for (int k = 0; k < 4; ++k) prev[k] = ld(p + k * d);
      } else if (!PK && h0 != nullptr) {
        const TX* p = h0 + static_cast<size_t>(b) * row4 + c0 + lane;
#pragma unroll
        for (int k = 0; k < 4; ++k) prev[k] = ld(p + k * d);
      }
    }
    // steps past the end lie outside the resources and read zeros
    const rsrc_t rx = make_rsrc(wx + first * row4 + c0, span);
    const rsrc_t rs = make_rsrc(states + first * row4 + c0, span);
    uint32_t xw[L][XS::N], hw[L][XS::N];
#pragma unroll
    for (int s = 0; s < L; ++s) {
      XS::load(rx, voff, s * row4 * SZ, d * SZ, xw[s]);
      XS::load(rs, voff, s * row4 * SZ, d * SZ, hw[s]);
    }
#pragma unroll
    for (int s = 0; s < L; ++s) {
      if (s < n) {
        if (PK && hd.at(s)) head_state(pk, h0, hd.seq(s), d, c0 + lane, live, prev);
        float x[4], h[4];
        XS::get(xw[s], x);
        XS::get(hw[s], h);
        const CellJE J = cell_jac_eager<TX>(prev, x, r, eps);
        const float p[4] = {J.pc, J.pn, J.pm, J.ph};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const unsigned f = __float_as_uint(round_to<TX>(p[k] - h[k])) & 0x7fffffffu;
          if (live) top = max(top, f);
          prev[k] = h[k];
        }
      }
    }
  }
#pragma unroll
  for (int k = 32; k >= 1; k >>= 1)
    top = max(top, static_cast<unsigned>(__shfl_xor(static_cast<int>(top), k)));
  if (lane == 0) s_max[wave] = top;
  __syncthreads();
  if (threadIdx.x == 0) {
    top = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
    atomicMax(out, top);
  }
}

}  // namespace slstm
}  // namespace prnn

using namespace prnn;

extern "C" PRNN_API int prnn_slstm_residual(const void* wx, const void* r, const void* h0,
                                            const void* states, float* out, int B, int T, int d,
                                            float eps, int dtype, const int* cu_seqlens,
                                            int n_seq, void* stream) {
  int rc = slstm::check_dims(B, T, d, dtype);
  if (rc != PRNN_OK) return rc;
  const bool packed = cu_seqlens != nullptr;
  if (packed && (B != 1 || n_seq < 1 || n_seq > T))
    return fail(PRNN_ERR_VALUE, "a packed stream has B = 1 and n_seq in [1, T], got B=%d n_seq=%d",
                B, n_seq);
  if (!wx || !r || !states || !out)
    return fail(PRNN_ERR_VALUE, "wx, r, states and out must be non-null");
  hipStream_t s = static_cast<hipStream_t>(stream);
  rc = clear_words(reinterpret_cast<int*>(out), 1, s);
  if (rc != PRNN_OK) return rc;
  const slstm::Packed pk{cu_seqlens, nullptr, n_seq};
  return with_storage(dtype, [&](auto tag) {
    using TX = decltype(tag);
    const int n_cb = (d + slstm::kCB - 1) / slstm::kCB;
    const int n_seg = (T + slstm::kResSteps<TX> - 1) / slstm::kResSteps<TX>;
    const int n_tasks = B * n_cb * n_seg;
    const dim3 grid(std::min((n_tasks + 3) / 4, slstm::kResBlocks)), block(256);
    unsigned* o = reinterpret_cast<unsigned*>(out);
    const TX *x = static_cast<const TX*>(wx), *rr = static_cast<const TX*>(r),
             *h = static_cast<const TX*>(h0), *st = static_cast<const TX*>(states);
    if (packed)
      slstm::slstm_residual_kernel<TX, true><<<grid, block, 0, s>>>(x, rr, h, st, o, T, d, n_cb,
                                                                    n_seg, n_tasks, eps, pk);
    else
      slstm::slstm_residual_kernel<TX, false><<<grid, block, 0, s>>>(x, rr, h, st, o, T, d, n_cb,
                                                                     n_seg, n_tasks, eps, pk);
    PRNN_HIP(hipGetLastError());
    return static_cast<int>(PRNN_OK);
  });
}
