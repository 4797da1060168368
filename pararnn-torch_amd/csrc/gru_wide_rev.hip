// The eq. 2.6 adjoint walk of the wide-head tier (64 < d_head <= 128).  Laid out
// like the forward walks (gru_wide.hip, which says what bounds a step and what it
// measured).
#include "gru_wide.h"

namespace prnn {
namespace gruw {

// Adjoint walk at H* (eq. 2.6): from the last step down,
//   mu_t = g_t + nu_{t+1},  nu_t = J_t^T mu_t
// through the cell's VJP (reference kernels/gru_head_factor.py:68-112):
//   d_zpre = mu (n - h) z(1-z),  d_npre = mu z(1-n^2),  d_u = A_n d_npre,
//   d_rpre = d_u h r(1-r),  nu = (1-z) mu + A_z d_zpre + r d_u + A_r d_rpre.
// Writes the pre-activation gradients (dL/dwx, gate blocks z, r, n) in fp32
// and, at each sequence's first step, nu = dL/dh0 of that sequence's row.
template <typename TX, typename TG>
__global__ __launch_bounds__(kThreads) void gruw_reverse_kernel(
    const float* __restrict__ z, const float* __restrict__ r, const float* __restrict__ n,
    const float* __restrict__ hp, const TG* __restrict__ grad, const TX* __restrict__ a_z,
    const TX* __restrict__ a_r, const TX* __restrict__ a_n, float* __restrict__ g_wx,
    float* __restrict__ g_h0, int T, int H, int dh, const int* __restrict__ cu) {
  __shared__ float4 s_a[2][kS][DW];  // d1, d2, d3, g
  __shared__ float2 s_b[2][kS][DW];  // r, d5
  // the pre-activation gradients of a block's steps: the vectors the products
  // read, stored whole rows at a time at the end of the block
  __shared__ __attribute__((aligned(16))) float s_g[3][kS][kVec];
  const Role rl = role();
  const int c = rl.c;
  const int sc = slot(c);
  const int head = blockIdx.x % H;
  const Span sp = span_of(blockIdx.x / H, T, cu);
  const size_t hoff = static_cast<size_t>(head) * dh * dh;
  float az[kK], ar[kK], an[kK];
  load_group<TX, false>(a_z + hoff, dh, rl, az);
  load_group<TX, false>(a_r + hoff, dh, rl, ar);
  load_group<TX, false>(a_n + hoff, dh, rl, an);
  const int d = H * dh;
  const bool live = c < dh;
  const size_t col = static_cast<size_t>(head) * dh + c;
  float nu = 0.f;
  if (sp.t0 >= sp.t1) return;
  const size_t row_base = static_cast<size_t>(sp.row) * T * d;
  auto load = [&](int t_first) {
    return load_block(z, r, n, hp, grad, row_base, d, head, dh, t_first, -1, sp.t0, sp.t1 - 1);
  };
  auto take = [&](const Staged& st, int to) {
    take_block(st, dh, [&](int s, int cc, float zt, float rt, float nt, float ht, float gt) {
      const Scalars k = scalars(zt, rt, nt, ht);
      s_a[to][s][cc] = float4{k.d1, k.d2, k.d3, gt};
      s_b[to][s][cc] = float2{rt, k.d5};
    });
  };
  // rows tb, tb - 1, ..., of dL/dwx from s_g
  const int fc = static_cast<int>(threadIdx.x) & (DW - 1), fs = static_cast<int>(threadIdx.x) / DW;
  float* g_col = g_wx + row_base * 3 + static_cast<size_t>(head) * dh + fc;
  auto flush = [&](int tb, int ns) {
    if (fc >= dh) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = fs + 4 * j;
      if (s < ns) {
        float* p = g_col + static_cast<size_t>(tb - s) * 3 * d;
#pragma unroll
        for (int q = 0; q < 3; ++q) p[static_cast<size_t>(q) * d] = s_g[q][s][slot(fc)];
      }
    }
  };
  take(load(sp.t1 - 1), 0);
  __syncthreads();
  int buf = 0;
  for (int tb = sp.t1 - 1; tb >= sp.t0; tb -= kS) {
    const bool more = tb - kS >= sp.t0;
    Staged next;
    if (more) next = load(tb - kS);
    const int ns = min(kS, tb - sp.t0 + 1);
    float4 ka = s_a[buf][0][c];
    float2 kb = s_b[buf][0][c];
    for (int s = 0; s < ns; ++s) {
      const float mu = ka.w + nu;
      if (rl.wr) {
        s_g[2][s][sc] = mu * ka.z;
        s_g[0][s][sc] = mu * ka.y;
      }
      __syncthreads();
      const Seg nv = load_seg(s_g[2][s], rl), zv = load_seg(s_g[0][s], rl);
      // the next step's scalars, behind the vectors in the LDS queue
      const int sn = min(s + 1, kS - 1);
      const float4 kan = s_a[buf][sn][c];
      const float2 kbn = s_b[buf][sn][c];
      const float du = dot_seg(an, nv);
      const float dr = du * kb.y;
      if (rl.wr) s_g[1][s][sc] = dr;
      __builtin_amdgcn_sched_barrier(0);
      const float base = ka.x * mu + (kb.x * du + dot_seg(az, zv));
      ka = kan;
      kb = kbn;
      __syncthreads();
      nu = base + dot(ar, s_g[1][s], rl);
    }
    flush(tb, ns);
    // (the other staging buffer was last read a block ago, before this
    // block's barriers)
    if (more) take(next, buf ^ 1);
    __syncthreads();  // s_g is rewritten after this
    buf ^= 1;
  }
  // nu at the sequence's first step: dL/dh0 of its row
  if (rl.wr && live && g_h0 != nullptr) g_h0[static_cast<size_t>(sp.seq) * d + col] = nu;
}

}  // namespace gruw
}  // namespace prnn

using namespace prnn;

extern "C" PRNN_API int prnn_gru_wide_reverse(const float* z, const float* r, const float* n,
                                              const float* hp, const void* grad, int grad_f32,
                                              const void* a_z, const void* a_r, const void* a_n,
                                              float* g_wx, float* g_h0, int B, int T,
                                              int n_heads, int d_head, int dtype,
                                              const int* cu_seqlens, int n_seq, void* stream) {
  int rc = gruw::check(B, T, n_heads, d_head, dtype, cu_seqlens, n_seq);
  if (rc != PRNN_OK) return rc;
  if (!z || !r || !n || !hp || !grad || !a_z || !a_r || !a_n || !g_wx)
    return fail(PRNN_ERR_VALUE, "z, r, n, hp, grad, a_z, a_r, a_n and g_wx must be non-null");
  const int seqs = (cu_seqlens ? n_seq : B) * n_heads;
  hipStream_t s = static_cast<hipStream_t>(stream);
  with_storage(dtype, [&](auto tag) {
    using TX = decltype(tag);
    const TX* az = static_cast<const TX*>(a_z);
    const TX* ar = static_cast<const TX*>(a_r);
    const TX* an = static_cast<const TX*>(a_n);
    if (grad_f32)
      gruw::gruw_reverse_kernel<TX, float><<<dim3(seqs), dim3(gruw::kThreads), 0, s>>>(
          z, r, n, hp, static_cast<const float*>(grad), az, ar, an, g_wx, g_h0, T, n_heads,
          d_head, cu_seqlens);
    else
      gruw::gruw_reverse_kernel<TX, TX><<<dim3(seqs), dim3(gruw::kThreads), 0, s>>>(
          z, r, n, hp, static_cast<const TX*>(grad), az, ar, an, g_wx, g_h0, T, n_heads,
          d_head, cu_seqlens);
    return PRNN_OK;
  });
  PRNN_HIP(hipGetLastError());
  return PRNN_OK;
}
