// ParaGRU mix='head', 64-wide heads, as walks over time: the tier for many
// or short sequences, beside the chunked scan of gru_head.hip.
//
// The chunked scan is parallel in time and pays for it with a 64 x 64 transfer
// matrix per chunk, 64 times the arithmetic of the recurrence itself.  When
// the (sequence, head) pairs alone fill the chip that parallelism buys
// nothing: a walk per pair does the recurrence's own three 64-wide products
// per step.  What bounds it is the latency of a step (two broadcasts through
// LDS and a barrier each), so everything else is kept off that chain (see
// gru_walk.h).
//
// gruk_newton_kernel: all K Newton iterations in one launch, a workgroup per
// (iteration, sequence, head).  Iteration k needs H_{k-1} at steps t - 1 and t
// only, so it runs a few blocks behind k - 1; the iterates pass through the
// workspace as tagged words {value, tag}, 8 bytes per element written once
// and read once (iteration 0 forms the initial guess from wx, the last one
// writes `out`).  Workgroups take their place from a ticket, iteration-major,
// so a workgroup only waits on running or finished ones; waits are bounded
// (status word, NaN for what never came).
//
// gruk_reverse_kernel: the eq. 2.6 adjoint at H*, one walk per (sequence, head)
// from the last step down.
//
// Measured (fp32 / bf16 alike): 0.40 us per Newton step and 0.45 us per adjoint
// step while every walk has a CU to itself, of which the gate products take
// 0.05 (8 parts of 2 channels instead of 16 of 4, twice the LDS words read per
// product: 0.41 and 0.49); 440 walks advance per step time when they are more
// (two workgroups per CU).  K = 3, 128 walks of 1024 steps: 0.61 ms against 1.63 ms chunked, 512
// walks: 1.5 against 4.6; adjoint, 512 walks of 1024: 0.8 against 1.85 ms.
// With the outputs stored step by step from the lanes that hold them instead
// of whole rows per block a step took 0.43 and 0.55 us.
//
// fp32 throughout; the reference's streamed tier walks the same way, one
// program per (b, head) (kernels/newton_gru_head.py:765-960).
#include "gru_walk.h"

#include <algorithm>
#include <type_traits>

namespace prnn {
namespace gruk {

using gruw::Span;
using gruw::span_of;

struct WaitLimit {
  int* status;
  int limit;
};

struct NewtonShared {
  float4 a[2][kBlk][DH];   // d1, d2, d3, F
  float2 b[2][kBlk][DH];   // r, d5
  // H_{k-1}: rows 1 .. 16 a block's steps, row 0 the step before it
  __attribute__((aligned(16))) float h[2][kBlk + 1][kPad];
  __attribute__((aligned(16))) float hr[kBlk][kPad];
  // delta of a block's steps: the vector that the next step reads, and at the
  // end of the block what its outputs are made of
  __attribute__((aligned(16))) float d[kBlk][DH];
  __attribute__((aligned(16))) float w[DH];
};

// One block's inputs as loaded: wx at the lane's MFMA output positions, and
// either the tagged words of H_{k-1} or the two gates of the initial guess at
// the lane's staging positions (step tid / 64 + 4 j, channel tid % 64).
template <typename TX>
struct WxRegs {
  TX x[3][4];
};
template <typename TX, bool TAGGED>
struct HRegs {
  typename std::conditional<TAGGED, unsigned long long, TX>::type v[4];
  TX n[TAGGED ? 1 : 4];
};

template <typename TX, bool TAGGED, bool LAST>
__device__ __forceinline__ void newton_walk(
    NewtonShared& sh, const TX* __restrict__ wx, const TX* __restrict__ a_z,
    const TX* __restrict__ a_r, const TX* __restrict__ a_n, const TX* __restrict__ h0,
    const unsigned long long* __restrict__ src, int src_tag, unsigned long long* __restrict__ dst,
    int dst_tag, TX* __restrict__ out, int T, int H, int head, const Span& sp, float omega,
    const WaitLimit& spin) {
  const Lane l = lane_roles();
  const int d = H * DH;
  const size_t row_base = static_cast<size_t>(sp.row) * T;
  const size_t hcol = static_cast<size_t>(head) * DH;
  float az[kKeep], ar[kKeep], an[kKeep];
  load_group<TX, true>(a_z, l, az);
  load_group<TX, true>(a_r, l, ar);
  load_group<TX, true>(a_n, l, an);
  GateOps ops;
  ops.load(a_z, a_r, a_n, l);

  const int sc = threadIdx.x & (DH - 1), ss = threadIdx.x >> 6;  // staging channel, first step
  // steps past the end are clamped to the last one: computed, never used
  auto step_at = [&](int t) { return row_base + min(t, sp.t1 - 1); };
  auto load_wx = [&](int tb, WxRegs<TX>& x) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const TX* p = wx + step_at(tb + 4 * l.g + v) * 3 * d + hcol + l.col;
#pragma unroll
      for (int q = 0; q < 3; ++q) x.x[q][v] = p[static_cast<size_t>(q) * d];
    }
  };
  auto load_h = [&](int tb, HRegs<TX, TAGGED>& h) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t row = step_at(tb + ss + 4 * j);
      if constexpr (TAGGED) {
        h.v[j] = __hip_atomic_load(src + row * d + hcol + sc, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
      } else {
        const TX* p = wx + row * 3 * d + hcol + sc;
        h.v[j] = p[0];
        h.n[j] = p[2 * static_cast<size_t>(d)];
      }
    }
  };
  // rows 1 .. 16 of buffer `to` from the loaded values; tagged words are
  // tested here, not at the load, and reloaded until they have come
  bool gave_up = false;
  auto store_h = [&](int tb, HRegs<TX, TAGGED>& h, int to) {
    float v[4];
    if constexpr (TAGGED) {
      int rounds = 0;
      while (true) {
        bool ok = true;
#pragma unroll
        for (int j = 0; j < 4; ++j) ok = ok && static_cast<int>(h.v[j] >> 32) == src_tag;
        if (ok) break;
        if (gave_up || ++rounds > spin.limit) {
          if (!gave_up)
            __hip_atomic_fetch_or(spin.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          gave_up = true;
          break;
        }
        __builtin_amdgcn_s_sleep(2);
        load_h(tb, h);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = static_cast<int>(h.v[j] >> 32) == src_tag
                   ? __uint_as_float(static_cast<uint32_t>(h.v[j]))
                   : __builtin_nanf("");
    } else {
      // the initial guess f(0, x) (reference solvers/newton/__init__.py:925-940)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = lerp_t(0.f, ftanh(to_f32(h.n[j])), fsigmoid(to_f32(h.v[j])));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) sh.h[to][1 + ss + 4 * j][sc] = v[j];
  };
  GateAcc acc;
  // scalars of the block whose rows are sh.h[hb], into buffer `to`
  auto finish = [&](int hb, int to) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 4 * l.g + v;
      const float z = acc.z[v], r = acc.r[v], n = acc.n[v];
      const float hp = sh.h[hb][row][l.col], hin = sh.h[hb][row + 1][l.col];
      const Scalars k = scalars(z, r, n, hp);
      sh.a[to][row][l.col] = float4{k.d1, k.d2, k.d3, lerp_t(hp, n, z) - hin};
      sh.b[to][row][l.col] = float2{r, k.d5};
    }
  };

  // ---- the first two blocks' rows and the first block's scalars ----
  WxRegs<TX> xr;
  load_wx(sp.t0, xr);
  {
    HRegs<TX, TAGGED> ha, hb;
    load_h(sp.t0, ha);
    load_h(sp.t0 + kBlk, hb);
    if (threadIdx.x < DH) {
      sh.h[0][0][threadIdx.x] =
          h0 != nullptr ? ld(h0 + static_cast<size_t>(sp.seq) * d + hcol + threadIdx.x) : 0.f;
      sh.d[kBlk - 1][threadIdx.x] = 0.f;
    }
    store_h(sp.t0, ha, 0);
    if (sp.t1 - sp.t0 > kBlk) store_h(sp.t0 + kBlk, hb, 1);
  }
  __syncthreads();
  if (!TAGGED && h0 != nullptr) {
    // the guess of the first step is the cell at h0
    const TX* p = wx + (row_base + sp.t0) * 3 * d + hcol + l.c;
    const Seg h = load_seg(sh.h[0][0], l);
    const float z = fsigmoid(ld(p) + dot_seg(az, h));
    const float r = fsigmoid(ld(p + d) + dot_seg(ar, h));
    const float hp = sh.h[0][0][l.c];
    if (l.wr) sh.w[l.c] = hp * r;
    __syncthreads();
    const float n = ftanh(ld(p + 2 * static_cast<size_t>(d)) + dot_seg(an, load_seg(sh.w, l)));
    if (l.wr) sh.h[0][1][l.c] = lerp_t(hp, n, z);
    __syncthreads();
  }
  if (threadIdx.x < DH) sh.h[1][0][threadIdx.x] = sh.h[0][kBlk][threadIdx.x];
#pragma unroll
  for (int s = 0; s < kSlices; ++s) {
    if (s == 17) __syncthreads();
    gate_slice(s, ops, acc, sh.h[0], sh.hr, xr.x, l, [&] { finish(0, 0); });
  }
  load_wx(sp.t0 + kBlk, xr);
  __syncthreads();

  // ---- the walk ----
  float delta = 0.f;
  // H_k = H_{k-1} + omega delta of a block's `ns` steps: whole rows at a time
  auto flush = [&](int tb, int buf, int ns) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = ss + 4 * j;
      if (s < ns) {
        const float h = sh.h[buf][1 + s][sc] + omega * sh.d[s][sc];
        const size_t at = (row_base + tb + s) * d + hcol + sc;
        if constexpr (LAST)
          st(out + at, h);
        else
          st_tagged(dst + at, h, dst_tag);
      }
    }
  };
  float4 ka = sh.a[0][0][l.c];
  float2 kb = sh.b[0][0][l.c];
  auto step = [&](int buf, int s, auto&& beside) {
    const Seg dv = load_seg(sh.d[s > 0 ? s - 1 : kBlk - 1], l);
    beside(2 * s);
    const float w = kb.x * delta + kb.y * dot_seg(ar, dv);
    if (l.wr) sh.w[l.c] = w;
    __builtin_amdgcn_sched_barrier(0);
    const float base = ka.x * delta + (ka.y * dot_seg(az, dv) + ka.w);
    __syncthreads();
    const Seg wv = load_seg(sh.w, l);
    // the next step's scalars, behind the vector in the LDS queue
    const int sn = s + 1 < kBlk ? s + 1 : 0, bn = s + 1 < kBlk ? buf : buf ^ 1;
    const float4 kan = sh.a[bn][sn][l.c];
    const float2 kbn = sh.b[bn][sn][l.c];
    beside(2 * s + 1);
    delta = base + ka.z * dot_seg(an, wv);
    if (l.wr) sh.d[s][l.c] = delta;
    ka = kan;
    kb = kbn;
    __syncthreads();
  };
  int buf = 0;
  for (int tb = sp.t0; tb < sp.t1; tb += kBlk, buf ^= 1) {
    if (tb + kBlk >= sp.t1) {  // the last block: nothing to prepare
      const int ns = sp.t1 - tb;
      for (int s = 0; s < ns; ++s) step(buf, s, [](int) {});
      flush(tb, buf, ns);
      break;
    }
    // this block's steps beside the next block's gates; the inputs of the
    // block after that are on their way
    const int t2 = tb + 2 * kBlk;
    const bool more = t2 < sp.t1;
    HRegs<TX, TAGGED> hn;
    if (more) load_h(t2, hn);
#pragma unroll
    for (int s = 0; s < kBlk; ++s)
      step(buf, s, [&](int q) {
        gate_slice(q, ops, acc, sh.h[buf ^ 1], sh.hr, xr.x, l,
                   [&] { finish(buf ^ 1, buf ^ 1); });
        if (q == 28 && more) load_wx(t2, xr);
      });
    flush(tb, buf, kBlk);
    if (more) {
      // the rows of two blocks on replace this block's: a lane rewrites the
      // elements it has just flushed, and row 0 is no longer read
      if (threadIdx.x < DH) sh.h[buf][0][threadIdx.x] = sh.h[buf ^ 1][kBlk][threadIdx.x];
      store_h(t2, hn, buf);
    }
    __syncthreads();
  }
}

template <typename TX>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void
gruk_newton_kernel(const TX* __restrict__ wx, const TX* __restrict__ a_z,
                   const TX* __restrict__ a_r, const TX* __restrict__ a_n,
                   const TX* __restrict__ h0, unsigned long long* __restrict__ iters,
                   TX* __restrict__ out, int B, int T, int H, int n_rows, int K, float omega,
                   const int* __restrict__ cu, int* __restrict__ ticket, int tag_base,
                   WaitLimit spin) {
  __shared__ NewtonShared sh;
  __shared__ int s_ticket;
  if (threadIdx.x == 0)
    s_ticket = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int units = n_rows * H;
  const int task = __builtin_amdgcn_readfirstlane(s_ticket);
  const int k = task / units, unit = task % units;
  const int head = unit % H;
  const Span sp = span_of(unit / H, T, cu);
  if (sp.t0 >= sp.t1) return;
  const size_t plane = static_cast<size_t>(B) * T * H * DH, hoff = static_cast<size_t>(head) * DH * DH;
  unsigned long long* dst = k == K - 1 ? nullptr : iters + k * plane;
  const unsigned long long* src = k == 0 ? nullptr : iters + (k - 1) * plane;
  auto walk = [&](auto tagged, auto last) {
    newton_walk<TX, decltype(tagged)::value, decltype(last)::value>(
        sh, wx, a_z + hoff, a_r + hoff, a_n + hoff, h0, src, tag_base + k, dst, tag_base + 1 + k,
        out, T, H, head, sp, omega, spin);
  };
  if (k == 0 && K == 1)
    walk(std::false_type{}, std::true_type{});
  else if (k == 0)
    walk(std::false_type{}, std::false_type{});
  else if (k == K - 1)
    walk(std::true_type{}, std::true_type{});
  else
    walk(std::true_type{}, std::false_type{});
}

// ---------------------------------------------------------------------------
// The adjoint walk: with nu_t = J_t^T mu_t, from the last step down
//   mu = g + nu,  d_z = mu (n - h) z (1 - z),  d_n = mu z (1 - n^2),
//   d_u = A_n d_n,  d_r = d_u h r (1 - r),
//   nu <- (1 - z) mu + A_z d_z + r d_u + A_r d_r
// (reference kernels/gru_head_factor.py:68-112).  Row i of a block is step
// tb - i; the gates are those of the forward step at H*, made the same way.
// Writes d_z, d_r, d_n (= dL/dwx), r in the layout the dL/dA reduction reads
// ([sequence chunk][step][channel]), and at the sequence's first step
// nu = dL/dh0.
// ---------------------------------------------------------------------------
struct ReverseShared {
  float4 a[2][kBlk][DH];  // d1, d2, d3, g
  float2 b[2][kBlk][DH];  // r, d5
  __attribute__((aligned(16))) float h[2][kBlk][kPad];
  __attribute__((aligned(16))) float hr[kBlk][kPad];
  // the pre-activation gradients of a block's steps: the vectors the products
  // read, stored whole rows at a time at the end of the block
  __attribute__((aligned(16))) float g[3][kBlk][DH];
};

template <typename TX>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void
gruk_reverse_kernel(const TX* __restrict__ wx, const TX* __restrict__ a_z,
                    const TX* __restrict__ a_r, const TX* __restrict__ a_n,
                    const TX* __restrict__ h0, const TX* __restrict__ states,
                    const TX* __restrict__ grad, TX* __restrict__ g_wx, float* __restrict__ r_out,
                    float* __restrict__ g_h0, int T, int H, int n_chunks, int chunk,
                    const int* __restrict__ cu) {
  __shared__ ReverseShared sh;
  const Lane l = lane_roles();
  const int head = blockIdx.x % H;
  const Span sp = span_of(blockIdx.x / H, T, cu);
  if (sp.t0 >= sp.t1) return;
  const int d = H * DH;
  const size_t row_base = static_cast<size_t>(sp.row) * T;
  const size_t hcol = static_cast<size_t>(head) * DH, hoff = hcol * DH;
  float az[kKeep], ar[kKeep], an[kKeep];
  load_group<TX, false>(a_z + hoff, l, az);
  load_group<TX, false>(a_r + hoff, l, ar);
  load_group<TX, false>(a_n + hoff, l, an);
  GateOps ops;
  ops.load(a_z + hoff, a_r + hoff, a_n + hoff, l);

  const int sc = threadIdx.x & (DH - 1), ss = threadIdx.x >> 6;
  // steps before the start are clamped to it: computed, never used
  TX xr[3][4], gr[4], hn[4];
  auto load_x = [&](int tb) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const size_t row = row_base + max(tb - 4 * l.g - v, sp.t0);
      const TX* p = wx + row * 3 * d + hcol + l.col;
#pragma unroll
      for (int q = 0; q < 3; ++q) xr[q][v] = p[static_cast<size_t>(q) * d];
      gr[v] = grad[row * d + hcol + l.col];
    }
  };
  auto load_h = [&](int tb) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = max(tb - ss - 4 * j, sp.t0);
      hn[j] = TX{};
      if (t > sp.t0)
        hn[j] = states[(row_base + t - 1) * d + hcol + sc];
      else if (h0 != nullptr)
        hn[j] = h0[static_cast<size_t>(sp.seq) * d + hcol + sc];
    }
  };
  auto store_h = [&](int to) {
#pragma unroll
    for (int j = 0; j < 4; ++j) sh.h[to][ss + 4 * j][sc] = to_f32(hn[j]);
  };
  GateAcc acc;
  auto finish = [&](int tb, int to) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 4 * l.g + v, t = tb - row;
      const float r = acc.r[v];
      const Scalars k = scalars(acc.z[v], r, acc.n[v], sh.h[to][row][l.col]);
      sh.a[to][row][l.col] = float4{k.d1, k.d2, k.d3, to_f32(gr[v])};
      sh.b[to][row][l.col] = float2{r, k.d5};
      if (t >= sp.t0) {
        const size_t task = (static_cast<size_t>(sp.row) * H + head) * n_chunks + t / chunk;
        r_out[(task * chunk + t % chunk) * DH + l.col] = r;
      }
    }
  };
  load_x(sp.t1 - 1);
  load_h(sp.t1 - 1);
  store_h(0);
  load_h(sp.t1 - 1 - kBlk);
  __syncthreads();
#pragma unroll
  for (int s = 0; s < kSlices; ++s) {
    if (s == 17) __syncthreads();
    gate_slice(s, ops, acc, sh.h[0], sh.hr, xr, l, [&] { finish(sp.t1 - 1, 0); });
  }
  load_x(sp.t1 - 1 - kBlk);
  store_h(1);
  __syncthreads();

  float nu = 0.f;
  auto flush = [&](int tb, int ns) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = ss + 4 * j;
      if (s < ns) {
        TX* p = g_wx + (row_base + tb - s) * 3 * d + hcol + sc;
#pragma unroll
        for (int q = 0; q < 3; ++q) st(p + static_cast<size_t>(q) * d, sh.g[q][s][sc]);
      }
    }
  };
  float4 ka = sh.a[0][0][l.c];
  float2 kb = sh.b[0][0][l.c];
  // (every lane of a channel writes the same word here: masking the writes to
  // one lane, which the forward walk gains 2% from, cost this one 1%)
  auto step = [&](int buf, int s, auto&& beside) {
    const float mu = ka.w + nu;
    sh.g[2][s][l.c] = mu * ka.z;
    sh.g[0][s][l.c] = mu * ka.y;
    __syncthreads();
    const Seg nv = load_seg(sh.g[2][s], l), zv = load_seg(sh.g[0][s], l);
    // the next step's scalars, behind the vectors in the LDS queue
    const int sn = s + 1 < kBlk ? s + 1 : 0, bn = s + 1 < kBlk ? buf : buf ^ 1;
    const float4 kan = sh.a[bn][sn][l.c];
    const float2 kbn = sh.b[bn][sn][l.c];
    beside(2 * s);
    const float du = dot_seg(an, nv);
    sh.g[1][s][l.c] = du * kb.y;
    __builtin_amdgcn_sched_barrier(0);
    const float base = ka.x * mu + (kb.x * du + dot_seg(az, zv));
    ka = kan;
    kb = kbn;
    __syncthreads();
    const Seg rv = load_seg(sh.g[1][s], l);
    beside(2 * s + 1);
    nu = base + dot_seg(ar, rv);
  };
  int buf = 0;
  for (int tb = sp.t1 - 1; tb >= sp.t0; tb -= kBlk, buf ^= 1) {
    const int tn = tb - kBlk;
    if (tn < sp.t0) {
      const int ns = tb - sp.t0 + 1;
      for (int s = 0; s < ns; ++s) step(buf, s, [](int) {});
      flush(tb, ns);
      break;
    }
    const bool more = tn - kBlk >= sp.t0;
    if (more) load_h(tn - kBlk);
#pragma unroll
    for (int s = 0; s < kBlk; ++s)
      step(buf, s, [&](int q) {
        gate_slice(q, ops, acc, sh.h[buf ^ 1], sh.hr, xr, l, [&] { finish(tn, buf ^ 1); });
        if (q == 28 && more) load_x(tn - kBlk);
      });
    flush(tb, kBlk);
    if (more) store_h(buf);
    __syncthreads();
  }
  if (l.wr && g_h0 != nullptr) g_h0[static_cast<size_t>(sp.seq) * d + hcol + l.c] = nu;
}

template <typename TX>
void launch_walk_reverse(const TX* wx, const TX* az, const TX* ar, const TX* an, const TX* h0,
                         const TX* states, const TX* grad, TX* g_wx, float* r_out, float* g_h0,
                         int T, int H, int n_rows, int n_chunks, int chunk, const int* cu,
                         hipStream_t stream) {
  gruk_reverse_kernel<TX><<<dim3(n_rows * H), dim3(kThreads), 0, stream>>>(
      wx, az, ar, an, h0, states, grad, g_wx, r_out, g_h0, T, H, n_chunks, chunk, cu);
}
#define PRNN_INSTANTIATE(TX)                                                                     \
  template void launch_walk_reverse<TX>(const TX*, const TX*, const TX*, const TX*, const TX*,   \
                                        const TX*, const TX*, TX*, float*, float*, int, int, int, \
                                        int, int, const int*, hipStream_t);
PRNN_INSTANTIATE(float)
PRNN_INSTANTIATE(bf16)
PRNN_INSTANTIATE(f16)
#undef PRNN_INSTANTIATE

// Workspace: PRNN_TAG_SPAN ticket counters (the first is used) and the status
// word, then the tagged iterates H_0 .. H_{K-2}.
struct NewtonWs {
  int* counters;
  unsigned long long* iters;
  size_t clear_words;
};

static NewtonWs carve(void* base, long long rows, int d, int K, size_t* total) {
  Carver cv(base);
  NewtonWs w;
  w.counters = static_cast<int*>(cv.take(sizeof(int) * (PRNN_TAG_SPAN + 1)));
  w.iters = static_cast<unsigned long long*>(
      cv.take(sizeof(unsigned long long) * static_cast<size_t>(K - 1) * rows * d));
  w.clear_words = cv.used / sizeof(int);
  *total = cv.used;
  return w;
}

static int check_newton(int B, int T, int H, int K, int dtype, const int* cu, int n_seq) {
  if (K < 1 || K > PRNN_TAG_SPAN)
    return fail(PRNN_ERR_VALUE, "max_iters must be in [1, %d], got %d", PRNN_TAG_SPAN, K);
  const long long rows = cu != nullptr ? n_seq : B;
  if (B >= 1 && T >= 1 && H >= 1 && rows * H * K > (1ll << 30))
    return fail(PRNN_ERR_VALUE, "problem too large");
  if (B < 1 || T < 1 || H < 1)
    return fail(PRNN_ERR_VALUE, "B, T, n_heads must be >= 1, got B=%d T=%d n_heads=%d", B, T, H);
  if (check_dtype(dtype) != PRNN_OK) return PRNN_ERR_TYPE;
  if (cu != nullptr && (B != 1 || n_seq < 1 || n_seq > T))
    return fail(PRNN_ERR_VALUE, "a packed stream has B = 1 and n_seq in [1, T], got B=%d n_seq=%d",
                B, n_seq);
  return PRNN_OK;
}

}  // namespace gruk
}  // namespace prnn

using namespace prnn;

extern "C" PRNN_API size_t prnn_gru_head_walk_newton_workspace_size(int B, int T, int n_heads,
                                                                    int max_iters) {
  if (gruk::check_newton(B, T, n_heads, max_iters, PRNN_F32, nullptr, 0) != PRNN_OK) return 0;
  size_t total = 0;
  gruk::carve(nullptr, static_cast<long long>(B) * T, n_heads * gruk::DH, max_iters, &total);
  return total;
}

extern "C" PRNN_API int prnn_gru_head_walk_newton(const void* wx, const void* a_z,
                                                  const void* a_r, const void* a_n,
                                                  const void* h0, void* out, int B, int T,
                                                  int n_heads, int max_iters, float omega,
                                                  int dtype, const int* cu_seqlens, int n_seq,
                                                  void* workspace, size_t workspace_bytes,
                                                  int tag_base, void* stream) {
  int rc = gruk::check_newton(B, T, n_heads, max_iters, dtype, cu_seqlens, n_seq);
  if (rc != PRNN_OK) return rc;
  if (tag_base < 0 || tag_base > PRNN_TAG_BASE_MAX)
    return fail(PRNN_ERR_VALUE, "tag_base must be in [0, %d], got %d", PRNN_TAG_BASE_MAX,
                tag_base);
  if (!wx || !a_z || !a_r || !a_n || !out || !workspace)
    return fail(PRNN_ERR_VALUE, "wx, a_z, a_r, a_n, out and workspace must be non-null");
  size_t need = 0;
  const gruk::NewtonWs w = gruk::carve(workspace, static_cast<long long>(B) * T,
                                       n_heads * gruk::DH, max_iters, &need);
  if (workspace_bytes < need)
    return fail(PRNN_ERR_VALUE, "workspace too small: %zu < %zu bytes", workspace_bytes, need);
  hipStream_t s = static_cast<hipStream_t>(stream);
  // tag_base > 0: every word holds a tag below tag_base + 1, only the counters
  // need zeroing (as for the sLSTM workspaces)
  rc = clear_words(w.counters, tag_base > 0 ? PRNN_TAG_SPAN + 1 : w.clear_words, s);
  if (rc != PRNN_OK) return rc;
  const int rows = cu_seqlens ? n_seq : B;
  const gruk::WaitLimit lim{w.counters + PRNN_TAG_SPAN, spin_limit()};
  timing_begin(s);
  with_storage(dtype, [&](auto tag) {
    using TX = decltype(tag);
    gruk::gruk_newton_kernel<TX><<<dim3(max_iters * rows * n_heads), dim3(gruk::kThreads), 0, s>>>(
        static_cast<const TX*>(wx), static_cast<const TX*>(a_z), static_cast<const TX*>(a_r),
        static_cast<const TX*>(a_n), static_cast<const TX*>(h0), w.iters, static_cast<TX*>(out),
        B, T, n_heads, rows, max_iters, omega, cu_seqlens, w.counters, tag_base, lim);
    return PRNN_OK;
  });
  timing_end(s);
  PRNN_HIP(hipGetLastError());
  return PRNN_OK;
}
