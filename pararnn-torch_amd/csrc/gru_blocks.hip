// Heads narrower than 64 channels in 64-channel blocks: channels and weights
// into the block layout of the head-GRU kernels, and results out of it, every
// array of a call in one launch.
//
// per = 64 / d_head heads share a block.  Block b holds the w = per d_head
// channels [b w, b w + w) of a row at its first w places (fewer in a partly
// filled last block) and zeros behind them; the 64 x 64 matrix of a block has
// its heads' matrices on the diagonal and zeros elsewhere.
//
// A wave moves whole 64-place rows of the block layout: place j of row
// (r, b) is channel b w + j of row r, so a lane needs no division of its own, and
// both sides are read and written contiguously.  Bound: launches for the
// weights (a few KB to a few MB), memory for the activations.  Index arithmetic,
// zero fills and index_copy / index_select took most of a training step's 98
// launches; packed N = 9001 rows, H = 8, d_head = 24, fp32: 28 launches, the step
// 1.83 -> 1.37 ms, of which the moves in take 37 us (129 MB, 3.5 TB/s) and the
// moves out 22 us.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "prnn_host.h"

namespace prnn {
namespace gru {

constexpr int kMaxMoves = 8;
constexpr int kMoveRows = 8;  // block rows per wave, all in flight
struct Moves {
  const void* src[kMaxMoves];
  void* dst[kMaxMoves];
  long long units[kMaxMoves];   // block rows
  unsigned first[kMaxMoves];    // first workgroup
  int matrix[kMaxMoves], two[kMaxMoves];
  int n;
};

template <typename T, bool TO>
__device__ __forceinline__ void move_rows(const T* __restrict__ src, T* __restrict__ dst,
                                          long long units, long long u0, bool matrix, int nb,
                                          int H, int dh) {
  const int lane = threadIdx.x & 63;
  const int per = 64 / dh, w = per * dh;
  T v[kMoveRows];
  long long at[kMoveRows];  // the lane's place in the packed array, -1: a zero
  long long row = u0 / nb;
  int b = static_cast<int>(u0 - row * nb);
#pragma unroll
  for (int q = 0; q < kMoveRows; ++q) {
    const long long u = u0 + q;
    bool in;
    if (matrix) {
      // u = (matrix g, block b, row i of 64)
      const long long gb = u / 64;
      const int i = static_cast<int>(u - gb * 64), sub = i / dh;
      const long long g = gb / nb;
      const int head = static_cast<int>(gb - g * nb) * per + sub, j = lane - sub * dh;
      in = sub < per && head < H && j >= 0 && j < dh;
      at[q] = ((g * H + head) * dh + (i - sub * dh)) * dh + j;
    } else {
      in = lane < w && b * w + lane < H * dh;
      at[q] = row * (static_cast<long long>(H) * dh) + b * w + lane;
      if (++b == nb) {
        b = 0;
        ++row;
      }
    }
    in = in && u < units;
    v[q] = T(0);
    if (TO && in) v[q] = src[at[q]];
    if (!TO && in) v[q] = src[u * 64 + lane];
    if (!in) at[q] = -1;
  }
#pragma unroll
  for (int q = 0; q < kMoveRows; ++q) {
    const long long u = u0 + q;
    if (TO && u < units) dst[u * 64 + lane] = v[q];
    if (!TO && at[q] >= 0) dst[at[q]] = v[q];
  }
}

template <bool TO>
__global__ __launch_bounds__(256) void gru_blocks_kernel(Moves m, int nb, int H, int dh) {
  int k = 0;
  while (k + 1 < m.n && blockIdx.x >= m.first[k + 1]) ++k;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long u0 =
      (static_cast<long long>(blockIdx.x - m.first[k]) * 4 + wave) * kMoveRows;
  if (m.two[k])
    move_rows<unsigned short, TO>(static_cast<const unsigned short*>(m.src[k]),
                                  static_cast<unsigned short*>(m.dst[k]), m.units[k], u0,
                                  m.matrix[k], nb, H, dh);
  else
    move_rows<unsigned, TO>(static_cast<const unsigned*>(m.src[k]),
                            static_cast<unsigned*>(m.dst[k]), m.units[k], u0, m.matrix[k], nb, H,
                            dh);
}

}  // namespace gru
}  // namespace prnn

using namespace prnn;

extern "C" PRNN_API int prnn_gru_head_blocks(const prnn_block_move* moves, int n_moves,
                                             int n_heads, int d_head, int to_blocks,
                                             void* stream) {
  if (n_heads < 1 || n_heads > (1 << 20))
    return fail(PRNN_ERR_VALUE, "n_heads must be in [1, 2^20], got %d", n_heads);
  if (d_head < 1 || d_head > 64)
    return fail(PRNN_ERR_TYPE, "d_head must be in [1, 64], got %d", d_head);
  if (!moves || n_moves < 1 || n_moves > gru::kMaxMoves)
    return fail(PRNN_ERR_VALUE, "n_moves must be in [1, %d], got %d", gru::kMaxMoves, n_moves);
  const int per = 64 / d_head, nb = (n_heads + per - 1) / per;
  gru::Moves m{};
  long long wgs = 0;
  for (int k = 0; k < n_moves; ++k) {
    const prnn_block_move& v = moves[k];
    if (!v.src || !v.dst) return fail(PRNN_ERR_VALUE, "src and dst must be non-null");
    if (v.elem_bytes != 2 && v.elem_bytes != 4)
      return fail(PRNN_ERR_TYPE, "elements of 2 or 4 bytes, got %d", v.elem_bytes);
    if (v.rows < 1 || v.rows > (1ll << 40) / nb)
      return fail(PRNN_ERR_VALUE, "rows out of range: %lld", v.rows);
    m.src[k] = v.src;
    m.dst[k] = v.dst;
    m.units[k] = v.rows * nb * (v.matrix ? 64 : 1);
    m.matrix[k] = v.matrix != 0;
    m.two[k] = v.elem_bytes == 2;
    m.first[k] = static_cast<unsigned>(wgs);
    wgs += (m.units[k] + 4 * gru::kMoveRows - 1) / (4 * gru::kMoveRows);
    if (wgs > (1ll << 31) - 1) return fail(PRNN_ERR_VALUE, "too many rows: %lld", v.rows);
  }
  m.n = n_moves;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<unsigned>(wgs));
  if (to_blocks)
    gru::gru_blocks_kernel<true><<<grid, dim3(256), 0, s>>>(m, nb, n_heads, d_head);
  else
    gru::gru_blocks_kernel<false><<<grid, dim3(256), 0, s>>>(m, nb, n_heads, d_head);
  PRNN_HIP(hipGetLastError());
  return PRNN_OK;
}
