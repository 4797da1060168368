// ParaSLSTM mix='diag' launches for packed streams (cu_seqlens), fp32 and
// bf16 storage (launchers in slstm_packed_impl.h).  Kept apart from
// slstm_diag.hip so the two sets of kernel instantiations compile in parallel.
#include "slstm_packed_impl.h"

namespace prnn {
namespace slstm {

template void launch_picard_packed<float>(const float*, const float*, const float*, float*, int,
                                          int, int, float, const Lookback&, unsigned long long*,
                                          hipStream_t, const Packed&);
template void launch_picard_packed<bf16>(const bf16*, const bf16*, const bf16*, bf16*, int, int,
                                         int, float, const Lookback&, unsigned long long*,
                                         hipStream_t, const Packed&);
template void launch_newton_fused_packed<float>(const float*, const float*, const float*,
                                                const float*, float*, int, int, int, float,
                                                float, const Lookback&, unsigned long long*,
                                                hipStream_t, const Packed&);
template void launch_newton_fused_packed<bf16>(const bf16*, const bf16*, const bf16*,
                                               const bf16*, bf16*, int, int, int, float, float,
                                               const Lookback&, unsigned long long*, hipStream_t,
                                               const Packed&);
// K = 1 (result in the storage dtype) and the early-exit step (fp32 result)
template void launch_newton_packed<float, float, float>(const float*, const float*, const float*,
                                                        const float*, float*, int, int, float,
                                                        float, const Lookback&, int, hipStream_t,
                                                        const Packed&);
template void launch_newton_packed<bf16, bf16, bf16>(const bf16*, const bf16*, const bf16*,
                                                     const bf16*, bf16*, int, int, float, float,
                                                     const Lookback&, int, hipStream_t,
                                                     const Packed&);
template void launch_newton_packed<bf16, bf16, float>(const bf16*, const bf16*, const bf16*,
                                                      const bf16*, float*, int, int, float, float,
                                                      const Lookback&, int, hipStream_t,
                                                      const Packed&);
template void launch_newton_packed<bf16, float, float>(const bf16*, const bf16*, const bf16*,
                                                       const float*, float*, int, int, float,
                                                       float, const Lookback&, int, hipStream_t,
                                                       const Packed&);

}  // namespace slstm
}  // namespace prnn
