// One tile configuration of the int8 GEMM for one output type: the build script compiles this file once for each pair
// (I8F_TU_CFG, I8F_TU_OUT; I8F_TU_GROUPED where the configuration also serves the grouped launch).
#include "gemm_i8_impl.hpp"

namespace i8f {
namespace gemm {
template int launch_cfg<I8F_TU_CFG, I8F_TU_OUT>(GemmArgs &, hipStream_t);
#if I8F_TU_GROUPED
template int launch_cfg_grouped<I8F_TU_CFG, I8F_TU_OUT>(const GemmArgs *, int, hipStream_t);
#endif
}  // namespace gemm
}  // namespace i8f
