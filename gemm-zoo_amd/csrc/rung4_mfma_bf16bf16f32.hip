// MFMA rung, bf16bf16f32 instantiation (one translation unit per type bundle keeps the build parallel).
#include "rung4_mfma.hpp"

namespace gz {
template int launch_mfma<GZ_BF16BF16F32>(const GemmArgs<GZ_BF16BF16F32>&, int, hipStream_t);
template int launch_splitk<GZ_BF16BF16F32>(const GemmArgs<GZ_BF16BF16F32>&, const SplitKPlan&, hipStream_t);
}  // namespace gz
