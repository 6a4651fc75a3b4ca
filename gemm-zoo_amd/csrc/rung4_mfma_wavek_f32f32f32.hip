// Small tiles of the MFMA rung, f32f32f32 instantiation (one translation unit per type bundle keeps the build parallel).
#include "rung4_mfma_wavek.hpp"

namespace gz {
template int launch_wavek<GZ_F32F32F32>(const GemmArgs<GZ_F32F32F32>&, int, const SplitK&, hipStream_t);
}  // namespace gz
