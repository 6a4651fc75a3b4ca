// Small tiles of the MFMA rung, s8s8s32 instantiation (one translation unit per type bundle keeps the build parallel).
#include "rung4_mfma_wavek.hpp"

namespace gz {
template int launch_wavek<GZ_S8S8S32>(const GemmArgs<GZ_S8S8S32>&, int, const SplitK&, hipStream_t);
}  // namespace gz
