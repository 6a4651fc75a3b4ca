// Small tiles of the MFMA rung, f16f16f16 instantiation (one translation unit per type bundle keeps the build parallel).
#include "rung4_mfma_wavek.hpp"

namespace gz {
template int launch_wavek<GZ_F16F16F16>(const GemmArgs<GZ_F16F16F16>&, int, const SplitK&, hipStream_t);
}  // namespace gz
