// Small tiles of the MFMA rung, e5m2e5m2f16 instantiation (one translation unit per type bundle keeps the build parallel).
#include "rung4_mfma_wavek.hpp"

namespace gz {
template int launch_wavek<GZ_E5M2E5M2F16>(const GemmArgs<GZ_E5M2E5M2F16>&, int, const SplitK&, hipStream_t);
}  // namespace gz
