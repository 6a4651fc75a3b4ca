// Small tiles of the MFMA rung, bf16bf16bf16 instantiation (one translation unit per type bundle keeps the build parallel).
#include "rung4_mfma_wavek.hpp"

namespace gz {
template int launch_wavek<GZ_BF16BF16BF16>(const GemmArgs<GZ_BF16BF16BF16>&, int, const SplitK&, hipStream_t);
}  // namespace gz
