// Single-surface wavefront kernels, float.
#include "ar_wave_kernels.hpp"

namespace arma_hip {

const void* ar_wave_kernel_f32(int P0, const WaveVariant& v) {
	return wave_kernel_by_order<float, true>(P0, v);
}

}  // namespace arma_hip
