// Single-surface wavefront kernels, double.
#include "ar_wave_kernels.hpp"

namespace arma_hip {

const void* ar_wave_kernel_f64(int P0, const WaveVariant& v) {
	return wave_kernel_by_order<double, false>(P0, v);
}

}  // namespace arma_hip
