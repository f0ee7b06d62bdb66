// Batch wavefront kernels, float: many surfaces in one persistent launch.
#include "ar_batch_kernels.hpp"

namespace arma_hip {

const void* ar_batch_kernel_f32(int tile_x, bool buf, bool dense) {
	if (dense && buf && tile_x == 16) return ar_batch_dense_f32();
	return batch_kernel_by_tile<float, true>(tile_x, buf);
}

}  // namespace arma_hip
