// Batch wavefront kernels whose known shapes all fit two workgroups per CU.
#include "ar_batch_kernels.hpp"

namespace arma_hip {

const void* ar_batch_dense_f32() {
	return reinterpret_cast<const void*>(&ar_batch_kernel<float, 16, true, 2, true, true>);
}

const void* ar_batch_dense_f64() {
	return reinterpret_cast<const void*>(&ar_batch_kernel<double, 16, false, 2, true, true>);
}

}  // namespace arma_hip
