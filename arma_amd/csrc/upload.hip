// Host-to-device copies of the tables that precede a launch.
#include "common.hpp"

#include <cstring>

namespace arma_hip {
namespace {

// What one launch carries: the arguments of a kernel go along with it, so the
// caller's buffer is free again at once and nobody waits.
constexpr size_t kChunkWords = 896;
constexpr size_t kMostChunks = 4;

struct Chunk {
	unsigned w[kChunkWords];
};

__global__ __launch_bounds__(256) void store_kernel(Chunk c, unsigned* __restrict__ dst, int n) {
	for (int i = threadIdx.x; i < n; i += 256) dst[i] = c.w[i];
}

}  // namespace

// Tables of up to 14 KB (a surface's coefficients, seeds and records, the time
// indices of a potential) travel as kernel arguments: a copy from pageable memory
// waits for the copy engine and then for the stream, 25-35 us between the kernels
// on both sides, a launch of this kernel about 5.  Larger ones, and any that a
// capture would have to refuse, are copied, complete on return.
void upload(arma_hip_ctx* ctx, void* dst, const void* src, size_t bytes) {
	if (bytes == 0) return;
	if (bytes <= kMostChunks * sizeof(Chunk) && bytes % 4 == 0 &&
	    reinterpret_cast<uintptr_t>(dst) % 4 == 0) {
		hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
		ARMA_HIP_CHECK(hipStreamIsCapturing(ctx->stream, &cap));
		if (cap == hipStreamCaptureStatusNone) {
			for (size_t at = 0; at < bytes; at += sizeof(Chunk)) {
				Chunk c;
				const size_t n = std::min(bytes - at, sizeof(Chunk));
				std::memcpy(c.w, (const unsigned char*)src + at, n);
				store_kernel<<<1, 256, 0, ctx->stream>>>(c, (unsigned*)((unsigned char*)dst + at),
				                                         int(n / 4));
				ARMA_HIP_CHECK(hipGetLastError());
			}
			return;
		}
	}
	ARMA_HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
	ARMA_HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

}  // namespace arma_hip
