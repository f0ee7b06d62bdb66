// The batch kernel of the one-lane wavefront tile.  DENSE: two workgroups per
// CU, for batches whose known shapes all fit kDenseRegs (15 FP32 surfaces of
// orders up to 5: 490 us against 635 with one).
#pragma once

#include "ar_tile.hpp"

namespace arma_hip {
namespace {

// Workgroups take the queue's entries in order, each the next one when it is
// done with its last.  An entry only waits on earlier ones, so the earliest
// unfinished entry is always being marched: the launch cannot deadlock.  The
// waits are bounded all the same (abortw, limit), so that a launch that lost its
// CUs ends with an error instead of hanging.
//
// A tile whose turn came before its neighbours let it start holds its CU
// waiting, so the order matters as much as the tile: with entries w, w + G, ...
// dealt to workgroup w of G, tiles in rows, 12 FP32 surfaces of
// 111-476 slices took 2.62 ms, with a surface's tiles by X + Y 2.40 ms, with the
// next entry to whoever is free and the surfaces by their longest chain 1.33 ms.
template <class T, int TX, bool KAHAN, int G, bool BUF, bool DENSE>
__global__ __launch_bounds__(kThreads * G, G == 1 ? 1 : DENSE ? 4 : 2) void ar_batch_kernel(
	T* __restrict__ arena, const T* __restrict__ coef, const int* __restrict__ taps,
	const T* __restrict__ zero, T* __restrict__ sink, T* __restrict__ mbox,
	const BatchSurface* __restrict__ surf, const int2* __restrict__ queue, int nqueue,
	int* __restrict__ next, int* __restrict__ abortw, long long limit) {
	extern __shared__ __align__(16) unsigned char smem_raw[];
	__shared__ int taken;
	for (;;) {
		if (threadIdx.x == 0)
			taken = __hip_atomic_fetch_add(next, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		__syncthreads();
		const int item = __builtin_amdgcn_readfirstlane(taken);
		if (item >= nqueue) break;
		const int si = queue[item].x;
		const int b = queue[item].y;
		const BatchSurface& sf = surf[si];
		T* const z = arena + sf.zoff;
		const T* const c0 = coef + sf.coff;
		const int* const tp = taps + sf.toff;
		T* const mb = mbox + sf.moff;
#define ARMA_BATCH_TILE(P, N, S)                                                              \
	wave_tile<T, TX, P, KAHAN, G, N, S, BUF>(z, sf.nt, sf.nx, sf.ny, c0, c0 + kNear, tp, sf.P1, \
	                                         sf.P2, sf.nY, zero, sink, mb, sf.NB,             \
	                                         sf.total_steps, sf.t0, b, BatchWait{abortw, limit},  \
	                                         smem_raw)
#define ARMA_BATCH_BODY(I)                                                                    \
	case I:                                                                                   \
		ARMA_BATCH_TILE(kBatchP0[I], 0, kAnyShape);                                           \
		break;
#define ARMA_BATCH_SHAPED(P)                                                                  \
	case kBatchBuckets + P - kShapedMin:                                                      \
		if constexpr (G == 2 && two_columns_fit(sizeof(T), P) &&                              \
		              (!DENSE || is_dense(sizeof(T), P, kTwoColumns)))                        \
			ARMA_BATCH_TILE(P, 2 * P - 1, kTwoColumns);                                           \
		break;                                                                                \
	case kBatchBuckets + kShaped + P - kShapedMin:                                            \
		if constexpr (G == 2 && (!DENSE || is_dense(sizeof(T), P, kSquare)))                  \
			ARMA_BATCH_TILE(P, square_taps(sizeof(T), P), kSquare);                           \
		break;
		switch (sf.body) {
			ARMA_BATCH_BODY(0)
			ARMA_BATCH_BODY(1)
			ARMA_BATCH_BODY(2)
			ARMA_BATCH_BODY(3)
			ARMA_BATCH_BODY(4)
			ARMA_BATCH_BODY(5)
			ARMA_BATCH_SHAPED(3)
			ARMA_BATCH_SHAPED(4)
			ARMA_BATCH_SHAPED(5)
			ARMA_BATCH_SHAPED(6)
			ARMA_BATCH_SHAPED(7)
			ARMA_BATCH_SHAPED(8)
			ARMA_BATCH_SHAPED(9)
		}
#undef ARMA_BATCH_TILE
#undef ARMA_BATCH_BODY
#undef ARMA_BATCH_SHAPED
		__syncthreads();  // the next tile clears the LDS that this one's lanes may still read
	}
}

// (the dense kernels are a translation unit of their own)
template <class T, bool KAHAN>
const void* batch_kernel_by_tile(int tile_x, bool buf) {
	auto fn = [](auto* k) { return reinterpret_cast<const void*>(k); };
	if (tile_x == 8)
		return buf ? fn(&ar_batch_kernel<T, 8, KAHAN, 1, true, false>)
		           : fn(&ar_batch_kernel<T, 8, KAHAN, 1, false, false>);
	if (tile_x == 32)
		return buf ? fn(&ar_batch_kernel<T, 32, KAHAN, 1, true, false>)
		           : fn(&ar_batch_kernel<T, 32, KAHAN, 1, false, false>);
	return buf ? fn(&ar_batch_kernel<T, 16, KAHAN, 2, true, false>)
	           : fn(&ar_batch_kernel<T, 16, KAHAN, 1, false, false>);
}

}  // namespace

const void* ar_batch_dense_f32();
const void* ar_batch_dense_f64();

}  // namespace arma_hip
