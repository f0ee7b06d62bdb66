// The kernels of the one-lane wavefront tile: one surface, or a queue of
// (surface, tile) entries of a batch.
#pragma once

#include "ar_tile.hpp"

namespace arma_hip {
namespace {

// Kernel arguments stay plain restrict-qualified pointers: the coefficient
// reads are then provably unclobbered by the kernel's stores and compile to
// scalar loads (a struct argument costs 30-60 VGPRs per lane).
template <class T, int TX, int P0, bool KAHAN, int G, int NTR, TapShape SH, bool BUF>
__global__ __launch_bounds__(kThreads * G, G == 1 ? 1 : is_dense(sizeof(T), P0, SH) ? 4 : 2) void ar_wave_kernel(
	T* __restrict__ zeta, int nt, int nx, int ny, const T* __restrict__ near,
	const T* __restrict__ coef, const int* __restrict__ offs, int P1, int P2, int nY,
	const T* __restrict__ zero, T* __restrict__ sink, T* __restrict__ mbox, int NB,
	int total_steps, int* check, int limit) {
	extern __shared__ __align__(16) unsigned char smem_raw[];
	// tiles wait only on tiles with smaller workgroup ids, which were dispatched
	// before them
	wave_tile<T, TX, P0, KAHAN, G, NTR, SH, BUF>(zeta, nt, nx, ny, near, coef, offs, P1, P2, nY,
	                                             zero, sink, mbox, NB, total_steps, 0,
	                                             diagonal_tile(blockIdx.x, (nx + TX - 1) / TX, nY),
	                                             CheckedWait{check, limit}, smem_raw);
}

// The single-surface kernel of order P0 in t for a variant.
template <class T, int P0, bool KAHAN>
const void* wave_kernel_of(const WaveVariant& v) {
	auto fn = [](auto* k) { return reinterpret_cast<const void*>(k); };
	constexpr int es = int(sizeof(T));
	if constexpr (P0 > 1) {
		if (v.buf && v.groups == 2) {
			if constexpr (two_columns_fit(es, P0))
				if (v.shape == kTwoColumns)
					return fn(&ar_wave_kernel<T, 16, P0, KAHAN, 2, 2 * P0 - 1, kTwoColumns, true>);
			if (v.shape == kSquare)
				return fn(&ar_wave_kernel<T, 16, P0, KAHAN, 2, square_taps(es, P0), kSquare, true>);
			return fn(&ar_wave_kernel<T, 16, P0, KAHAN, 2, 0, kAnyShape, true>);
		}
	}
	if (v.buf) return fn(&ar_wave_kernel<T, 16, P0, KAHAN, 1, 0, kAnyShape, true>);
	return fn(&ar_wave_kernel<T, 16, P0, KAHAN, 1, 0, kAnyShape, false>);
}

template <class T, bool KAHAN>
const void* wave_kernel_by_order(int P0, const WaveVariant& v) {
	switch (P0) {
	case 1: return wave_kernel_of<T, 1, KAHAN>(v);
	case 2: return wave_kernel_of<T, 2, KAHAN>(v);
	case 3: return wave_kernel_of<T, 3, KAHAN>(v);
	case 4: return wave_kernel_of<T, 4, KAHAN>(v);
	case 5: return wave_kernel_of<T, 5, KAHAN>(v);
	case 6: return wave_kernel_of<T, 6, KAHAN>(v);
	case 7: return wave_kernel_of<T, 7, KAHAN>(v);
	case 8: return wave_kernel_of<T, 8, KAHAN>(v);
	case 9: return wave_kernel_of<T, 9, KAHAN>(v);
	case 10: return wave_kernel_of<T, 10, KAHAN>(v);
	}
	return nullptr;
}

}  // namespace
}  // namespace arma_hip
