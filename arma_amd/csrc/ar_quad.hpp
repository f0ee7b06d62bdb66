// What the host and the kernels of the quad tile (ar_quad.hip) share.
#pragma once

#include "ar_tile.hpp"

namespace arma_hip {
namespace {

constexpr int kQuad = 4;
constexpr int kQThreads = kThreads * kQuad;
constexpr int kQD = 4;  // prefetch distance of the queue loads, in steps

// Taps per lane of the quad tile for an in-slice order of P12 taps, 0 when
// the tile does not take it.
__host__ __device__ constexpr int quad_taps(int p12) { return p12 <= 8 ? 2 : p12 <= 16 ? 4 : 0; }

// 32-bit registers a lane of the quad tile may spend on its coefficients
// (four waves per SIMD leave 128 per lane in all).
constexpr int kQuadCoefRegs = 56;

__host__ __device__ constexpr bool quad_fits(int es, int P0, int nt) {
	return nt > 0 && P0 * nt * (es / 4) <= kQuadCoefRegs;
}

}  // namespace
}  // namespace arma_hip
