// The quad tile: four lanes per column (ARMA_HIP_QUAD_TILE=1).
#include "ar_quad.hpp"

namespace arma_hip {
namespace {

// Spin until *p >= need and return the value seen: relaxed device-coherent
// polls, with an acquire load every 64 polls.  With limit > 0 the wait is
// bounded: every 256 polls it gives up (returning need) once *abortw is set,
// or sets *abortw itself when it has spun for more than limit ticks of the
// constant-rate wall clock.  A launch that gives up still runs every tile to
// its end; the host reads *abortw afterwards and reports the launch as
// failed.
__device__ __forceinline__ int wait_progress(const int* p, int need, int* abortw,
                                             long long limit) {
	long long start = 0;
	for (int n = 1;; ++n) {
		const int v = (n & 63) ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
		                       : __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
		if (v >= need) return v;
		if (limit > 0 && (n & 255) == 0) {
			if (__hip_atomic_load(abortw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
				return need;
			const long long now = wall_clock64();
			if (start == 0) {
				start = now;
			} else if (now - start > limit) {
				__hip_atomic_store(abortw, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				return need;
			}
		}
		__builtin_amdgcn_s_sleep(1);
	}
}

// A consumed halo value of a slice in range: flag it when it is the sentinel.
template <class T>
__device__ __forceinline__ void check_halo(int* check, T v) {
	if (is_sentinel(v)) __hip_atomic_store(check, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int pmod(int a, int r) {
	const int m = a % r;
	return m < 0 ? m + r : m;
}

// ---- four lanes per column ----
//
// With one lane per column (wave_tile) every step streams all P0*P1*P2
// coefficients through the scalar cache, and a tile is one wave per SIMD:
// the step is a chain of scalar-load and LDS waits with little to overlap.
// For in-slice orders of at most 16 taps quad_tile gives each column a quad
// of four adjacent lanes.  Lane g of the quad owns the in-slice taps
// m = g + 4n (n < NT), keeps their coefficients for every k in registers and
// keeps its own partial accumulators; the quad's partial sums of the point
// being completed are added with two DPP butterfly stages, in a fixed lane
// order, so the value of a point does not depend on the tile shape or the
// schedule.  A tile of 256 columns is 1024 lanes, four waves per SIMD.
// Tap m = 0 (i = j = 0) sits on lane 0 of the quad: its k = 0 coefficient is
// zero in the table (phi(0,0,0) multiplies the noise of the completed point
// instead), and its k >= 1 terms take the completed value itself.
// Lane 0 of a quad loads the noise and stores the surface, lane 1 stores
// the mailbox, lanes 1 and 2 carry one halo slot each; the ring, mailbox,
// progress protocol and halo geometry are those of wave_tile.
// Measured on MI355X: one tile alone steps in 0.78 us against 1.13 us for
// wave_tile (1024 x 16 x 16, phi (7,7,2), FP64), but a full grid of tiles is
// set by the inter-tile fill and the memory traffic of 1024 lanes: wave_tile
// is faster on full grids (2048 x 512 x 512 FP32: 7.5 ms with its per-lane
// line; FP64 1024 x 256 x 256: 2.2 against 3.0 ms), so the quad tile runs
// only when ARMA_HIP_QUAD_TILE=1 asks for it (FP32 surfaces).
// quad_perm DPP controls: lanes (1,0,3,2), lanes (2,3,0,1), all from lane 0
constexpr int kDppXor1 = 0xb1, kDppXor2 = 0x4e, kDppLane0 = 0x00;

template <int CTRL>
__device__ __forceinline__ double quad_dpp(double v) {
	const int lo = __double2loint(v), hi = __double2hiint(v);
	return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, false),
	                        __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, false));
}

template <int CTRL>
__device__ __forceinline__ float quad_dpp(float v) {
	return __int_as_float(
		__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// Sum over the quad, the same bits on all four lanes (each stage adds two
// values in either order, which rounds the same).
template <class T>
__device__ __forceinline__ T quad_sum(T s) {
	s = s + quad_dpp<kDppXor1>(s);
	return s + quad_dpp<kDppXor2>(s);
}

// Compensated sum over the quad of the pairs (s, c): TwoSum of the leading
// parts (its error term is exact, so either operand order gives the same
// bits), the compensations and the error added to c.
template <class T>
__device__ __forceinline__ T quad_sum2(T s, T c) {
	auto stage = [&](T s2, T c2) {
		const T r = s + s2;
		const T bb = r - s;
		const T e = (s - (r - bb)) + (s2 - bb);
		c = (c + c2) + e;
		s = r;
	};
	stage(quad_dpp<kDppXor1>(s), quad_dpp<kDppXor1>(c));
	stage(quad_dpp<kDppXor2>(s), quad_dpp<kDppXor2>(c));
	return s + c;
}

template <class T, int TX, int P0, int NT, bool KAHAN>
__device__ __forceinline__ void quad_tile(
	T* __restrict__ zeta, int nt, int nx, int ny, const T* __restrict__ qcoef,
	const int* __restrict__ qoff, int P1, int P2, int nY, int* __restrict__ progress,
	const T* __restrict__ zero, T* __restrict__ sink, T* __restrict__ mbox, int NB,
	int total_steps, int t0, int b, int* abortw, long long limit, int* check,
	unsigned char* smem_raw) {
	constexpr int kTX = TX, kTY = kThreads / TX;
	static_assert(kTX * kTY == kThreads && kTX >= 8 && kTY >= 8, "tile shape");
	T* ring = reinterpret_cast<T*>(smem_raw);
	const int HX = P1 - 1, HY = P2 - 1;
	const int WX = kTX + HX, WY = kTY + HY;
	const int R = P1 + P2 - 1;
	const int slot = WX * WY;
	const int X = b / nY, Y = b - (b / nY) * nY;
	const int X0 = X * kTX, Y0 = Y * kTY;
	const int tid = threadIdx.x;
	const int g = tid & (kQuad - 1), col = tid / kQuad;
	const int lx = col / kTY, ly = col - (col / kTY) * kTY;
	const bool active = (X0 + lx < nx) && (Y0 + ly < ny);
	const size_t sxy = size_t(nx) * ny;
	const size_t own_off = size_t(X0 + lx) * ny + (Y0 + ly);
	const int own_lds = (lx + HX) * WY + (ly + HY);

	// the halo slot of quad lanes 1 and 2 (top band, then left band; at most
	// 2 * 256 positions for orders up to 10)
	const int H = WX * WY - kThreads;
	const int h = g == 1 ? col : (g == 2 ? col + kThreads : H);
	const bool hval = h < H;
	int hsk = 0, hlds = 0, hnb = 0, hm = 0, hdu = 0;
	bool hin = false;
	if (hval) {
		int hx, hy;
		if (h < HX * WY) {
			hx = -HX + h / WY;
			hy = -HY + (h - (h / WY) * WY);
		} else {
			const int q = h - HX * WY;
			hx = q / HY;
			hy = -HY + (q - (q / HY) * HY);
		}
		hsk = hx + hy;
		hlds = (hx + HX) * WY + (hy + HY);
		const int gx = X0 + hx, gy = Y0 + hy;
		hin = gx >= 0 && gy >= 0 && gx < nx && gy < ny;
		const int px = hx < 0 ? kTX + hx : hx, py = hy < 0 ? kTY + hy : hy;
		hnb = b - (hx < 0 ? nY : 0) - (hy < 0 ? 1 : 0);
		hm = mbox_column<TX>(px, py, HX, HY);
		hdu = (hx < 0 ? kTX : 0) + (hy < 0 ? kTY : 0);
	}
	const int nb_top = X > 0 ? b - nY : -1;
	const int nb_left = Y > 0 ? b - 1 : -1;
	int* const my_prog = progress + size_t(b) * kProgStride;
	const int* const top_prog = progress + size_t(max(nb_top, 0)) * kProgStride;
	const int* const left_prog = progress + size_t(max(nb_left, 0)) * kProgStride;

	// this lane's taps: coefficients [n][k] and LDS byte distances
	T c[NT][P0];
	int toff[NT];
#pragma unroll
	for (int n = 0; n < NT; ++n) {
		toff[n] = qoff[g * NT + n];
#pragma unroll
		for (int k = 0; k < P0; ++k) c[n][k] = qcoef[(g * NT + n) * P0 + k];
	}
	const T phi000 = qcoef[kQuad * NT * P0];

	Acc<T, KAHAN> acc[P0];
#pragma unroll
	for (int k = 0; k < P0; ++k) acc[k].zero();

	const int s0 = -(HX + HY);
	const int total_u = total_steps - s0;
	auto need_top = [&](int u) { return min(u + kTX + 1, total_u); };
	auto need_left = [&](int u) { return min(u + kTY + 1, total_u); };

	for (int q = tid; q < R * slot; q += kQThreads) ring[q] = T(0);
	int rs_own = pmod(s0 - lx - ly, R);
	int rs_h = pmod(s0 - hsk, R);

	const int my_m = mbox_column<TX>(lx, ly, HX, HY);
	// Memory traffic per lane and step, the same four instructions on every
	// lane (so that the compiler's vector-memory counter waits exactly for
	// the queue slot consumed):
	//  * quad lane 0 loads the noise and stores the surface with ordinary
	//    accesses; the other lanes load and store their own slot of the
	//    tile's sink, which stays in the L2;
	//  * quad lanes 1 and 2 load a halo value and lane 1 of a boundary
	//    column stores the mailbox, device-coherently, through one buffer
	//    descriptor spanning the mailboxes from the corner neighbour's to this
	//    tile's; every other lane passes the offset just past its end, which
	//    the hardware drops without a memory access.
	T* const my_sink = sink + size_t(b) * kQThreads + tid;
	const int bb0 = max(b - nY - 1, 0);
	const size_t tile_mb = size_t(total_u) * NB;  // elements of one tile's mailbox
	const unsigned mb_end = unsigned((size_t(b - bb0) + 1) * tile_mb * sizeof(T));
	const __amdgpu_buffer_rsrc_t mrsrc = __builtin_amdgcn_make_buffer_rsrc(
		mbox + size_t(bb0) * tile_mb, 0, int(mb_end), kBufferDword3);
	const bool mstore = g == 1 && my_m >= 0;
	unsigned moff = mstore ? unsigned((size_t(b - bb0) * tile_mb + my_m) * sizeof(T)) : mb_end;
	const unsigned mstep = mstore ? unsigned(NB * sizeof(T)) : 0u;
	// the noise of slice te and the halo of slice th_ld are the next to load;
	// both advance by one slice per step (a slice in range implies a step in
	// range)
	const bool eps_lane = g == 0 && active;
	int te = s0 - lx - ly, th_ld = s0 - hsk;
	T* pe = zeta + own_off + ptrdiff_t(te) * ptrdiff_t(sxy);
	unsigned hoff = hin ? unsigned(((size_t(hnb - bb0) * total_u + hdu) * NB + hm) * sizeof(T)) : 0u;
	const unsigned hstep = unsigned(NB * sizeof(T));
	auto issue_load = [=, &te, &th_ld, &pe, &hoff](T& qe, T& qh) {
		const bool ve = eps_lane && unsigned(te) < unsigned(nt);
		const bool vh = hin && unsigned(th_ld) < unsigned(nt);
		qe = *(ve ? pe : my_sink);
		qh = buffer_load_coherent<T>(mrsrc, vh ? hoff : mb_end);
		++te;
		++th_ld;
		pe += sxy;
		hoff += hstep;
	};

	int known_t = total_u, known_l = total_u;
	if (tid == 0) {
		known_t = nb_top >= 0 ? wait_progress(top_prog, need_top(kQD - 1), abortw, limit) : total_u;
		known_l =
			nb_left >= 0 ? wait_progress(left_prog, need_left(kQD - 1), abortw, limit) : total_u;
	}
	__syncthreads();
	T qe[kQD], qh[kQD];
	int qt[kQD], ql[kQD];  // neighbour progress loaded kQD steps earlier (lane 0)
#pragma unroll
	for (int d = 0; d < kQD; ++d) {
		issue_load(qe[d], qh[d]);
		qt[d] = known_t;
		ql[d] = known_l;
	}

	auto step = [&](int u, T& qe_q, T& qh_q, int& t_q, int& l_q) {
		const int s = u + s0;
		// 1. the halo value of step s into the ring
		{
			const int th = s - hsk;
			if (hval && th >= 0 && th < nt) {
				ring[rs_h * slot + hlds] = qh_q;
				if (check && hin) check_halo(check, qh_q);
			}
		}
		// 2. own point, slice t = s - lx - ly
		const int t = s - lx - ly;
		const bool live = active && t >= 0 && t < nt;
		const char* bb = reinterpret_cast<const char*>(ring + rs_own * slot + own_lds);
		T v[NT];
#pragma unroll
		for (int n = 0; n < NT; ++n) v[n] = *reinterpret_cast<const T*>(bb - toff[n]);
		// zero outside the column's slices (what the idle loads returned is
		// whatever the sink held), so that the steps before a column's first
		// slice push exact zeros into its accumulators
		const T eps_in = quad_dpp<kDppLane0>(qe_q);
		const T eps = live ? eps_in : T(0);
		T sum;
		if constexpr (KAHAN) {
			T p = T(0);
#pragma unroll
			for (int n = 0; n < NT; ++n) p = fma(c[n][0], v[n], p);
			acc[0].add(p);
			sum = quad_sum2(acc[0].s, acc[0].c);
		} else {
#pragma unroll
			for (int n = 0; n < NT; ++n) acc[0].s = fma(c[n][0], v[n], acc[0].s);
			sum = quad_sum(acc[0].s);
		}
		// slices t < t0 are given: they feed later sums unchanged
		const T zc = eps + (sum + phi000 * eps);
		const T z = t < t0 ? eps : zc;
		const bool zlive = g == 0 && live;
		if (zlive) ring[rs_own * slot + own_lds] = z;
		// (the noise of slice t + kQD is the next to load)
		*(zlive ? pe - ptrdiff_t(kQD) * ptrdiff_t(sxy) : my_sink) = z;
		buffer_store_coherent(mrsrc, moff, z);
		moff += mstep;
		// the terms of points t+1 .. t+P0-1 (tap 0 of quad lane 0 is the
		// point itself)
		const T v0 = g == 0 ? z : v[0];
#pragma unroll
		for (int k = 1; k < P0; ++k) {
			if constexpr (KAHAN) {
				T p = T(0);
#pragma unroll
				for (int n = 1; n < NT; ++n) p = fma(c[n][k], v[n], p);
				acc[k].add(fma(c[0][k], v0, p));
			} else {
#pragma unroll
				for (int n = 1; n < NT; ++n) acc[k].s = fma(c[n][k], v[n], acc[k].s);
				acc[k].s = fma(c[0][k], v0, acc[k].s);
			}
		}
#pragma unroll
		for (int k = 0; k + 1 < P0; ++k) acc[k] = acc[k + 1];
		acc[P0 - 1].zero();
		rs_own = wrap_inc(rs_own, R);
		rs_h = wrap_inc(rs_h, R);
		// keep this step's sums in this step: left free, the compiler defers
		// the k >= 1 terms to the step that completes their point, holding
		// the ring values of up to P0 - 1 steps in registers
#pragma unroll
		for (int k = 0; k < P0; ++k) acc[k].pin();
		// 3. lane 0: may the loads of step u + kQD go out?
		const int u2 = u + kQD;
		if (tid == 0) {
			known_t = max(known_t, t_q);
			known_l = max(known_l, l_q);
			if (u2 < total_u) {
				if (known_t < need_top(u2))
					known_t = wait_progress(top_prog, need_top(u2), abortw, limit);
				if (known_l < need_left(u2))
					known_l = wait_progress(left_prog, need_left(u2), abortw, limit);
			}
			t_q = nb_top >= 0 ? coherent_load(top_prog) : total_u;
			l_q = nb_left >= 0 ? coherent_load(left_prog) : total_u;
		}
		__syncthreads();
		// 4. publish: every wave consumed at this step a load issued after
		//    its stores of step u - kQD
		if (tid == 0 && u >= kQD) coherent_store(my_prog, u - kQD + 1);
		// 5. the loads of step u + kQD into the queue slot just consumed
		issue_load(qe_q, qh_q);
	};

	int u = 0;
	for (; u + kQD <= total_u; u += kQD) {
#pragma unroll
		for (int d = 0; d < kQD; ++d) step(u + d, qe[d], qh[d], qt[d], ql[d]);
	}
#pragma unroll
	for (int d = 0; d < kQD; ++d)
		if (u + d < total_u) step(u + d, qe[d], qh[d], qt[d], ql[d]);
	__builtin_amdgcn_s_waitcnt(0);
	__syncthreads();
	if (tid == 0) coherent_store(my_prog, total_u);
}

template <class T, int P0, int NT, bool KAHAN>
__global__ __launch_bounds__(kQThreads) void ar_quad_kernel(
	T* __restrict__ zeta, int nt, int nx, int ny, const T* __restrict__ qcoef,
	const int* __restrict__ qoff, int P1, int P2, int nY, int* __restrict__ progress,
	const T* __restrict__ zero, T* __restrict__ sink, T* __restrict__ mbox, int NB,
	int total_steps, int* check) {
	extern __shared__ __align__(16) unsigned char smem_raw[];
	quad_tile<T, 16, P0, NT, KAHAN>(zeta, nt, nx, ny, qcoef, qoff, P1, P2, nY, progress, zero,
	                                sink, mbox, NB, total_steps, 0, blockIdx.x, nullptr, 0,
	                                check, smem_raw);
}

// The same queue walk over surfaces on the quad tile (1024 lanes): the
// switch is over (P0 bucket, taps per lane), for the pairs whose
// coefficients fit the register budget.
template <class T, int TX, bool KAHAN>
__global__ __launch_bounds__(kQThreads) void ar_quad_batch_kernel(
	T* __restrict__ arena, const T* __restrict__ coef, const int* __restrict__ taps,
	int* __restrict__ progress, const T* __restrict__ zero, T* __restrict__ sink,
	T* __restrict__ mbox, const BatchSurface* __restrict__ surf, const int2* __restrict__ queue,
	int nqueue, int* __restrict__ abortw, long long limit) {
	extern __shared__ __align__(16) unsigned char smem_raw[];
	for (int item = blockIdx.x; item < nqueue; item += gridDim.x) {
		const int si = queue[item].x;
		const int b = queue[item].y;
		const BatchSurface& sf = surf[si];
		T* const z = arena + sf.zoff;
		const T* const qc = coef + sf.coff;
		const int* const qo = taps + sf.toff;
		int* const pr = progress + size_t(sf.poff) * kProgStride;
		T* const mb = mbox + sf.moff;
		const int wide = quad_taps(sf.P1 * sf.P2) == 4 ? 1 : 0;
		switch (2 * sf.body + wide) {
#define ARMA_QBATCH_BODY(I, N)                                                                   \
	case 2 * I + (N == 4 ? 1 : 0):                                                               \
		if constexpr (quad_fits(int(sizeof(T)), kBatchP0[I], N))                                 \
			quad_tile<T, TX, kBatchP0[I], N, KAHAN>(z, sf.nt, sf.nx, sf.ny, qc, qo, sf.P1, sf.P2,  \
			                                        sf.nY, pr, zero, sink, mb, sf.NB,              \
			                                        sf.total_steps, sf.t0, b, abortw, limit,       \
			                                        nullptr, smem_raw);                            \
		break;
			ARMA_QBATCH_BODY(0, 2)
			ARMA_QBATCH_BODY(0, 4)
			ARMA_QBATCH_BODY(1, 2)
			ARMA_QBATCH_BODY(1, 4)
			ARMA_QBATCH_BODY(2, 2)
			ARMA_QBATCH_BODY(2, 4)
			ARMA_QBATCH_BODY(3, 2)
			ARMA_QBATCH_BODY(3, 4)
			ARMA_QBATCH_BODY(4, 2)
			ARMA_QBATCH_BODY(4, 4)
			ARMA_QBATCH_BODY(5, 2)
			ARMA_QBATCH_BODY(5, 4)
#undef ARMA_QBATCH_BODY
		}
	}
}

template <int P0>
const void* quad_kernel_of(int nt) {
	if (nt == 2) {
		if constexpr (quad_fits(4, P0, 2))
			return reinterpret_cast<const void*>(&ar_quad_kernel<float, P0, 2, true>);
	} else {
		if constexpr (quad_fits(4, P0, 4))
			return reinterpret_cast<const void*>(&ar_quad_kernel<float, P0, 4, true>);
	}
	return nullptr;
}

}  // namespace

const void* ar_quad_kernel_f32(int P0, int nt) {
	switch (P0) {
	case 1: return quad_kernel_of<1>(nt);
	case 2: return quad_kernel_of<2>(nt);
	case 3: return quad_kernel_of<3>(nt);
	case 4: return quad_kernel_of<4>(nt);
	case 5: return quad_kernel_of<5>(nt);
	case 6: return quad_kernel_of<6>(nt);
	case 7: return quad_kernel_of<7>(nt);
	case 8: return quad_kernel_of<8>(nt);
	case 9: return quad_kernel_of<9>(nt);
	case 10: return quad_kernel_of<10>(nt);
	}
	return nullptr;
}

const void* ar_quad_batch_kernel_f32(int tile_x) {
	if (tile_x == 8) return reinterpret_cast<const void*>(&ar_quad_batch_kernel<float, 8, true>);
	if (tile_x == 32) return reinterpret_cast<const void*>(&ar_quad_batch_kernel<float, 32, true>);
	return reinterpret_cast<const void*>(&ar_quad_batch_kernel<float, 16, true>);
}

}  // namespace arma_hip
