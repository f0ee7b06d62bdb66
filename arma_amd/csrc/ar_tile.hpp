// Persistent wavefront kernel for the 3-D AR recurrence
//   zeta(t,x,y) = eps(t,x,y) + sum_{k,i,j} phi(k,i,j) zeta(t-k, x-i, y-j)
// (src/generator/ar_model_surf.cc:3-36; zero outside the grid, which is the
// reference's truncated causal boundary).
//
// Decomposition:
//  * Every tile of TX x TY columns (x, y) is marched over the whole t axis by
//    256 lanes, one per column, or by two groups of 256 that share the work of
//    a column.  Lane (x, y) completes slice t = s - x - y at step s, so every
//    in-slice dependency (x-i, y-j) was finished at an earlier step: the skew
//    replaces the reference's partition DAG inside the tile.
//  * "Push" form of the sum: each value zeta(t, x-i, y-j) is read once from LDS
//    by each group and feeds the partial sums of the points (t+k, x, y), k < P0,
//    which the lanes keep in registers: P1*P2 LDS reads feed P0*P1*P2 FMAs.
//  * LDS holds a ring of planes, one per step, of the tile plus its causal halo
//    (P1-1 rows above, P2-1 columns to the left).
//  * Halo values come from the neighbouring tiles through HBM.  Each tile keeps
//    a mailbox with one row per step of the values its boundary lanes (the
//    bottom P1-1 rows and right P2-1 columns) computed at that step, stored
//    device-coherently (past the per-XCD L2) as contiguous rows; the surface
//    itself goes out with ordinary write-back stores.  A neighbour computed the
//    value at a halo position at its own step u + TX and / or + TY, so a
//    consumer reads a fixed mailbox row per step, kD steps ahead.  The launch
//    fills the mailboxes with a signalling NaN first, which arithmetic never
//    produces, so the value says itself whether it is there: no counters, no
//    fences, no polls while it is.  Tiles only wait on tiles that were started
//    before them, so the launch cannot deadlock.
//  * FP32 mode keeps every partial sum as a compensated (Kahan/TwoSum) pair;
//    each step adds one P1*P2-term FP32 partial to it.
//
// What bounds it: a step is a chain from the last step's values to this one's,
// write - barrier - read - part[0] - write, about 0.3 us, plus the FMAs of one
// step (P0*P1*P2 of four cycles per wave and SIMD), which go to twice the waves.
// 1024 x 256 x 256 FP64, phi (7, 7, 2): 2.16 ms with one lane per column,
// coefficients streamed through the scalar cache and progress counters polled at
// every step, 0.84 ms so; phi (7, 7, 7) 3.84 and 2.77 ms; 512^3 FP32 (7, 7, 7) 6.5 and
// 2.6 ms, 2048 x 512 x 512 FP32 (7, 7, 2) 7.65 and 2.88 ms.
#pragma once

#include "common.hpp"

#include <type_traits>
#include <utility>
#include <vector>

namespace arma_hip {

// What the compiler knows of the in-slice order: nothing, P0 x 2 (a
// propagating wave's) or P0 x P0 (a standing wave's).
enum TapShape { kAnyShape, kTwoColumns, kSquare };

// The form of the one-lane tile that a launch takes.
struct WaveVariant {
	bool buf = false;  // accesses through buffer descriptors
	int groups = 1;
	int ntr = 0;       // resident taps
	TapShape shape = kAnyShape;
};

// The kernels, one translation unit each (they take the compiler a while).
const void* ar_wave_kernel_f32(int P0, const WaveVariant& v);
const void* ar_wave_kernel_f64(int P0, const WaveVariant& v);
const void* ar_batch_kernel_f32(int tile_x, bool buf, bool dense);
const void* ar_batch_kernel_f64(int tile_x, bool buf, bool dense);
const void* ar_quad_kernel_f32(int P0, int taps_per_lane);
const void* ar_quad_batch_kernel_f32(int tile_x);

namespace {

// Tiles are TX x TY columns with TX * TY = kThreads: 8 x 32, 16 x 16 or
// 32 x 8 (the halo of a 10 x 10 in-slice order then needs at most two slots
// per lane).
constexpr int kThreads = 256;
constexpr int kD = 4;  // prefetch distance of the noise and halo loads, in steps
constexpr int kMaxP12 = 10;  // largest P1, P2 handled
constexpr int kProgStride = 32;  // ints between tile progress counters: one per 128-byte line

template <class T, bool KAHAN>
struct Acc;

template <class T>
struct Acc<T, false> {
	T s;
	__device__ void zero() { s = T(0); }
	__device__ void add(T v) { s += v; }
	__device__ T value() const { return s; }
	__device__ void pin() { asm volatile("" : "+v"(s)); }
};

template <class T>
struct Acc<T, true> {
	T s, c;
	__device__ void zero() {
		s = T(0);
		c = T(0);
	}
	__device__ void add(T v) {
		// TwoSum(s, v); the rounding error goes to the compensation term
		const T r = s + v;
		const T bb = r - s;
		c += (s - (r - bb)) + (v - bb);
		s = r;
	}
	__device__ T value() const { return s + c; }
	__device__ void pin() { asm volatile("" : "+v"(s), "+v"(c)); }
};

__global__ void reset_progress(int* p, int n) {
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) p[i] = 0;
}

template <class T>
__device__ __forceinline__ T coherent_load(const T* p) {
	return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <class T>
__device__ __forceinline__ void coherent_store(T* p, T v) {
	__hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Device-coherent loads and stores through a buffer descriptor (the
// instruction form of the agent-scope relaxed atomics above: sc1).  An
// offset past the descriptor's byte range loads zero and stores nothing,
// without a memory access.  Word 3 of the descriptor: raw 32-bit data for
// gfx9-class buffer instructions.
constexpr int kBufferDword3 = 0x00020000;
constexpr int kCoherentSc1 = 16;
typedef unsigned int uint2v __attribute__((ext_vector_type(2)));

template <class T>
__device__ __forceinline__ T buffer_load_coherent(__amdgpu_buffer_rsrc_t r, unsigned off) {
	if constexpr (sizeof(T) == 8)
		return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kCoherentSc1));
	else
		return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, kCoherentSc1));
}

template <class T>
__device__ __forceinline__ void buffer_store_coherent(__amdgpu_buffer_rsrc_t r, unsigned off, T v) {
	if constexpr (sizeof(T) == 8)
		__builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, v), r, off, 0, kCoherentSc1);
	else
		__builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0,
		                                      kCoherentSc1);
}

// The same without device coherence.
template <class T>
__device__ __forceinline__ T buffer_load(__amdgpu_buffer_rsrc_t r, unsigned off) {
	if constexpr (sizeof(T) == 8)
		return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
	else
		return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

template <class T>
__device__ __forceinline__ void buffer_store(__amdgpu_buffer_rsrc_t r, unsigned off, T v) {
	if constexpr (sizeof(T) == 8)
		__builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, v), r, off, 0, 0);
	else
		__builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 0);
}

// Every mailbox is filled with this signalling NaN before a launch; arithmetic
// only produces quiet NaNs, and given values are stored there without it
// (quieted), so a consumer that reads it for a slice in range has read a mailbox
// row before its producer stored it.
constexpr unsigned long long kHaloSentinel64 = 0x7ff4a5a5a5a5a5a5ull;
constexpr unsigned kHaloSentinel32 = 0x7fa5a5a5u;

// (the high word tells: no quiet NaN and no number has it)
__device__ __forceinline__ bool is_sentinel(double v) {
	return unsigned(__double2hiint(v)) == unsigned(kHaloSentinel64 >> 32);
}
__device__ __forceinline__ bool is_sentinel(float v) { return __float_as_uint(v) == kHaloSentinel32; }

__device__ __forceinline__ double quieted(double v) {
	return is_sentinel(v) ? __hiloint2double(__double2hiint(v) | 0x00080000, __double2loint(v)) : v;
}
__device__ __forceinline__ float quieted(float v) {
	return is_sentinel(v) ? __uint_as_float(kHaloSentinel32 | 0x00400000u) : v;
}

// n elements at a 16-byte aligned address, 16 bytes per lane.
template <class T>
__global__ void fill_sentinel(T* p, size_t n) {
	constexpr unsigned lo = sizeof(T) == 8 ? unsigned(kHaloSentinel64) : kHaloSentinel32;
	constexpr unsigned hi = sizeof(T) == 8 ? unsigned(kHaloSentinel64 >> 32) : kHaloSentinel32;
	constexpr size_t per = 16 / sizeof(T);
	const size_t i0 = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
	const size_t step = size_t(gridDim.x) * blockDim.x;
	for (size_t i = i0; i < n / per; i += step)
		reinterpret_cast<uint4*>(p)[i] = make_uint4(lo, hi, lo, hi);
	for (size_t i = n / per * per + i0; i < n; i += step) {
		if constexpr (sizeof(T) == 8)
			p[i] = __longlong_as_double((long long)kHaloSentinel64);
		else
			p[i] = __uint_as_float(kHaloSentinel32);
	}
}

inline size_t div_ceil_z(size_t a, size_t b) { return a / b + (a % b ? 1 : 0); }

__device__ __forceinline__ int wrap_inc(int v, int r) { return v + 1 == r ? 0 : v + 1; }

// ---- tables of one surface ----
//
// At step s a lane completes a point of slice t = s - x - y.  By then everything
// that its neighbours (x - i, y - j), i + j > 0, have of slice t was completed at
// earlier steps, so the step adds up the slice's part of the sums of all slices
// t + k, k < P0, before the point itself is known:
//   part[k] = sum of phi(k, i, j) zeta(t, x - i, y - j), (i, j) != (0, 0)
// as a chain of FMAs from zero over the taps in row-major order; the point takes
// acc[0] + part[0], and acc[k] of the others gets part[k] + phi(k, 0, 0) times the
// point, one addition per slice.  In FP32 that addition is compensated.
//
// The order is part of the result: fitted coefficients of a standing wave are
// large and cancel (sum of |phi| 13-20 for a variance of 1), so that sums taken in
// another order differ by more than the rounding of their results, and a
// transform of the surface that is flat or not monotone (NIT) makes visible steps
// of it.  Adding the nearest terms apart from the others leaves only a few
// operations between the last step's values and a point, 0.79 in place of
// 0.84 ms above, but came out up to 1.4 times as far from 64 bits in FP32.
//
// The accumulators may be split between two groups of waves (256 lanes each, the
// same columns): group 0 has k < K0, the point and the memory traffic, group 1
// has k >= K0.  Group 1 takes its points a step late, from LDS, and hands slice
// t + K0 to group 0 through LDS at every step: the sum so far and part[K0], to
// which group 0, which has the point, adds phi(K0, 0, 0) times it.  The split
// changes no sum.
//
// Tables: near[k] = phi(k, 0, 0), k < P0, then per group the coefficients
// [tap][k] of its accumulators, taps (0, 1), (0, 2), ... in row-major order padded
// with zero coefficients.  Offsets: LDS holds the last R steps' values of the tile
// and its halo, one plane per step (step s in plane s mod R), so a tap's distance
// is uniform over the tile but turns with the step: row s mod R of the offset
// table has the byte offsets of [this step's plane, the last step's, unused, unused,
// the taps].

// The first NTR taps' coefficients (a template parameter) stay in vector
// registers, the others are streamed through the scalar cache in chunks of
// chunk_taps taps, whose coefficients fit the scalar registers.
__host__ __device__ constexpr int chunk_taps(int es, int k) {
	int c = 16;
	while (c > 1 && c * k * es > 256) c /= 2;
	return c;
}
constexpr int kNear = 16;  // elements before the coefficients, phi(k, 0, 0) in the first
constexpr int kOffHead = 4;

// n taps padded to the kernel's units.
__host__ __device__ constexpr int padded_taps(int n, int ntr, int chunk) {
	return n <= ntr ? ntr : ntr + (n - ntr + chunk - 1) / chunk * chunk;
}
// Planes of the LDS ring: the farthest tap of a step was completed
// P1 + P2 - 2 steps before it.  Of two columns a multiple of the prefetch
// distance, as the steady steps are unrolled over the planes; not otherwise: with
// FP64 orders of 9 x 10 the planes between would not fit beside the line of an 8 x 32
// tile.
__host__ __device__ constexpr int ring_planes(int P1, int P2) {
	const int n = P1 + P2 - 1 > 2 ? P1 + P2 - 1 : 2;
	return P2 == 2 ? (n + kD - 1) / kD * kD : n;
}
// Row pitch of a plane, in elements.  A wave reads a tap from four rows of 16
// lanes; in FP32 a pitch of 48 keeps the rows in separate banks where the tight
// pitch TY + P2 - 1 does not (1024 x 16 x 16, phi (5, 5, 5): 611 against 529 us,
// phi (7, 7, 7): 1110 against 935 us).  In FP64 it measured the same as the
// tight one (1570 against 1557 us), which leaves more LDS.
__host__ __device__ constexpr int ring_pitch(int es, int TX, int P1, int P2, int groups) {
	const int TY = kThreads / TX, tight = TY + P2 - 1;
	if (es != 4 || TX != 16 || groups == 1) return tight;
	const int rest = (TY + 1) * kThreads * es + 6 * kThreads * es;  // line, hand-over
	return ring_planes(P1, P2) * (TX + P1 - 1) * 48 * es + rest <= 160 * 1024 ? 48 : tight;
}

// Accumulators of group 0 of two.  Group 0 also has the point and the memory
// traffic, about 60 instructions a step, so with few taps it takes the
// fewest accumulators that leave group 1's coefficients room in its registers;
// with many the halves are even.
constexpr int kCoefRegs = 196;  // 32-bit registers for coefficients, of 256 at two waves per SIMD
constexpr int kDenseRegs = 84;  // of 128 at four
__host__ __device__ constexpr int group_split(int es, int p0, TapShape shape) {
	const int half = p0 > 2 ? (p0 - 1) / 2 : 1;
	if (shape != kTwoColumns) return half;
	const int most = (2 * p0 - 1) * (p0 - half) * (es / 4) <= kDenseRegs ? kDenseRegs : kCoefRegs;
	int k = p0 / 4 > 1 ? p0 / 4 : 1;
	while (k < half && (2 * p0 - 1) * (p0 - k) * (es / 4) > most) ++k;
	return k;
}
__host__ __device__ constexpr int group_most(int es, int p0, int groups, TapShape shape) {
	const int k = group_split(es, p0, shape);
	return groups == 1 ? p0 : p0 - k > k ? p0 - k : k;
}
// Resident taps of the kernels with known shapes.  Of a square order, as many as
// leave room for the sums, parts and row offsets of its P0: with more the kernels
// kept 5 to 80 registers in scratch memory (512 x 256 x 256 FP64, phi (9, 9, 9): 19
// taps 5.28 ms, 13 3.47 ms; (7, 7, 7): 24 taps 2.28 ms, 19 1.91 ms, 13 2.05 ms).
__host__ __device__ constexpr bool two_columns_fit(int es, int p0) {
	return p0 > 1 && (2 * p0 - 1) * group_most(es, p0, 2, kTwoColumns) * (es / 4) <= kCoefRegs;
}
__host__ __device__ constexpr int square_taps(int es, int p0) {
	const int w = es / 4, n = (238 - 6 * p0 * w) / (group_most(es, p0, 2, kSquare) * w);
	return n < p0 * p0 - 1 ? n : p0 * p0 - 1;
}
// Whether two workgroups of two groups share a CU: all coefficients of a known
// shape within kDenseRegs, or none resident.
__host__ __device__ constexpr bool is_dense(int es, int p0, TapShape shape) {
	return shape == kAnyShape ||
	       ((shape == kTwoColumns ? 2 : p0) * p0 - 1) * group_most(es, p0, 2, shape) * (es / 4) <=
	           kDenseRegs;
}

// Mailbox column of tile-local lane (x, y), or -1 when no neighbour reads it:
// the bottom HX rows first (row-major), then the right HY columns of the
// rows above them.
template <int TX>
__host__ __device__ __forceinline__ int mbox_column(int x, int y, int HX, int HY) {
	constexpr int TY = kThreads / TX;
	if (x >= TX - HX) return (x - (TX - HX)) * TY + y;
	if (y >= TY - HY) return TY * HX + x * HY + (y - (TY - HY));
	return -1;
}

template <int TX>
__host__ __device__ constexpr int mbox_width(int HX, int HY) {
	return (kThreads / TX) * HX + (TX - HX) * HY;
}

inline int mbox_width_rt(int TX, int HX, int HY) { return (kThreads / TX) * HX + (TX - HX) * HY; }

// The LDS byte offsets of phase PH for an in-slice order of P0 x 2.
template <class T, int kTX, int P0, int PH>
struct PhaseRow {
	static constexpr int R = ring_planes(P0, 2), WY = ring_pitch(sizeof(T), kTX, P0, 2, 2),
	                     kPlane = (kTX + P0 - 1) * WY;
	static __device__ constexpr unsigned at(int steps, int i, int j) {
		return unsigned((((PH - steps) % R + R) % R * kPlane - i * WY - j) * int(sizeof(T)));
	}
	__device__ constexpr unsigned head(int e) const { return at(e, 0, 0); }
	__device__ constexpr unsigned tap(int e) const {
		const int i = (e + 1) / 2, j = (e + 1) % 2;
		return at(i + j, i, j);
	}
};

// f(integral_constant<0>) ... f(integral_constant<N - 1>)
template <int N, class F, int... I>
__device__ __forceinline__ void unrolled_seq(F&& f, std::integer_sequence<int, I...>) {
	(f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unrolled(F&& f) {
	unrolled_seq<N>(f, std::make_integer_sequence<int, N>{});
}

// The b-th tile in order of X + Y, then X, of nX rows of nY tiles, as its index
// X * nY + Y.  The tiles before a diagonal of the short side form a triangle,
// those after the last full diagonal one from the other end.
__host__ __device__ inline int diagonal_tile(int b, int nX, int nY) {
	const int m = nX < nY ? nX : nY, ntiles = nX * nY;
	const int tri = m * (m - 1) / 2;  // tiles of the diagonals 0 .. m - 2
	const bool tail = b >= ntiles - tri;
	const int c = tail ? ntiles - 1 - b : b;
	int d, e;  // diagonal, place on it
	if (c < tri) {
		d = int((sqrtf(8.0f * float(c) + 1.0f) - 1.0f) * 0.5f);
		while (d * (d + 1) / 2 > c) --d;
		while ((d + 1) * (d + 2) / 2 <= c) ++d;
		e = c - d * (d + 1) / 2;
	} else {
		d = m - 1 + (c - tri) / m;
		e = (c - tri) % m;
	}
	int X = e + (d >= nY ? d - nY + 1 : 0);
	int Y = d - X;
	if (tail) {
		X = nX - 1 - e;
		Y = nY - 1 - (d - e);
	}
	return X * nY + Y;
}

// How long a tile waits for a neighbour's value; gives_up after poll n of a wait
// that began with start = 0.
//
// The batch kernel's: every 256 polls it gives up once *abortw is set, or sets
// *abortw itself when it has spun for more than limit ticks of the constant-rate
// wall clock.  The host reads *abortw afterwards.
struct BatchWait {
	int* abortw;
	long long limit;
	__device__ __forceinline__ bool gives_up(int n, long long& start) {
		if ((n & 255) != 0 || limit <= 0) return false;
		if (__hip_atomic_load(abortw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return true;
		const long long now = wall_clock64();
		if (start == 0) {
			start = now;
		} else if (now - start > limit) {
			__hip_atomic_store(abortw, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			return true;
		}
		return false;
	}
};

// A single surface's: for ever, but in a checked launch limit polls, once per wave
// and tile, since later waits of a wave that gave up end with their first.  Then
// *check is set.  (Nothing more is in the loop, which is unrolled with the steps: with
// the clock and *abortw in it a step took 2 % longer, at order 1 in t 10 %.)
struct CheckedWait {
	int* check;
	int limit;  // 0: none
	__device__ __forceinline__ bool gives_up(int n, long long&) {
		if (n != limit) return false;
		limit = 1;
		__hip_atomic_store(check, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		return true;
	}
};

// The march of one tile over all of t (P0 accumulators; a surface of lower
// order in t has zero coefficients past its own order).  G groups of 256 lanes;
// the first NTR taps resident.  With SH = kTwoColumns (all taps resident) LDS
// offsets are constants of the step's phase, and the steady steps are unrolled
// over the phases; with SH = kSquare the taps of one distance i + j share a
// base that turns with the step, at constant offsets.
template <class T, int TX, int P0, bool KAHAN, int G, int NTR, TapShape SH, bool BUF, class Wait>
__device__ __forceinline__ void wave_tile(
	T* __restrict__ zeta, int nt, int nx, int ny, const T* __restrict__ near,
	const T* __restrict__ coef, const int* __restrict__ offs, int P1_, int P2_, int nY,
	const T* __restrict__ zero, T* __restrict__ sink, T* __restrict__ mbox, int NB,
	int total_steps, int t0, int b, Wait wait, unsigned char* smem_raw) {
	constexpr int kTX = TX, kTY = kThreads / TX;
	static_assert(kTX * kTY == kThreads && kTX >= 8 && kTY >= 8, "tile shape");
	static_assert(G == 1 || P0 > 1, "two groups need two accumulators");
	constexpr bool TWO = SH == kTwoColumns, SQ = SH == kSquare;
	static_assert(!TWO || NTR == 2 * P0 - 1, "all taps of a P0 x 2 order are resident");
	static_assert(!SQ || NTR < P0 * P0, "no more taps than the order has");
	static_assert(P0 <= kNear, "phi(k, 0, 0) before the coefficients");
	constexpr int KD = kD;
	const int P1 = SH == kAnyShape ? P1_ : P0, P2 = TWO ? 2 : SQ ? P0 : P2_;
	constexpr int kCH = chunk_taps(sizeof(T), group_most(sizeof(T), P0, G, SH));
	constexpr int K0 = G == 1 ? P0 : group_split(sizeof(T), P0, SH), K1 = P0 - K0;
	const int HX = P1 - 1, HY = P2 - 1;
	const int WX = kTX + HX, WY = kTY + HY;
	const int R = ring_planes(P1, P2);
	const int pitch = ring_pitch(sizeof(T), TX, P1, P2, G);
	const int plane = WX * pitch;
	const int X = b / nY, Y = b - (b / nY) * nY;
	const int X0 = X * kTX, Y0 = Y * kTY;
	// opaque, so that the bodies of a batch kernel do not keep each other's
	// lane constants in registers across its queue loop
	int thread = threadIdx.x;
	asm volatile("" : "+v"(thread));
	const int group = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(thread / kThreads);
	const int tid = thread % kThreads;
	const int lx = tid / kTY, ly = tid - (tid / kTY) * kTY;
	const int ntap = padded_taps(P1 * P2 - 1, NTR, kCH);
	const int orow = kOffHead + ntap;  // ints per row of the offset table

	// LDS: the ring of planes, a line of kDL slots per lane, and with two
	// groups the hand-over of two steps (a part, and the sum that it goes to)
	unsigned char* const ring = smem_raw;
	constexpr int kDL = kTY + 1;
	T* const line = reinterpret_cast<T*>(smem_raw + size_t(R) * plane * sizeof(T)) + tid;
	using Hand = std::conditional_t<KAHAN, T[3], T[2]>;
	Hand* const hand = reinterpret_cast<Hand*>(line - tid + kDL * kThreads) + tid;
	const unsigned own = unsigned(((lx + HX) * pitch + (ly + HY)) * sizeof(T));
	auto lds = [&](unsigned at) -> T& { return *reinterpret_cast<T*>(ring + at); };

	// Step u of the loop is skew step s = u + s0; s0 < 0 lets the halo positions
	// (negative skew hx + hy) deliver their first slices and the first noise
	// arrive.  Every tile uses the same s0.
	const int s0 = -max(HX + HY, 1);
	const int total_u = total_steps - s0;

	// everything in LDS starts zeroed: halo positions outside the grid, slices
	// before the first and their noise stay zero
	{
		const int words = R * plane + kDL * kThreads + (G > 1 ? 2 * kThreads * (KAHAN ? 3 : 2) : 0);
		for (int q = thread; q < words; q += G * kThreads) reinterpret_cast<T*>(smem_raw)[q] = T(0);
	}
	int ph = s0 % R;  // plane of this step
	if (ph < 0) ph += R;

	// A step's LDS byte offsets from a lane's own position: a row of the offset
	// table, read a step ahead into scalar registers (the head and the resident
	// taps; for a square order the head and one base per distance), or
	// constants of the phase.
	constexpr int kP2 = TWO ? 2 : P0, kW = ring_pitch(sizeof(T), TX, P0, kP2, G);
	constexpr int kBases = P0 > 1 ? 2 * P0 - 2 : 1;  // distances of a square order's taps
	constexpr int kRow = 2 + (SQ ? kBases : NTR);
	struct Row {
		int o[kRow];
		__device__ unsigned head(int e) const { return unsigned(o[e]); }
		__device__ unsigned tap(int m) const {
			return unsigned(o[SQ ? 0 : 2 + m]);
		}
	};
	auto read_row = [&](int phase, Row& r) {
		const int* const p = offs + phase * orow;
#pragma unroll
		for (int e = 0; e < 2; ++e) r.o[e] = p[e];
		if constexpr (SQ) {
			// tap (0, d) or (d - P0 + 1, P0 - 1) of each distance d, without its
			// distance within the plane
#pragma unroll
			for (int d = 1; d <= kBases; ++d) {
				const int i = d < P0 ? 0 : d - P0 + 1, j = d < P0 ? d : P0 - 1;
				r.o[1 + d] = p[kOffHead + i * P0 + j - 1] + (i * kW + j) * int(sizeof(T));
			}
		} else {
#pragma unroll
			for (int e = 0; e < NTR; ++e) r.o[2 + e] = p[kOffHead + e];
		}
	};
	auto hold_row = [](Row& r) {
#pragma unroll
		for (int e = 0; e < kRow; ++e) asm volatile("" : "+s"(r.o[e]));
	};
	// a tap's value from base, the farthest in-plane distance before own, so that
	// a known order's constant offsets are nonnegative
	constexpr unsigned kBack = SH == kAnyShape ? 0u : unsigned(((P0 - 1) * kW + kP2 - 1) * sizeof(T));
	auto at_tap = [&](const auto& row, int e, unsigned base) {
		if constexpr (SQ) {
			const int i = (e + 1) / P0, j = (e + 1) % P0;
			return lds(base + unsigned(row.o[1 + i + j]) + (kBack - unsigned((i * kW + j) * sizeof(T))));
		} else {
			return lds(base + (kBack + row.tap(e)));
		}
	};
	// the parts of one group's K accumulators, with the coefficients cf
	auto parts_of = [&](auto kc, const T* __restrict__ cf, auto& creg, auto& part, int phase,
	                    const auto& row) {
		constexpr int K = decltype(kc)::value;
		// opaque in every step where two workgroups share a CU: the addresses of the
		// unrolled phases, kept over the loop, did not fit beside the coefficients
		unsigned base = own - kBack;
		if constexpr (TWO && is_dense(sizeof(T), P0, SH)) asm volatile("" : "+v"(base));
#pragma unroll
		for (int r = 0; r < K; ++r) part[r] = T(0);
		if constexpr (NTR > 0) {
			// the values in runs of 16, so that they do not crowd out the
			// coefficients
#pragma unroll
			for (int m0 = 0; m0 < NTR; m0 += 16) {
				T v[16];
#pragma unroll
				for (int m = 0; m < 16; ++m)
					if (m0 + m < NTR) v[m] = at_tap(row, m0 + m, base);
#pragma unroll
				for (int m = 0; m < 16; ++m)
					if (m0 + m < NTR) {
#pragma unroll
						for (int r = 0; r < K; ++r)
							part[r] = fma(creg[(m0 + m) * K + r], v[m], part[r]);
					}
			}
		}
		if constexpr (!TWO && !(SQ && NTR == P0 * P0 - 1)) {
			const int* to = offs + phase * orow + kOffHead + NTR;
			cf += NTR * K;
#pragma unroll 1
			for (int c = NTR; c < ntap; c += kCH, cf += kCH * K, to += kCH) {
				T v[kCH];
#pragma unroll
				for (int m = 0; m < kCH; ++m) v[m] = lds(own + unsigned(to[m]));
#pragma unroll
				for (int m = 0; m < kCH; ++m)
#pragma unroll
					for (int r = 0; r < K; ++r) part[r] = fma(cf[m * K + r], v[m], part[r]);
			}
		}
	};
	// keeps a step's sums in the step: left free, the compiler defers them to
	// the step that completes their point
	auto pin = [](auto& acc) {
		for (auto& a : acc) a.pin();
	};
	// phi(k, 0, 0) of accumulator k of the group
	auto near_of = [&](int k) { return k < P0 ? near[k] : T(0); };
	// coefficients kept in registers: loaded once, and opaque to the compiler,
	// which would otherwise keep uniform values in (and spill them from) the
	// scalar registers
	auto load_coef = [&](auto kc, const T* __restrict__ cf, auto& creg) {
		constexpr int K = decltype(kc)::value;
		if constexpr (NTR > 0) {
#pragma unroll
			for (int e = 0; e < NTR * K; ++e) {
				creg[e] = cf[e];
				asm volatile("" : "+v"(creg[e]));
			}
		}
	};

	if (G > 1 && group == 1) {
		using KC = std::integral_constant<int, K1 < 1 ? 1 : K1>;
		const T* const cf = coef + ntap * K0;
		T creg[NTR > 0 ? NTR * KC::value : 1];
		load_coef(KC{}, cf, creg);
		T c00[KC::value], part[KC::value];
		Acc<T, KAHAN> acc[KC::value];
#pragma unroll
		for (int r = 0; r < KC::value; ++r) {
			acc[r].zero();
			part[r] = T(0);
			c00[r] = near_of(K0 + r);
		}
		Row o;
		read_row(ph, o);
		__syncthreads();
		auto step = [&](const auto& row, int u) {
			constexpr bool kConst = !std::is_same_v<std::decay_t<decltype(row)>, Row>;
			const int pn = wrap_inc(ph, R);
			Row on;
			if constexpr (!kConst) read_row(pn, on);
			// the last step's point completes that step's sums; accumulator r of
			// this step is r + 1 of the last
			const T zl = lds(own + row.head(1));
#pragma unroll
			for (int r = 1; r < KC::value; ++r) {
				acc[r].add(fma(c00[r], zl, part[r]));
				acc[r - 1] = acc[r];
			}
			acc[KC::value - 1].zero();
			Hand& h = hand[(u & 1) * kThreads];
			h[1] = acc[0].s;
			if constexpr (KAHAN) h[2] = acc[0].c;
			parts_of(KC{}, cf, creg, part, ph, row);
			h[0] = part[0];
			pin(acc);
#pragma unroll
			for (int r = 1; r < KC::value; ++r) asm volatile("" : "+v"(part[r]));
			if constexpr (!kConst) {
				ph = pn;
				hold_row(on);
				o = on;
			}
			__syncthreads();
		};
		int u = 0;
		if constexpr (TWO) {
			// whole turns of the ring
			constexpr int kU = ring_planes(P0, 2);
			for (; u + kU <= total_u; u += kU)
				unrolled<kU>([&](auto d) {
					step(PhaseRow<T, kTX, P0, (kU * 16 - P0 + d) % kU>{}, u + d);
				});
			ph = (kU * 16 - P0) % kU;
			read_row(ph, o);
		}
		for (; u + KD <= total_u; u += KD) {
#pragma unroll
			for (int d = 0; d < KD; ++d) step(o, u + d);
		}
		for (; u < total_u; ++u) step(o, u);
		return;
	}

	// ---- group 0 ----
	const bool active = (X0 + lx < nx) && (Y0 + ly < ny);
	const size_t sxy = size_t(nx) * ny;
	const size_t own_off = size_t(X0 + lx) * ny + (Y0 + ly);

	// halo positions: top band (hx < 0, all hy), then left band (hx >= 0, hy < 0)
	const int H = WX * WY - kTX * kTY;
	const bool two_halos = H > kThreads;  // a second slot per lane
	int hsk[2];          // skew hx + hy of each halo slot
	unsigned hlds[2];    // its byte offset in a plane
	int hnb[2], hm[2], hdu[2];  // producing tile, its mailbox column, step offset
	bool hval[2], hin[2];
#pragma unroll
	for (int r = 0; r < 2; ++r) {
		const int h = tid + r * kThreads;
		int hx = 0, hy = 0;
		hin[r] = false;
		hval[r] = h < H;
		hsk[r] = 0;
		hlds[r] = 0;
		hnb[r] = 0;
		hm[r] = 0;
		hdu[r] = 0;
		if (hval[r]) {
			if (h < HX * WY) {
				hx = -HX + h / WY;
				hy = -HY + (h - (h / WY) * WY);
			} else {
				const int q = h - HX * WY;
				hx = q / HY;
				hy = -HY + (q - (q / HY) * HY);
			}
			hsk[r] = hx + hy;  // step s carries slice s - hx - hy
			hlds[r] = unsigned(((hx + HX) * pitch + (hy + HY)) * sizeof(T));
			const int gx = X0 + hx, gy = Y0 + hy;
			hin[r] = gx >= 0 && gy >= 0 && gx < nx && gy < ny;
			// the producing tile computed this position at its lane (px, py),
			// at u-step u + kTX and / or + kTY
			const int px = hx < 0 ? kTX + hx : hx, py = hy < 0 ? kTY + hy : hy;
			hnb[r] = b - (hx < 0 ? nY : 0) - (hy < 0 ? 1 : 0);
			hm[r] = mbox_column<TX>(px, py, HX, HY);
			hdu[r] = (hx < 0 ? kTX : 0) + (hy < 0 ? kTY : 0);
		}
	}
	// Boundary lanes (the bottom HX rows and the right HY columns, which the
	// tiles below and to the right read as halo) store every step's value into
	// this tile's mailbox, row u, column my_m: whole rows per step, so the
	// device-coherent stores are contiguous.  The surface itself goes out with
	// ordinary (write-back) stores.
	const int my_m = mbox_column<TX>(lx, ly, HX, HY);
	// BUF: every access goes through a buffer descriptor, where an offset past
	// its end loads zero and stores nothing, without a memory access: the
	// mailboxes from the corner neighbour's to this tile's through one (the
	// host chooses BUF when that span fits 31 bits), and the surface through one
	// whose base moves by a slice per step.  Every lane issues the same
	// instructions at every step, so the vector memory counter waits for
	// exactly the queue slot being consumed.  Without BUF idle lanes load the
	// zero word and store to their slot of the tile's sink.
	const int bb0 = max(b - nY - 1, 0);
	const size_t tile_mb = size_t(total_u) * NB;  // elements of one tile's mailbox
	const unsigned mb_end = unsigned((size_t(b - bb0) + 1) * tile_mb * sizeof(T));
	const __amdgpu_buffer_rsrc_t mrsrc = __builtin_amdgcn_make_buffer_rsrc(
		mbox + size_t(bb0) * tile_mb, 0, int(mb_end), kBufferDword3);
	unsigned moff = my_m >= 0 ? unsigned((size_t(b - bb0) * tile_mb + my_m) * sizeof(T)) : mb_end;
	const unsigned mstep = my_m >= 0 ? unsigned(NB * sizeof(T)) : 0u;
	unsigned hoff[2], hstep[2];
#pragma unroll
	for (int r = 0; r < 2; ++r) {
		hoff[r] = hin[r] ? unsigned(((size_t(hnb[r] - bb0) * total_u + hdu[r]) * NB + hm[r]) * sizeof(T))
		                 : mb_end;
		hstep[r] = hin[r] ? unsigned(NB * sizeof(T)) : 0u;
	}
	T* const my_sink = sink + size_t(b) * kThreads + tid;
	T* const my_mbox = my_m >= 0 ? mbox + size_t(b) * total_u * NB + my_m : my_sink;
	// The surface goes through a line of kDL slots per lane in LDS, so that a
	// wave's loads and stores cover whole row segments of one slice per tile
	// row instead of 64 cache lines of as many slices: lane (lx, ly) computes
	// slice t at step t + lx + ly; its noise is loaded for step t + lx - 1, as if
	// ly were 0, waits in slot (t + lx - 1) mod kDL, is read one step ahead of
	// its use, and the value that takes its place is stored at step t + lx + kTY.
	// kSurf lets the descriptor's base precede every lane's slice.
	constexpr int kSurf = kTX - 1;
	constexpr unsigned kNone = 0x80000000u;  // past every surface descriptor's end
	const unsigned soff = active ? unsigned((size_t(kSurf - lx) * sxy + own_off) * sizeof(T)) : kNone;
	auto surface = [&](T* base) {
		return __builtin_amdgcn_make_buffer_rsrc(base, 0, 0x7fffffff, kBufferDword3);
	};
	// bases of the next loads (step 0's: slice s0 + 1) and stores (slice s0 - kTY)
	T* zload = zeta + ptrdiff_t(s0 + 1 - kSurf) * ptrdiff_t(sxy);
	T* zstore = zeta + ptrdiff_t(s0 - kTY - kSurf) * ptrdiff_t(sxy);
	// mailbox element of halo slot r at u-step u2 (without BUF)
	auto halo_at = [&](int r, int u2) {
		return mbox + (size_t(hnb[r]) * total_u + u2 + hdu[r]) * NB + hm[r];
	};
	// A halo value that its producer has not stored yet reads as the sentinel
	// that the launch filled the mailboxes with: the lane reads it again until
	// it is there.  Rarely entered once a tile has fallen far enough behind its
	// neighbours.  Where the wait is bounded it may end without the value; a launch
	// that gave up still runs every tile to its end.
	auto await_halo = [&](int u, T& h0, T& h1) {
		long long start = 0;
		for (int n = 1; __any(is_sentinel(h0) || is_sentinel(h1)); ++n) {
			const bool w0 = is_sentinel(h0), w1 = is_sentinel(h1);
			if constexpr (BUF) {
				const T a = buffer_load_coherent<T>(mrsrc, w0 ? hoff[0] - KD * hstep[0] : mb_end);
				const T c = buffer_load_coherent<T>(mrsrc, w1 ? hoff[1] - KD * hstep[1] : mb_end);
				h0 = w0 ? a : h0;
				h1 = w1 ? c : h1;
			} else {
				if (w0) h0 = coherent_load(halo_at(0, u));
				if (w1) h1 = coherent_load(halo_at(1, u));
			}
			if (wait.gives_up(n, start)) break;
			__builtin_amdgcn_s_sleep(1);
		}
	};
	// loads of step u2 (in order of u2); steady: every slice involved is in the
	// grid, else each lane checks its own
	auto issue_loads = [&](auto steady, int u2, T& e, T& h0, T& h1) {
		const int s2 = u2 + s0;
		const int t = s2 + 1 - lx, ta = s2 - hsk[0], tb = s2 - hsk[1];
		if constexpr (BUF) {
			unsigned oe = soff, o0 = hoff[0], o1 = hoff[1];
			if constexpr (!decltype(steady)::value) {
				const bool in = u2 < total_u;
				oe = in && unsigned(t) < unsigned(nt) ? oe : kNone;
				o0 = in && unsigned(ta) < unsigned(nt) ? o0 : mb_end;
				o1 = in && unsigned(tb) < unsigned(nt) ? o1 : mb_end;
			}
			e = buffer_load<T>(surface(zload), oe);
			zload += sxy;
			h0 = buffer_load_coherent<T>(mrsrc, o0);
			h1 = T(0);
			if (two_halos) h1 = buffer_load_coherent<T>(mrsrc, o1);
			hoff[0] += hstep[0];
			hoff[1] += hstep[1];
		} else {
			const bool in = u2 < total_u;
			const bool ve = in && active && unsigned(t) < unsigned(nt);
			const bool v0 = in && hin[0] && unsigned(ta) < unsigned(nt);
			const bool v1 = in && hin[1] && unsigned(tb) < unsigned(nt);
			e = *(ve ? zeta + size_t(t) * sxy + own_off : zero);
			h0 = coherent_load(v0 ? halo_at(0, u2) : zero);
			h1 = coherent_load(v1 ? halo_at(1, u2) : zero);
		}
	};

	using KC = std::integral_constant<int, K0>;
	T creg[NTR > 0 ? NTR * K0 : 1];
	load_coef(KC{}, coef, creg);
	Acc<T, KAHAN> acc[K0];
#pragma unroll
	for (int r = 0; r < K0; ++r) acc[r].zero();
	T c00[K0 + 1];
#pragma unroll
	for (int r = 0; r < K0 + 1; ++r) c00[r] = near_of(r);
	T eps = T(0);  // the noise of the lane's next point
	T zl = T(0);   // its last point
	// line slots: this step's (the noise arriving, the value leaving), the next
	// point's, and this point's
	int dl = s0 % kDL, dn = (s0 - ly) % kDL, dw = (s0 - ly - 1) % kDL;
	dl += dl < 0 ? kDL : 0;
	dn += dn < 0 ? kDL : 0;
	dw += dw < 0 ? kDL : 0;

	Row o;
	read_row(ph, o);
	__syncthreads();
	T qe[KD], qh0[KD], qh1[KD];
#pragma unroll
	for (int d = 0; d < KD; ++d) issue_loads(std::false_type{}, d, qe[d], qh0[d], qh1[d]);

	auto step = [&](auto steady, const auto& row, int u, T& e_q, T& h0_q, T& h1_q) {
		constexpr bool kSteady = decltype(steady)::value;
		constexpr bool kConst = !std::is_same_v<std::decay_t<decltype(row)>, Row>;
		const int s = u + s0;
		const int pn = wrap_inc(ph, R);
		Row on;
		if constexpr (!kConst) read_row(pn, on);
		const unsigned here = row.head(0);
		// 1. the point: the parts of its slice, group 1's sum
		if constexpr (G > 1) {
			const Hand& h = hand[((u & 1) ^ 1) * kThreads];
			acc[K0 - 1].s = h[1];
			if constexpr (KAHAN) acc[K0 - 1].c = h[2];
			acc[K0 - 1].add(fma(c00[K0], zl, h[0]));
		}
		T part[K0];
		parts_of(KC{}, coef, creg, part, ph, row);
		acc[0].add(part[0]);
		// slice t = s - lx - ly; slices before the first come out as zero (zero
		// noise, sums and neighbours), and what lanes outside the grid or past
		// the last slice compute reaches no lane that is in it
		T z = eps + (acc[0].value() + c00[0] * eps);
		// slices t < t0 are given (a realtime stream's history): they feed the
		// sums of later slices unchanged, but must not read as missing elsewhere
		T zm = z;
		if constexpr (!kSteady) {
			z = s - lx - ly < t0 ? eps : z;
			zm = t0 > 0 ? quieted(z) : z;
		}
		lds(own + here) = z;
		// 2. halo values of step s
		if (__any(is_sentinel(h0_q) || is_sentinel(h1_q))) await_halo(u, h0_q, h1_q);
		if (hval[0]) lds(hlds[0] + here) = h0_q;
		if (two_halos && hval[1]) lds(hlds[1] + here) = h1_q;
		// 3. the line: a value leaves, noise arrives in its slot, this point
		//    takes the place of its noise, the next point's noise is read
		const T zd = line[dl * kThreads];
		line[dl * kThreads] = e_q;
		line[dw * kThreads] = z;
		eps = line[dn * kThreads];
		dw = dn;
		dn = wrap_inc(dn, kDL);
		dl = wrap_inc(dl, kDL);
		const int ts = s - lx - kTY;
		if constexpr (BUF) {
			unsigned os = soff;
			if constexpr (!kSteady) os = unsigned(ts) < unsigned(nt) ? os : kNone;
			buffer_store<T>(surface(zstore), os, zd);
			zstore += sxy;
			buffer_store_coherent(mrsrc, moff, zm);
			moff += mstep;
		} else {
			*(active && unsigned(ts) < unsigned(nt) ? zeta + size_t(ts) * sxy + own_off : my_sink) = zd;
			coherent_store(my_mbox + (my_m >= 0 ? size_t(u) * NB : 0), zm);
		}
		// 4. the point completes the sums of the slices after it
#pragma unroll
		for (int r = 1; r < K0; ++r) {
			acc[r].add(fma(c00[r], z, part[r]));
			acc[r - 1] = acc[r];
		}
		acc[K0 - 1].zero();
		zl = z;
		pin(acc);
		if constexpr (!kConst) {
			ph = pn;
			hold_row(on);
			o = on;
		}
		__syncthreads();
		// 5. loads for step u + KD into the queue slot just consumed
		issue_loads(steady, u + KD, e_q, h0_q, h1_q);
	};

	// steps from which, and up to which, every slice a step or its loads touch
	// is in the grid on every lane
	const int lead = max(HX + HY, 1);
	const int ua = max(kTX + kTY - 1, t0 + kTX + kTY - 2) - s0, ub = nt - lead - KD - s0;
	int u = 0;
	auto run_to = [&](auto steady, int end) {
		for (; u + KD <= end; u += KD) {
#pragma unroll
			for (int d = 0; d < KD; ++d)
				step(steady, o, u + d, qe[d], qh0[d], qh1[d]);
		}
	};
	if constexpr (BUF) {
		if (ua < ub) {
			if constexpr (TWO) {
				// whole turns of the ring, from a multiple of its planes
				constexpr int kU = ring_planes(P0, 2);
				run_to(std::false_type{}, (ua + kU - 1) / kU * kU);
				for (; u + kU <= ub; u += kU)
					unrolled<kU>([&](auto d) {
						step(std::true_type{}, PhaseRow<T, kTX, P0, (kU * 16 - P0 + d) % kU>{},
						     u + d, qe[d % KD], qh0[d % KD], qh1[d % KD]);
					});
				ph = (kU * 16 - P0) % kU;
				read_row(ph, o);
			} else {
				run_to(std::false_type{}, ua + KD - 1);
				run_to(std::true_type{}, ub);
			}
		}
	}
	run_to(std::false_type{}, total_u);
	// the last steps (fewer than KD), each on its own queue slot; the
	// condition is the same on every lane
#pragma unroll
	for (int d = 0; d < KD; ++d)
		if (u + d < total_u)
			step(std::false_type{}, o, u + d, qe[d], qh0[d], qh1[d]);
	// the stores due at step total_steps (slice nt - 1 of the tile's last row;
	// every other row's last slice was stored inside the loop)
	const int ts = total_steps - lx - kTY;
	if (active && unsigned(ts) < unsigned(nt)) zeta[size_t(ts) * sxy + own_off] = line[dl * kThreads];
}

struct BatchSurface {
	long long zoff;  // first element of the surface in the arena
	long long moff;  // first element of its mailboxes
	int nt, nx, ny;
	int P1, P2;
	int body;    // the tile body that marches it (batch_body)
	int nY;      // tiles along y
	int coff;    // coefficient block (elements): the nearest terms, then the bulk's
	int toff;    // offset table (ints)
	int poff;    // first progress counter (the quad tile's)
	int NB, total_steps;
	int t0;  // leading slices that are given, not generated
	int pad;
};

constexpr int kBatchP0[] = {2, 3, 5, 7, 9, 10};
constexpr int kBatchBuckets = 6;

inline int batch_bucket(int P0) {
	for (int i = 0; i < kBatchBuckets; ++i)
		if (P0 <= kBatchP0[i]) return i;
	return -1;
}

// Tile bodies of the two-group batch kernel: one per bucket for orders of any
// shape, then P0 x 2 and P0 x P0 in-slice orders of P0 = kShapedMin .. kShapedMax.
constexpr int kShapedMin = 3, kShapedMax = 9, kShaped = kShapedMax - kShapedMin + 1;
inline int batch_body(int bucket, TapShape shape, int P0) {
	if (shape == kAnyShape) return bucket;
	return kBatchBuckets + (shape == kSquare ? kShaped : 0) + P0 - kShapedMin;
}
// Groups of the batch kernel: two for 16 x 16 tiles behind buffer descriptors.
inline int batch_groups(int tile_x, bool buf) { return tile_x == 16 && buf ? 2 : 1; }

}  // namespace
}  // namespace arma_hip
