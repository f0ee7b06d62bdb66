// White noise on the GPU: dynamic-creator Mersenne Twister streams feeding
// the libstdc++ polar normal transform.
//
// Reference semantics:
//   genrand_mt / sgenrand_mt ........ src/parallel_mt.hh:217-262 (libdcmt)
//   generate_canonical, polar normal  /usr/include/c++/11/bits/random.tcc:
//                                     3348-3380, 1802-1836
//   whole-grid noise (framework=none) src/white_noise.hh:23-58,
//                                     src/generator/basic_arma_model.cc:36-48
//   per-partition noise ............. src/generator/ar_model_wn.cc:3-18 with
//                                     partitions of ar_model_parallel.cc:51-72
//
// Every stream is sequential by definition (the polar method rejects a
// data-dependent number of draws), but only in two things: the recurrence of
// its words, and the count of the pairs accepted before a place.  Which
// kernels draw a launch's streams depends on what their records allow and on
// how many there are (plan_noise, launch_streams):
//   many p = 521 streams   noise_wave_kernel, four streams per wave
//   few, long p = 521      cut into segments by jumping the generator ahead
//                          (noise_jump_kernel), counted, then filled by
//                          noise_wave_kernel, a row per segment
//   few large states       words drawn ahead by one workgroup per stream
//                          (noise_words_kernel), attempts over the whole GPU
//   other small states     noise_seg_kernel, noise_stream_kernel
//   many large states      noise_partitioned_kernel, one stream per thread
//
// All arithmetic is compiled without FP contraction, so every draw is
// computed with the roundings the reference source writes.  The FP64 polar
// step's logarithm is log_dd (log_dd.hpp): correctly rounded, where the
// device library's log is within an ulp, so a draw differs from the host's
// only where the host's log is not correctly rounded.
#include "common.hpp"
#include "log_dd.hpp"
#include "mt_jump.hpp"

#include <algorithm>
#include <type_traits>
#include <vector>

namespace arma_hip {
namespace {

constexpr int kMaxNN = 1392;  // largest dcmt state (p = 44497)

// The log table staged in LDS by the whole workgroup (before any lane leaves).
__device__ __forceinline__ void stage_log_table(double* lt) {
	for (int i = threadIdx.x; i < kLogDdRows * 3; i += blockDim.x) lt[i] = kLogDdTable[i];
	__syncthreads();
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t x, const arma_mt_params& p) {
	x ^= x >> p.shift0;
	x ^= (x << p.shiftB) & p.maskB;
	x ^= (x << p.shiftC) & p.maskC;
	x ^= x >> p.shift1;
	return x;
}

__device__ __forceinline__ uint32_t mt_twist_word(uint32_t hi, uint32_t lo, uint32_t src,
                                                  const arma_mt_params& p) {
	const uint32_t x = (hi & p.umask) | (lo & p.lmask);
	return src ^ (x >> 1) ^ ((x & 1u) ? p.aaa : 0u);
}

// Generator whose nn state words live in LDS at st[k * stride].
struct LdsMt {
	uint32_t* st;
	int stride;
	int i;
	arma_mt_params p;

	__device__ __forceinline__ uint32_t get(int k) const { return st[k * stride]; }
	__device__ __forceinline__ void set(int k, uint32_t v) { st[k * stride] = v; }

	__device__ void seed(uint32_t s) {
		for (int k = 0; k < p.nn; ++k) {
			set(k, s & p.wmask);
			s = 1812433253u * (s ^ (s >> 30)) + uint32_t(k + 1);
		}
		i = p.nn;
	}

	__device__ uint32_t next() {
		if (i >= p.nn) {
			const int n = p.nn, m = p.mm;
			int k = 0;
			for (; k < n - m; ++k) set(k, mt_twist_word(get(k), get(k + 1), get(k + m), p));
			for (; k < n - 1; ++k) set(k, mt_twist_word(get(k), get(k + 1), get(k + m - n), p));
			set(n - 1, mt_twist_word(get(n - 1), get(0), get(m - 1), p));
			i = 0;
		}
		return mt_temper(get(i++), p);
	}
};

// generate_canonical<double,53> over a 32-bit engine: two draws.
__device__ __forceinline__ double canonical_from(uint32_t u0, uint32_t u1) {
	double sum = double(u0);
	sum = sum + double(u1) * 4294967296.0;
	double ret = sum / 18446744073709551616.0;
	if (ret >= 1.0) ret = 0x1.fffffffffffffp-1;  // nextafter(1, 0)
	return ret;
}

// generate_canonical<float,24>: one draw.
__device__ __forceinline__ float canonical_from_f(uint32_t u0) {
	float sum = float(u0);
	float ret = sum / 4294967296.0f;
	if (ret >= 1.0f) ret = 0x1.fffffep-1f;
	return ret;
}

// One polar attempt from its words: the point and whether it is accepted.
template <int SEM>
struct Attempt {
	using R = std::conditional_t<SEM == ARMA_NOISE_DOUBLE, double, float>;
	R x, y, r2;
	bool accept;
	Attempt() = default;
	__device__ __forceinline__ Attempt(const uint32_t* wv, const arma_mt_params& p) {
		if constexpr (SEM == ARMA_NOISE_DOUBLE) {
			const uint4 w = *reinterpret_cast<const uint4*>(wv);
			x = 2.0 * canonical_from(mt_temper(w.x, p), mt_temper(w.y, p)) - 1.0;
			y = 2.0 * canonical_from(mt_temper(w.z, p), mt_temper(w.w, p)) - 1.0;
		} else {
			const uint2 w = *reinterpret_cast<const uint2*>(wv);
			x = 2.0f * canonical_from_f(mt_temper(w.x, p)) - 1.0f;
			y = 2.0f * canonical_from_f(mt_temper(w.y, p)) - 1.0f;
		}
		r2 = x * x + y * y;
		accept = !(r2 > R(1) || r2 == R(0));
	}
};

template <class G>
__device__ __forceinline__ double canonical_d(G& g) {
	const uint32_t u0 = g.next();
	const uint32_t u1 = g.next();
	return canonical_from(u0, u1);
}

// Polar normal generator with the libstdc++ cache of the second variate.
struct PolarD {
	bool saved_available = false;
	double saved = 0.0;

	template <class G>
	__device__ double next(G& g, double stddev, const double* ltab) {
		double ret;
		if (saved_available) {
			saved_available = false;
			ret = saved;
		} else {
			double x, y, r2;
			do {
				x = 2.0 * canonical_d(g) - 1.0;
				y = 2.0 * canonical_d(g) - 1.0;
				r2 = x * x + y * y;
			} while (r2 > 1.0 || r2 == 0.0);
			const double mult = sqrt(-2.0 * log_dd(r2, ltab) / r2);
			saved = x * mult;
			saved_available = true;
			ret = y * mult;
		}
		return ret * stddev + 0.0;
	}
};

struct PolarF {
	bool saved_available = false;
	float saved = 0.0f;

	template <class G>
	__device__ float next(G& g, float stddev) {
		float ret;
		if (saved_available) {
			saved_available = false;
			ret = saved;
		} else {
			float x, y, r2;
			do {
				x = 2.0f * canonical_from_f(g.next()) - 1.0f;
				y = 2.0f * canonical_from_f(g.next()) - 1.0f;
				r2 = x * x + y * y;
			} while (r2 > 1.0f || r2 == 0.0f);
			const float mult = sqrtf(-2.0f * logf(r2) / r2);
			saved = x * mult;
			saved_available = true;
			ret = y * mult;
		}
		return ret * stddev + 0.0f;
	}
};

// The block of the output one stream fills: its origin and extents inside a
// surface, the surface's row lengths and the standard deviation.
template <class OutT>
struct StreamBlock {
	OutT* out;   // element (0, 0, 0) of the surface
	int sy, sz;  // surface extents along x and y
	int lo0, lo1, lo2;
	int e0, e1, e2;
	double sd;
	float sdf;
};

// One surface: stream p fills partition p (row-major partition index).
template <class OutT>
struct GridBlocks {
	OutT* out;
	int3 shape, part, np;
	double sd;
	float sdf;
	__device__ __forceinline__ StreamBlock<OutT> operator()(int p) const {
		const int a = p / (np.y * np.z), b = (p / np.z) % np.y, c = p % np.z;
		StreamBlock<OutT> k;
		k.out = out;
		k.sy = shape.y;
		k.sz = shape.z;
		k.lo0 = a * part.x;
		k.lo1 = b * part.y;
		k.lo2 = c * part.z;
		k.e0 = min(k.lo0 + part.x, shape.x) - k.lo0;
		k.e1 = min(k.lo1 + part.y, shape.y) - k.lo1;
		k.e2 = min(k.lo2 + part.z, shape.z) - k.lo2;
		k.sd = sd;
		k.sdf = sdf;
		return k;
	}
};

// Many surfaces: one record per stream.
template <class OutT>
struct TableBlocks {
	OutT* arena;
	const NoiseBlockRec* recs;
	__device__ __forceinline__ StreamBlock<OutT> operator()(int p) const {
		const NoiseBlockRec r = recs[p];
		return StreamBlock<OutT>{arena + r.base, r.sy, r.sz, r.lo0, r.lo1, r.lo2,
		                         r.e0,           r.e1, r.e2, r.sd,  r.sdf};
	}
};

// One thread per partition; partitions in row-major order (stream p fills
// partition p), noise row-major inside each partition.
template <class OutT, int SEM, class Geo>
__global__ void noise_partitioned_kernel(const arma_mt_params* __restrict__ params,
                                         const uint32_t* __restrict__ seeds, Geo geo,
                                         int ntotal) {
	extern __shared__ uint32_t lds_state[];
	const int tid = threadIdx.x;
	const int p = blockIdx.x * blockDim.x + tid;
	if (p >= ntotal) return;
	LdsMt g;
	g.st = lds_state + tid;
	g.stride = blockDim.x;
	g.p = params[p];
	g.seed(seeds ? seeds[p] : 0u);
	const StreamBlock<OutT> k = geo(p);
	PolarD nd;
	PolarF nf;
	for (int t = 0; t < k.e0; ++t) {
		for (int x = 0; x < k.e1; ++x) {
			OutT* row = k.out + ((size_t)(k.lo0 + t) * k.sy + (k.lo1 + x)) * k.sz + k.lo2;
			for (int y = 0; y < k.e2; ++y) {
				if (SEM == ARMA_NOISE_DOUBLE) {
					row[y] = OutT(nd.next(g, k.sd, kLogDdTable));
				} else {
					row[y] = OutT(nf.next(g, k.sdf));
				}
			}
		}
	}
}

// Raw tempered draws, one thread per stream.
__global__ void mt_raw_kernel(const arma_mt_params* __restrict__ params,
                              const uint32_t* __restrict__ seeds, int n_streams, int draws,
                              uint32_t* __restrict__ out) {
	extern __shared__ uint32_t lds_state[];
	const int tid = threadIdx.x;
	const int s = blockIdx.x * blockDim.x + tid;
	if (s >= n_streams) return;
	LdsMt g;
	g.st = lds_state + tid;
	g.stride = blockDim.x;
	g.p = params[s];
	g.seed(seeds ? seeds[s] : 0u);
	for (int k = 0; k < draws; ++k) out[(size_t)s * draws + k] = g.next();
}

// ---- one stream per workgroup: cooperative twist, parallel polar attempts ----
//
// A workgroup owns one stream and the block of the grid it fills (the whole
// grid for framework=none, one partition otherwise).  The twist runs in
// chunks of c = nn - mm words (within a chunk every new word depends only on
// old words and on earlier chunks); each round evaluates THREADS polar
// attempts in parallel, compacts the accepted ones with a ballot prefix sum
// and writes their two variates at the positions the sequential generator
// would have given them.

// Streams whose words are drawn ahead into memory (noise_words_kernel): words
// per stream, and the blocks of kBlockAttempts attempts they hold.
struct WordPlan {
	int words = 0, blocks = 0;
};

// Sum of v[0 .. n-1] on every thread of the workgroup (tot: one int per wave).
template <int THREADS>
__device__ int block_sum(const int* v, int n, int* tot) {
	int s = 0;
	for (int i = threadIdx.x; i < n; i += THREADS) s += v[i];
#pragma unroll
	for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m);
	if ((threadIdx.x & 63) == 0) tot[threadIdx.x >> 6] = s;
	__syncthreads();
	s = 0;
#pragma unroll
	for (int w = 0; w < THREADS / 64; ++w) s += tot[w];
	__syncthreads();
	return s;
}

template <int THREADS, int MAXNN>
__device__ void twist_parallel(uint32_t* st, const arma_mt_params& p, int tid) {
	constexpr int PER = (MAXNN + THREADS - 1) / THREADS;
	const int n = p.nn, m = p.mm, c = n - m;
	for (int k0 = 0; k0 < n; k0 += c) {
		const int k1 = min(k0 + c, n);
		uint32_t v[PER];
#pragma unroll
		for (int j = 0; j < PER; ++j) {
			const int k = k0 + tid + j * THREADS;
			if (k < k1) {
				if (k < n - m) v[j] = mt_twist_word(st[k], st[k + 1], st[k + m], p);
				else if (k < n - 1) v[j] = mt_twist_word(st[k], st[k + 1], st[k + m - n], p);
				else v[j] = mt_twist_word(st[n - 1], st[0], st[m - 1], p);
			}
		}
		__syncthreads();
#pragma unroll
		for (int j = 0; j < PER; ++j) {
			const int k = k0 + tid + j * THREADS;
			if (k < k1) st[k] = v[j];
		}
		__syncthreads();
	}
}

template <class OutT, int SEM, int THREADS, int MAXNN, class Geo>
__global__ __launch_bounds__(THREADS) void noise_stream_kernel(
	const arma_mt_params* __restrict__ params, const uint32_t* __restrict__ seeds, Geo geo,
	WordPlan wp, const uint32_t* __restrict__ drawn, const int* __restrict__ counts) {
	constexpr int words_per_attempt = SEM == ARMA_NOISE_DOUBLE ? 4 : 2;
	constexpr int round_words = THREADS * words_per_attempt;
	constexpr int KEEP = (MAXNN + THREADS - 1) / THREADS;
	__shared__ uint32_t st[MAXNN];
	__shared__ uint32_t buf[round_words + MAXNN];
	__shared__ int wave_tot[THREADS / 64];
	__shared__ double ltab[kLogDdRows * 3];
	stage_log_table(ltab);
	const int tid = threadIdx.x;
	const int lane = tid & 63, wave = tid >> 6;
	const int pid = blockIdx.x;
	const arma_mt_params p = params[pid];
	// the block of the grid this stream fills, row-major
	const StreamBlock<OutT> blk = geo(pid);
	OutT* const out = blk.out;
	const int sy = blk.sy, sz = blk.sz;
	const int lo0 = blk.lo0, lo1 = blk.lo1, lo2 = blk.lo2;
	const int e2 = blk.e2;
	const double stddev = blk.sd;
	const float stddev_f = blk.sdf;
	const long long e12 = (long long)blk.e1 * e2;
	const long long n = (long long)blk.e0 * e12;
	// position -> (t, x, y) inside the block; 32-bit quotients through a
	// double reciprocal (exact after one correction) while positions fit
	const double r12 = 1.0 / double(e12), r2 = 1.0 / double(e2);
	const bool small = n < (1ll << 31);
	auto put = [&](long long q, OutT v) {
		long long t;
		int x, y;
		if (small) {
			const uint32_t uq = uint32_t(q), u12 = uint32_t(e12), u2 = uint32_t(e2);
			uint32_t qt = uint32_t(double(uq) * r12);
			if (uint64_t(qt) * u12 > uq) --qt;
			else if (uint64_t(qt + 1) * u12 <= uq) ++qt;
			const uint32_t rr = uq - qt * u12;
			uint32_t qx = uint32_t(double(rr) * r2);
			if (uint64_t(qx) * u2 > rr) --qx;
			else if (uint64_t(qx + 1) * u2 <= rr) ++qx;
			t = qt;
			x = int(qx);
			y = int(rr - qx * u2);
		} else {
			t = q / e12;
			const long long r = q - t * e12;
			x = int(r / e2);
			y = int(r - (long long)x * e2);
		}
		out[(size_t(lo0 + t) * sy + (lo1 + x)) * sz + (lo2 + y)] = v;
	};
	long long produced = 0;
	if (drawn) {
		// what is left of a block after the words drawn for it were used up
		// (usually nothing): the generator goes on from the last nn of them
		produced = 2ll * block_sum<THREADS>(counts + size_t(pid) * wp.blocks, wp.blocks, wave_tot);
		if (produced >= n) return;
		for (int k = tid; k < p.nn; k += THREADS)
			st[k] = drawn[size_t(pid) * wp.words + wp.words - p.nn + k];
	} else if (tid == 0) {
		uint32_t s = seeds ? seeds[pid] : 0u;
		for (int k = 0; k < p.nn; ++k) {
			st[k] = s & p.wmask;
			s = 1812433253u * (s ^ (s >> 30)) + uint32_t(k + 1);
		}
	}
	__syncthreads();
	int avail = 0;
	while (produced < n) {
		while (avail < round_words) {
			twist_parallel<THREADS, MAXNN>(st, p, tid);
			for (int k = tid; k < p.nn; k += THREADS) buf[avail + k] = mt_temper(st[k], p);
			avail += p.nn;
			__syncthreads();
		}
		const uint32_t* w = buf + tid * words_per_attempt;
		bool accept;
		double xd = 0, yd = 0, r2d = 0;
		float xf = 0, yf = 0, r2f = 0;
		if (SEM == ARMA_NOISE_DOUBLE) {
			xd = 2.0 * canonical_from(w[0], w[1]) - 1.0;
			yd = 2.0 * canonical_from(w[2], w[3]) - 1.0;
			r2d = xd * xd + yd * yd;
			accept = !(r2d > 1.0 || r2d == 0.0);
		} else {
			xf = 2.0f * canonical_from_f(w[0]) - 1.0f;
			yf = 2.0f * canonical_from_f(w[1]) - 1.0f;
			r2f = xf * xf + yf * yf;
			accept = !(r2f > 1.0f || r2f == 0.0f);
		}
		const unsigned long long mask = __ballot(accept);
		const int below = __popcll(mask & ((1ull << lane) - 1ull));
		if (lane == 0) wave_tot[wave] = __popcll(mask);
		__syncthreads();
		int before = 0, total = 0;
		for (int q = 0; q < THREADS / 64; ++q) {
			if (q < wave) before += wave_tot[q];
			total += wave_tot[q];
		}
		if (accept) {
			const long long pos = produced + 2ll * (before + below);
			if (pos < n) {
				if (SEM == ARMA_NOISE_DOUBLE) {
					const double mult = sqrt(-2.0 * log_dd(r2d, ltab) / r2d);
					put(pos, OutT(yd * mult * stddev + 0.0));
					if (pos + 1 < n) put(pos + 1, OutT(xd * mult * stddev + 0.0));
				} else {
					const float mult = sqrtf(-2.0f * logf(r2f) / r2f);
					put(pos, OutT(yf * mult * stddev_f + 0.0f));
					if (pos + 1 < n) put(pos + 1, OutT(xf * mult * stddev_f + 0.0f));
				}
			}
		}
		produced += 2ll * total;
		__syncthreads();
		// drop the consumed words
		const int left = avail - round_words;
		uint32_t keep[KEEP];
#pragma unroll
		for (int j = 0; j < KEEP; ++j) {
			const int k = tid + j * THREADS;
			if (k < left) keep[j] = buf[round_words + k];
		}
		__syncthreads();
#pragma unroll
		for (int j = 0; j < KEEP; ++j) {
			const int k = tid + j * THREADS;
			if (k < left) buf[k] = keep[j];
		}
		avail = left;
		__syncthreads();
	}
}

// ---- large states: words drawn ahead, attempts over the whole GPU ----
//
// One workgroup that twists, tempers, transforms and stores a large-state
// stream took 8.7 ns per normal (4.56 ms for the 524288 normals of a
// 128x64x64 surface from one MT19937).  Only the words are sequential:
// noise_words_kernel draws them untempered into memory, one workgroup per
// stream, and the attempts (a fixed number of words each) are then counted
// and transformed by workgroups of 1024 attempts, as for the segments of
// noise_wave_kernel's streams.
//
// The recurrence x_(k+n) = x_(k+m) ^ y_k, y_k = y(x_k, x_(k+1)), allows n - m
// words at a time.  Substituting it twice,
//   x_(k+n) = x_(k+3m-2n) ^ y_(k-2(n-m)) ^ y_(k-(n-m)) ^ y_k,
// allows min(n - 1, 3 (n - m)): 623 instead of 227 words of MT19937 per
// workgroup barrier.
//
// The words drawn are those that a block needs on average; noise_stream_kernel
// afterwards makes up what a stream's rejections left short.

// y is linear over GF(2), so the three cost one: the arguments are summed
// first.  The state moves through a straight LDS buffer (no index wraps) whose
// tail goes back to its start when it is full.  1.34 M words of MT19937: 0.79
// ms with three y and a ring of wrapped indices (65 VALU instructions per
// word), 0.48 ms so, 0.22 us per chunk of 623: what remains is the chain LDS
// read, twist, LDS write, barrier.  Several words per lane in fewer waves were
// slower (320 lanes of two words 0.62 ms, 256 of three 0.86).

constexpr int kWordThreads = 640;
constexpr int kWordBuffer = 16384;  // words in LDS
constexpr int kBlockAttempts = 1024, kBlockThreads = 256;

__global__ __launch_bounds__(kWordThreads) void noise_words_kernel(
	const arma_mt_params* __restrict__ params, const uint32_t* __restrict__ seeds, WordPlan wp,
	uint32_t* __restrict__ drawn) {
	__shared__ uint32_t buf[kWordBuffer];
	// room for the words a chunk reads (n + 2d, d = n - m) and one chunk
	// beyond what a move takes
	static_assert(2 * (3 * kMaxNN) + kMaxNN <= kWordBuffer, "buffer too small");
	const int tid = threadIdx.x;
	const arma_mt_params p = params[blockIdx.x];
	uint32_t* const out = drawn + size_t(blockIdx.x) * wp.words;
	const int n = p.nn, d = p.nn - p.mm;
	if (tid == 0) {
		uint32_t s = seeds ? seeds[blockIdx.x] : 0u;
		for (int k = 0; k < n; ++k) {
			buf[k] = s & p.wmask;
			s = 1812433253u * (s ^ (s >> 30)) + uint32_t(k + 1);
		}
	}
	__syncthreads();
	// k0 words are drawn (word j of the output is x_(n+j)) and x_(k0) is at
	// buf[at]; single steps until 2d words lie before x_(k0)
	int k0 = 0, at = 0;
	const int c1 = min(d, n - 1);
	while (k0 < wp.words && k0 < 2 * d) {
		for (int j = tid; j < c1; j += kWordThreads) {
			const uint32_t* x = buf + at + j;
			const uint32_t v = mt_twist_word(x[0], x[1], x[p.mm], p);
			buf[at + n + j] = v;
			if (k0 + j < wp.words) out[k0 + j] = v;
		}
		__syncthreads();
		k0 += c1;
		at += c1;
	}
	const int c = min(n - 1, 3 * d);
	while (k0 < wp.words) {
		if (at + n + max(c, kWordThreads) > kWordBuffer) {
			// x_(k0-2d) .. x_(k0+n-1) to the start of the buffer, far below
			for (int j = tid; j < 2 * d + n; j += kWordThreads) buf[j] = buf[at - 2 * d + j];
			__syncthreads();
			at = 2 * d;
		}
		auto word = [&](int j) {
			const uint32_t *x0 = buf + at + j, *x1 = x0 - d, *x2 = x1 - d;
			return mt_twist_word(x0[0] ^ x1[0] ^ x2[0], x0[1] ^ x1[1] ^ x2[1], x0[n - 3 * d], p);
		};
		if (c <= kWordThreads && k0 + kWordThreads <= wp.words) {
			const uint32_t v = word(tid);
			if (tid < c) {
				buf[at + n + tid] = v;
				out[k0 + tid] = v;
			}
		} else {
			for (int j = tid; j < c; j += kWordThreads) {
				const uint32_t v = word(j);
				buf[at + n + j] = v;
				if (k0 + j < wp.words) out[k0 + j] = v;
			}
		}
		__syncthreads();
		k0 += c;
		at += c;
	}
}

// Pairs accepted by each block of attempts.
template <int SEM>
__global__ __launch_bounds__(kBlockThreads) void noise_block_count_kernel(
	const arma_mt_params* __restrict__ params, WordPlan wp, const uint32_t* __restrict__ drawn,
	int* __restrict__ counts) {
	constexpr int WPA = SEM == ARMA_NOISE_DOUBLE ? 4 : 2;
	__shared__ int tot[kBlockThreads / 64];
	const int pid = blockIdx.y;
	const arma_mt_params p = params[pid];
	const uint32_t* w =
		drawn + size_t(pid) * wp.words + size_t(blockIdx.x) * (kBlockAttempts * WPA);
	int mine = 0;
#pragma unroll
	for (int a = 0; a < kBlockAttempts / kBlockThreads; ++a) {
		const Attempt<SEM> t(w + (a * kBlockThreads + threadIdx.x) * WPA, p);
		mine += t.accept;
	}
#pragma unroll
	for (int m = 32; m > 0; m >>= 1) mine += __shfl_xor(mine, m);
	if ((threadIdx.x & 63) == 0) tot[threadIdx.x >> 6] = mine;
	__syncthreads();
	if (threadIdx.x == 0) {
		int s = 0;
		for (int q = 0; q < kBlockThreads / 64; ++q) s += tot[q];
		counts[size_t(pid) * wp.blocks + blockIdx.x] = s;
	}
}

// The normals of each block of attempts, from the position that the counts of
// the stream's earlier blocks give it.
template <class OutT, int SEM, class Geo>
__global__ __launch_bounds__(kBlockThreads) void noise_block_fill_kernel(
	const arma_mt_params* __restrict__ params, Geo geo, WordPlan wp,
	const uint32_t* __restrict__ drawn, const int* __restrict__ counts) {
	constexpr int WPA = SEM == ARMA_NOISE_DOUBLE ? 4 : 2;
	constexpr int A = kBlockAttempts / kBlockThreads;
	__shared__ int tot[A][kBlockThreads / 64];
	__shared__ double ltab[kLogDdRows * 3];
	stage_log_table(ltab);
	const int pid = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const StreamBlock<OutT> blk = geo(pid);
	const long long e12 = (long long)blk.e1 * blk.e2, n = blk.e0 * e12;
	const long long before = 2ll * block_sum<kBlockThreads>(counts + size_t(pid) * wp.blocks,
	                                                        int(blockIdx.x), tot[0]);
	if (before >= n) return;
	const arma_mt_params p = params[pid];
	const uint32_t* w =
		drawn + size_t(pid) * wp.words + size_t(blockIdx.x) * (kBlockAttempts * WPA);
	Attempt<SEM> t[A];
	int below[A];
#pragma unroll
	for (int a = 0; a < A; ++a) {
		t[a] = Attempt<SEM>(w + (a * kBlockThreads + threadIdx.x) * WPA, p);
		const unsigned long long mask = __ballot(t[a].accept);
		below[a] = __popcll(mask & ((1ull << lane) - 1ull));
		if (lane == 0) tot[a][wave] = __popcll(mask);
	}
	__syncthreads();
	int run = 0;
#pragma unroll
	for (int a = 0; a < A; ++a)
		for (int q = 0; q < kBlockThreads / 64; ++q) {
			if (q == wave) below[a] += run;
			run += tot[a][q];
		}
	auto put = [&](long long q, OutT v) {
		const uint32_t t0 = uint32_t(q) / uint32_t(e12), r = uint32_t(q) - t0 * uint32_t(e12);
		const uint32_t x = r / uint32_t(blk.e2);
		blk.out[(size_t(blk.lo0 + t0) * blk.sy + (blk.lo1 + x)) * blk.sz +
		        (blk.lo2 + (r - x * uint32_t(blk.e2)))] = v;
	};
#pragma unroll
	for (int a = 0; a < A; ++a) {
		const long long pos = before + 2ll * below[a];
		double v0, v1;
		if (SEM == ARMA_NOISE_DOUBLE) {
			const double r2 = t[a].accept ? double(t[a].r2) : 0.5;
			const double mult = sqrt(-2.0 * log_dd(r2, ltab) / r2);
			v0 = t[a].y * mult * blk.sd + 0.0;
			v1 = t[a].x * mult * blk.sd + 0.0;
		} else {
			const float r2 = t[a].accept ? float(t[a].r2) : 0.5f;
			const float mult = sqrtf(-2.0f * logf(r2) / r2);
			v0 = float(t[a].y) * mult * blk.sdf + 0.0f;
			v1 = float(t[a].x) * mult * blk.sdf + 0.0f;
		}
		if (t[a].accept && pos < n) {
			put(pos, OutT(v0));
			if (pos + 1 < n) put(pos + 1, OutT(v1));
		}
	}
}

// ---- two streams per wave: one-round twist, 32 polar attempts per stream ----
//
// For small dcmt states (nn <= 32, 2*mm <= nn, e.g. p = 521, 607) a wave
// runs two streams on 32 lanes each.  Every twist is a single LDS round:
// lane k computes word k of the new state from old words only, evaluating
// the one or two new words it depends on (k + mm - nn, and 0 and mm - 1 for
// the last word) itself, which are themselves functions of old words when
// 2*mm <= nn.  Each round then tempers whole twists into a word buffer until
// 32 attempts' worth of words is there, evaluates the attempts in parallel
// and places the accepted pairs at the positions the sequential generator
// gives them (prefix count over the 32-lane half of the wave ballot).

constexpr int kSegLanes = 32;

__device__ __forceinline__ uint32_t twist_word_old(const uint32_t* st, int k,
                                                   const arma_mt_params& p) {
	// new word k < nn - mm: old words k, k+1, k+mm
	return mt_twist_word(st[k], st[k + 1], st[k + p.mm], p);
}

template <class OutT, int SEM, class Geo>
__global__ __launch_bounds__(64) void noise_seg_kernel(
	const arma_mt_params* __restrict__ params, const uint32_t* __restrict__ seeds, Geo geo,
	int nstreams) {
	constexpr int WPA = SEM == ARMA_NOISE_DOUBLE ? 4 : 2;  // words per attempt
	constexpr int RW = kSegLanes * WPA;                     // words per round
	__shared__ uint32_t st_all[2][32];
	__shared__ uint32_t buf_all[2][RW + 32];
	__shared__ double ltab[kLogDdRows * 3];
	stage_log_table(ltab);
	const int seg = threadIdx.x >> 5;
	const int lane = threadIdx.x & 31;
	const int pid = blockIdx.x * 2 + seg;
	const bool valid = pid < nstreams;
	uint32_t* st = st_all[seg];
	uint32_t* buf = buf_all[seg];
	arma_mt_params p = params[valid ? pid : 0];
	const int nn = p.nn;
	// the block of the grid this stream fills, row-major
	const StreamBlock<OutT> blk = geo(valid ? pid : 0);
	OutT* const out = blk.out;
	const int sy = blk.sy, sz = blk.sz;
	const int lo0 = blk.lo0, lo1 = blk.lo1, lo2 = blk.lo2;
	const int e2 = blk.e2;
	const double stddev = blk.sd;
	const float stddev_f = blk.sdf;
	const long long e12 = (long long)blk.e1 * e2;
	const long long n = valid ? (long long)blk.e0 * e12 : 0;
	const double r12 = 1.0 / double(e12), r2 = 1.0 / double(e2);
	// block extents that are powers of two (full partitions of the usual
	// shapes) split a position with shifts and masks
	const bool pow2 = (e2 & (e2 - 1)) == 0 && (e12 & (e12 - 1)) == 0;
	const int s2 = __ffs(unsigned(e2)) - 1, s12 = __ffsll((unsigned long long)e12) - 1;
	auto put = [&](long long q, OutT v) {
		// q < 2^31: 32-bit quotients
		const uint32_t uq = uint32_t(q), u12 = uint32_t(e12), u2 = uint32_t(e2);
		uint32_t qt, rr, qx;
		if (pow2) {
			qt = uq >> s12;
			rr = uq & (u12 - 1u);
			qx = rr >> s2;
		} else {
			// through a double reciprocal, corrected
			qt = uint32_t(double(uq) * r12);
			if (uint64_t(qt) * u12 > uq) --qt;
			else if (uint64_t(qt + 1) * u12 <= uq) ++qt;
			rr = uq - qt * u12;
			qx = uint32_t(double(rr) * r2);
			if (uint64_t(qx) * u2 > rr) --qx;
			else if (uint64_t(qx + 1) * u2 <= rr) ++qx;
		}
		out[(size_t(lo0 + qt) * sy + (lo1 + qx)) * sz + (lo2 + (rr - qx * u2))] = v;
	};
	if (lane == 0) {
		uint32_t sd = valid && seeds ? seeds[pid] : 0u;
		for (int k = 0; k < nn; ++k) {
			st[k] = sd & p.wmask;
			sd = 1812433253u * (sd ^ (sd >> 30)) + uint32_t(k + 1);
		}
	}
	__syncthreads();
	int avail = 0;
	long long produced = 0;
	// the workgroup is one wave: loop conditions are wave votes, and the
	// barriers below only order LDS accesses between lanes
	while (__any(produced < n)) {
		// twists until a round of words is buffered (avail is the same on
		// every lane of a segment)
		while (__any(avail < RW)) {
			const bool mine = avail < RW;
			uint32_t w = 0;
			if (mine && lane < nn) {
				const int k = lane, m = p.mm;
				if (k < nn - m) {
					w = twist_word_old(st, k, p);
				} else if (k < nn - 1) {
					w = mt_twist_word(st[k], st[k + 1], twist_word_old(st, k + m - nn, p), p);
				} else {
					w = mt_twist_word(st[nn - 1], twist_word_old(st, 0, p),
					                  twist_word_old(st, m - 1, p), p);
				}
			}
			__syncthreads();
			if (mine && lane < nn) {
				st[lane] = w;
				buf[avail + lane] = mt_temper(w, p);
			}
			if (mine) avail += nn;
			__syncthreads();
		}
		// one attempt per lane
		const uint32_t* wv = buf + lane * WPA;
		bool accept;
		double xd = 0, yd = 0, r2d = 0;
		float xf = 0, yf = 0, r2f = 0;
		if (SEM == ARMA_NOISE_DOUBLE) {
			xd = 2.0 * canonical_from(wv[0], wv[1]) - 1.0;
			yd = 2.0 * canonical_from(wv[2], wv[3]) - 1.0;
			r2d = xd * xd + yd * yd;
			accept = !(r2d > 1.0 || r2d == 0.0);
		} else {
			xf = 2.0f * canonical_from_f(wv[0]) - 1.0f;
			yf = 2.0f * canonical_from_f(wv[1]) - 1.0f;
			r2f = xf * xf + yf * yf;
			accept = !(r2f > 1.0f || r2f == 0.0f);
		}
		const unsigned long long mask = __ballot(accept);
		const uint32_t half = uint32_t(mask >> (32 * seg));
		const int below = __popc(half & ((1u << lane) - 1u));
		const int total = __popc(half);
		if (accept && produced < n) {
			const long long pos = produced + 2ll * below;
			if (pos < n) {
				if (SEM == ARMA_NOISE_DOUBLE) {
					const double mult = sqrt(-2.0 * log_dd(r2d, ltab) / r2d);
					put(pos, OutT(yd * mult * stddev + 0.0));
					if (pos + 1 < n) put(pos + 1, OutT(xd * mult * stddev + 0.0));
				} else {
					const float mult = sqrtf(-2.0f * logf(r2f) / r2f);
					put(pos, OutT(yf * mult * stddev_f + 0.0f));
					if (pos + 1 < n) put(pos + 1, OutT(xf * mult * stddev_f + 0.0f));
				}
			}
		}
		produced += 2ll * total;
		// drop the consumed words (fewer than 32 remain)
		const int left = avail - RW;
		const uint32_t keep = lane < left ? buf[RW + lane] : 0u;
		__syncthreads();
		if (lane < left) buf[lane] = keep;
		avail = left;
		__syncthreads();
	}
}

// ---- MT521 streams in registers: producer and consumer waves ----
//
// For the dynamic-creator records of p = 521 with 32-bit words (nn = 17,
// mm = 8, the records the partitioned configurations use), each 16-lane row
// of a producer wave runs one stream's twist: lane k of the row holds state
// word k (k < 16) and lane 15 also holds word 16.  A twist, in genrand_mt's
// sequential order (src/parallel_mt.hh:236), is
//   new[k]  = tw(old[k], old[k+1], old[k+8])     k = 0..8
//   new[k]  = tw(old[k], old[k+1], new[k-9])     k = 9..15
//   new[16] = tw(old[16], new[0], new[7])
// where tw(a, b, s) = s ^ y(a, b) and y depends on old words only, so a twist
// is one y per lane, the row shifts that bring old[k+1], old[k+8], new[k-9],
// new[0] and new[7] into place (DPP within each row, so the four streams of
// a wave never mix), and two XORs: 68 words for about the instructions the
// 17 words of one stream per wave took.
//
// The untempered words go into a 1024-word ring per stream in LDS.  A
// consumer wave takes the same four streams: lane k of a row evaluates
// attempts 16a + k (a < 4 in FP64 semantics, a < 8 in FP32) of its stream's
// round of 256 words, tempering the words it reads, with the attempts'
// chains interleaved, and stores the accepted pairs where
// the sequential generator puts them (prefix counts over the row's 16 bits of
// the wave ballots).  Both roles step through rounds together, one workgroup
// barrier per round: while the consumers use round r the producers twist
// round r + 1, so a twist's dependent chain and the attempts' transcendental
// chains issue side by side.  A workgroup is eight waves, four stream groups,
// with the roles ordered P0 C1 P2 C3 C0 P1 C2 P3 so that waves w and w + 4
// (the same SIMD when waves are placed round-robin) are one producer and one
// consumer.  The consumers publish per round whether their streams are
// complete (flags alternating by round parity, so a flag is rewritten only
// after every wave has read it); all waves leave after the same barrier.

constexpr int kWaveNN = 17, kWaveMM = 8;
constexpr int kRingWords = 1024;  // >= a round in use + a round + 17 written ahead
constexpr int kRoundWords = 256;  // words per round per stream
constexpr int kPcThreads = 512;

template <int CTRL>
__device__ __forceinline__ uint32_t row_move(uint32_t v) {
	return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), CTRL, 0xf, 0xf, true));
}
// as row_move, with lanes whose source falls outside the row keeping old
template <int CTRL>
__device__ __forceinline__ uint32_t row_move_or(uint32_t old, uint32_t v) {
	return uint32_t(__builtin_amdgcn_update_dpp(int(old), int(v), CTRL, 0xf, 0xf, false));
}
constexpr int kRowShl1 = 0x101, kRowShl7 = 0x107, kRowShl8 = 0x108;  // lane k <- lane k + n
constexpr int kRowShr8 = 0x118, kRowShr9 = 0x119, kRowShr15 = 0x11f;  // lane k <- lane k - n

// y(a, b) = ((a & upper) | (b & lower)) >> 1, xor aaa when the low bit is set
__device__ __forceinline__ uint32_t mt_twist_y(uint32_t a, uint32_t b, const arma_mt_params& p) {
	const uint32_t x = (a & p.umask) | (b & p.lmask);
	return (x >> 1) ^ ((x & 1u) ? p.aaa : 0u);
}

// The state of one stream on a 16-lane row and its twist.
struct Twist521 {
	uint32_t s, t;
	__device__ __forceinline__ void next(int k, const arma_mt_params& p) {
		const uint32_t nx1 = row_move_or<kRowShl1>(t, s);  // old[k + 1]; lane 15: old[16]
		const uint32_t t8 = row_move<kRowShl7>(t);          // lane 8 <- old[16]
		const uint32_t nx8 = row_move_or<kRowShl8>(t8, s);  // old[k + 8]; lane 8: old[16]
		const uint32_t y = mt_twist_y(s, nx1, p);
		const uint32_t a = nx8 ^ y;                  // new[k], k <= 8
		const uint32_t a9 = row_move<kRowShr9>(a);   // new[k - 9]
		const uint32_t a0 = row_move<kRowShr15>(a);  // lane 15 <- new[0]
		const uint32_t a7 = row_move<kRowShr8>(a);   // lane 15 <- new[7]
		t = a7 ^ mt_twist_y(t, a0, p);               // new[16] (lane 15)
		s = k <= kWaveMM ? a : (a9 ^ y);
	}
};

// Orders a wave's LDS stores before its later loads of them (LDS operations
// of one wave complete in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_order() {
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// How streams are cut: per_stream segments at most, of L = e0 2^squarings
// words (rounds rounds of kRoundWords) each, the last one open-ended.
struct SegmentPlan {
	int per_stream = 1, e0 = 0, squarings = 0, rounds = 0;
	// Segments of a stream of n normals: its expected words (a pair takes
	// 4 / pi attempts on average) over the segment length, rounded up.
	__host__ __device__ int segments(long long n, int words_per_attempt) const {
		const long long words = (n * words_per_attempt * 41722 >> 16) + 1;
		const long long len = (long long)rounds * kRoundWords;
		const long long k = (words + len - 1) / len;
		return k < 1 ? 1 : k < per_stream ? int(k) : per_stream;
	}
};

// SEG: a row's work is not a whole stream but one of the segments a long
// stream is cut into (see noise_jump_kernel).  Every segment but a stream's
// last is seg.rounds rounds long; the last runs until the block is full.
template <class OutT, int SEM, bool SEG, class Geo>
__global__ __launch_bounds__(kPcThreads) void noise_wave_kernel(
	const arma_mt_params* __restrict__ params, const uint32_t* __restrict__ seeds, Geo geo,
	int nstreams, SegmentPlan seg, const uint32_t* __restrict__ states,
	const int* __restrict__ counts) {
	constexpr int WPA = SEM == ARMA_NOISE_DOUBLE ? 4 : 2;  // words per attempt
	constexpr int A = kRoundWords / (16 * WPA);            // attempts per lane per round
	static_assert(A * 16 * WPA == kRoundWords, "a round is whole attempts");
	static_assert(3 * kRoundWords + kWaveNN <= kRingWords, "ring too small");
	// rows 16 words (16 banks) apart, so the four rows' stores of a twist and
	// reads of a round fall on different banks
	__shared__ __align__(16) uint32_t ring_all[4][4][kRingWords + 16];  // [group][row][word]
	__shared__ int gdone[2][4];
	__shared__ double ltab[kLogDdRows * 3];
	stage_log_table(ltab);
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
	const int row = lane >> 4, k = lane & 15;
	const int g = wave & 3;
	const bool producer = ((wave >> 2) ^ (wave & 1)) == 0;
	const int rid = (int(blockIdx.x) * 4 + g) * 4 + row;
	const int pid = !SEG ? rid : rid / seg.per_stream;
	const int sid = !SEG ? 0 : rid - pid * seg.per_stream;
	const bool valid = pid < nstreams;
	uint32_t* ring = ring_all[g][row];
	const arma_mt_params p = params[valid ? pid : 0];

	// producer: the state (lane k: word k; word 16 on lane 15, held by all)
	Twist521 tw{0, 0};
	uint32_t &s = tw.s, &t = tw.t;
	int wpos = 0;
	auto twist = [&]() {
		tw.next(k, p);
		ring[(wpos + k) & (kRingWords - 1)] = s;
		if (k == 15) ring[(wpos + 16) & (kRingWords - 1)] = t;
		wpos += kWaveNN;
	};

	// consumer: the block of the grid this row's stream fills
	const StreamBlock<OutT> blk = geo(valid ? pid : 0);
	OutT* const out = blk.out;
	const int sy = blk.sy, sz = blk.sz;
	const int lo0 = blk.lo0, lo1 = blk.lo1, lo2 = blk.lo2;
	const int e2 = blk.e2;
	const double stddev = blk.sd;
	const float stddev_f = blk.sdf;
	const long long e12 = (long long)blk.e1 * e2;
	long long n = valid ? (long long)blk.e0 * e12 : 0;
	// rounds of this row: unbounded (until the block is full) for a whole
	// stream and a stream's last segment
	int rounds = 0x7fffffff;
	if constexpr (SEG) {
		const int nseg = seg.segments(n, WPA);
		if (sid < nseg - 1) rounds = seg.rounds;
		if (sid > nseg - 1) n = 0;
	}
	const double r12 = 1.0 / double(e12), r2 = 1.0 / double(e2);
	const bool pow2 = (e2 & (e2 - 1)) == 0 && (e12 & (e12 - 1)) == 0;
	const int s2 = __ffs(unsigned(e2)) - 1, s12 = __ffsll((unsigned long long)e12) - 1;
	auto index = [&](long long q) {
		// q < 2^31: 32-bit quotients
		const uint32_t uq = uint32_t(q), u12 = uint32_t(e12), u2 = uint32_t(e2);
		uint32_t qt, rr, qx;
		if (pow2) {
			qt = uq >> s12;
			rr = uq & (u12 - 1u);
			qx = rr >> s2;
		} else {
			qt = uint32_t(double(uq) * r12);
			if (uint64_t(qt) * u12 > uq) --qt;
			else if (uint64_t(qt + 1) * u12 <= uq) ++qt;
			rr = uq - qt * u12;
			qx = uint32_t(double(rr) * r2);
			if (uint64_t(qx) * u2 > rr) --qx;
			else if (uint64_t(qx + 1) * u2 <= rr) ++qx;
		}
		return (size_t(lo0 + qt) * sy + (lo1 + qx)) * sz + (lo2 + (rr - qx * u2));
	};
	// the pair at positions q (even) and q + 1: with an even row length the
	// second is the next element of the same row
	const bool even_rows = (e2 & 1) == 0;
	auto put_pair = [&](long long q, OutT v0, OutT v1) {
		const size_t i0 = index(q);
		out[i0] = v0;
		if (q + 1 < n) out[even_rows ? i0 + 1 : index(q + 1)] = v1;
	};
	long long produced = 0;
	if constexpr (SEG) {
		// the pairs of the stream's earlier segments
		if (!producer && n > 0) {
			int before = 0;
			for (int i = k; i < sid; i += 16) before += counts[rid - sid + i];
#pragma unroll
			for (int m = 8; m > 0; m >>= 1) before += __shfl_xor(before, m, 16);
			produced = 2ll * before;
		}
	}
	auto consume = [&](int r) {
		// attempts a * 16 + k (a < A) of the row's stream in round r; the
		// transform is evaluated on every lane (a rejected attempt on a
		// stand-in radius) and only accepted pairs are stored
		const uint32_t* words = ring + ((r * kRoundWords) & (kRingWords - 1));
		bool acc[A];
		double xd[A], yd[A], r2d[A];
		float xf[A], yf[A], r2f[A];
#pragma unroll
		for (int a = 0; a < A; ++a) {
			const uint32_t* wv = words + (a * 16 + k) * WPA;
			if (SEM == ARMA_NOISE_DOUBLE) {
				const uint4 w = *reinterpret_cast<const uint4*>(wv);
				xd[a] = 2.0 * canonical_from(mt_temper(w.x, p), mt_temper(w.y, p)) - 1.0;
				yd[a] = 2.0 * canonical_from(mt_temper(w.z, p), mt_temper(w.w, p)) - 1.0;
				r2d[a] = xd[a] * xd[a] + yd[a] * yd[a];
				acc[a] = !(r2d[a] > 1.0 || r2d[a] == 0.0);
			} else {
				const uint2 w = *reinterpret_cast<const uint2*>(wv);
				xf[a] = 2.0f * canonical_from_f(mt_temper(w.x, p)) - 1.0f;
				yf[a] = 2.0f * canonical_from_f(mt_temper(w.y, p)) - 1.0f;
				r2f[a] = xf[a] * xf[a] + yf[a] * yf[a];
				acc[a] = !(r2f[a] > 1.0f || r2f[a] == 0.0f);
			}
		}
		int below[A];
		int total = 0;
#pragma unroll
		for (int a = 0; a < A; ++a) {
			if constexpr (SEG) acc[a] = acc[a] && r < rounds;
			const uint32_t bits = uint32_t(__ballot(acc[a]) >> (16 * row)) & 0xffffu;
			below[a] = total + __popc(bits & ((1u << k) - 1u));
			total += __popc(bits);
		}
#pragma unroll
		for (int a = 0; a < A; ++a) {
			const long long pos = produced + 2ll * below[a];
			if (SEM == ARMA_NOISE_DOUBLE) {
				const double rr2 = acc[a] ? r2d[a] : 0.5;
				const double mult = sqrt(-2.0 * log_dd(rr2, ltab) / rr2);
				if (acc[a] && pos < n)
					put_pair(pos, OutT(yd[a] * mult * stddev + 0.0), OutT(xd[a] * mult * stddev + 0.0));
			} else {
				const float rr2 = acc[a] ? r2f[a] : 0.5f;
				const float mult = sqrtf(-2.0f * logf(rr2) / rr2);
				if (acc[a] && pos < n)
					put_pair(pos, OutT(yf[a] * mult * stddev_f + 0.0f),
					         OutT(xf[a] * mult * stddev_f + 0.0f));
			}
		}
		produced += 2ll * total;
	};

	if (producer) {
		// sgenrand_mt: word w of the recurrence from the seed; lane k keeps
		// word k, every lane keeps word 16 (lane 15's copy is the one used)
		if constexpr (!SEG) {
			uint32_t x = valid && seeds ? seeds[pid] : 0u;
			for (int w = 0; w < kWaveNN; ++w) {
				const uint32_t v = x & p.wmask;
				if (w == k) s = v;
				if (w == kWaveNN - 1) t = v;
				x = 1812433253u * (x ^ (x >> 30)) + uint32_t(w + 1);
			}
		} else if (n > 0) {
			s = states[size_t(rid) * kWaveNN + k];
			t = states[size_t(rid) * kWaveNN + kWaveNN - 1];
		}
		while (wpos < kRoundWords) twist();
	}
	__syncthreads();  // round 0 is in the rings
	for (int r = 0;; ++r) {
		if (producer) {
			while (wpos < (r + 2) * kRoundWords) twist();  // round r + 1
		} else {
			consume(r);
			bool more = produced < n;
			if constexpr (SEG) more = more && r + 1 < rounds;
			const bool mine_done = !__any(more);
			if (lane == 0) gdone[r & 1][g] = mine_done;
		}
		__syncthreads();
		if (gdone[r & 1][0] && gdone[r & 1][1] && gdone[r & 1][2] && gdone[r & 1][3]) break;
	}
}

// ---- long MT521 streams cut into segments ----
//
// With few streams the launch time of noise_wave_kernel is the length of one
// stream (29 ns per normal: a twist is a dependent chain), whatever the GPU
// could do beside it: 2.12 ms for streams of 73728 normals, one or 4096 of
// them.  Cut in segments, 64 such streams take 0.14 ms, 1000 0.79 ms.  A polar
// attempt always takes the same number of words, accepted or not, so a stream's
// words can be cut anywhere between attempts once the generator's state there is
// known: segment j of a stream starts at its word j L.
//
// noise_jump_kernel finds those states, one workgroup per stream.  With the
// residue g = t^(mL) mod chi (mt_jump.hpp) the state m segments further on is
// a correlation of g with the 538 words after a segment's start, so the
// states double in number per level: from segments 0..m-1 to m..2m-1, g
// squared in between.  Each 16-lane row twists one segment's 538 words into
// LDS and correlates them (lane k: state word k, lane 15 also word 16), or, where
// a level has fewer states than the workgroup rows, its share of g's words.
// noise_count_kernel then counts what each segment accepts, and
// noise_wave_kernel writes the normals of all segments side by side, each
// from the sum of the counts before it.  The words, and so the noise, are
// those of the sequential generator.

// Streams cut into at most this many segments take one-wave workgroups, many
// per CU: their polynomial work is what costs, not the segments.
constexpr int kJumpFew = 8;
// words of a row's window: 521 + 17 rounded up to whole twists; the row
// stride keeps a wave's four rows on different banks
constexpr int kJumpWindow = 544, kJumpStride = 560;

__constant__ const JumpTable kJumpPolys = jump_table();

template <int THREADS>
__global__ __launch_bounds__(THREADS) void noise_jump_kernel(
	const arma_mt_params* __restrict__ params, const uint32_t* __restrict__ seeds,
	SegmentPlan seg, uint32_t* __restrict__ states) {
	constexpr int kRows = THREADS / 16;
	constexpr int kGroups = THREADS / kJumpWords < 8 ? THREADS / kJumpWords : 8;
	__shared__ uint32_t win[kRows][kJumpStride];
	// The large workgroup (few streams, much to jump) keeps the residues of all
	// powers that a square can have above chi's degree: three barriers a square
	// instead of 34.  With the rows that share a state it took the noise of a 32^3
	// FP32 surface in 8 streams from 146 to 104 us; many streams in one-wave
	// workgroups do not miss the barriers, but would the LDS.
	constexpr bool kTable = THREADS >= 512;
	constexpr int kSquareRows = (kJumpDegree - 1) / 2;  // t^522, t^524, ..., t^1040
	__shared__ uint32_t high[kTable ? kSquareRows : 1][kJumpWords];
	__shared__ uint32_t shift[32][kJumpWords];  // t^(521 + b) mod chi
	__shared__ uint32_t sq[2 * kJumpWords + 2];
	__shared__ uint32_t g[kJumpWords], next_g[kJumpWords];
	__shared__ uint32_t part[kRows][kWaveNN + 1];
	const int tid = threadIdx.x;
	const int row = tid >> 4, k = tid & 15;
	const arma_mt_params p = params[blockIdx.x];
	uint32_t* const st = states + size_t(blockIdx.x) * seg.per_stream * kWaveNN;
	if (tid == 0) {
		// sgenrand_mt: the state of segment 0
		uint32_t x = seeds ? seeds[blockIdx.x] : 0u;
		for (int w = 0; w < kWaveNN; ++w) {
			st[w] = x & p.wmask;
			x = 1812433253u * (x ^ (x >> 30)) + uint32_t(w + 1);
		}
	}
	if (seg.per_stream == 1) return;
	// t^521 mod chi
	if (tid < kJumpWords) {
		uint32_t v = kJumpPolys.base.w[tid];
		for (int i = 0; i < 32; ++i) v ^= ((p.aaa >> i) & 1u) ? kJumpPolys.a[i].w[tid] : 0u;
		shift[0][tid] = v;
		// t^e0, e0 at most 512
		g[tid] = seg.e0 >> 5 == tid ? 1u << (seg.e0 & 31) : 0u;
		next_g[tid] = 0;
	}
	__syncthreads();
	for (int b = 1; b < 32; ++b) {
		if (tid < kJumpWords) {
			const uint32_t top = (shift[b - 1][kJumpWords - 1] >> (kJumpTop - 1)) & 1u;
			uint32_t v = (shift[b - 1][tid] << 1) | (tid ? shift[b - 1][tid - 1] >> 31 : 0u);
			if (tid == kJumpWords - 1) v &= (1u << kJumpTop) - 1u;
			shift[b][tid] = v ^ (top ? shift[0][tid] : 0u);
		}
		__syncthreads();
	}
	if constexpr (kTable) {
		// t^(521 + b + 32) from t^(521 + b): a word up, the bits past the degree
		// reduced by shift.  Row r = 16 c + q is t^(521 + 2 q + 1 + 32 c).
		static_assert(16 * kJumpWords <= THREADS, "a lane per word of 16 rows");
		const int q = tid / kJumpWords, w = tid % kJumpWords;
		if (q < 16) high[q][w] = shift[2 * q + 1][w];
		__syncthreads();
		for (int r0 = 16; r0 < kSquareRows; r0 += 16) {
			if (q < 16 && r0 + q < kSquareRows) {
				const uint32_t* from = high[r0 - 16 + q];
				const uint32_t v =
					(from[kJumpWords - 2] >> kJumpTop) | (from[kJumpWords - 1] << (32 - kJumpTop));
				uint32_t x = w ? from[w - 1] : 0u;
				if (w == kJumpWords - 1) x &= (1u << kJumpTop) - 1u;
#pragma unroll
				for (int b = 0; b < 32; ++b) x ^= shift[b][w] & (0u - ((v >> b) & 1u));
				high[r0 + q][w] = x;
			}
			__syncthreads();
		}
	}
	// g <- g^2 mod chi
	auto square = [&]() {
		if (tid < kJumpWords) {
			// bit i to bit 2 i
			auto spread = [](uint32_t v) {
				v = (v | (v << 8)) & 0x00ff00ffu;
				v = (v | (v << 4)) & 0x0f0f0f0fu;
				v = (v | (v << 2)) & 0x33333333u;
				return (v | (v << 1)) & 0x55555555u;
			};
			sq[2 * tid] = spread(g[tid] & 0xffffu);
			sq[2 * tid + 1] = spread(g[tid] >> 16);
		}
		__syncthreads();
		if constexpr (kTable) {
			constexpr int kShare = THREADS / kJumpWords;
			const int q = tid / kJumpWords, w = tid % kJumpWords;
			if (q < kShare) {
				uint32_t x = 0;
				for (int r = q; r < kSquareRows; r += kShare) {
					const int bit = kJumpDegree + 1 + 2 * r;
					x ^= high[r][w] & (0u - ((sq[bit >> 5] >> (bit & 31)) & 1u));
				}
				uint32_t low = 0;
				if (q == 0) {
					low = sq[w];
					if (w == kJumpWords - 1) low &= (1u << kJumpTop) - 1u;
				}
				atomicXor(&next_g[w], x ^ low);
			}
			__syncthreads();
			if (tid < kJumpWords) {
				g[tid] = next_g[tid];
				next_g[tid] = 0;
			}
			__syncthreads();
			return;
		}
		// 32 bits at a time from the top (the square has degree at most 1040):
		// bits 521 + 32c .. 521 + 32c + 31 select rows of shift
		for (int c = 16; c >= 0; --c) {
			const uint32_t v =
				(sq[16 + c] >> kJumpTop) | (sq[17 + c] << (32 - kJumpTop));
			__syncthreads();
			if (tid < kGroups * kJumpWords) {
				const int w = tid % kJumpWords, b0 = tid / kJumpWords;
				uint32_t x = 0;
#pragma unroll
				for (int q = 0; q < (32 + kGroups - 1) / kGroups; ++q) {
					const int b = min(b0 + kGroups * q, 31);
					x ^= b0 + kGroups * q < 32 && ((v >> b) & 1u) ? shift[b][w] : 0u;
				}
				if (x) atomicXor(&sq[c + w], x);
			}
			__syncthreads();
		}
		if (tid < kJumpWords)
			g[tid] = tid == kJumpWords - 1 ? sq[tid] & ((1u << kJumpTop) - 1u) : sq[tid];
		__syncthreads();
	};
	for (int q = 0; q < seg.squarings; ++q) square();
	uint32_t* const mine = win[row];
	for (int m = 1; m < seg.per_stream; m *= 2) {
		if (m > 1) square();
		const int end = min(2 * m, seg.per_stream);
		// a level of few states takes several rows for each, which share the words
		// of g (all of them twist the window)
		int split = 1;
		while (split < 16 && 2 * split * (end - m) <= kRows) split *= 2;
		for (int t0 = m; t0 < end; t0 += kRows / split) {
			const int to = t0 + row / split, first = row % split;
			const bool act = to < end;
			if (__any(act)) {
				const uint32_t* const from = st + size_t(act ? to - m : 0) * kWaveNN;
				Twist521 tw{from[k], from[kWaveNN - 1]};
				mine[k] = tw.s;
				if (k == 15) mine[16] = tw.t;
				for (int w = kWaveNN; w < kJumpWindow; w += kWaveNN) {
					tw.next(k, p);
					mine[w + k] = tw.s;
					if (k == 15) mine[w + 16] = tw.t;
				}
				wave_lds_order();
				// state word k: sum of g_i x_(i+k); word 16 one word behind on lane 15
				uint32_t acc = 0, acc16 = 0;
				for (int w = first; w < kJumpWords; w += split) {
					const uint32_t gw = g[w];
					const uint32_t* x = mine + 32 * w + k;
					uint32_t prev = 0;
					if (w < kJumpWords - 1) {
#pragma unroll
						for (int b = 0; b < 32; ++b) {
							const uint32_t mask = 0u - ((gw >> b) & 1u);
							acc ^= x[b] & mask;
							acc16 ^= x[b] & prev;
							prev = mask;
						}
						acc16 ^= x[32] & prev;
					} else {
#pragma unroll
						for (int b = 0; b < kJumpTop; ++b) {
							const uint32_t mask = 0u - ((gw >> b) & 1u);
							acc ^= x[b] & mask;
							acc16 ^= x[b] & prev;
							prev = mask;
						}
						acc16 ^= x[kJumpTop] & prev;
					}
				}
				if (split == 1) {
					if (act) {
						st[size_t(to) * kWaveNN + k] = acc;
						if (k == 15) st[size_t(to) * kWaveNN + 16] = acc16;
					}
				} else {
					part[row][k] = acc;
					if (k == 15) part[row][16] = acc16;
				}
				wave_lds_order();
			}
			if (split > 1) {  // one turn of the loop
				__syncthreads();
				if (act && first == 0) {
					for (int w = k; w < kWaveNN; w += 16) {
						uint32_t x = 0;
						for (int r = 0; r < split; ++r) x ^= part[row + r][w];
						st[size_t(to) * kWaveNN + w] = x;
					}
				}
			}
		}
		__syncthreads();  // the level's states are the next level's starts
	}
}

// Pairs that each segment but a stream's last accepts.  Four segments per
// wave, one per 16-lane row; a wave twists a round of words of its rows into
// LDS and tests their attempts, without the producer and consumer roles of
// noise_wave_kernel: the twists are most of the work and the waves of a
// SIMD fill each other's stalls.  In FP64 semantics an attempt is decided by
// the high words of its two uniforms (each within 2^-31 of the uniform's
// value, so r^2 within 2^-28) unless r^2 is that close to 1 or may be zero.
constexpr int kCountRows = 16;  // rows per workgroup

template <int SEM, class Geo>
__global__ __launch_bounds__(16 * kCountRows) void noise_count_kernel(
	const arma_mt_params* __restrict__ params, Geo geo, int nstreams, SegmentPlan seg,
	const uint32_t* __restrict__ states, int* __restrict__ counts) {
	constexpr int WPA = SEM == ARMA_NOISE_DOUBLE ? 4 : 2;
	constexpr int A = kRoundWords / (16 * WPA);
	constexpr int kRing = 512;  // a round and the 16 words written ahead
	__shared__ __align__(16) uint32_t ring_all[kCountRows][kRing + 16];
	const int lrow = threadIdx.x >> 4, k = threadIdx.x & 15;
	const int rid = int(blockIdx.x) * kCountRows + lrow;
	const int pid = rid / seg.per_stream, sid = rid - pid * seg.per_stream;
	bool live = false;
	if (pid < nstreams) {
		const auto blk = geo(pid);
		live = sid < seg.segments((long long)blk.e0 * blk.e1 * blk.e2, WPA) - 1;
	}
	if (!__any(live)) return;
	const arma_mt_params p = params[live ? pid : 0];
	uint32_t* const ring = ring_all[lrow];
	Twist521 tw{0, 0};
	if (live) {
		tw.s = states[size_t(rid) * kWaveNN + k];
		tw.t = states[size_t(rid) * kWaveNN + kWaveNN - 1];
	}
	const int row = lrow & 3;  // of the wave
	int wpos = 0, total = 0;
	for (int r = 0; r < seg.rounds; ++r) {
		while (wpos < (r + 1) * kRoundWords) {
			tw.next(k, p);
			ring[(wpos + k) & (kRing - 1)] = tw.s;
			if (k == 15) ring[(wpos + 16) & (kRing - 1)] = tw.t;
			wpos += kWaveNN;
		}
		wave_lds_order();
		const uint32_t* words = ring + ((r * kRoundWords) & (kRing - 1));
		bool acc[A];
#pragma unroll
		for (int a = 0; a < A; ++a) {
			const uint32_t* wv = words + (a * 16 + k) * WPA;
			if (SEM == ARMA_NOISE_DOUBLE) {
				const uint4 w = *reinterpret_cast<const uint4*>(wv);
				const uint32_t u = mt_temper(w.y, p), v = mt_temper(w.w, p);
				const double x = double(int(u ^ 0x80000000u)), y = double(int(v ^ 0x80000000u));
				const double q = fma(x, x, y * y);  // r^2 * 2^62
				acc[a] = q <= 0x1p62;
				if (__builtin_expect(fabs(q - 0x1p62) < 0x1p35 || q < 0x1p12, 0)) {
					const double xd = 2.0 * canonical_from(mt_temper(w.x, p), u) - 1.0;
					const double yd = 2.0 * canonical_from(mt_temper(w.z, p), v) - 1.0;
					const double r2 = xd * xd + yd * yd;
					acc[a] = !(r2 > 1.0 || r2 == 0.0);
				}
			} else {
				const uint2 w = *reinterpret_cast<const uint2*>(wv);
				const float x = 2.0f * canonical_from_f(mt_temper(w.x, p)) - 1.0f;
				const float y = 2.0f * canonical_from_f(mt_temper(w.y, p)) - 1.0f;
				const float r2 = x * x + y * y;
				acc[a] = !(r2 > 1.0f || r2 == 0.0f);
			}
		}
#pragma unroll
		for (int a = 0; a < A; ++a)
			total += __popc(uint32_t(__ballot(acc[a]) >> (16 * row)) & 0xffffu);
		wave_lds_order();
	}
	if (live && k == 0) counts[rid] = total;
}

bool wave_kernel_fits(const arma_mt_params* mts, int n) {
	for (int i = 0; i < n; ++i)
		if (mts[i].nn != kWaveNN || mts[i].mm != kWaveMM) return false;
	return true;
}

// Streams whose states noise_jump_kernel can advance: the records of p = 521
// with the dynamic creator's masks.
bool jump_fits(const arma_mt_params* mts, int n) {
	for (int i = 0; i < n; ++i) {
		const arma_mt_params& q = mts[i];
		if (q.nn != kJumpN || q.mm != kJumpM || q.umask != 0xffffffffu << kJumpR ||
		    q.lmask != ~(0xffffffffu << kJumpR))
			return false;
	}
	return true;
}

// Rows a segmented launch aims at (two workgroups of 16 rows per CU), the
// most segments of one stream, and the shortest segment in words.
constexpr int kSegRowsPerCu = 32, kMaxSegments = 256, kMinSegmentWords = 1024;
// Measured on MI355X, in ns: per word of a row filling its block and counting
// (one workgroup of rows per CU), the jump's fixed part, each of its levels
// or squarings, and its share per stream where many jump side by side.
constexpr double kWordNs = 11.4, kCountWordNs = 4.5, kJumpNs = 30e3, kJumpLevelNs = 6e3,
                 kJumpStreamNs = 40.0;

// How to cut nstreams streams whose longest block has n normals.
SegmentPlan plan_segments(const arma_hip_ctx* ctx, int sem, int nstreams, long long n,
                          const arma_mt_params* mts, bool small_blocks) {
	SegmentPlan seg;
	const int wpa = sem == ARMA_NOISE_DOUBLE ? 4 : 2;
	const int rows = kSegRowsPerCu * std::max(ctx->num_cus, 1);
	const int most = std::min(kMaxSegments, rows / std::max(nstreams, 1));
	if (!small_blocks || most < 2) return seg;
	// segment lengths e0 2^q, whole rounds of words: the shortest that keeps
	// the launch within rows
	for (int q = 2; q < 40; ++q)
		for (int e0 : {256, 320, 384, 448}) {
			const long long len = (long long)e0 << q;
			if (len < kMinSegmentWords || len > (1ll << 30)) continue;
			seg.e0 = e0;
			seg.squarings = q;
			seg.rounds = int(len / kRoundWords);
			seg.per_stream = kMaxSegments + 1;
			const int k = seg.segments(n, wpa);
			if (k > most) continue;
			seg.per_stream = k;
			int levels = 0;
			while ((1 << levels) < k) ++levels;
			const double words = double(n) * wpa * 0.6366;
			const double whole = kWordNs * words;
			// two workgroups on a CU share its issue slots
			const double share =
				std::max(1.0, 0.85 * 2.0 * double(nstreams) * k / double(rows));
			const double cut = kJumpNs + kJumpLevelNs * (levels + q) + kJumpStreamNs * nstreams +
			                   (kWordNs + kCountWordNs) * double(len) * share;
			// one stream of 32768 normals: 146 us cut in 82 against 905 whole;
			// 1000 of 73728: 0.79 against 2.12 ms; 2700 of 8192, which this
			// line leaves whole, 279 against 241 us
			// (the records last: there may be thousands)
			if (k < 2 || cut > 0.93 * whole || !jump_fits(mts, nstreams)) return SegmentPlan();
			return seg;
		}
	return SegmentPlan();
}

// Streams of large states take their words from noise_words_kernel when they
// have at least kAheadNormals normals (below, the extra launches cost what the
// stream does) and all words fit kAheadBytes, or in a batch, whose requests a
// server admits by bytes that do not count them, kBatchAheadBytes.  Beyond a stream per
// CU its workgroups, which fill most of a CU's LDS and seed their state word by
// word, run one after another, and the one-workgroup streams, four to a CU, are the
// faster ones up to so many normals per state word (us, whole against ahead: MT19937,
// 512 streams of 8192 132 and 118, 768 of 8192 140 and 153, 768 of 32768 403 and 333;
// 1392 words of state, 256 of 8192 107 and 88, 512 of 8192 122 and 144, 512 of 32768
// 285 and 264, 768 of 32768 321 and 380).
constexpr long long kAheadNormals = 8192, kAheadBytes = 256ll << 20,
                    kBatchAheadBytes = 16ll << 20;
constexpr int kAheadPerWord[] = {0, 16, 64, 64};  // by streams per CU, rounded up, less one

WordPlan plan_ahead(const arma_hip_ctx* ctx, int sem, int nstreams, long long n,
                    const arma_mt_params* mts, bool small_blocks, long long most) {
	WordPlan wp;
	const int cus = std::max(ctx->num_cus, 1);
	if (!small_blocks || n < kAheadNormals || nstreams > 4 * cus) return wp;
	int nn_max = 0;
	for (int i = 0; i < nstreams; ++i) nn_max = std::max(nn_max, int(mts[i].nn));
	if (nn_max <= 64 || n < (long long)kAheadPerWord[(nstreams - 1) / cus] * nn_max) return wp;
	const int wpa = sem == ARMA_NOISE_DOUBLE ? 4 : 2;
	// 4 / pi attempts per pair on average, in whole blocks
	const long long blocks = (n * 41722 / 65536 + kBlockAttempts) / kBlockAttempts;
	const long long words = blocks * kBlockAttempts * wpa;
	if (words * 4 * nstreams > most || blocks > 65535) return wp;
	wp.words = int(words);
	wp.blocks = int(blocks);
	return wp;
}

// How a launch draws its streams: whole (neither set), by segments, or with
// the words drawn ahead.
struct NoisePlan {
	SegmentPlan seg;
	WordPlan ahead;
	// device bytes beside the parameters and seeds
	size_t bytes(int nstreams) const {
		if (ahead.words > 0)
			return size_t(nstreams) * (size_t(ahead.words) + ahead.blocks) * sizeof(uint32_t);
		if (seg.per_stream > 1)
			return size_t(nstreams) * seg.per_stream * (kWaveNN + 1) * sizeof(uint32_t);
		return 0;
	}
};

NoisePlan plan_noise(const arma_hip_ctx* ctx, int sem, int nstreams, long long n,
                     const arma_mt_params* mts, bool small_blocks, long long ahead_bytes) {
	NoisePlan plan;
	plan.ahead = plan_ahead(ctx, sem, nstreams, n, mts, small_blocks, ahead_bytes);
	if (plan.ahead.words == 0)
		plan.seg = plan_segments(ctx, sem, nstreams, n, mts, small_blocks);
	return plan;
}

// The two-per-wave kernel applies to states of at most 32 words whose twist
// needs only old words for its redundant evaluations.
bool seg_kernel_fits(const arma_mt_params* mts, int n) {
	for (int i = 0; i < n; ++i)
		if (mts[i].nn > kSegLanes || 2 * mts[i].mm > mts[i].nn) return false;
	return true;
}

int threads_for_state(int nn) {
	// per-thread LDS state of nn words; at most 64 KiB per workgroup
	int t = 256;
	while (t > 1 && size_t(t) * nn * 4 > 65536) t >>= 1;
	return t;
}

void validate_params(const arma_mt_params* mts, int n) {
	for (int i = 0; i < n; ++i) {
		const arma_mt_params& q = mts[i];
		ARMA_HIP_REQUIRE(q.nn > 1 && q.nn <= kMaxNN && q.mm > 0 && q.mm < q.nn &&
		                     q.shift0 >= 0 && q.shift0 < 32 && q.shift1 >= 0 && q.shift1 < 32 &&
		                     q.shiftB >= 0 && q.shiftB < 32 && q.shiftC >= 0 && q.shiftC < 32,
		                 ARMA_HIP_EINVAL, "bad Mersenne Twister parameter record");
	}
}

// Launches the noise of nstreams streams whose output blocks geo describes:
// as the plan says, or whole streams with the kernel their parameter sets
// allow: four streams per wave for p = 521, a whole workgroup for another
// single stream, two streams per wave for small dcmt states, one wave per
// stream up to 64 state words, one workgroup per stream for a few large
// states, else one thread per stream.
template <class OutT, int SEM, class Geo>
void launch_streams(arma_hip_ctx* ctx, const arma_mt_params* hparams,
                    const arma_mt_params* dparams, const uint32_t* dseeds, Geo geo, int nstreams,
                    bool small_blocks, const NoisePlan& plan, void* buf) {
	const SegmentPlan& seg = plan.seg;
	const WordPlan& wp = plan.ahead;
	if (wp.words > 0) {
		uint32_t* drawn = (uint32_t*)buf;
		int* counts = (int*)(drawn + size_t(nstreams) * wp.words);
		noise_words_kernel<<<nstreams, kWordThreads, 0, ctx->stream>>>(dparams, dseeds, wp, drawn);
		ARMA_HIP_CHECK(hipGetLastError());
		noise_block_count_kernel<SEM><<<dim3(wp.blocks, nstreams), kBlockThreads, 0, ctx->stream>>>(
			dparams, wp, drawn, counts);
		ARMA_HIP_CHECK(hipGetLastError());
		noise_block_fill_kernel<OutT, SEM, Geo>
			<<<dim3(wp.blocks, nstreams), kBlockThreads, 0, ctx->stream>>>(dparams, geo, wp, drawn,
			                                                           counts);
		ARMA_HIP_CHECK(hipGetLastError());
		noise_stream_kernel<OutT, SEM, 256, kMaxNN, Geo>
			<<<nstreams, 256, 0, ctx->stream>>>(dparams, dseeds, geo, wp, drawn, counts);
		ARMA_HIP_CHECK(hipGetLastError());
		return;
	}
	if (seg.per_stream > 1) {
		const int rows = nstreams * seg.per_stream;
		uint32_t* states = (uint32_t*)buf;
		int* counts = (int*)(states + size_t(rows) * kWaveNN);
		if (seg.per_stream <= kJumpFew)
			noise_jump_kernel<64><<<nstreams, 64, 0, ctx->stream>>>(dparams, dseeds, seg, states);
		else
			noise_jump_kernel<512><<<nstreams, 512, 0, ctx->stream>>>(dparams, dseeds, seg, states);
		ARMA_HIP_CHECK(hipGetLastError());
		noise_count_kernel<SEM, Geo><<<div_ceil(rows, kCountRows), 16 * kCountRows, 0, ctx->stream>>>(
			dparams, geo, nstreams, seg, states, counts);
		ARMA_HIP_CHECK(hipGetLastError());
		noise_wave_kernel<OutT, SEM, true, Geo>
			<<<div_ceil(rows, 16), kPcThreads, 0, ctx->stream>>>(dparams, dseeds, geo, nstreams,
			                                                   seg, states, counts);
		ARMA_HIP_CHECK(hipGetLastError());
		return;
	}
	int nn_max = 0;
	for (int i = 0; i < nstreams; ++i) nn_max = std::max(nn_max, int(hparams[i].nn));
	if (small_blocks && wave_kernel_fits(hparams, nstreams)) {
		noise_wave_kernel<OutT, SEM, false, Geo>
			<<<div_ceil(nstreams, 16), kPcThreads, 0, ctx->stream>>>(dparams, dseeds, geo,
			                                                       nstreams, seg, nullptr, nullptr);
	} else if (nstreams == 1) {
		// the whole grid from one stream (framework=none)
		noise_stream_kernel<OutT, SEM, 256, kMaxNN, Geo>
			<<<1, 256, 0, ctx->stream>>>(dparams, dseeds, geo, wp, nullptr, nullptr);
	} else if (small_blocks && seg_kernel_fits(hparams, nstreams)) {
		noise_seg_kernel<OutT, SEM, Geo>
			<<<div_ceil(nstreams, 2), 64, 0, ctx->stream>>>(dparams, dseeds, geo, nstreams);
	} else if (nn_max <= 64) {
		noise_stream_kernel<OutT, SEM, 64, 64, Geo>
			<<<nstreams, 64, 0, ctx->stream>>>(dparams, dseeds, geo, wp, nullptr, nullptr);
	} else if (nstreams <= 4 * std::max(ctx->num_cus, 1)) {
		noise_stream_kernel<OutT, SEM, 256, kMaxNN, Geo>
			<<<nstreams, 256, 0, ctx->stream>>>(dparams, dseeds, geo, wp, nullptr, nullptr);
	} else {
		const int tpb = std::min(threads_for_state(nn_max), 64);
		noise_partitioned_kernel<OutT, SEM, Geo>
			<<<div_ceil(nstreams, tpb), tpb, size_t(tpb) * nn_max * 4, ctx->stream>>>(
				dparams, dseeds, geo, nstreams);
	}
	ARMA_HIP_CHECK(hipGetLastError());
}

template <class Geo2>
void launch_by_type(arma_hip_ctx* ctx, bool fp32, int sem, const arma_mt_params* hparams,
                    const arma_mt_params* dparams, const uint32_t* dseeds, void* out,
                    const Geo2& g, int nstreams, bool small_blocks, const NoisePlan& plan,
                    void* buf) {
	if (fp32) {
		auto geo = g.template make<float>((float*)out);
		if (sem == ARMA_NOISE_DOUBLE)
			launch_streams<float, ARMA_NOISE_DOUBLE>(ctx, hparams, dparams, dseeds, geo, nstreams,
			                                         small_blocks, plan, buf);
		else
			launch_streams<float, ARMA_NOISE_FLOAT>(ctx, hparams, dparams, dseeds, geo, nstreams,
			                                        small_blocks, plan, buf);
	} else {
		auto geo = g.template make<double>((double*)out);
		if (sem == ARMA_NOISE_DOUBLE)
			launch_streams<double, ARMA_NOISE_DOUBLE>(ctx, hparams, dparams, dseeds, geo,
			                                          nstreams, small_blocks, plan, buf);
		else
			launch_streams<double, ARMA_NOISE_FLOAT>(ctx, hparams, dparams, dseeds, geo,
			                                         nstreams, small_blocks, plan, buf);
	}
}

struct GridSpec {
	int3 shape, part, np;
	double sd;
	float sdf;
	template <class OutT>
	GridBlocks<OutT> make(OutT* out) const {
		return GridBlocks<OutT>{out, shape, part, np, sd, sdf};
	}
};

struct TableSpec {
	const NoiseBlockRec* recs;
	template <class OutT>
	TableBlocks<OutT> make(OutT* arena) const {
		return TableBlocks<OutT>{arena, recs};
	}
};

}  // namespace

void launch_white_noise(arma_hip_ctx* ctx, const arma_ar_desc* d, void* eps) {
	ARMA_HIP_REQUIRE(d->varwn >= 0.0, ARMA_HIP_EINVAL, "variance is less than zero");
	ARMA_HIP_REQUIRE(d->shape[0] > 0 && d->shape[1] > 0 && d->shape[2] > 0, ARMA_HIP_EINVAL,
	                 "bad output grid shape");
	const bool fp32 = d->precision == ARMA_FP32;
	const int sem = d->noise_semantics;
	ARMA_HIP_REQUIRE(sem == ARMA_NOISE_DOUBLE || sem == ARMA_NOISE_FLOAT, ARMA_HIP_EINVAL,
	                 "bad noise semantics");
	GridSpec g;
	g.shape = int3{d->shape[0], d->shape[1], d->shape[2]};
	g.sd = std::sqrt(d->varwn);
	g.sdf = std::sqrt(float(d->varwn));
	if (d->noise_mode == ARMA_NOISE_SEQUENTIAL) {
		g.part = g.shape;
		g.np = int3{1, 1, 1};
	} else {
		ARMA_HIP_REQUIRE(d->noise_mode == ARMA_NOISE_PARTITIONED, ARMA_HIP_EINVAL,
		                 "bad noise mode");
		ARMA_HIP_REQUIRE(d->partition[0] > 0 && d->partition[1] > 0 && d->partition[2] > 0,
		                 ARMA_HIP_EINVAL, "bad partition shape");
		g.part = int3{d->partition[0], d->partition[1], d->partition[2]};
		g.np = int3{div_ceil(g.shape.x, g.part.x), div_ceil(g.shape.y, g.part.y),
		            div_ceil(g.shape.z, g.part.z)};
	}
	const int ntotal = g.np.x * g.np.y * g.np.z;
	ARMA_HIP_REQUIRE(d->n_mts >= ntotal && d->mts, ARMA_HIP_EPRNG, "bad number of MT configs");
	validate_params(d->mts, ntotal);
	auto* dparams = (arma_mt_params*)work_buffer(ctx, ctx->params, sizeof(arma_mt_params) * ntotal);
	upload(ctx, dparams, d->mts, sizeof(arma_mt_params) * ntotal);
	uint32_t* dseeds = nullptr;
	if (d->seeds) {
		dseeds = (uint32_t*)work_buffer(ctx, ctx->seeds, sizeof(uint32_t) * ntotal);
		upload(ctx, dseeds, d->seeds, sizeof(uint32_t) * ntotal);
	}
	// every stream's block must fit 32-bit positions for the fast kernels
	const bool small_blocks = (long long)g.part.x * g.part.y * g.part.z < (1ll << 31);
	KernelTimer timer(ctx, d->noise_mode == ARMA_NOISE_SEQUENTIAL ? "noise_sequential"
	                                                               : "noise_partitioned");
	// (not within a borrowed region, whose size callers reckon without it)
	NoisePlan plan;
	if (!ctx->borrow_base)
		plan = plan_noise(ctx, sem, ntotal,
		                  (long long)std::min(g.part.x, g.shape.x) *
		                      std::min(g.part.y, g.shape.y) * std::min(g.part.z, g.shape.z),
		                  d->mts, small_blocks, kAheadBytes);
	void* buf = plan.bytes(ntotal) ? ctx->noise_tmp.try_get(plan.bytes(ntotal)) : nullptr;
	if (!buf) plan = NoisePlan();  // whole streams need no buffer
	launch_by_type(ctx, fp32, sem, d->mts, dparams, dseeds, eps, g, ntotal, small_blocks, plan,
	               buf);
}

size_t white_noise_work_bytes(const arma_ar_desc* d) {
	size_t n = 1;
	if (d->noise_mode == ARMA_NOISE_PARTITIONED && d->partition[0] > 0 && d->partition[1] > 0 &&
	    d->partition[2] > 0)
		n = size_t(div_ceil(d->shape[0], d->partition[0])) * div_ceil(d->shape[1], d->partition[1]) *
		    div_ceil(d->shape[2], d->partition[2]);
	const size_t params = (sizeof(arma_mt_params) * n + 255) / 256 * 256;
	return params + (d->seeds ? sizeof(uint32_t) * n : 0);
}

void launch_mt_raw(arma_hip_ctx* ctx, const arma_mt_params* mts, const uint32_t* seeds,
                   int n_streams, int draws, uint32_t* out) {
	ARMA_HIP_REQUIRE(n_streams > 0 && draws >= 0 && mts, ARMA_HIP_EINVAL, "bad stream count");
	validate_params(mts, n_streams);
	int nn_max = 0;
	for (int i = 0; i < n_streams; ++i) nn_max = std::max(nn_max, int(mts[i].nn));
	auto* dparams = (arma_mt_params*)ctx->params.get(sizeof(arma_mt_params) * n_streams);
	upload(ctx, dparams, mts, sizeof(arma_mt_params) * n_streams);
	uint32_t* dseeds = nullptr;
	if (seeds) {
		dseeds = (uint32_t*)ctx->seeds.get(sizeof(uint32_t) * n_streams);
		upload(ctx, dseeds, seeds, sizeof(uint32_t) * n_streams);
	}
	const int tpb = std::min(threads_for_state(nn_max), 64);
	mt_raw_kernel<<<div_ceil(n_streams, tpb), tpb, size_t(tpb) * nn_max * 4, ctx->stream>>>(
		dparams, dseeds, n_streams, draws, out);
	ARMA_HIP_CHECK(hipGetLastError());
}

struct NoiseBatch {
	int precision = 0;
	int sem = ARMA_NOISE_DOUBLE;
	int nstreams = 0;
	bool small_blocks = true;
	NoisePlan plan;
	std::vector<arma_mt_params> hparams;
	Scratch params, seeds, recs, parts;
};

NoiseBatch* noise_batch_create(arma_hip_ctx* ctx, int precision,
                               const std::vector<BatchMember>& m) {
	auto* b = new NoiseBatch;
	try {
		noise_batch_build(ctx, b, precision, m);
	} catch (...) {
		delete b;
		throw;
	}
	return b;
}

NoiseBatch* noise_batch_new() { return new NoiseBatch; }

void noise_batch_build(arma_hip_ctx* ctx, NoiseBatch* b, int precision,
                       const std::vector<BatchMember>& m) {
	{
		b->precision = precision;
		b->small_blocks = true;
		b->hparams.clear();
		ARMA_HIP_REQUIRE(!m.empty(), ARMA_HIP_EINVAL, "empty batch");
		b->sem = m[0].d->noise_semantics;
		std::vector<uint32_t> seeds;
		std::vector<NoiseBlockRec> recs;
		for (const BatchMember& x : m) {
			const arma_ar_desc* d = x.d;
			ARMA_HIP_REQUIRE(d->varwn >= 0.0, ARMA_HIP_EINVAL, "variance is less than zero");
			ARMA_HIP_REQUIRE(d->noise_semantics == b->sem, ARMA_HIP_EINVAL,
			                 "every surface of a batch needs the same noise semantics");
			// the generated block: slices t0 .. nt-1
			const int gt = d->shape[0] - x.t0;
			ARMA_HIP_REQUIRE(x.t0 >= 0 && gt > 0, ARMA_HIP_EINVAL, "bad history length");
			int3 part{gt, d->shape[1], d->shape[2]};
			if (d->noise_mode == ARMA_NOISE_PARTITIONED) {
				ARMA_HIP_REQUIRE(d->partition[0] > 0 && d->partition[1] > 0 && d->partition[2] > 0,
				                 ARMA_HIP_EINVAL, "bad partition shape");
				part = int3{d->partition[0], d->partition[1], d->partition[2]};
			} else {
				ARMA_HIP_REQUIRE(d->noise_mode == ARMA_NOISE_SEQUENTIAL, ARMA_HIP_EINVAL,
				                 "bad noise mode");
			}
			const int np0 = div_ceil(gt, part.x), np1 = div_ceil(d->shape[1], part.y),
			          np2 = div_ceil(d->shape[2], part.z);
			const int n = np0 * np1 * np2;
			ARMA_HIP_REQUIRE(d->n_mts >= n && d->mts, ARMA_HIP_EPRNG, "bad number of MT configs");
			validate_params(d->mts, n);
			b->small_blocks = b->small_blocks && (long long)part.x * part.y * part.z < (1ll << 31);
			const double sd = std::sqrt(d->varwn);
			const float sdf = std::sqrt(float(d->varwn));
			for (int p = 0; p < n; ++p) {
				const int a = p / (np1 * np2), bb = (p / np2) % np1, c = p % np2;
				NoiseBlockRec r;
				r.base = (long long)(x.zoff + size_t(x.t0) * d->shape[1] * d->shape[2]);
				r.sy = d->shape[1];
				r.sz = d->shape[2];
				r.lo0 = a * part.x;
				r.lo1 = bb * part.y;
				r.lo2 = c * part.z;
				r.e0 = std::min(r.lo0 + part.x, gt) - r.lo0;
				r.e1 = std::min(r.lo1 + part.y, d->shape[1]) - r.lo1;
				r.e2 = std::min(r.lo2 + part.z, d->shape[2]) - r.lo2;
				r.sd = sd;
				r.sdf = sdf;
				recs.push_back(r);
				b->hparams.push_back(d->mts[p]);
				seeds.push_back(d->seeds ? d->seeds[p] : 0u);
			}
		}
		b->nstreams = int(recs.size());
		long long longest = 0;
		for (const NoiseBlockRec& r : recs)
			longest = std::max(longest, (long long)r.e0 * r.e1 * r.e2);
		b->plan = plan_noise(ctx, b->sem, b->nstreams, longest, b->hparams.data(),
		                     b->small_blocks, kBatchAheadBytes);
		if (b->plan.bytes(b->nstreams) && !b->parts.try_get(b->plan.bytes(b->nstreams)))
			b->plan = NoisePlan();
		b->params.get(sizeof(arma_mt_params) * recs.size());
		b->seeds.get(sizeof(uint32_t) * recs.size());
		b->recs.get(sizeof(NoiseBlockRec) * recs.size());
		upload(ctx, b->params.ptr, b->hparams.data(), sizeof(arma_mt_params) * recs.size());
		upload(ctx, b->seeds.ptr, seeds.data(), sizeof(uint32_t) * recs.size());
		upload(ctx, b->recs.ptr, recs.data(), sizeof(NoiseBlockRec) * recs.size());
	}
}

void noise_batch_launch(arma_hip_ctx* ctx, NoiseBatch* b, void* arena) {
	KernelTimer timer(ctx, "noise_batch");
	TableSpec g{(const NoiseBlockRec*)b->recs.ptr};
	launch_by_type(ctx, b->precision == ARMA_FP32, b->sem, b->hparams.data(),
	               (const arma_mt_params*)b->params.ptr, (const uint32_t*)b->seeds.ptr, arena, g,
	               b->nstreams, b->small_blocks, b->plan, b->parts.ptr);
}

void noise_batch_destroy(NoiseBatch* b) { delete b; }

}  // namespace arma_hip
