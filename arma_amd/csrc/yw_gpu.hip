// Yule-Walker coefficients by Choi's order recursion, and the white-noise
// variance, in FP64 on the GPU (src/yule_walker.cc:420-539,
// src/generator/ar_model.cc:55-61).
//
// The recursion is a chain of small dense products and inverses (matrices of
// at most shell(l) = 3l^2 + 3l + 1 rows: 169 for l = 7, 271 for l = 9) with a
// data-dependent stop.  Every operation keeps the order of the host solver's
// arithmetic (products summed over k in order, LU with the first largest pivot,
// substitutions column by column, dot products in order) and no contraction
// into FMAs, so the GPU result is the host result to the last bit.
//
// What bounds it is latency, so the chain is cut where the arithmetic allows:
//  * A matrix that is multiplied from the left only ever meets its own columns.
//    All of an order's updates of Phi (and Theta's products) therefore go by
//    strips of kStrip columns, each strip's whole chain over m in one workgroup
//    with workgroup barriers only, and the strips on as many CUs.
//  * Left operands are stored with a column's rows side by side, so that a wave
//    reads 64 rows of a column in one go, and a lane holds the sums of one row and
//    all columns of the strip.
//  * The LU works by panels of 16 columns, a panel in the registers of one wave
//    (no barrier and no memory between its columns), and the rest of the matrix
//    takes the panel's updates with all waves.
//  * The triangular solves take 16 columns per workgroup, 16 lanes per column.
// Each order is five launches, whose boundaries are the only waits between
// workgroups; a model that is finished (or failed) makes the rest return at once.
// A solve that goes through all orders up to 7 takes 1.76 ms, call and copies
// included, 9.66 when one workgroup walked the matrices; about half of it is LU,
// then the triangular solves and Phi.
#include "common.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

namespace arma_hip {
namespace {

__host__ __device__ inline int shell(int a) { return 3 * a * a + 3 * a + 1; }

struct YwArgs {
	const double* rho;  // rho(i,j,k) = gamma / gamma000 on an n^3 cube
	int n;
	int M;              // largest order tried
	double var_eps;
	int determine;
	double variance;    // gamma000
	// point tables: row points of a and shell points of b (i, j, k triples)
	const int* rows;
	const int* rows_off;
	const int* cols;
	const int* cols_off;
	// storage; every matrix but lu has its columns contiguous
	double* phi;            // Phi blocks
	const long long* phi_off;  // by key ((p * (M + 2)) + a) * (M + 2) + j
	double* pi0;            // Pi of this order and the last, by turns, blocks per m at pi_off[m]
	double* pi1;
	const long long* pi_off;
	double* theta;          // Theta_l^-1 at theta_off[l] (R_{1,1}^-1 for l = 1)
	const long long* theta_off;
	double* r;              // R_{m,q}, q < m
	const long long* r_off; // by m * (M + 2) + q
	double* lu;             // Theta_l, then its factors, row-major
	double* h;
	int* where;             // the row of the factors that a row of Theta_l went to
	double* state;          // lambda, variance of the last order
	double* out;            // l, varwn, then the l^3 coefficients
	int* status;            // 1 while the recursion runs
};

constexpr int kRunning = 1;

__device__ inline double rho_at(const YwArgs& a, int i, int j, int k) {
	i = i < 0 ? -i : i;
	j = j < 0 ? -j : j;
	k = k < 0 ? -k : k;
	return a.rho[(size_t(i) * a.n + j) * a.n + k];
}

// Element (r, c) of R_{a,b} (shell(a) x shell(b)).
__device__ inline double R_at(const YwArgs& y, int a, int b, int r, int c) {
	const int* rp = y.rows + 3 * (y.rows_off[a] + r);
	const int* cp = y.cols + 3 * (y.cols_off[b] + c);
	return rho_at(y, rp[0] - b + cp[0], rp[1] - b + cp[1], rp[2] - b + cp[2]);
}

__device__ inline double Rb0_at(const YwArgs& y, int a, int r) {
	const int* rp = y.rows + 3 * (y.rows_off[a] + r);
	return rho_at(y, rp[0], rp[1], rp[2]);
}

__device__ inline double Ra0_at(const YwArgs& y, int b, int c) {
	const int* cp = y.cols + 3 * (y.cols_off[b] + c);
	return rho_at(y, -b + cp[0], -b + cp[1], -b + cp[2]);
}

// Phi[p, a, j] (shell(a) x shell(p + j))
__device__ inline double* phi_block(const YwArgs& y, int p, int a, int j) {
	return y.phi + y.phi_off[(size_t(p) * (y.M + 2) + a) * (y.M + 2) + j];
}

// Pi of the last order (old) and of this one, l
__device__ inline double* pi_old(const YwArgs& y, int l, int m) {
	return (l & 1 ? y.pi1 : y.pi0) + y.pi_off[m];
}
__device__ inline double* pi_new(const YwArgs& y, int l, int m) {
	return (l & 1 ? y.pi0 : y.pi1) + y.pi_off[m];
}

// All R_{m,q}, q < m, of a model: grid (any, (M + 1) (M + 2), models).
__global__ void choi_r_kernel(const YwArgs* __restrict__ ys) {
	const YwArgs y = ys[blockIdx.z];
	const int m = blockIdx.y / (y.M + 2), q = blockIdx.y % (y.M + 2);
	if (m > y.M || q < 1 || q >= m) return;
	const int nr = shell(m), nc = shell(q);
	double* dst = y.r + y.r_off[m * (y.M + 2) + q];
	for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nr * nc; e += gridDim.x * blockDim.x)
		dst[e] = R_at(y, m, q, e % nr, e / nr);
}

// ---- products by strips of columns ----

constexpr int kStripThreads = 256;

// s[c] = sum over k of A(i, k) B(k, c) in order, A with its columns contiguous
// (rows of them), B in LDS with the strip's C columns side by side.
template <int C>
__device__ __forceinline__ void strip_row(double (&s)[C], const double* __restrict__ A, int rows,
                                          int K, int i, const double* B) {
	constexpr int kAhead = 16;  // loads in flight while as many terms are summed
	const double* a = A + i;
	double x[kAhead], next[kAhead];
#pragma unroll
	for (int u = 0; u < kAhead; ++u) x[u] = a[size_t(min(u, K - 1)) * rows];
#pragma unroll
	for (int c = 0; c < C; ++c) s[c] = 0.0;
	for (int k = 0; k < K; k += kAhead) {
		if (k + kAhead < K) {
#pragma unroll
			for (int u = 0; u < kAhead; ++u) next[u] = a[size_t(min(k + kAhead + u, K - 1)) * rows];
		}
		if (k + kAhead <= K) {
#pragma unroll
			for (int u = 0; u < kAhead; ++u)
#pragma unroll
				for (int c = 0; c < C; ++c) s[c] = s[c] + x[u] * B[(k + u) * C + c];
		} else {
#pragma unroll
			for (int u = 0; u < kAhead; ++u)
				if (k + u < K)
#pragma unroll
					for (int c = 0; c < C; ++c) s[c] = s[c] + x[u] * B[(k + u) * C + c];
		}
#pragma unroll
		for (int u = 0; u < kAhead; ++u) x[u] = next[u];
	}
}

// Columns j0 .. j0 + C - 1 (zero from column n on) of a matrix of K rows to LDS.
template <int C>
__device__ __forceinline__ void stage_strip(double* B, const double* __restrict__ src, int K,
                                            int j0, int n) {
	for (int e = threadIdx.x; e < K * C; e += kStripThreads) {
		const int c = e / K, k = e - c * K;
		B[k * C + c] = j0 + c < n ? src[size_t(j0 + c) * K + k] : 0.0;
	}
}

// Theta_l = R_{l,l} - sum_m R_{l,m} Phi[l,m,0] into lu, and as one more column
// h = R_b0(l) - sum_m R_{l,m} Pi[m], in strips of C columns: grid (strips, models).
// cap: rows of B that LDS holds.
template <int C>
__global__ __launch_bounds__(kStripThreads) void choi_theta_kernel(const YwArgs* __restrict__ ys,
                                                                   int l, int cap) {
	extern __shared__ double smem[];
	const YwArgs y = ys[blockIdx.y];
	if (*y.status != kRunning || l > y.M) return;
	const int n = shell(l), j0 = blockIdx.x * C;
	if (j0 > n) return;
	for (int i0 = 0; i0 < n; i0 += kStripThreads) {
		const int i = i0 + threadIdx.x;
		double t[C];
#pragma unroll
		for (int c = 0; c < C; ++c)
			t[c] = i < n && j0 + c <= n ? (j0 + c < n ? R_at(y, l, l, i, j0 + c) : Rb0_at(y, l, i))
			                            : 0.0;
		for (int m = 1; m < l;) {
			// the operands of as many m as fit
			int me = m, rows = 0;
			__syncthreads();
			for (; me < l && rows + shell(me) <= cap; ++me) {
				const int K = shell(me);
				stage_strip<C>(smem + rows * C, phi_block(y, l, me, 0), K, j0, n);
				if (j0 + C > n) {
					__syncthreads();
					const double* pv = pi_old(y, l, me);
					for (int k = threadIdx.x; k < K; k += kStripThreads)
						smem[(rows + k) * C + n - j0] = pv[k];
				}
				rows += K;
			}
			__syncthreads();
			for (const double* B = smem; m < me; B += shell(m) * C, ++m)
				if (i < n) {
					double s[C];
					strip_row<C>(s, y.r + y.r_off[l * (y.M + 2) + m], n, shell(m), i, B);
#pragma unroll
					for (int c = 0; c < C; ++c) t[c] = t[c] - s[c];
				}
		}
#pragma unroll
		for (int c = 0; c < C; ++c)
			if (i < n && j0 + c <= n) *(j0 + c < n ? y.lu + size_t(i) * n + j0 + c : y.h + i) = t[c];
	}
}

// Phi[2, 1, j] = R_{1,1}^-1 R_{1,2+j} for every j: grid (any, models).
__global__ void choi_phi1_kernel(const YwArgs* __restrict__ ys) {
	const YwArgs y = ys[blockIdx.y];
	if (*y.status != kRunning) return;
	const double* inv = y.theta + y.theta_off[1];
	constexpr int K = 7;  // shell(1)
	for (int j = 0; j + 2 <= y.M; ++j) {
		double* dst = phi_block(y, 2, 1, j);
		for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < K * shell(2 + j);
		     e += gridDim.x * blockDim.x) {
			double s = 0.0;
			for (int k = 0; k < K; ++k) s = s + inv[k * K + e % K] * R_at(y, 1, 2 + j, k, e / K);
			dst[e] = s;
		}
	}
}

// The blocks of order l + 1: for m = 2 .. l
//   Phi[m+1, m, l-m] = Theta_m^-1 (R_{m,l+1} - sum_q R_{m,q} Phi[m, q, l-m+1])
//   Phi[m+1, a, l-m] = Phi[m, a, l-m+1] - Phi[m, a, 0] Phi[m+1, m, l-m], a < m,
// in strips of C of their shell(l + 1) columns: grid (strips, models).
template <int C>
__global__ __launch_bounds__(kStripThreads) void choi_phi_kernel(const YwArgs* __restrict__ ys,
                                                                 int l, int cap) {
	extern __shared__ double smem[];
	const YwArgs y = ys[blockIdx.y];
	if (*y.status != kRunning || l >= y.M) return;
	const int n = shell(l + 1), j0 = blockIdx.x * C;
	if (j0 >= n) return;
	double* const rhs = smem + cap * C;
	double* const top = rhs + shell(l) * C;  // the strip of Phi[m+1, m, l-m]
	const int tid = threadIdx.x;
	for (int m = 2; m <= l; ++m) {
		const int M = shell(m), j = l - m;
		for (int i0 = 0; i0 < M; i0 += kStripThreads) {
			const int i = i0 + tid;
			double t[C];
#pragma unroll
			for (int c = 0; c < C; ++c)
				t[c] = i < M && j0 + c < n ? R_at(y, m, l + 1, i, j0 + c) : 0.0;
			for (int q = 1; q < m;) {
				int qe = q, rows = 0;
				__syncthreads();
				for (; qe < m && rows + shell(qe) <= cap; ++qe) {
					stage_strip<C>(smem + rows * C, phi_block(y, m, qe, j + 1), shell(qe), j0, n);
					rows += shell(qe);
				}
				__syncthreads();
				for (const double* B = smem; q < qe; B += shell(q) * C, ++q)
					if (i < M) {
						double s[C];
						strip_row<C>(s, y.r + y.r_off[m * (y.M + 2) + q], M, shell(q), i, B);
#pragma unroll
						for (int c = 0; c < C; ++c) t[c] = t[c] - s[c];
					}
			}
			if (i < M)
#pragma unroll
				for (int c = 0; c < C; ++c) rhs[i * C + c] = t[c];
		}
		__syncthreads();
		double* const out = phi_block(y, m + 1, m, j);
		for (int i = tid; i < M; i += kStripThreads) {
			double s[C];
			strip_row<C>(s, y.theta + y.theta_off[m], M, M, i, rhs);
#pragma unroll
			for (int c = 0; c < C; ++c) {
				top[i * C + c] = s[c];
				if (j0 + c < n) out[size_t(j0 + c) * M + i] = s[c];
			}
		}
		__syncthreads();
		// all rows of all a at once
		for (int e = tid; e < m * m * m - 1; e += kStripThreads) {
			int a = 1, i = e;
			for (; i >= shell(a); ++a) i -= shell(a);
			const int K = shell(a);
			double s[C];
			strip_row<C>(s, phi_block(y, m, a, 0), K, M, i, top);
			const double* d = phi_block(y, m, a, j + 1);
			double* o = phi_block(y, m + 1, a, j);
#pragma unroll
			for (int c = 0; c < C; ++c)
				if (j0 + c < n) o[size_t(j0 + c) * K + i] = d[size_t(j0 + c) * K + i] - s[c];
		}
	}
}

// ---- LU factorisation with partial pivoting ----

constexpr int kLuThreads = 512;
constexpr int kPanel = 16;
constexpr int kPanelRows = 5;               // rows of a panel per lane at most
constexpr int kLuPanelN = 64 * kPanelRows;  // largest matrix that goes by panels

template <int CTRL>
__device__ __forceinline__ double dpp_max(double v) {
	const int lo = __double2loint(v), hi = __double2hiint(v);
	const double o = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false),
	                                  __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false));
	return o > v ? o : v;
}

// The largest value of a wave (none is a NaN).
__device__ __forceinline__ double wave_max(double v) {
	v = dpp_max<0x111>(v);  // row_shr:1, 2, 4, 8
	v = dpp_max<0x112>(v);
	v = dpp_max<0x114>(v);
	v = dpp_max<0x118>(v);
	v = dpp_max<0x142>(v);  // row_bcast:15, 31
	v = dpp_max<0x143>(v);
	return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
	                        __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// LDS written before it by one lane of a wave is read after it by the others
// (a wave's LDS operations execute in order; the compiler must keep them so).
__device__ __forceinline__ void wave_sync() {
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
}

// Columns k0 .. k0 + 15 of rows k0 .. n - 1, RPL rows per lane of one wave:
// register row r of a lane is row k0 + lane + 64 r, and its columns move up by
// one with every step, so that a step's code is the same for all (unrolled over
// the columns it did not stay in the instruction cache).  Rows are not moved:
// place[r] is the row that it has become, and a row that has been a pivot (place
// below the current column) takes no further updates.  The pivot is the first
// largest by place, as in a sequential scan that keeps a row only when a later
// one is strictly larger; a NaN diagonal stays, a NaN elsewhere is never picked.
// The finished columns go to lp[column][row] (by register row, at the end by
// place).  Returns false when a pivot is exactly zero.
template <int RPL>
__device__ __forceinline__ bool factor_panel(double* lu, int n, int k0, double* lp, double* pivot_row,
                                             int* piv, int* moves, int* nmoves) {
	const int lane = threadIdx.x;
	double v[RPL][kPanel];
	int place[RPL];
	const int w = min(kPanel, n - k0);
#pragma unroll
	for (int r = 0; r < RPL; ++r) {
		const int i = k0 + lane + 64 * r;
		place[r] = i < n ? i : -1;  // no row: as one that is done
#pragma unroll
		for (int t = 0; t < kPanel; ++t) v[r][t] = i < n && t < w ? lu[size_t(i) * n + k0 + t] : 0.0;
	}
#pragma unroll 1
	for (int t = 0; t < w; ++t) {
		const int k = k0 + t;
		// a lane's best row, of equal ones the first
		double best = -1.0;
		int at = n, row = 0;
		bool nan_diag = false;
#pragma unroll
		for (int r = 0; r < RPL; ++r) {
			const double x = place[r] >= k ? fabs(v[r][0]) : -1.0;
			const bool better = x > best || (x == best && place[r] < at);
			best = better ? x : best;
			at = better ? place[r] : at;
			row = better ? r : row;
			nan_diag = nan_diag || (place[r] == k && isnan(v[r][0]));
		}
		const double most = wave_max(best);
		if (__any(nan_diag) || most < 0.0) {  // the diagonal it is
			at = n;
#pragma unroll
			for (int r = 0; r < RPL; ++r)
				if (place[r] == k) {
					at = k;
					row = r;
				}
			best = at == k ? most : -2.0;
		}
		unsigned long long hit = __ballot(best == most);
		int pl = __builtin_ctzll(hit);
		int p = __builtin_amdgcn_readlane(at, pl);
		for (hit &= hit - 1; hit; hit &= hit - 1) {
			const int hl = __builtin_ctzll(hit), hp = __builtin_amdgcn_readlane(at, hl);
			if (hp < p) {
				p = hp;
				pl = hl;
			}
		}
		const int pr = __builtin_amdgcn_readlane(row, pl);
		// its row to every lane, and as the row of U that it is from here on
#pragma unroll
		for (int r = 0; r < RPL; ++r)
			if (r == pr && lane == pl)
#pragma unroll
				for (int c = 0; c < kPanel; ++c) {
					pivot_row[c] = v[r][c];
					lp[(t + c) * kLuPanelN + lane + 64 * r] = v[r][c];
				}
		wave_sync();
		double u[kPanel];
#pragma unroll
		for (int c = 0; c < kPanel; ++c) u[c] = pivot_row[c];
		wave_sync();
		if (u[0] == 0.0) return false;
		if (lane == 0) piv[k] = p;
#pragma unroll
		for (int r = 0; r < RPL; ++r) {
			const bool is_pivot = r == pr && lane == pl;
			place[r] = is_pivot ? k : place[r] == k ? p : place[r];
			if (place[r] > k) {
				const double m = v[r][0] / u[0];
				lp[t * kLuPanelN + lane + 64 * r] = m;
#pragma unroll
				for (int c = 1; c < kPanel; ++c) v[r][c - 1] = v[r][c] - m * u[c];
			}
		}
	}
	// the rows to their places; which rows of the other columns move (at most two
	// per pivot)
	int count = 0;
#pragma unroll
	for (int r = 0; r < RPL; ++r)
#pragma unroll
		for (int t = 0; t < kPanel; ++t) v[r][t] = t < w ? lp[t * kLuPanelN + lane + 64 * r] : 0.0;
#pragma unroll
	for (int r = 0; r < RPL; ++r) {
		const int i = k0 + lane + 64 * r;
		const bool moved = i < n && place[r] != i;
		if (i < n) {
#pragma unroll
			for (int t = 0; t < kPanel; ++t)
				if (t < w) {
					lu[size_t(place[r]) * n + k0 + t] = v[r][t];
					lp[t * kLuPanelN + place[r]] = v[r][t];
				}
		}
		const unsigned long long mv = __ballot(moved);
		if (moved) {
			const int at = count + __popcll(mv & ((1ull << lane) - 1));
			moves[2 * at] = i;
			moves[2 * at + 1] = place[r];
		}
		count += __popcll(mv);
	}
	// (the list's rest repeats its first entry)
	wave_sync();
	if (lane >= count && lane < 2 * kPanel && count > 0) {
		moves[2 * lane] = moves[0];
		moves[2 * lane + 1] = moves[1];
	}
	if (lane == 0) *nmoves = count;
	return true;
}

// The factors of the n x n matrix at lu, n <= kLuPanelN, the pivots to piv (LDS).
// An element's updates come one at a time in the order of the columns, whichever
// panel they are in.
__device__ __forceinline__ bool lu_panels(double* lu, int n, int* piv) {
	// the panel, [column][row] (a pivot's row is written whole, past the last)
	__shared__ double pool[3 * kPanel * kLuPanelN];
	double* const lp = pool;
	double* const up = pool + 2 * kPanel * kLuPanelN;  // the rows of U beside it, [row][column]
	double* const tmp = pool + kPanel * kLuPanelN;     // rows on the move, a column per lane
	__shared__ double pivot_row[kPanel];
	__shared__ int moves[4 * kPanel], nmoves, good;
	const int tid = threadIdx.x;
	for (int k0 = 0; k0 < n; k0 += kPanel) {
		if (tid < 64) {
			bool ok;
			switch ((n - k0 + 63) / 64) {
			case 1: ok = factor_panel<1>(lu, n, k0, lp, pivot_row, piv, moves, &nmoves); break;
			case 2: ok = factor_panel<2>(lu, n, k0, lp, pivot_row, piv, moves, &nmoves); break;
			case 3: ok = factor_panel<3>(lu, n, k0, lp, pivot_row, piv, moves, &nmoves); break;
			case 4: ok = factor_panel<4>(lu, n, k0, lp, pivot_row, piv, moves, &nmoves); break;
			default: ok = factor_panel<5>(lu, n, k0, lp, pivot_row, piv, moves, &nmoves); break;
			}
			if (tid == 0) good = ok;
		}
		__syncthreads();
		if (!good) return false;
		const int w = min(kPanel, n - k0), k1 = k0 + w, nm = nmoves;
		// the other columns: the panel's row moves, then right of it its rows of U
		for (int c = tid; c < n - w; c += kLuThreads) {
			const int j = c < k0 ? c : c + w;
			for (int e0 = 0; e0 < nm; e0 += 8)
#pragma unroll
				for (int e = 0; e < 8; ++e) tmp[(e0 + e) * kLuPanelN + j] = lu[moves[2 * (e0 + e)] * n + j];
			for (int e0 = 0; e0 < nm; e0 += 8)
#pragma unroll
				for (int e = 0; e < 8; ++e) lu[moves[2 * (e0 + e) + 1] * n + j] = tmp[(e0 + e) * kLuPanelN + j];
			if (j >= k1) {
				// a row at a time, the ones below it moving up
				double u[kPanel];
#pragma unroll
				for (int t = 0; t < kPanel; ++t) u[t] = t < w ? lu[(k0 + t) * n + j] : 0.0;
#pragma unroll 1
				for (int q = 0; q < w; ++q) {
					lu[(k0 + q) * n + j] = u[0];
					up[q * kLuPanelN + j] = u[0];
					const double* l = lp + q * kLuPanelN + k0 + q;
					const double top = u[0];
#pragma unroll
					for (int t = 1; t < kPanel; ++t) u[t - 1] = u[t] - l[t] * top;
				}
			}
		}
		__syncthreads();
		// everything below and right of it, tiles of 64 x 32 per wave, 8 rows and 4
		// columns per lane (a lane with a row of 64 columns to itself and 8 rows of
		// broadcast factors was bound by its reads of LDS)
		constexpr int kR = 8, kC = 4;
		const int nj = (n - k1 + 8 * kC - 1) / (8 * kC), ni = (n - k1 + 8 * kR - 1) / (8 * kR);
		for (int e = tid / 64; e < nj * ni; e += kLuThreads / 64) {
			const int i = k1 + 8 * kR * (e / nj) + kR * (tid % 64 / 8);
			const int j = k1 + 8 * kC * (e % nj) + tid % 8;  // and 8, 16, 24 on
			if (i >= n) continue;
			double x[kR][kC];
#pragma unroll
			for (int r = 0; r < kR; ++r)
#pragma unroll
				for (int c = 0; c < kC; ++c) x[r][c] = lu[min(i + r, n - 1) * n + min(j + 8 * c, n - 1)];
#pragma unroll 2
			for (int t = 0; t < kPanel; ++t) {
				double l[kR], u[kC];
#pragma unroll
				for (int r = 0; r < kR; ++r) l[r] = lp[t * kLuPanelN + i + r];
#pragma unroll
				for (int c = 0; c < kC; ++c) u[c] = up[t * kLuPanelN + min(j + 8 * c, n - 1)];
#pragma unroll
				for (int r = 0; r < kR; ++r)
#pragma unroll
					for (int c = 0; c < kC; ++c) x[r][c] = x[r][c] - l[r] * u[c];
			}
#pragma unroll
			for (int r = 0; r < kR; ++r)
#pragma unroll
				for (int c = 0; c < kC; ++c)
					if (i + r < n && j + 8 * c < n) lu[(i + r) * n + j + 8 * c] = x[r][c];
		}
		__syncthreads();
	}
	return true;
}

// The same column by column in device memory, for larger matrices.
__device__ __forceinline__ bool lu_columns(double* lu, int n, int* piv) {
	__shared__ int pk;
	__shared__ int bad;
	__shared__ double wbest[kLuThreads / 64];
	__shared__ int wbidx[kLuThreads / 64];
	if (threadIdx.x == 0) bad = 0;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	for (int k = 0; k < n; ++k) {
		// pivot: the first row i >= k of largest |lu(i, k)| (the host's
		// sequential scan keeps a row only when a later one is strictly
		// larger), as a lane scan, a wave reduction and a fold of the waves,
		// each preferring the smaller row on ties
		double bv = -1.0;
		int bi = n;
		for (int i = k + threadIdx.x; i < n; i += blockDim.x) {
			const double v = fabs(lu[size_t(i) * n + k]);
			if (v > bv) {
				bv = v;
				bi = i;
			}
		}
		for (int off = 32; off > 0; off >>= 1) {
			const double ov = __shfl_xor(bv, off);
			const int oi = __shfl_xor(bi, off);
			if (ov > bv || (ov == bv && oi < bi)) {
				bv = ov;
				bi = oi;
			}
		}
		if (lane == 0) {
			wbest[wave] = bv;
			wbidx[wave] = bi;
		}
		__syncthreads();
		if (threadIdx.x == 0) {
			int p = wbidx[0];
			double pv = wbest[0];
			for (int q = 1; q < int(blockDim.x) / 64; ++q)
				if (wbest[q] > pv || (wbest[q] == pv && wbidx[q] < p)) {
					pv = wbest[q];
					p = wbidx[q];
				}
			// the scan never leaves a NaN diagonal (no value compares larger)
			// and never picks a NaN row
			if (p >= n || isnan(lu[size_t(k) * n + k])) p = k;
			if (lu[size_t(p) * n + k] == 0.0) bad = 1;
			pk = p;
			piv[k] = p;
		}
		__syncthreads();
		if (bad) return false;
		const int p = pk;
		if (p != k)
			for (int j = threadIdx.x; j < n; j += blockDim.x) {
				const double t = lu[size_t(k) * n + j];
				lu[size_t(k) * n + j] = lu[size_t(p) * n + j];
				lu[size_t(p) * n + j] = t;
			}
		__syncthreads();
		const double d = lu[size_t(k) * n + k];
		for (int i = k + 1 + threadIdx.x; i < n; i += blockDim.x) lu[size_t(i) * n + k] /= d;
		__syncthreads();
		// the rank-1 update, four consecutive elements of a row per lane:
		// every operand is loaded before any of the four is stored (an updated
		// element (i > k, j > k) is never an operand of another: those are
		// column k, row k and the element itself)
		const int w = n - k - 1, wb = (w + 3) / 4;
		for (int e = threadIdx.x; e < w * wb; e += blockDim.x) {
			const int i = k + 1 + e / wb, j0 = k + 1 + 4 * (e - (e / wb) * wb);
			const int cnt = min(4, n - j0);
			double* row = lu + size_t(i) * n;
			const double* rk = lu + size_t(k) * n;
			const double l = row[k];
			double a[4], u[4];
#pragma unroll
			for (int r = 0; r < 4; ++r) {
				const int j = r < cnt ? j0 + r : j0;
				a[r] = row[j];
				u[r] = rk[j];
			}
#pragma unroll
			for (int r = 0; r < 4; ++r)
				if (r < cnt) row[j0 + r] = a[r] - l * u[r];
		}
		__syncthreads();
	}
	return true;
}

// Theta_l at lu to its factors, one workgroup per model.
__global__ __launch_bounds__(kLuThreads) void choi_lu_kernel(const YwArgs* __restrict__ ys, int l) {
	const YwArgs y = ys[blockIdx.x];
	if (*y.status != kRunning || l > y.M) return;
	__shared__ int piv[kLuPanelN];
	const int n = shell(l), tid = threadIdx.x;
	const bool panels = n <= kLuPanelN;
	int* const pv = panels ? piv : y.where + n;
	if (!(panels ? lu_panels(y.lu, n, piv) : lu_columns(y.lu, n, pv))) {
		__syncthreads();
		if (tid == 0) *y.status = ARMA_HIP_ERUNTIME;
		return;
	}
	__syncthreads();
	// where the interchanges took each row
	for (int c = tid; c < n; c += kLuThreads) {
		int pos = c;
		for (int k = 0; k < n; ++k) {
			const int p = pv[k];
			pos = pos == k ? p : pos == p ? k : pos;
		}
		y.where[c] = pos;
	}
}

// ---- triangular solves ----

constexpr int kSubCols = 16;               // columns of the inverse per workgroup
constexpr int kSubRows = 16;               // rows of a block, one lane each per column
constexpr int kSubThreads = kSubCols * kSubRows;
constexpr int kSubChunk = 256;             // columns of the factors in LDS at a time
constexpr int kSubPitch = kSubChunk + 1;
constexpr int kSubX = 320;                 // rows of the solution that LDS holds

template <int T>
__device__ __forceinline__ double row_bcast(double v) {
	return __hiloint2double(
		__builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x150 + T, 0xf, 0xf, true),
		__builtin_amdgcn_update_dpp(0, __double2loint(v), 0x150 + T, 0xf, 0xf, true));
}

template <int T, int E, class F>
__device__ __forceinline__ void up_to(F&& f) {
	if constexpr (T < E) {
		f(std::integral_constant<int, T>{});
		up_to<T + 1, E>(f);
	}
}

// Theta_l^-1 from the factors: column c of it starts as e_c through the row
// interchanges, then
//   forward  x_i = b_i - sum_{j<i} L_ij x_j      (j ascending)
//   backward x_i = (y_i - sum_{j>i} U_ij x_j) / U_ii  (j descending),
// each row's terms subtracted one at a time in that order, as the host solver
// does.  Rows go in blocks of 16: the terms with j outside the block come first
// in either order and the block's rows take them side by side, a lane each; then
// the block's own rows hand their values on across the 16 lanes.  The solution is
// in LDS where it fits, else it stays in the result's columns.
__global__ __launch_bounds__(kSubThreads) void choi_solve_kernel(const YwArgs* __restrict__ ys,
                                                                 int l) {
	__shared__ double f[kSubRows * kSubPitch];     // rows of the factors
	__shared__ double xs[kSubCols * (kSubX + 1)];
	const YwArgs y = ys[blockIdx.y];
	if (*y.status != kRunning || l > y.M) return;
	const int n = shell(l), c = blockIdx.x * kSubCols + threadIdx.x / kSubRows;
	const int r = threadIdx.x % kSubRows;
	if (int(blockIdx.x) * kSubCols >= n) return;
	const double* __restrict__ lu = y.lu;
	double* const inv = y.theta + y.theta_off[l];
	const bool act = c < n;
	const bool in_lds = n <= kSubX;
	double* const x = in_lds ? xs + (threadIdx.x / kSubRows) * (kSubX + 1) : inv + size_t(act ? c : 0) * n;
	const int pos = act ? y.where[c] : -1;
	// Columns j0 .. j0 + kSubChunk - 1 of rows I .. I + 15 of the factors, on their
	// way to LDS while the last ones are in use.
	constexpr int kEach = kSubRows * kSubChunk / kSubThreads;
	double ahead[kEach];
	auto fetch = [&](int I, int j0, int jn) {
#pragma unroll
		for (int e = 0; e < kEach; ++e) {
			const int q = j0 + threadIdx.x;
			ahead[e] = I + e < n && q < jn ? lu[size_t(I + e) * n + q] : 0.0;
		}
	};
	static_assert(kSubThreads == kSubChunk, "a lane fetches a column of the chunk");
	auto put = [&] {
		__syncthreads();
#pragma unroll
		for (int e = 0; e < kEach; ++e) f[e * kSubPitch + threadIdx.x] = ahead[e];
		__syncthreads();
	};
	const double* const fr = f + r * kSubPitch;
	fetch(0, 0, kSubRows);
	for (int I = 0; I < n; I += kSubRows) {
		double v = I + r == pos ? 1.0 : 0.0;
		const int jend = I + kSubRows;  // columns of the lower triangle
		for (int j0 = 0; j0 < jend; j0 += kSubChunk) {
			put();
			if (j0 + kSubChunk < jend)
				fetch(I, j0 + kSubChunk, jend);
			else if (jend < n)
				fetch(jend, 0, jend + kSubRows);
			const int je = min(kSubChunk, I - j0);
			if (act) {
#pragma unroll 8
				for (int q = 0; q < je; ++q) v = v - fr[q] * x[j0 + q];
			}
			if (I < j0 + kSubChunk) {
				up_to<0, kSubRows>([&](auto t) {
					const double xt = row_bcast<t.value>(v);
					const double d = v - fr[I - j0 + t.value] * xt;
					v = r > t.value ? d : v;
				});
			}
		}
		if (act && I + r < n) x[I + r] = v;
	}
	const int last = (n - 1) / kSubChunk * kSubChunk;
	fetch((n - 1) / kSubRows * kSubRows, last, n);
	for (int I = (n - 1) / kSubRows * kSubRows; I >= 0; I -= kSubRows) {
		const int nb = min(kSubRows, n - I), first = I / kSubChunk * kSubChunk;
		double v = 0.0;
		for (int j0 = last; j0 >= first; j0 -= kSubChunk) {
			put();
			if (j0 > first)
				fetch(I, j0 - kSubChunk, n);
			else if (I > 0)
				fetch(I - kSubRows, last, n);
			if (j0 == last) v = act && r < nb ? x[I + r] : 0.0;
			const int qlo = max(0, I + nb - j0);
			if (act) {
#pragma unroll 8
				for (int q = min(kSubChunk, n - j0) - 1; q >= qlo; --q) v = v - fr[q] * x[j0 + q];
			}
			if (j0 == first) {
				const double diag = r < nb ? fr[I - j0 + r] : 1.0;
				up_to<0, kSubRows>([&](auto tt) {
					constexpr int t = kSubRows - 1 - decltype(tt)::value;
					const double q = v / diag;
					const double xt = row_bcast<t>(q);
					const double d = v - fr[I - j0 + t] * xt;
					if (t < nb) v = r == t ? q : r < t ? d : v;
				});
			}
		}
		if (act && r < nb) {
			x[I + r] = v;
			inv[size_t(c) * n + I + r] = v;
		}
	}
}

// Pi of order l, the variance, and whether the recursion ends: one workgroup per
// model.
constexpr int kPiThreads = 512;

__global__ __launch_bounds__(kPiThreads) void choi_pi_kernel(const YwArgs* __restrict__ ys, int l) {
	extern __shared__ double smem[];
	const YwArgs y = ys[blockIdx.x];
	if (*y.status != kRunning || l > y.M) return;
	const int n = shell(l), tid = threadIdx.x;
	double* const h = smem;
	double* const top = smem + n;
	__shared__ int over;
	__shared__ int changed;
	for (int i = tid; i < n; i += kPiThreads) h[i] = y.h[i];
	__syncthreads();
	for (int i = tid; i < n; i += kPiThreads) {
		double s[1];
		strip_row<1>(s, y.theta + y.theta_off[l], n, n, i, h);
		top[i] = s[0];
		pi_new(y, l, l)[i] = s[0];
	}
	__syncthreads();
	for (int e = tid; e < l * l * l - 1; e += kPiThreads) {
		int a = 1, i = e;
		for (; i >= shell(a); ++a) i -= shell(a);
		double s[1];
		strip_row<1>(s, phi_block(y, l, a, 0), shell(a), n, i, top);
		pi_new(y, l, a)[i] = pi_old(y, l, a)[i] - s[0];
	}
	// the first order's variance takes R_a0 for h
	if (l == 1) {
		for (int i = tid; i < n; i += kPiThreads) h[i] = Ra0_at(y, 1, i);
		__syncthreads();
	}
	if (tid == 0) {
		double s = 0.0;
		for (int i = 0; i < n; ++i) s += h[i] * top[i];
		const double lambda = (l == 1 ? 1.0 : y.state[0]) - s;
		const double var0 = l == 1 ? y.variance : y.state[1];
		const double var = y.variance * lambda;
		y.state[0] = lambda;
		y.state[1] = var;
		changed = !(y.determine && fabs(var - var0) < y.var_eps);
		over = l > 1 && !(l < y.M && changed);
		if (over) {
			y.out[0] = double(l);
			y.out[1] = changed ? var : var0;
		}
	}
	__syncthreads();
	if (!over) return;
	// phi(l x l x l) from the block vectors, in the order of the row points
	double* const coef = y.out + 2;
	for (int e = tid; e < l * l * l; e += kPiThreads) coef[e] = 0.0;
	__syncthreads();
	for (int e = tid; e < l * l * l - 1; e += kPiThreads) {
		int d = 1, i = e;
		for (; i >= shell(d); ++d) i -= shell(d);
		const int* rp = y.rows + 3 * (y.rows_off[d] + i);
		coef[(size_t(rp[0]) * l + rp[1]) * l + rp[2]] =
			(changed ? pi_new(y, l, d) : pi_old(y, l, d))[i];
	}
	__syncthreads();
	if (tid == 0) *y.status = ARMA_HIP_OK;
}

// sigma^2 = gamma000 - sum phi * gamma over phi's shape, summed in the host
// order by one lane from the products that the workgroup has formed (order 7:
// 28 us with that lane's loads behind one another, 5 us so).
__global__ __launch_bounds__(256) void varwn_kernel(const double* acf, int a1, int a2,
                                                    const double* phi, int p0, int p1, int p2,
                                                    double* out) {
	__shared__ double term[1024];
	const long long np = (long long)p0 * p1 * p2;
	double s = 0.0;
	for (long long e0 = 0; e0 < np; e0 += 1024) {
		const int m = int(min(np - e0, 1024ll));
		for (int e = threadIdx.x; e < m; e += 256) {
			const long long q = e0 + e, ab = q / p2;
			const int a = int(ab / p1), b = int(ab % p1), c = int(q % p2);
			term[e] = phi[q] * acf[(size_t(a) * a1 + b) * a2 + c];
		}
		__syncthreads();
		if (threadIdx.x == 0) {
#pragma unroll 8
			for (int e = 0; e < m; ++e) s += term[e];
		}
		__syncthreads();
	}
	if (threadIdx.x == 0) *out = acf[0] - s;
}

void push_points(std::vector<int>& v, int i, int j, int k) {
	v.push_back(i);
	v.push_back(j);
	v.push_back(k);
}

}  // namespace

namespace {

// Host tables and device layout of one model's recursion.
struct YwPlan {
	int n = 0, M = 0, MP = 0;
	double var_eps = 0.0, variance = 0.0;
	bool determine = true;
	std::vector<int> rows, cols, rows_off, cols_off;
	std::vector<long long> phi_off, pi_off, theta_off, r_off;
	std::vector<double> rho;
	long long nphi = 0, npi = 0, nth = 0, nr = 0, S = 0;
	// bytes that the host fills, and of the recursion's storage
	size_t host_bytes() const {
		const size_t b = 8 * (rho.size() + phi_off.size() + pi_off.size() + theta_off.size() + r_off.size()) +
		                 4 * (rows.size() + cols.size() + rows_off.size() + cols_off.size() + 1);
		return (b + 255) / 256 * 256;
	}
	size_t storage_bytes() const {
		const size_t b = 8 * (size_t(nphi) + 2 * size_t(npi) + size_t(nth) + size_t(nr) +
		                      size_t(S) * S + size_t(S) + 2 + out_len()) +
		                 4 * 2 * size_t(S);
		return (b + 255) / 256 * 256;
	}
	size_t out_len() const { return size_t(M + 1) * (M + 1) * (M + 1) + 2; }
};

YwPlan plan_model(const double* acf, int n, int max_order, double var_eps, bool determine) {
	YwPlan q;
	q.n = n;
	q.M = std::min(max_order, n - 1);
	ARMA_HIP_REQUIRE(q.M >= 2, ARMA_HIP_EINVAL, "AR order below 2 for Choi solver");
	ARMA_HIP_REQUIRE(acf[0] != 0.0, ARMA_HIP_EINVAL, "zero variance in the ACF");
	q.var_eps = var_eps;
	q.determine = determine;
	q.variance = acf[0];
	const int MP = q.MP = q.M + 2;
	// point tables up to M + 1
	q.rows_off.resize(MP);
	q.cols_off.resize(MP);
	for (int a = 0; a < MP; ++a) {
		q.rows_off[a] = int(q.rows.size() / 3);
		push_points(q.rows, a, a, a);
		for (int e = 1; e <= a; ++e) {
			for (int r = 0; r < e; ++r) push_points(q.rows, a - e, a - r, a);
			for (int r = 0; r < e; ++r) push_points(q.rows, a - e + r, a - e, a);
			for (int r = 0; r < e; ++r) push_points(q.rows, a, a - e, a - r);
			for (int r = 0; r < e; ++r) push_points(q.rows, a, a - e + r, a - e);
			for (int r = 0; r < e; ++r) push_points(q.rows, a - r, a, a - e);
			for (int r = 0; r < e; ++r) push_points(q.rows, a - e, a, a - e + r);
		}
		q.cols_off[a] = int(q.cols.size() / 3);
		push_points(q.cols, 0, 0, 0);
		for (int e = 1; e <= a; ++e) {
			for (int r = 0; r < e; ++r) push_points(q.cols, e, r, 0);
			for (int r = 0; r < e; ++r) push_points(q.cols, e - r, e, 0);
			for (int r = 0; r < e; ++r) push_points(q.cols, 0, e, r);
			for (int r = 0; r < e; ++r) push_points(q.cols, 0, e - r, e);
			for (int r = 0; r < e; ++r) push_points(q.cols, r, 0, e);
			for (int r = 0; r < e; ++r) push_points(q.cols, e, 0, e - r);
		}
	}
	// block offsets (in doubles)
	q.phi_off.assign(size_t(MP) * MP * MP, -1);
	q.pi_off.resize(MP);
	q.theta_off.resize(MP);
	for (int p = 2; p < MP; ++p)
		for (int a = 1; a < p; ++a)
			for (int j = 0; p + j < MP; ++j) {
				q.phi_off[(size_t(p) * MP + a) * MP + j] = q.nphi;
				q.nphi += (long long)shell(a) * shell(p + j);
			}
	for (int m = 0; m < MP; ++m) {
		q.pi_off[m] = q.npi;
		q.npi += shell(m);
		q.theta_off[m] = q.nth;
		q.nth += (long long)shell(m) * shell(m);
	}
	q.r_off.assign(size_t(MP) * MP, -1);
	for (int m = 2; m <= q.M; ++m)
		for (int p = 1; p < m; ++p) {
			q.r_off[size_t(m) * MP + p] = q.nr;
			q.nr += (long long)shell(m) * shell(p);
		}
	q.S = shell(q.M);
	const size_t n3 = size_t(n) * n * n;
	q.rho.resize(n3);
	for (size_t e = 0; e < n3; ++e) q.rho[e] = acf[e] / acf[0];
	return q;
}

// Lays the model out: what the host fills, from offset o1 of the host image
// (the same from device address dev1), then the recursion's storage from dev2.
YwArgs place_model(const YwPlan& q, unsigned char* dev1, unsigned char* img, unsigned char* dev2) {
	YwArgs y{};
	y.n = q.n;
	y.M = q.M;
	y.var_eps = q.var_eps;
	y.determine = q.determine ? 1 : 0;
	y.variance = q.variance;
	size_t at = 0;
	auto put = [&](auto& ptr, const auto& v) {
		std::memcpy(img + at, v.data(), v.size() * sizeof(v[0]));
		ptr = reinterpret_cast<std::decay_t<decltype(ptr)>>(dev1 + at);
		at += v.size() * sizeof(v[0]);
	};
	put(y.rho, q.rho);
	put(y.phi_off, q.phi_off);
	put(y.pi_off, q.pi_off);
	put(y.theta_off, q.theta_off);
	put(y.r_off, q.r_off);
	put(y.rows, q.rows);
	put(y.cols, q.cols);
	put(y.rows_off, q.rows_off);
	put(y.cols_off, q.cols_off);
	put(y.status, std::vector<int>{kRunning});
	at = 0;
	auto take = [&](auto& ptr, size_t n) {
		ptr = reinterpret_cast<std::decay_t<decltype(ptr)>>(dev2 + at);
		at += n * sizeof(*ptr);
	};
	take(y.phi, size_t(q.nphi));
	take(y.pi0, size_t(q.npi));
	take(y.pi1, size_t(q.npi));
	take(y.theta, size_t(q.nth));
	take(y.r, size_t(q.nr));
	take(y.lu, size_t(q.S) * q.S);
	take(y.h, size_t(q.S));
	take(y.state, 2);
	take(y.out, q.out_len());
	take(y.where, 2 * size_t(q.S));
	return y;
}

// Launches of the recursion over nm models of orders up to M.
template <int C>
void launch_choi(arma_hip_ctx* ctx, const YwArgs* ys, int nm, int M) {
	// rows of the right operands that a strip keeps in LDS: those of all lower
	// orders up to order 10, at least those of one block
	const int cap = std::max(shell(M), std::min(M * M * M, 1000));
	const size_t lds_theta = size_t(cap) * C * sizeof(double);
	const size_t lds_phi = lds_theta + 2 * size_t(shell(M)) * C * sizeof(double);
	const size_t lds_pi = 2 * size_t(shell(M)) * sizeof(double);
	if (lds_phi > 65536) {
		ARMA_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&choi_theta_kernel<C>),
		                                   hipFuncAttributeMaxDynamicSharedMemorySize, int(lds_theta)));
		ARMA_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&choi_phi_kernel<C>),
		                                   hipFuncAttributeMaxDynamicSharedMemorySize, int(lds_phi)));
	}
	hipStream_t st = ctx->stream;
	choi_r_kernel<<<dim3(8, (M + 1) * (M + 2), nm), 256, 0, st>>>(ys);
	for (int l = 1; l <= M; ++l) {
		choi_theta_kernel<C><<<dim3(div_ceil(shell(l) + 1, C), nm), kStripThreads, lds_theta, st>>>(
			ys, l, cap);
		choi_lu_kernel<<<nm, kLuThreads, 0, st>>>(ys, l);
		choi_solve_kernel<<<dim3(div_ceil(shell(l), kSubCols), nm), kSubThreads, 0, st>>>(ys, l);
		choi_pi_kernel<<<nm, kPiThreads, lds_pi, st>>>(ys, l);
		if (l == 1)
			choi_phi1_kernel<<<dim3(4, nm), 256, 0, st>>>(ys);
		else if (l < M)
			choi_phi_kernel<C><<<dim3(div_ceil(shell(l + 1), C), nm), kStripThreads, lds_phi, st>>>(
				ys, l, cap);
		ARMA_HIP_CHECK(hipGetLastError());
	}
}

}  // namespace

void yule_walker_choi_device_many(arma_hip_ctx* ctx, const std::vector<YwProblem>& probs,
                                  std::vector<YwSolution>& sols) {
	const size_t nm = probs.size();
	sols.assign(nm, YwSolution{});
	if (nm == 0) return;
	std::vector<YwPlan> plans;
	plans.reserve(nm);
	// the arguments, then what the host fills of every model, in one upload; the
	// storage after it
	const size_t args_bytes = (sizeof(YwArgs) * nm + 255) / 256 * 256;
	size_t filled = args_bytes, total = 0;
	int M = 0;
	for (const YwProblem& pr : probs) {
		plans.push_back(plan_model(pr.acf, pr.n, pr.max_order, pr.var_eps, pr.determine));
		filled += plans.back().host_bytes();
		total += plans.back().storage_bytes();
		M = std::max(M, plans.back().M);
	}
	total += filled;
	unsigned char* dev = (unsigned char*)ctx->yw.get(total);
	std::vector<unsigned char> img(filled, 0);
	std::vector<YwArgs> args(nm);
	size_t at1 = args_bytes, at2 = filled;
	for (size_t i = 0; i < nm; ++i) {
		args[i] = place_model(plans[i], dev + at1, img.data() + at1, dev + at2);
		at1 += plans[i].host_bytes();
		at2 += plans[i].storage_bytes();
	}
	std::memcpy(img.data(), args.data(), sizeof(YwArgs) * nm);
	upload(ctx, dev, img.data(), filled);
	{
		KernelTimer timer(ctx, "yule_walker_choi");
		// four columns per strip; single ones where their operands would not fit
		// LDS (orders above 20)
		if (M <= 20)
			launch_choi<4>(ctx, (const YwArgs*)dev, int(nm), M);
		else
			launch_choi<1>(ctx, (const YwArgs*)dev, int(nm), M);
	}
	// every model's status and results come back with one copy of the
	// whole buffer's result words
	std::vector<int> status(nm);
	std::vector<std::vector<double>> tails(nm);
	for (size_t i = 0; i < nm; ++i) {
		tails[i].resize(plans[i].out_len());
		ARMA_HIP_CHECK(hipMemcpyAsync(&status[i], args[i].status, 4, hipMemcpyDeviceToHost,
		                              ctx->stream));
		ARMA_HIP_CHECK(hipMemcpyAsync(tails[i].data(), args[i].out, tails[i].size() * 8,
		                              hipMemcpyDeviceToHost, ctx->stream));
	}
	ARMA_HIP_CHECK(hipStreamSynchronize(ctx->stream));
	for (size_t i = 0; i < nm; ++i) {
		YwSolution& r = sols[i];
		if (status[i] != ARMA_HIP_OK) {
			r.status = ARMA_HIP_ERUNTIME;  // getrf: a zero pivot
			continue;
		}
		r.l = int(tails[i][0]);
		if (!(r.l >= 2 && r.l <= plans[i].M)) {
			r.status = ARMA_HIP_ERUNTIME;
			continue;
		}
		r.status = ARMA_HIP_OK;
		r.varwn = tails[i][1];
		const size_t L3 = size_t(r.l) * r.l * r.l;
		r.phi.assign(tails[i].begin() + 2, tails[i].begin() + 2 + L3);
	}
}

void yule_walker_choi_device(arma_hip_ctx* ctx, const double* acf, int n, int max_order,
                             double var_eps, bool determine, std::vector<double>& phi, int& l,
                             double& varwn) {
	std::vector<YwSolution> sol;
	yule_walker_choi_device_many(ctx, {YwProblem{acf, n, max_order, var_eps, determine}}, sol);
	ARMA_HIP_REQUIRE(sol[0].status == ARMA_HIP_OK, ARMA_HIP_ERUNTIME, "getrf error");
	l = sol[0].l;
	varwn = sol[0].varwn;
	phi = std::move(sol[0].phi);
}

double white_noise_variance_device(arma_hip_ctx* ctx, const double* acf, const int32_t acf_shape[3],
                                   const double* phi, const int32_t phi_shape[3]) {
	const size_t na = numel3(acf_shape), np = numel3(phi_shape);
	double* d = (double*)ctx->yw.get((na + np + 1) * 8);
	upload(ctx, d, acf, na * 8);
	upload(ctx, d + na, phi, np * 8);
	varwn_kernel<<<1, 256, 0, ctx->stream>>>(d, acf_shape[1], acf_shape[2], d + na, phi_shape[0],
	                                        phi_shape[1], phi_shape[2], d + na + np);
	ARMA_HIP_CHECK(hipGetLastError());
	double v = 0.0;
	ARMA_HIP_CHECK(hipMemcpyAsync(&v, d + na + np, 8, hipMemcpyDeviceToHost, ctx->stream));
	ARMA_HIP_CHECK(hipStreamSynchronize(ctx->stream));
	return v;
}

}  // namespace arma_hip
