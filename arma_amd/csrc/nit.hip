// Non-linear inertialess transform (NIT) of the realisation on the GPU.
//
// Reference: NIT_transform<T>::transform_realisation
// (src/nonlinear/nit_transform.cc:127-164) -> transform_data
// (src/nonlinear/transforms.hh:58-75): every point x of the surface is
// replaced by the root c of F(c) = Phi(x / stdev), stdev = sqrt(acf(0,0,0)),
// where F is the target CDF, Gram-Charlier (src/stats/gram_charlier.hh:40-45)
// or skew normal (src/stats/skew_normal.hh:38-42, Owen's T by the symmetric
// 20-point Gauss-Legendre rule of src/apmath/owen_t.cc:38-55), and the root
// comes from the reference's bisection (src/linalg.hh:199-213): at most
// max_iter halvings of [a, b], stopping once b - a <= eps or |F(c) - y| <= eps,
// the last midpoint being the result.
//
// One thread per point; the bisection runs in FP64 for both precisions.  The
// reference evaluates F at a and at b again in every step; F is a pure
// function, so the kernel keeps F(a) and F(b) from the step that set them and
// evaluates F once per step, with identical results.  The Gauss-Legendre
// nodes are computed on the host (Newton's method on P_20) and passed in.
//
// The evaluations (an exp and an erf, or eleven exps, at each of about 25 steps)
// are the kernel's time.  Every point starts from the same interval, so its first
// steps visit the same few midpoints as all others': a launch first evaluates F
// at the midpoints of the first levels (nit_table_kernel, at most a sixteenth as
// many as there are points) and the points take those steps by look-up, with
// the same decisions.  4194304 points in FP64, error 1e-6, with a copy of the points
// beside it: Gram-Charlier 0.23 ms with 18 levels and 0.61 without, skew normal
// 0.39 and 1.54.
#include <hip/hip_runtime.h>

#include <cmath>

#include "common.hpp"

namespace arma_hip {
namespace {

struct NitParams {
	double stdev;  // deviation of the data's normal law
	double a, b, eps;
	int max_iter, dist;
	double skew, kurt;          // Gram-Charlier
	double mean, sigma, alpha;  // skew normal
	double gx[10], gw[10];      // positive nodes and weights of the 20-point rule
};

// The reference's 13-digit constants (src/physical_constants.hh:21-24).
constexpr double kSqrt2Pi = 2.506628274631;
constexpr double kSqrt2 = 1.4142135623731;
constexpr double kTwoPi = 6.283185307179586476925286766559;

// gsl_cdf_gaussian_P(x - mu, sigma)
__device__ __forceinline__ double normal_cdf(double x, double mu, double sigma) {
	return 0.5 * erfc(-((x - mu) / sigma) / 1.4142135623730951);
}

__device__ __forceinline__ double gram_charlier_cdf(double x, double s, double k) {
	return exp(-0.5 * x * x) * (k * (3.0 * x - x * x * x) + s * (4.0 - 4.0 * x * x) +
	                            3.0 * x * x * x - 9.0 * x) /
	           (24.0 * kSqrt2Pi) +
	       0.5 * erf(x / kSqrt2) + 0.5;
}

__device__ __forceinline__ double owen_t(const NitParams& p, double h, double alpha) {
	const double a2 = alpha * alpha, h2 = -0.5 * h * h;
	double r = 0.0;
#pragma unroll
	for (int i = 0; i < 10; ++i) {
		const double term = 1.0 + a2 * p.gx[i] * p.gx[i];
		r += p.gw[i] * exp(h2 * term) / term;
	}
	return r * alpha / kTwoPi;
}

__device__ __forceinline__ double target_cdf(const NitParams& p, double x) {
	if (p.dist == ARMA_NIT_GRAM_CHARLIER) return gram_charlier_cdf(x, p.skew, p.kurt);
	return normal_cdf(x, p.mean, p.sigma) - 2.0 * owen_t(p, (x - p.mean) / p.sigma, p.alpha);
}

// F at the midpoints of the first levels of the bisection: table[1] at the first,
// table[2 j] and table[2 j + 1] at those of the lower and upper half of the
// interval whose midpoint is table[j]'s; table[0] = F(a) and, past the last,
// F(b).
__global__ __launch_bounds__(256) void nit_table_kernel(double* __restrict__ table, int size,
                                                        NitParams p) {
	const int j = int(blockIdx.x) * 256 + int(threadIdx.x);
	if (j > size) return;
	double a = p.a, b = p.b;
	double c = j == 0 ? a : b;
	if (j > 0 && j < size) {
		c = 0.5 * (a + b);
		for (int bit = 30 - __clz(j); bit >= 0; --bit) {
			if (j >> bit & 1)
				a = c;
			else
				b = c;
			c = 0.5 * (a + b);
		}
	}
	table[j] = target_cdf(p, c);
}

// TABLE: the first steps by look-up.  One kernel for both, with the table's size
// tested, took 22 us for 512 points and a Gram-Charlier law where these take 18 with the
// table and 19 without.
template <class T, bool TABLE>
__global__ __launch_bounds__(256) void nit_kernel(T* __restrict__ data, size_t n, NitParams p,
                                                  const double* __restrict__ table, int size) {
	const size_t stride = size_t(gridDim.x) * blockDim.x;
	for (size_t q = size_t(blockIdx.x) * blockDim.x + threadIdx.x; q < n; q += stride) {
		const double y = normal_cdf(double(data[q]), 0.0, p.stdev);
		double a = p.a, b = p.b, c, fc;
		double fa = (TABLE ? table[0] : target_cdf(p, a)) - y;
		double fb = (TABLE ? table[size] : target_cdf(p, b)) - y;
		int i = 0;
		// one step from F(c) - y
		auto step = [&] {
			if (fa * fc < 0.0) {
				b = c;
				fb = fc;
			}
			if (fb * fc < 0.0) {
				a = c;
				fa = fc;
			}
			++i;
		};
		auto more = [&] { return i < p.max_iter && (b - a) > p.eps && fabs(fc) > p.eps; };
		if constexpr (TABLE) {
			bool on = true;
			for (int node = 1; on && node < size;) {
				c = 0.5 * (a + b);
				fc = table[node] - y;
				const bool lower = fa * fc < 0.0, upper = !lower && fb * fc < 0.0;
				step();
				node = lower ? 2 * node : upper ? 2 * node + 1 : node;
				on = more();
			}
			if (!on) {
				data[q] = T(c);
				continue;
			}
		}
		do {
			c = 0.5 * (a + b);
			fc = target_cdf(p, c) - y;
			step();
		} while (more());
		data[q] = T(c);
	}
}

// Positive nodes and weights of the 2m-point Gauss-Legendre rule (Newton's
// method on P_2m; w = 2 / ((1 - x^2) P'(x)^2)), ascending.
void gauss_legendre_half(int m, double* x, double* w) {
	const int n = 2 * m;
	for (int i = 0; i < m; ++i) {
		double z = std::cos(M_PI * (i + 0.75) / (n + 0.5)), dp = 0.0;
		for (int it = 0; it < 100; ++it) {
			double p0 = 1.0, p1 = z;
			for (int k = 2; k <= n; ++k) {
				const double p2 = ((2.0 * k - 1.0) * z * p1 - (k - 1.0) * p0) / k;
				p0 = p1;
				p1 = p2;
			}
			dp = n * (z * p1 - p0) / (z * z - 1.0);
			const double dz = p1 / dp;
			z -= dz;
			if (std::fabs(dz) < 1e-15) break;  // converged to within a few ulp
		}
		x[m - 1 - i] = z;
		w[m - 1 - i] = 2.0 / ((1.0 - z * z) * dp * dp);
	}
}

}  // namespace

void launch_nit_realisation(arma_hip_ctx* ctx, void* zeta, size_t n, int precision,
                            double gamma0, const arma_nit_desc* d) {
	NitParams p;
	p.stdev = std::sqrt(gamma0);
	p.a = d->interval[0];
	p.b = d->interval[1];
	p.eps = d->absolute_error;
	p.max_iter = d->max_iterations;
	p.dist = d->distribution;
	p.skew = d->skewness;
	p.kurt = d->kurtosis;
	p.mean = d->mean;
	p.sigma = d->stdev;
	p.alpha = d->alpha;
	gauss_legendre_half(10, p.gx, p.gw);
	if (n == 0) return;
	const int grid = int(std::min<size_t>((n + 255) / 256, size_t(1) << 20));
	KernelTimer t(ctx, "nit_realisation");
	// levels of the table: a sixteenth of the points at most, 2 MB, and no more
	// than the bisection can take.  A captured launch shares no buffer with the
	// context's other calls and evaluates every step
	int levels = 0;
	hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
	ARMA_HIP_CHECK(hipStreamIsCapturing(ctx->stream, &cap));
	if (cap == hipStreamCaptureStatusNone) {
		double width = p.b - p.a;
		while (levels < 18 && levels < p.max_iter && width > p.eps && (size_t(32) << levels) <= n) {
			++levels;
			width *= 0.5;
		}
		if (levels < 4) levels = 0;
	}
	int size = levels ? 1 << levels : 0;
	double* table = nullptr;
	if (size) table = (double*)ctx->nit_table.try_get(sizeof(double) * (size_t(size) + 1));
	if (!table) size = 0;
	if (size) {
		nit_table_kernel<<<size / 256 + 1, 256, 0, ctx->stream>>>(table, size, p);
		ARMA_HIP_CHECK(hipGetLastError());
	}
	auto launch = [&](auto* kernel, auto* data) {
		kernel<<<grid, 256, 0, ctx->stream>>>(data, n, p, table, size);
	};
	if (precision == ARMA_FP32)
		launch(size ? &nit_kernel<float, true> : &nit_kernel<float, false>, static_cast<float*>(zeta));
	else
		launch(size ? &nit_kernel<double, true> : &nit_kernel<double, false>,
		       static_cast<double*>(zeta));
	ARMA_HIP_CHECK(hipGetLastError());
}

}  // namespace arma_hip
