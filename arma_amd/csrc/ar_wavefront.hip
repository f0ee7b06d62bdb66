// Host side of the wavefront recurrence: tables, launches and batches.  The
// tile is in ar_tile.hpp, its kernels in ar_wave_*.hip and ar_batch_*.hip, the
// quad tile in ar_quad.hip.
#include "ar_quad.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <vector>

namespace arma_hip {
namespace {

// Whether a surface runs on the quad tile: at most 16 in-slice taps, the
// coefficients of its batch bucket's P0 within the register budget, and, for
// every tile shape, the mailboxes from a tile's corner neighbour to itself
// within the reach of one buffer descriptor.  Single surfaces and batch
// members follow the same rule, so a batch member's values equal those of
// the same surface alone.
bool quad_eligible(const arma_ar_desc* d) {
	const int P0 = d->phi_shape[0], P1 = d->phi_shape[1], P2 = d->phi_shape[2];
	const int b = batch_bucket(P0);
	const size_t es = d->precision == ARMA_FP32 ? 4 : 8;
	// The one-lane tile is the default in both precisions: with its mailbox
	// traffic behind a buffer descriptor it ran 2.38 ms against the quad
	// tile's 2.68 ms on 1024x256x256 FP32 and 16.7 against 17.2 ms on
	// 2048x512x512 FP32 (whose 262 144 columns fit at one lane each, four
	// workgroups per CU, but at four lanes each only a quarter at a time),
	// and 2.44 against 3.0 ms on 1024x256x256 FP64.  ARMA_HIP_QUAD_TILE=1
	// selects the quad tile for FP32 surfaces, single and batched alike (a
	// point's sum is added in another order there, so the choice must be the
	// same for a batch member and the single surface it is compared with).
	const char* e = std::getenv("ARMA_HIP_QUAD_TILE");
	if (!(e && e[0] == '1' && e[1] == 0)) return false;
	if (d->precision != ARMA_FP32) return false;
	if (b < 0 || P1 > kMaxP12 || P2 > kMaxP12 ||
	    !quad_fits(int(es), kBatchP0[b], quad_taps(P1 * P2)))
		return false;
	for (int TX : {8, 16, 32}) {
		const int TY = kThreads / TX;
		const size_t nY = size_t(div_ceil(d->shape[2], TY));
		const size_t total_u = size_t(d->shape[0]) + TX + TY - 2 + (P1 - 1) + (P2 - 1);
		const size_t NB = size_t(std::max(1, mbox_width_rt(TX, P1 - 1, P2 - 1)));
		if ((nY + 2) * total_u * NB * es >= (size_t(1) << 31) - 64) return false;
	}
	return true;
}

// Quad tile tables of one surface, appended to ph and offs: the
// coefficients [g][n][k] of tap m = g + 4n (k stride P0S, zero past P0 and
// past the last tap; zero for m = 0, k = 0), then phi(0,0,0); offs gets each
// (g, n) tap's LDS byte distance back from the own position for a ring row
// of WY slots (zero past the last tap).  Returns the taps per lane.
template <class T>
int append_quad_tables(const double* phi, int P0, int P1, int P2, int P0S, int WY,
                       std::vector<T>& ph, std::vector<int>& offs) {
	const int P12 = P1 * P2, NT = quad_taps(P12);
	const size_t base = ph.size();
	ph.resize(base + size_t(kQuad) * NT * P0S + 1, T(0));
	ph.resize((ph.size() + 15) / 16 * 16, T(0));
	const size_t ob = offs.size();
	offs.resize(ob + size_t(kQuad) * NT, 0);
	for (int g = 0; g < kQuad; ++g)
		for (int n = 0; n < NT; ++n) {
			const int m = g + kQuad * n;
			if (m >= P12) continue;
			for (int k = 0; k < P0; ++k)
				if (m > 0 || k > 0)
					ph[base + (size_t(g) * NT + n) * P0S + k] = T(phi[size_t(k) * P12 + m]);
			offs[ob + size_t(g) * NT + n] = ((m / P2) * WY + (m % P2)) * int(sizeof(T));
		}
	ph[base + size_t(kQuad) * NT * P0S] = T(phi[0]);
	return NT;
}

// Coefficient and offset tables of one surface (see "tables of one surface"),
// appended to ph and offs: P0S accumulators (the P0 the kernel is compiled
// for) in one or two groups, ntr resident taps, tiles TX columns wide.
template <class T>
void append_tables(const double* phi, int P0, int P1, int P2, int P0S, int groups, TapShape shape,
                   int ntr, int TX, std::vector<T>& ph, std::vector<int>& offs) {
	const int K0 = groups == 1 ? P0S : group_split(sizeof(T), P0S, shape);
	const int P12 = P1 * P2;
	const int chunk = chunk_taps(sizeof(T), group_most(sizeof(T), P0S, groups, shape));
	const int ntap = padded_taps(P12 - 1, ntr, chunk);
	auto at = [&](int k, int m) { return k < P0 ? T(phi[size_t(k) * P12 + m]) : T(0); };
	const size_t base = ph.size();
	ph.resize(base + kNear + size_t(ntap) * P0S, T(0));
	for (int k = 0; k < P0S; ++k) ph[base + k] = at(k, 0);
	for (int e = 0; e < P12 - 1; ++e)
		for (int k = 0; k < P0S; ++k)
			ph[base + kNear + (k < K0 ? size_t(e) * K0 + k
			                          : size_t(ntap) * K0 + size_t(e) * (P0S - K0) + (k - K0))] =
				at(k, e + 1);
	// keep every surface's block 16-element aligned
	ph.resize((ph.size() + 15) / 16 * 16, T(0));
	// a tap of distance d = i + j was completed d steps before this; the padding
	// repeats the last tap, so that its zero coefficients meet no value that the
	// point does not depend on
	const int R = ring_planes(P1, P2), es = int(sizeof(T));
	const int WY = ring_pitch(es, TX, P1, P2, groups), plane = (TX + P1 - 1) * WY * es;
	for (int s = 0; s < R; ++s) {
		auto back = [&](int steps) { return ((s - steps) % R + R) % R * plane; };
		offs.push_back(back(0));
		offs.push_back(back(1));
		offs.push_back(0);
		offs.push_back(0);
		for (int e = 0; e < ntap; ++e) {
			const int m = std::min(e + 1, P12 - 1), i = m / P2, j = m % P2;
			offs.push_back(back(i + j) - (i * WY + j) * es);
		}
	}
}

// LDS bytes of a one-lane tile: the ring, the line and the hand-over.
constexpr size_t tile_lds(int es, int TX, int P1, int P2, int G, bool kahan) {
	const int TY = kThreads / TX;
	return size_t(es) * (size_t(ring_planes(P1, P2)) * (TX + P1 - 1) * ring_pitch(es, TX, P1, P2, G) +
	                     size_t(TY + 1) * kThreads + (G > 1 ? 2 * kThreads * (kahan ? 3 : 2) : 0));
}

// Every order whose halo a tile's width admits (ar_batch_fits) has its LDS, beside
// the kernel's own few words: nothing else decides what a batch takes.
constexpr bool all_orders_fit() {
	for (int es : {4, 8})
		for (int TX : {8, 16, 32})
			for (int P1 = 1; P1 <= kMaxP12 && P1 - 1 <= TX; ++P1)
				for (int P2 = 1; P2 <= kMaxP12 && P2 - 1 <= kThreads / TX; ++P2)
					for (int G = 1; G <= (TX == 16 ? 2 : 1); ++G)
						if (tile_lds(es, TX, P1, P2, G, es == 4) + 256 > 160 * 1024) return false;
	return true;
}
static_assert(all_orders_fit(), "an order's LDS exceeds the CU's");

// Whether a surface's accesses go through buffer descriptors: the mailboxes
// from a tile's corner neighbour to itself, and the slices of a step's noise
// loads, within 31 bits.
bool buffer_fits(size_t es, int TX, int nx, int ny, int nY, size_t total_u, size_t NB) {
	const size_t most = (size_t(1) << 31) - 64;
	return (size_t(nY) + 2) * total_u * NB * es < most && size_t(TX) * nx * ny * es < most;
}

// Fills n mailbox elements with the sentinel that await_halo waits for to be
// replaced, on the launch's stream before it.
template <class T>
void fill_mailboxes(hipStream_t stream, T* mbox, size_t n) {
	const size_t blocks = std::min<size_t>(std::max<size_t>(div_ceil_z(n * sizeof(T), 16 * 256 * 4), 1),
	                                       65536);
	fill_sentinel<T><<<unsigned(blocks), 256, 0, stream>>>(mbox, n);
	ARMA_HIP_CHECK(hipGetLastError());
}

// Checked launches of single surfaces: ARMA_HIP_CHECK_HALO set (and not "0")
// in the environment.  arm() points the kernel at a check word in the launch's
// cleared zero-word line; verify() reads the word back after the launch and fails
// the call if it was set.  The one-lane tile sets it when a halo value has not been
// stored after kCheckPolls polls (ARMA_HIP_CHECK_HALO_POLLS: another number) instead of
// waiting for it for ever; the quad tile, whose mailboxes are filled only in a
// checked launch, when a consumer reads one that its producer has not stored.
constexpr int kCheckPolls = 1 << 23;  // some ten seconds
struct HaloCheck {
	int* word = nullptr;
	int limit = 0;
	void arm(unsigned char* zero_line) {
		const char* e = std::getenv("ARMA_HIP_CHECK_HALO");
		if (!e || !*e || (e[0] == '0' && e[1] == 0)) return;
		word = reinterpret_cast<int*>(zero_line + 128);
		const char* polls = std::getenv("ARMA_HIP_CHECK_HALO_POLLS");
		limit = polls && std::atoi(polls) > 0 ? std::atoi(polls) : kCheckPolls;
	}
	void verify(arma_hip_ctx* ctx) const {
		if (!word) return;
		int v = 0;
		ARMA_HIP_CHECK(hipMemcpyAsync(&v, word, sizeof v, hipMemcpyDeviceToHost, ctx->stream));
		ARMA_HIP_CHECK(hipStreamSynchronize(ctx->stream));
		ARMA_HIP_REQUIRE(v == 0, ARMA_HIP_ERUNTIME,
		                 "checked launch: a halo value was not there when it was needed");
	}
};

// Launches a kernel of another translation unit; the arguments' types must be
// exactly the kernel's.
template <class... A>
void launch_kernel(const void* fn, int grid, int threads, size_t lds, hipStream_t stream,
                   A... args) {
	void* list[] = {(void*)&args...};
	// above 64 KiB: the larger LDS of gfx950
	if (lds > 65536)
		ARMA_HIP_CHECK(
			hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
	ARMA_HIP_CHECK(hipLaunchKernel(fn, dim3(grid), dim3(threads), list, lds, stream));
}

// The form of a surface's tile.  Two groups of waves always paid where they
// were measured (one lane per column: 1024 x 256 x 256 FP64 (7, 7, 2) 1.92 ms
// against 0.84); resident coefficients where the shape of phi is one that the
// fitted models have, P0 x P0 x 2 or P0 x P0 x P0 (streamed: that 1.34 ms, and FP32
// (5, 5, 5) 1.7 times as long).  Beyond a buffer descriptor's reach, and of order 1
// in t, one group.
WaveVariant wave_variant(int es, int P0, int P1, int P2, bool buf) {
	WaveVariant v;
	v.buf = buf;
	if (!buf || P0 < 2) return v;
	v.groups = 2;
	if (P1 == P0 && P2 == 2 && two_columns_fit(es, P0)) {
		v.shape = kTwoColumns;
		v.ntr = 2 * P0 - 1;
	} else if (P1 == P0 && P2 == P0) {
		v.shape = kSquare;
		v.ntr = square_taps(es, P0);
	}
	return v;
}

// One surface on the quad tile (16 x 16 columns, 1024 lanes per tile).
void launch_quad(arma_hip_ctx* ctx, const arma_ar_desc* d, float* zeta) {
	using T = float;
	const int nt = d->shape[0], nx = d->shape[1], ny = d->shape[2];
	const int P0 = d->phi_shape[0], P1 = d->phi_shape[1], P2 = d->phi_shape[2];
	constexpr int kTX = 16, kTY = kThreads / kTX;
	std::vector<T> ph;
	std::vector<int> offs;
	const int NT = append_quad_tables(d->phi, P0, P1, P2, P0, kTY + P2 - 1, ph, offs);
	const size_t phi_bytes = (ph.size() * sizeof(T) + 255) / 256 * 256;
	unsigned char* dbuf =
		(unsigned char*)work_buffer(ctx, ctx->phi, phi_bytes + offs.size() * sizeof(int));
	T* dphi = (T*)dbuf;
	int* doffs = (int*)(dbuf + phi_bytes);
	upload(ctx, dphi, ph.data(), ph.size() * sizeof(T));
	upload(ctx, doffs, offs.data(), offs.size() * sizeof(int));
	const int nY = div_ceil(ny, kTY);
	const int ntiles = div_ceil(nx, kTX) * nY;
	const int total_steps = nt + kTX + kTY - 2;
	// flags buffer: progress counters, a zero word for idle loads and a
	// per-tile sink for idle stores
	const size_t prog_bytes = sizeof(int) * kProgStride * size_t(ntiles);
	const size_t zero_bytes = 256;
	unsigned char* fb = (unsigned char*)work_buffer(
		ctx, ctx->flags, prog_bytes + zero_bytes + size_t(ntiles) * kQThreads * sizeof(T));
	int* prog = (int*)fb;
	const T* zero = (const T*)(fb + prog_bytes);
	T* sink = (T*)(fb + prog_bytes + zero_bytes);
	const int NB = std::max(1, mbox_width<kTX>(P1 - 1, P2 - 1));
	const int total_u = total_steps + (P1 - 1) + (P2 - 1);
	T* mbox = (T*)work_buffer(ctx, ctx->mbox, sizeof(T) * size_t(ntiles) * total_u * NB);
	const int nclear = int((prog_bytes + zero_bytes) / sizeof(int));
	reset_progress<<<div_ceil(nclear, 256), 256, 0, ctx->stream>>>(prog, nclear);
	ARMA_HIP_CHECK(hipGetLastError());
	HaloCheck hc;
	hc.arm(fb + prog_bytes);
	if (hc.word) fill_mailboxes(ctx->stream, mbox, size_t(ntiles) * total_u * NB);
	const int R = P1 + P2 - 1;
	const size_t lds = size_t(R) * (kTX + P1 - 1) * (kTY + P2 - 1) * sizeof(T);
	ARMA_HIP_REQUIRE(lds <= 160 * 1024, ARMA_HIP_EINVAL, "AR order too large for the LDS ring");
	KernelTimer timer(ctx, "ar_wavefront");
	const void* fn = ar_quad_kernel_f32(P0, NT);
	ARMA_HIP_REQUIRE(fn != nullptr, ARMA_HIP_EINVAL, "AR order outside the quad tile");
	launch_kernel(fn, ntiles, kQThreads, lds, ctx->stream, zeta, nt, nx, ny, (const T*)dphi,
	              (const int*)doffs, P1, P2, nY, prog, zero, sink, mbox, NB, total_steps, hc.word);
	hc.verify(ctx);
}

// A surface's launch on the one-lane tile and the buffers that it takes.
struct WavePlan {
	static constexpr int kTX = 16, kTY = kThreads / kTX;
	int nY, ntiles, total_steps, NB;
	size_t total_u;
	WaveVariant var;
	size_t coef_bytes, table_bytes;  // coefficients; with the offsets
	size_t flag_bytes, mbox_elems;
	explicit WavePlan(const arma_ar_desc* d) {
		const size_t es = d->precision == ARMA_FP32 ? 4 : 8;
		const int nt = d->shape[0], nx = d->shape[1], ny = d->shape[2];
		const int P0 = d->phi_shape[0], P1 = d->phi_shape[1], P2 = d->phi_shape[2];
		nY = div_ceil(ny, kTY);
		ntiles = div_ceil(nx, kTX) * nY;
		total_steps = nt + kTX + kTY - 2;
		NB = std::max(1, mbox_width<kTX>(P1 - 1, P2 - 1));
		total_u = size_t(total_steps) + std::max(P1 + P2 - 2, 1);
		var = wave_variant(int(es), P0, P1, P2, buffer_fits(es, kTX, nx, ny, nY, total_u, NB));
		// (as append_tables lays them out)
		const int chunk = chunk_taps(int(es), group_most(int(es), P0, var.groups, var.shape));
		const size_t ntap = size_t(padded_taps(P1 * P2 - 1, var.ntr, chunk));
		coef_bytes = ((kNear + ntap * P0 + 15) / 16 * 16 * es + 255) / 256 * 256;
		table_bytes = coef_bytes + size_t(ring_planes(P1, P2)) * (kOffHead + ntap) * sizeof(int);
		// a zero word for out-of-range loads (and the check word) and, without
		// buffer descriptors, a sink per tile for out-of-range stores
		flag_bytes = 256 + (var.buf ? 0 : size_t(ntiles) * kThreads * es);
		mbox_elems = size_t(ntiles) * total_u * NB;  // a row of boundary values per tile and step
	}
};

template <class T, bool KAHAN>
void launch_typed(arma_hip_ctx* ctx, const arma_ar_desc* d, T* zeta) {
	const int nt = d->shape[0], nx = d->shape[1], ny = d->shape[2];
	const int P0 = d->phi_shape[0], P1 = d->phi_shape[1], P2 = d->phi_shape[2];
	ARMA_HIP_REQUIRE(P1 <= kMaxP12 && P2 <= kMaxP12 && P0 <= 10, ARMA_HIP_EINVAL,
	                 "AR order above 10 is not supported by the wavefront kernel");
	if constexpr (sizeof(T) == 4) {
		if (quad_eligible(d)) {
			launch_quad(ctx, d, zeta);
			return;
		}
	}
	const WavePlan p(d);
	std::vector<T> ph;
	std::vector<int> offs;
	append_tables(d->phi, P0, P1, P2, P0, p.var.groups, p.var.shape, p.var.ntr, p.kTX, ph, offs);
	std::vector<unsigned char> tables(p.table_bytes);
	ARMA_HIP_REQUIRE(ph.size() * sizeof(T) <= p.coef_bytes &&
	                     p.coef_bytes + offs.size() * sizeof(int) == p.table_bytes,
	                 ARMA_HIP_ERUNTIME, "wavefront tables and plan differ");
	std::memcpy(tables.data(), ph.data(), ph.size() * sizeof(T));
	std::memcpy(tables.data() + p.coef_bytes, offs.data(), offs.size() * sizeof(int));
	unsigned char* dbuf = (unsigned char*)work_buffer(ctx, ctx->phi, p.table_bytes);
	upload(ctx, dbuf, tables.data(), tables.size());
	unsigned char* fb = (unsigned char*)work_buffer(ctx, ctx->flags, p.flag_bytes);
	T* mbox = (T*)work_buffer(ctx, ctx->mbox, p.mbox_elems * sizeof(T));
	HaloCheck hc;
	hc.arm(fb);
	if (!p.var.buf || hc.word) {  // (behind descriptors the zero word is not read)
		reset_progress<<<1, 256, 0, ctx->stream>>>((int*)fb, 256 / int(sizeof(int)));
		ARMA_HIP_CHECK(hipGetLastError());
	}
	KernelTimer timer(ctx, "ar_wavefront");
	fill_mailboxes(ctx->stream, mbox, p.mbox_elems);
	const size_t lds = tile_lds(sizeof(T), p.kTX, P1, P2, p.var.groups, KAHAN);
	ARMA_HIP_REQUIRE(lds <= 160 * 1024, ARMA_HIP_EINVAL, "AR order too large for the LDS ring");
	const void* fn = sizeof(T) == 4 ? ar_wave_kernel_f32(P0, p.var) : ar_wave_kernel_f64(P0, p.var);
	ARMA_HIP_REQUIRE(fn != nullptr, ARMA_HIP_EINVAL, "bad AR order");
	launch_kernel(fn, p.ntiles, kThreads * p.var.groups, lds, ctx->stream, zeta, nt, nx, ny,
	              (const T*)dbuf, (const T*)dbuf + kNear, (const int*)(dbuf + p.coef_bytes), P1, P2,
	              p.nY, (const T*)fb, (T*)(fb + (p.var.buf ? 0 : 256)), mbox, p.NB, p.total_steps,
	              hc.word, hc.limit);
	hc.verify(ctx);
}

// The kernel a batch part launches: the quad tile, or the one-lane tile with
// or without buffer descriptors.
const void* batch_kernel_fn(int precision, int tx, bool quad, bool buf, bool dense) {
	if (quad) return ar_quad_batch_kernel_f32(tx);
	return precision == ARMA_FP32 ? ar_batch_kernel_f32(tx, buf, dense)
	                               : ar_batch_kernel_f64(tx, buf, dense);
}

}  // namespace

namespace {

// A batch launch is complete when its event has fired.  Events are shared so
// that the chain below can outlive the batch that recorded them.
struct LaunchEvent {
	hipEvent_t ev = nullptr;
	LaunchEvent() { ARMA_HIP_CHECK(hipEventCreateWithFlags(&ev, hipEventDisableTiming)); }
	~LaunchEvent() {
		if (ev) (void)hipEventDestroy(ev);
	}
	LaunchEvent(const LaunchEvent&) = delete;
	LaunchEvent& operator=(const LaunchEvent&) = delete;
};

// The last batch launch enqueued on each device, on any stream.
std::mutex g_batch_mu;
std::map<int, std::shared_ptr<LaunchEvent>> g_batch_last;

// Bounded waits give up after this long without progress.
constexpr double kBatchWaitLimitS = 10.0;

}  // namespace

// One persistent launch over the members of one tile kind: the classic tile
// (256 lanes) or the quad tile (1024 lanes).  A batch has one part per kind
// its members need; the parts run one after the other.
struct ArBatchPart {
	bool quad = false;
	bool buf = true;    // every member's accesses fit buffer descriptors
	bool dense = true;  // every member's coefficients leave room for two workgroups per CU
	int nqueue = 0, grid = 0, max_slots = 0;
	size_t lds = 0;
	size_t nclear = 0;  // ints cleared before a launch: the abort word line, progress, zero word
	Scratch coef, taps, surf, queue, flags, mbox;
	int* clear_base = nullptr;  // start of the words cleared before a launch
	int* next = nullptr;        // entries taken of the queue
	int* abortw = nullptr;      // set by a launch whose bounded waits gave up
	int* progress = nullptr;  // quad tiles' counters
	size_t mbox_elems = 0;
	void* zero = nullptr;
	void* sink = nullptr;
};

struct ArBatch {
	int precision = 0;
	BatchArConfig cfg;
	ArBatchPart part[2];  // classic, quad
	long long limit = 0;  // wall-clock ticks of kBatchWaitLimitS
	std::shared_ptr<LaunchEvent> done;
};

namespace {

template <class T>
void build_part(arma_hip_ctx* ctx, const ArBatch* ab, ArBatchPart* pt,
                const std::vector<BatchMember>& all, const std::vector<int>& idx) {
	const int TX = ab->cfg.tile_x, TY = kThreads / TX;
	std::vector<T> coef;
	std::vector<int> taps;
	std::vector<BatchSurface> surf(idx.size());
	std::vector<double> work(idx.size());
	std::vector<int> ntiles(idx.size());
	long long tiles = 0, mbox_elems = 0;
	int max_tiles = 0;
	size_t lds = 0;
	pt->buf = pt->dense = true;
	for (int m : idx) {
		const arma_ar_desc* d = all[m].d;
		const int HX = d->phi_shape[1] - 1, HY = d->phi_shape[2] - 1;
		const size_t total_u = size_t(d->shape[0]) + TX + TY - 2 + std::max(HX + HY, 1);
		pt->buf = pt->buf && buffer_fits(sizeof(T), TX, d->shape[1], d->shape[2],
		                                 div_ceil(d->shape[2], TY), total_u,
		                                 size_t(std::max(1, mbox_width_rt(TX, HX, HY))));
	}
	const int groups = pt->quad ? 1 : batch_groups(TX, pt->buf);
	const int lanes = pt->quad ? kQThreads : kThreads * groups;
	for (size_t i = 0; i < idx.size(); ++i) {
		const arma_ar_desc* d = all[idx[i]].d;
		const int nt = d->shape[0], nx = d->shape[1], ny = d->shape[2];
		const int P0 = d->phi_shape[0], P1 = d->phi_shape[1], P2 = d->phi_shape[2];
		ARMA_HIP_REQUIRE(P1 <= kMaxP12 && P2 <= kMaxP12 && P0 <= 10, ARMA_HIP_EINVAL,
		                 "AR order above 10 is not supported by the wavefront kernel");
		// a tile's halo comes from its direct neighbours only
		ARMA_HIP_REQUIRE(P1 - 1 <= TX && P2 - 1 <= TY, ARMA_HIP_EINVAL,
		                 "AR order wider than the batch tile");
		const int bucket = batch_bucket(P0);
		BatchSurface& sf = surf[i];
		sf.zoff = (long long)all[idx[i]].zoff;
		sf.nt = nt;
		sf.nx = nx;
		sf.ny = ny;
		sf.P1 = P1;
		sf.P2 = P2;
		const WaveVariant var =
			groups == 2 && P0 >= kShapedMin && P0 <= kShapedMax
				? wave_variant(sizeof(T), P0, P1, P2, true)
				: WaveVariant{};
		pt->dense = pt->dense && is_dense(sizeof(T), P0, var.shape);
		const int P0S = var.shape == kAnyShape ? kBatchP0[bucket] : P0;
		sf.body = pt->quad ? bucket : batch_body(bucket, var.shape, P0);
		sf.nY = div_ceil(ny, TY);
		sf.coff = int(coef.size());
		sf.toff = int(taps.size());
		if (pt->quad)
			append_quad_tables(d->phi, P0, P1, P2, kBatchP0[bucket], TY + P2 - 1, coef, taps);
		else
			append_tables(d->phi, P0, P1, P2, P0S, groups, var.shape, var.ntr, TX, coef, taps);
		ntiles[i] = div_ceil(nx, TX) * sf.nY;
		sf.poff = int(tiles);
		sf.total_steps = nt + TX + TY - 2;
		sf.t0 = all[idx[i]].t0;
		sf.pad = 0;
		sf.NB = std::max(1, mbox_width_rt(TX, P1 - 1, P2 - 1));
		const long long total_u = sf.total_steps + std::max(P1 + P2 - 2, 1);
		sf.moff = mbox_elems;
		mbox_elems += (long long)ntiles[i] * total_u * sf.NB;
		mbox_elems = (mbox_elems + 63) / 64 * 64;
		tiles += ntiles[i];
		max_tiles = std::max(max_tiles, ntiles[i]);
		lds = std::max(lds, pt->quad ? size_t(P1 + P2 - 1) * (TX + P1 - 1) * (TY + P2 - 1) * sizeof(T)
		                             : tile_lds(sizeof(T), TX, P1, P2, groups, sizeof(T) == 4));
		// the time from a surface's first tile to the end of its last, in us: 16
		// steps and the way through memory per tile of its longest chain
		const double step = 0.25 + 0.002 * P0 * P1 * P2;
		work[i] = nt * step + (div_ceil(nx, TX) + sf.nY) * (16 * step + 4.5);
	}
	ARMA_HIP_REQUIRE(lds <= 160 * 1024, ARMA_HIP_EINVAL, "AR order too large for the LDS ring");
	ARMA_HIP_REQUIRE(tiles < (1ll << 31) / kProgStride && coef.size() < (1u << 31) &&
	                     taps.size() < (1u << 31),
	                 ARMA_HIP_EINVAL, "batch too large");
	// the queue: surfaces by decreasing work; a surface's tiles by X + Y, the
	// order in which they can start, so every tile follows the tiles it waits on
	std::vector<int> order(idx.size());
	for (size_t i = 0; i < idx.size(); ++i) order[i] = int(i);
	std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return work[a] > work[b]; });
	std::vector<int2> queue;
	queue.reserve(size_t(tiles));
	if (ab->cfg.schedule == ARMA_BATCH_INTERLEAVED) {
		for (int diagonal = 0; queue.size() < size_t(tiles); ++diagonal)
			for (int i : order) {
				const int nY = surf[i].nY, nX = ntiles[i] / nY;
				const int X0 = std::max(0, diagonal - nY + 1), X1 = std::min(nX - 1, diagonal);
				for (int X = X0; X <= X1; ++X) queue.push_back(make_int2(i, X * nY + diagonal - X));
			}
	} else {
		for (int i : order) {
			const int nY = surf[i].nY, nX = ntiles[i] / nY;
			for (int b = 0; b < ntiles[i]; ++b)
				queue.push_back(make_int2(i, diagonal_tile(b, nX, nY)));
		}
	}
	pt->nqueue = int(queue.size());
	pt->lds = lds;
	// device tables
	pt->coef.get(std::max<size_t>(coef.size(), 16) * sizeof(T));
	pt->taps.get(std::max<size_t>(taps.size(), 16) * sizeof(int));
	pt->surf.get(surf.size() * sizeof(BatchSurface));
	pt->queue.get(std::max<size_t>(queue.size(), 1) * sizeof(int2));
	upload(ctx, pt->coef.ptr, coef.data(), coef.size() * sizeof(T));
	upload(ctx, pt->taps.ptr, taps.data(), taps.size() * sizeof(int));
	upload(ctx, pt->surf.ptr, surf.data(), surf.size() * sizeof(BatchSurface));
	upload(ctx, pt->queue.ptr, queue.data(), queue.size() * sizeof(int2));
	// flags: the queue counter and the abort word (a line each), the quad tiles'
	// progress counters, a zero word, and a sink for idle stores sized for the
	// largest surface (behind buffer descriptors the one-lane tile stores none)
	const size_t head = 256;
	const size_t prog_bytes = pt->quad ? sizeof(int) * kProgStride * size_t(tiles) : 0;
	const size_t zero_bytes = 256;
	const size_t sink_lanes = pt->quad ? kQThreads : pt->buf ? 0 : kThreads;
	unsigned char* fb = (unsigned char*)pt->flags.get(head + prog_bytes + zero_bytes +
	                                                  size_t(max_tiles) * sink_lanes * sizeof(T));
	pt->clear_base = (int*)fb;
	pt->next = (int*)fb;
	pt->abortw = (int*)(fb + 128);
	pt->progress = (int*)(fb + head);
	pt->zero = fb + head + prog_bytes;
	pt->sink = sink_lanes ? fb + head + prog_bytes + zero_bytes : pt->zero;
	pt->nclear = (head + prog_bytes + zero_bytes) / sizeof(int);
	pt->mbox_elems = size_t(mbox_elems);
	pt->mbox.get(std::max<size_t>(size_t(mbox_elems), 64) * sizeof(T));
	const void* fn = batch_kernel_fn(ab->precision, TX, pt->quad, pt->buf, pt->dense);
	if (lds > 65536)
		ARMA_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
		                                   int(lds)));
	int per_cu = 0;
	ARMA_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, lanes, lds));
	pt->max_slots = std::max(per_cu, 1);
	const int slots = ab->cfg.slots_per_cu > 0 ? std::min(ab->cfg.slots_per_cu, pt->max_slots)
	                                           : pt->max_slots;
	pt->grid = int(std::min<long long>(pt->nqueue, (long long)slots * std::max(ctx->num_cus, 1)));
}

// Members whose order fits the quad tile go to the quad part, the others to
// the classic part (the same rule as single surfaces).
template <class T>
void build_batch(arma_hip_ctx* ctx, ArBatch* ab, const std::vector<BatchMember>& m) {
	std::vector<int> idx[2];
	for (size_t i = 0; i < m.size(); ++i) {
		// the member as a single surface at the batch's precision
		arma_ar_desc d = *m[i].d;
		d.precision = ab->precision;
		idx[quad_eligible(&d) ? 1 : 0].push_back(int(i));
	}
	for (int k = 0; k < 2; ++k) {
		ab->part[k].quad = k == 1;
		ab->part[k].nqueue = 0;
		if (!idx[k].empty()) build_part<T>(ctx, ab, &ab->part[k], m, idx[k]);
	}
	int khz = 0;
	ARMA_HIP_CHECK(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, ctx->device));
	ab->limit = (long long)(double(std::max(khz, 1)) * 1e3 * kBatchWaitLimitS);
	if (!ab->done) ab->done = std::make_shared<LaunchEvent>();
}

template <class T>
void batch_go(arma_hip_ctx* ctx, const ArBatch* ab, const ArBatchPart* pt, T* arena) {
	const void* fn = batch_kernel_fn(ab->precision, ab->cfg.tile_x, pt->quad, pt->buf, pt->dense);
	const T* coef = (const T*)pt->coef.ptr;
	const int* taps = (const int*)pt->taps.ptr;
	T* mbox = (T*)pt->mbox.ptr;
	const BatchSurface* surf = (const BatchSurface*)pt->surf.ptr;
	const int2* queue = (const int2*)pt->queue.ptr;
	if (pt->quad) {
		launch_kernel(fn, pt->grid, kQThreads, pt->lds, ctx->stream, arena, coef, taps, pt->progress,
		              (const T*)pt->zero, (T*)pt->sink, mbox, surf, queue, pt->nqueue, pt->abortw,
		              ab->limit);
	} else {
		fill_mailboxes(ctx->stream, mbox, pt->mbox_elems);
		launch_kernel(fn, pt->grid, kThreads * batch_groups(ab->cfg.tile_x, pt->buf), pt->lds,
		              ctx->stream, arena, coef, taps, (const T*)pt->zero, (T*)pt->sink, mbox, surf,
		              queue, pt->nqueue, pt->next, pt->abortw, ab->limit);
	}
}

void batch_enqueue(arma_hip_ctx* ctx, ArBatch* ab, void* arena) {
	KernelTimer timer(ctx, "ar_batch");
	for (const ArBatchPart& pt : ab->part) {
		if (pt.nqueue == 0) continue;
		const int nclear = int(pt.nclear);
		reset_progress<<<div_ceil(nclear, 256), 256, 0, ctx->stream>>>(pt.clear_base, nclear);
		ARMA_HIP_CHECK(hipGetLastError());
		if (ab->precision == ARMA_FP32)
			batch_go(ctx, ab, &pt, (float*)arena);
		else
			batch_go(ctx, ab, &pt, (double*)arena);
		ARMA_HIP_CHECK(hipGetLastError());
	}
}

}  // namespace

void launch_ar_wavefront(arma_hip_ctx* ctx, const arma_ar_desc* d, void* zeta) {
	if (d->precision == ARMA_FP32)
		launch_typed<float, true>(ctx, d, (float*)zeta);
	else
		launch_typed<double, false>(ctx, d, (double*)zeta);
}

size_t ar_wavefront_work_bytes(const arma_ar_desc* d) {
	// the buffers launch_quad or launch_typed takes, in their order, each
	// 256-byte aligned
	auto al = [](size_t b) { return (b + 255) / 256 * 256; };
	const size_t es = d->precision == ARMA_FP32 ? 4 : 8;
	const WavePlan p(d);
	const size_t mbox = p.mbox_elems * es;
	if (quad_eligible(d)) {
		const size_t nq = size_t(kQuad) * quad_taps(d->phi_shape[1] * d->phi_shape[2]);
		const size_t tables = al((nq * d->phi_shape[0] + 1 + 15) / 16 * 16 * es) + nq * sizeof(int);
		const size_t flags = (sizeof(int) * kProgStride + kQThreads * es) * size_t(p.ntiles) + 256;
		return al(tables) + al(flags) + mbox;
	}
	return al(p.table_bytes) + al(p.flag_bytes) + mbox;
}

bool ar_batch_fits(const std::vector<BatchMember>& m, int tile_x) {
	for (const BatchMember& x : m)
		if (x.d->phi_shape[1] - 1 > tile_x || x.d->phi_shape[2] - 1 > kThreads / tile_x)
			return false;
	return true;
}

void ar_batch_build(arma_hip_ctx* ctx, ArBatch* ab, int precision,
                    const std::vector<BatchMember>& m, const BatchArConfig& cfg) {
	ARMA_HIP_REQUIRE(cfg.tile_x == 8 || cfg.tile_x == 16 || cfg.tile_x == 32, ARMA_HIP_EINVAL,
	                 "batch tile width must be 8, 16 or 32");
	ARMA_HIP_REQUIRE(cfg.schedule == ARMA_BATCH_SURFACE_MAJOR ||
	                     cfg.schedule == ARMA_BATCH_INTERLEAVED,
	                 ARMA_HIP_EINVAL, "bad batch schedule");
	ARMA_HIP_REQUIRE(!m.empty(), ARMA_HIP_EINVAL, "empty batch");
	ab->precision = precision;
	ab->cfg = cfg;
	if (precision == ARMA_FP32)
		build_batch<float>(ctx, ab, m);
	else
		build_batch<double>(ctx, ab, m);
}

ArBatch* ar_batch_create(arma_hip_ctx* ctx, int precision, const std::vector<BatchMember>& m,
                         const BatchArConfig& cfg) {
	auto* ab = new ArBatch;
	try {
		ar_batch_build(ctx, ab, precision, m, cfg);
	} catch (...) {
		delete ab;
		throw;
	}
	return ab;
}

ArBatch* ar_batch_new() { return new ArBatch; }

// (a sink is counted for every member: whether there is one depends on the others)
size_t ar_batch_member_bytes(const arma_ar_desc* d, int tile_x) {
	const int TX = tile_x, TY = kThreads / TX;
	const size_t es = d->precision == ARMA_FP32 ? 4 : 8;
	const int P1 = d->phi_shape[1], P2 = d->phi_shape[2];
	const size_t tiles = size_t(div_ceil(d->shape[1], TX)) * div_ceil(d->shape[2], TY);
	const size_t total_u = size_t(d->shape[0]) + TX + TY - 2 + std::max(P1 + P2 - 2, 1);
	const size_t NB = std::max(1, mbox_width_rt(TX, P1 - 1, P2 - 1));
	const size_t lanes = quad_eligible(d) ? kQThreads : kThreads;
	const size_t progress = quad_eligible(d) ? sizeof(int) * kProgStride * tiles : 0;
	return es * (tiles * total_u * NB + tiles * lanes) + progress;
}

// Batch launches on one device run one after another, whatever stream they
// are enqueued on: each waits for the previous one's event.  Under graph
// capture the chain is left out (an event recorded outside the capture cannot
// be waited on inside it); the caller then keeps replays from overlapping
// other batch launches.
void ar_batch_launch(arma_hip_ctx* ctx, ArBatch* ab, void* arena) {
	hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
	ARMA_HIP_CHECK(hipStreamIsCapturing(ctx->stream, &cap));
	if (cap != hipStreamCaptureStatusNone) {
		batch_enqueue(ctx, ab, arena);
		return;
	}
	std::lock_guard<std::mutex> lock(g_batch_mu);
	std::shared_ptr<LaunchEvent>& last = g_batch_last[ctx->device];
	if (last && last != ab->done) ARMA_HIP_CHECK(hipStreamWaitEvent(ctx->stream, last->ev, 0));
	batch_enqueue(ctx, ab, arena);
	ARMA_HIP_CHECK(hipEventRecord(ab->done->ev, ctx->stream));
	last = ab->done;
}

void ar_batch_check(arma_hip_ctx* ctx, ArBatch* ab) {
	int stalled[2] = {0, 0};
	for (int k = 0; k < 2; ++k)
		if (ab->part[k].nqueue > 0)
			ARMA_HIP_CHECK(hipMemcpyAsync(&stalled[k], ab->part[k].abortw, sizeof(int),
			                              hipMemcpyDeviceToHost, ctx->stream));
	ARMA_HIP_CHECK(hipStreamSynchronize(ctx->stream));
	ARMA_HIP_REQUIRE(stalled[0] == 0 && stalled[1] == 0, ARMA_HIP_ERUNTIME,
	                 "batch recurrence launch stalled (its workgroups were not all resident); "
	                 "its surfaces are invalid");
}

void ar_batch_destroy(ArBatch* ab) { delete ab; }

// Workgroups of the batch's launches (the largest part's grid).
int ar_batch_grid(const ArBatch* ab) { return std::max(ab->part[0].grid, ab->part[1].grid); }

// Resident workgroups per CU of the batch's tile kinds (the most of its parts).
int ar_batch_max_slots(const ArBatch* ab) {
	int m = 0;
	for (const ArBatchPart& pt : ab->part)
		if (pt.nqueue > 0) m = std::max(m, pt.max_slots);
	return std::max(m, 1);
}

}  // namespace arma_hip
